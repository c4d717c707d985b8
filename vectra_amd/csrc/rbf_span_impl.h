// Long key axes of a few planes with a bias on gfx950 matrix cores: the kernel template,
// instantiated with the tile kernel's dtype pairs in rbf_tile_<in>_<out>.hip.
//
// A workgroup owns 16 or 32 query rows of one (b, h) plane and its waves share out
// the keys: wave w takes the 32-key pairs w, w + W, ... against all of
// its queries, with a softmax of its own (running shift, sum, accumulators), and
// one merge through LDS ends the rows.  The tile kernel's waves share out the
// queries instead and each walks the whole key axis: with fewer work items
// than CUs that walk is the launch's time and most of the chip is idle.
//
// The products, their lane layouts and the logits are rbf_block_kernel's:
//
//   S^T = K . Q^T     (16 keys x 16 queries per instruction, 32-deep steps)
//   O^T = V^T . P^T   (16 value dims x 16 queries)
//   x = coef (q.k - |q|^2 / 2) + c_j,  c_j = log2(e) (bias_j - gamma |k_j|^2)
//
// K's operands are loaded from memory as the products read them; V goes through a
// piece of LDS of the wave's own (no barrier in the loop) for the transposing
// read.  Weights are shifted by a running value that follows the query's
// largest logit when that has moved by more than 2^8, so a sum is at least 1
// and a weight at most 2^8, where the hi + lo split is accurate.
//
// Bound: the vector unit (exp2, the split, the running shift) on the CUs that
// have an item, with four waves per SIMD (two for 128-dim heads, by registers)
// to cover a pair's chain.  The weight sum is that of the hi + lo pairs (see
// rbf_block_impl.h), two per instruction after the products are issued: 1000 x
// 1000 x 64 17.0 -> 18.0 us, as a product of ones 19.3 (16 registers spilled
// for 12).  Measured, bf16 with ragged masks, streamed tiles
// and here: 8 planes of 700 x 700 x 64 20 and 15 us, of 1000 x 1000 x 64 26 and
// 18, four of 640 x 640 x 128 29 and 12, 16 of 340 x 1300 x 32 23 and 11, four of
// 1000 x 2000 x 64 (fp16) 48 and 16.  Items of 16 queries where every CU holds
// at most one: a plane of 1024 x 4096 x 64 25 us, 32 with items of 32.  Query
// operands are read from LDS: in registers 25 more spilled at 64 dims.

#pragma once

#include "rbf_common.h"
#include "rbf_kernels.h"
#include "rbf_mfma_ops.h"

namespace vectra {

template <int kD>
constexpr int span_waves() {
  return kD <= 64 ? 16 : 8;
}

// kCB: 16-query blocks of a workgroup.
template <typename T, typename OutT, int kD, int kCB>
__global__ __launch_bounds__(64 * span_waves<kD>()) void rbf_span_kernel(Problem p, int32_t q_blocks) {
  using Ops = MfmaOps<T>;
  using Qk = typename Ops::Qk;
  constexpr int kWaves = span_waves<kD>();
  constexpr int kRows = 16 * kCB;
  constexpr int kChunks = kD / 8;
  constexpr int kKSteps = kD / 32;
  constexpr int kDTiles = kD / 16;
  constexpr int kRowBytes = 2 * kD;
  constexpr int kRowsPerSpan = 256 / kRowBytes;
  constexpr int kVLoads = kChunks / 2;         // 16-byte chunks of V a lane stages per pair
  constexpr int kPassRows = 64 / kChunks;      // V rows of one of them over the wave
  constexpr int kVBytes = 32 * kRowBytes;      // a wave's piece of V
  constexpr float kMove = 8.f;
  constexpr uint32_t kOutSize = sizeof(OutT);

  // The waves' pieces of V and of c; then, per wave, the accumulators.
  constexpr int kStageBytes = kWaves * (kVBytes + 32 * 4);
  constexpr int kMergeBytes = kWaves * kRows * kD * 4;
  __shared__ __align__(16) unsigned char lds[kStageBytes > kMergeBytes ? kStageBytes : kMergeBytes];
  // Every wave's query operands (in registers they would spill at D = 64).
  __shared__ __align__(16) uint4 ql[kCB][kKSteps][kWave];
  __shared__ float part_shift[kWaves][kRows], part_total[kWaves][kRows];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15;
  const int grp = lane >> 4;
  const int32_t n_q = static_cast<int32_t>(p.Nq);
  const int32_t n_k = static_cast<int32_t>(p.Nk);
  const int32_t pairs = (n_k + 31) / 32;
  const int32_t bias_esize = p.bias_dtype == VECTRA_F32 ? 4 : 2;
  const uint32_t q_row_bytes = static_cast<uint32_t>(p.sq[2]) * 2u;
  const uint32_t k_row_bytes = static_cast<uint32_t>(p.sk[2]) * 2u;
  const uint32_t v_row_bytes = static_cast<uint32_t>(p.sv[2]) * 2u;

  // XCD-local order, as in rbf_block_kernel.
  const int32_t items = static_cast<int32_t>(gridDim.x);
  int32_t item = static_cast<int32_t>(blockIdx.x);
  if (items % 8 == 0) item = (item & 7) * (items / 8) + (item >> 3);
  const int32_t bh = static_cast<int32_t>(fast_div(static_cast<uint32_t>(item), p.nq_mul, p.nq_shift));
  const int32_t first_q = (item - bh * q_blocks) * kRows;
  const int32_t b = static_cast<int32_t>(fast_div(static_cast<uint32_t>(bh), p.h_mul, p.h_shift));
  const int32_t h = bh - b * static_cast<int32_t>(p.H);

  unsigned char* vl = lds + wave * kVBytes;
  float* cl = reinterpret_cast<float*>(lds + kWaves * kVBytes) + wave * 32;
  auto at = [](int row, int chunk) { return row * kRowBytes + ((chunk ^ ((row / kRowsPerSpan) & (kChunks - 1))) * 16); };

  const float coef = 2.f * kLog2e * load_any(p.scale, b * p.ssb + h * p.ssh, p.scale_dtype);
  const char* qp = static_cast<const char*>(p.q) + (b * p.sq[0] + h * p.sq[1]) * 2;
  const char* kp = static_cast<const char*>(p.k) + (b * p.sk[0] + h * p.sk[1]) * 2;
  const char* vp = static_cast<const char*>(p.v) + (b * p.sv[0] + h * p.sv[1]) * 2;
  const char* bp = static_cast<const char*>(p.bias) + (b * p.sbb + h * p.sbh) * bias_esize;
  const uint32_t misalign = base_misalign(bp);

  float q_half[kCB];
  uint4 kf[2][kKSteps], vf[kVLoads];
  uint32_t bias_word[2];
  // Rows past Nk read row Nk - 1; consume() replaces them.
  auto issue = [&](int32_t pair) __attribute__((always_inline)) {
#pragma unroll
    for (int hb = 0; hb < 2; ++hb) {
      const uint32_t row = static_cast<uint32_t>(min(32 * pair + 16 * hb + col, n_k - 1));
      bias_word[hb] = load_raw_scalar32(bp, misalign, row * static_cast<uint32_t>(p.sbn), p.bias_dtype).word;
#pragma unroll
      for (int ks = 0; ks < kKSteps; ++ks)
        kf[hb][ks] = load16(kp + row * k_row_bytes + static_cast<uint32_t>(64 * ks + 16 * grp));
    }
#pragma unroll
    for (int s = 0; s < kVLoads; ++s) {
      const uint32_t row = static_cast<uint32_t>(min(32 * pair + s * kPassRows + lane / kChunks, n_k - 1));
      vf[s] = load16(vp + row * v_row_bytes + static_cast<uint32_t>(lane % kChunks) * 16u);
    }
  };

  if (wave < pairs) issue(wave);
#pragma unroll
  for (int cb = 0; cb < kCB; ++cb) {
    // Rows past Nq read row Nq - 1 and are not stored.
    const uint32_t row = static_cast<uint32_t>(min(first_q + 16 * cb + col, n_q - 1));
    float sq = 0.f;
#pragma unroll
    for (int ks = 0; ks < kKSteps; ++ks) {
      const uint4 r = load16(qp + row * q_row_bytes + static_cast<uint32_t>(64 * ks + 16 * grp));
      if (wave == 0) ql[cb][ks][lane] = r;
      sq = dot_chunk<T>(r, r, sq);
    }
    q_half[cb] = -0.5f * allreduce_bit32(allreduce_bit16(sq, OpSum()), OpSum());
  }
  __syncthreads();

  f32x4 acc[kCB][kDTiles];
  float shift[kCB], total[kCB];
#pragma unroll
  for (int cb = 0; cb < kCB; ++cb) {
    shift[cb] = -INFINITY;
    total[cb] = 0.f;
#pragma unroll
    for (int u = 0; u < kDTiles; ++u) acc[cb][u] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  for (int32_t pair = wave; pair < pairs; pair += kWaves) {
    const bool ragged = 32 * pair + 32 > n_k;
    // Norms and c_j: every lane of a column ends with its two keys' values.
    float c[2];
#pragma unroll
    for (int hb = 0; hb < 2; ++hb) {
      const int32_t key = 32 * pair + 16 * hb + col;
      if (ragged && key >= n_k) {
#pragma unroll
        for (int ks = 0; ks < kKSteps; ++ks) kf[hb][ks] = make_uint4(0, 0, 0, 0);
      }
      float sq = 0.f;
#pragma unroll
      for (int ks = 0; ks < kKSteps; ++ks) sq = dot_chunk<T>(kf[hb][ks], kf[hb][ks], sq);
      sq = allreduce_bit32(allreduce_bit16(sq, OpSum()), OpSum());
      const uint32_t bytes =
          static_cast<uint32_t>(min(key, n_k - 1)) * static_cast<uint32_t>(p.sbn) * bias_esize + misalign;
      const float bias = decode_raw_scalar(RawScalar{bias_word[hb], (bytes & 2u) * 8u}, p.bias_dtype) * kLog2e;
      c[hb] = key < n_k ? fmaf(-0.5f * coef, sq, bias) : -INFINITY;
    }
    if (grp < 2) cl[16 * grp + col] = grp == 0 ? c[0] : c[1];
#pragma unroll
    for (int s = 0; s < kVLoads; ++s) {
      const int row = s * kPassRows + lane / kChunks;
      if (ragged && 32 * pair + row >= n_k) vf[s] = make_uint4(0, 0, 0, 0);
      *reinterpret_cast<uint4*>(vl + at(row, lane % kChunks)) = vf[s];
    }
    f32x4 st[kCB][2];
#pragma unroll
    for (int hb = 0; hb < 2; ++hb)
#pragma unroll
      for (int ks = 0; ks < kKSteps; ++ks)
#pragma unroll
        for (int cb = 0; cb < kCB; ++cb)
          st[cb][hb] = Ops::qk(__builtin_bit_cast(Qk, kf[hb][ks]), __builtin_bit_cast(Qk, ql[cb][ks][lane]),
                               ks == 0 ? f32x4{q_half[cb], q_half[cb], q_half[cb], q_half[cb]} : st[cb][hb]);
    // The registers are free for the next pair's loads.
    if (pair + kWaves < pairs) issue(pair + kWaves);

    // One wave's LDS operations complete in order; this keeps the compiler
    // from moving the reads above the writes.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    Qk p_hi[kCB], p_lo[kCB];
    float4 ch[2];
#pragma unroll
    for (int hb = 0; hb < 2; ++hb) ch[hb] = *reinterpret_cast<const float4*>(cl + 16 * hb + 4 * grp);
#pragma unroll
    for (int cb = 0; cb < kCB; ++cb) {
      __builtin_amdgcn_sched_barrier(0);  // one block's logits at a time: registers
      float x[2][4];
#pragma unroll
      for (int hb = 0; hb < 2; ++hb) {
        x[hb][0] = fmaf(coef, st[cb][hb][0], ch[hb].x);
        x[hb][1] = fmaf(coef, st[cb][hb][1], ch[hb].y);
        x[hb][2] = fmaf(coef, st[cb][hb][2], ch[hb].z);
        x[hb][3] = fmaf(coef, st[cb][hb][3], ch[hb].w);
      }
      float m = -INFINITY;
#pragma unroll
      for (int hb = 0; hb < 2; ++hb) m = fmaxf(m, fmaxf(fmaxf(x[hb][0], x[hb][1]), fmaxf(x[hb][2], x[hb][3])));
      m = allreduce_bit32(allreduce_bit16(m, OpMax()), OpMax());
      const bool moved = m > shift[cb] + kMove;
      if (__builtin_amdgcn_ballot_w64(moved) != 0) {
        // exp2(-inf) = 0 for a query without a key so far: its sums are 0.
        const float next = moved ? m : shift[cb];
        const float scale = moved ? __builtin_amdgcn_exp2f(shift[cb] - m) : 1.f;
        shift[cb] = next;
        total[cb] *= scale;
#pragma unroll
        for (int u = 0; u < kDTiles; ++u) acc[cb][u] *= scale;
      }
      const float off = shift[cb] == -INFINITY ? 0.f : shift[cb];
      uint32_t hi[4], lo[4];
#pragma unroll
      for (int hb = 0; hb < 2; ++hb) {
        float w[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) w[r] = __builtin_amdgcn_exp2f(x[hb][r] - off);
        Ops::split2(w[0], w[1], hi[2 * hb], lo[2 * hb]);
        Ops::split2(w[2], w[3], hi[2 * hb + 1], lo[2 * hb + 1]);
      }
      p_hi[cb] = __builtin_bit_cast(Qk, make_uint4(hi[0], hi[1], hi[2], hi[3]));
      p_lo[cb] = __builtin_bit_cast(Qk, make_uint4(lo[0], lo[1], lo[2], lo[3]));
    }
#pragma unroll
    for (int u = 0; u < kDTiles; ++u) {
      const int row = 4 * grp + col / 4;
      const int chunk = 2 * u + (col % 4) / 2;
      const int half = (col & 1) * 8;
      const unsigned char* from = vl + at(row, chunk) + half;
      const uint2 a0 = lds_read_tr16(from);
      const uint2 a1 = lds_read_tr16(from + 16 * kRowBytes);  // row + 16: the same permutation
      const Qk a = __builtin_bit_cast(Qk, make_uint4(a0.x, a0.y, a1.x, a1.y));
#pragma unroll
      for (int cb = 0; cb < kCB; ++cb) {
        acc[cb][u] = Ops::qk(a, p_hi[cb], acc[cb][u]);
        acc[cb][u] = Ops::qk(a, p_lo[cb], acc[cb][u]);
      }
    }
    // The sum of the same pairs, on the vector unit while the products run.
#pragma unroll
    for (int cb = 0; cb < kCB; ++cb) {
      const uint4 hi = __builtin_bit_cast(uint4, p_hi[cb]), lo = __builtin_bit_cast(uint4, p_lo[cb]);
      const float sum_lo = Ops::add2(lo.w, Ops::add2(lo.z, Ops::add2(lo.y, Ops::add2(lo.x, 0.f))));
      total[cb] = Ops::add2(hi.w, Ops::add2(hi.z, Ops::add2(hi.y, Ops::add2(hi.x, total[cb] + sum_lo))));
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }

#pragma unroll
  for (int cb = 0; cb < kCB; ++cb) {
    total[cb] = allreduce_bit32(allreduce_bit16(total[cb], OpSum()), OpSum());
    if (grp == 0) {
      part_shift[wave][16 * cb + col] = shift[cb];
      part_total[wave][16 * cb + col] = total[cb];
    }
  }
  __syncthreads();

  // ---- Merge: every wave's accumulators over the staging area.
  float* part = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int cb = 0; cb < kCB; ++cb) {
#pragma unroll
    for (int u = 0; u < kDTiles; ++u)
      *reinterpret_cast<float4*>(part + ((wave * kRows + 16 * cb + col) * kD + 4 * ((4 * u + grp) ^ (col & 7)))) =
          make_float4(acc[cb][u][0], acc[cb][u][1], acc[cb][u][2], acc[cb][u][3]);
  }
  __syncthreads();
  // A thread sums 4 dims of a query over the waves.
  char* out_plane = static_cast<char*>(p.out) + (b * p.so[0] + h * p.so[1]) * static_cast<int64_t>(kOutSize);
  for (int slot = tid; slot < kRows * kD / 4; slot += 64 * kWaves) {
    const int row = slot / (kD / 4);
    const int quad = slot % (kD / 4);
    if (first_q + row >= n_q) break;  // rows ascend
    float m = -INFINITY;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) m = fmaxf(m, part_shift[w][row]);
    if (m == -INFINITY) m = 0.f;
    float sum = 0.f, y[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int w = 0; w < kWaves; ++w) {
      // A wave without a key that counts holds shift -inf and zeros (or NaN).
      const float f = __builtin_amdgcn_exp2f(part_shift[w][row] - m);
      const float4 a = *reinterpret_cast<const float4*>(part + ((w * kRows + row) * kD + 4 * (quad ^ (row & 7))));
      sum = fmaf(part_total[w][row], f, sum);
      y[0] = fmaf(a.x, f, y[0]);
      y[1] = fmaf(a.y, f, y[1]);
      y[2] = fmaf(a.z, f, y[2]);
      y[3] = fmaf(a.w, f, y[3]);
    }
    // A fully masked row has sum 0 and ends as 0 * inf = NaN.
    const float inv = __builtin_amdgcn_rcpf(sum);
    const uint32_t off = (static_cast<uint32_t>(first_q + row) * static_cast<uint32_t>(p.so[2]) +
                          static_cast<uint32_t>(4 * quad) * static_cast<uint32_t>(p.so[3])) * kOutSize;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *reinterpret_cast<OutT*>(out_plane + off + r * static_cast<uint32_t>(p.so[3]) * kOutSize) =
          from_float<OutT>(y[r] * inv);
  }
}

template <typename T, typename OutT, int kD, int kCB>
hipError_t launch_span_k(Problem& p, hipStream_t s) {
  const int64_t q_blocks = (p.Nq + 16 * kCB - 1) / (16 * kCB);
  Problem k = p;  // the kernel divides work items by q_blocks with the Nq slots
  make_fast_div(q_blocks, &k.nq_mul, &k.nq_shift);
  int32_t qb = static_cast<int32_t>(q_blocks);
  void* args[] = {&k, &qb};
  return hipLaunchKernel(reinterpret_cast<const void*>(&rbf_span_kernel<T, OutT, kD, kCB>),
                         dim3(static_cast<unsigned>(p.B * p.H * q_blocks)), dim3(64 * span_waves<kD>()), args, 0, s);
}

// Items of 16 queries while the chip's CUs hold them all at once, else of 32.
template <typename T, typename OutT, int kD>
hipError_t launch_span(Problem& p, int64_t units, hipStream_t s) {
  if (p.B * p.H * ((p.Nq + 15) / 16) <= units) return launch_span_k<T, OutT, kD, 1>(p, s);
  return launch_span_k<T, OutT, kD, 2>(p, s);
}

}  // namespace vectra
