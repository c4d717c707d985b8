// Whole planes of up to a few hundred keys on gfx950 matrix cores: the kernel
// template, instantiated with the tile kernel's dtype pairs in
// rbf_tile_<in>_<out>.hip (a plane whose keys fit LDS takes this kernel, a
// longer one streams its tiles through rbf_tile_kernel).
//
// A workgroup stages one (b, h) plane's K and V in LDS once, behind one
// barrier, and its waves then take blocks of 16 queries (kCB at a time) in
// turn, each against every key, with no further barrier.  The products and
// their lane layouts are the tile kernel's:
//
//   S^T = K . Q^T     (16 keys x 16 queries per instruction, 32-deep steps)
//   O^T = V^T . P^T   (16 value dims x 16 queries)
//   x = coef (q.k - |q|^2 / 2) + c_j,  c_j = log2(e) (bias_j - gamma |k_j|^2)
//
// and weights go to the second product as hi + lo 16-bit pairs; a product of
// the same pairs with ones divides it, so that what the split drops of a
// dominant weight drops out, as in the tile kernel.  (The sum of the unsplit
// weights on the vector unit took the same time, 27.2 us for the first shape
// below, and left 1.2 to 1.7 times the error without a bias in fp16 and with
// an additive one in bf16.)  Without a bias and with gamma >= 0 the
// weights are used as they come (x <= 0); otherwise each query's weights are
// shifted by its largest logit over the first 32 keys that count.  Where a
// query's weight sum leaves the range in which the split is accurate (or a
// value overflows), the wave computes its blocks again with each query's
// exact maximum: no other wave is involved.
//
// Pairs of 16-key blocks without a key that counts (masked with a -inf bias,
// or past Nk; a masked key whose K norm or V row is not finite counts) are
// skipped: such weights are exactly 0.
//
// LDS: K and V rows without padding, their 16-byte chunks permuted by the
// row so that the operand reads of 16 rows fall into distinct bank groups
// (the rows one 256-byte span of banks holds share a permutation); padded
// rows would leave 64-dim planes of 257 keys one workgroup per CU instead of
// two.
//
// Bound: the staging latency and the arithmetic after it (a plane is read
// once from HBM).  Streaming the same planes through the tile kernel staged
// them once per 64-256 queries and split them into work items that a 257th
// query leaves half empty.  Measured, bf16 with ragged key masks, streamed
// (two passes, as masked planes took them) and here: 512 planes of 257 x 257 x
// 64 76 and 25 us (HBM: 13), 1,600 of 100 x 100 x 64 81 and 23, 1,200 of
// 130 x 130 x 128 110 and 55, 400 of 200 x 200 x 32 22 and 14.5.  Two query
// blocks per wave (107 registers, four waves per SIMD, against 88) halve the
// operand reads and were 5-30% slower.

#pragma once

#include "rbf_common.h"
#include "rbf_kernels.h"
#include "rbf_mfma_ops.h"
#include "rbf_tile_ops.h"

namespace vectra {

// LDS of a workgroup: two per CU fit up to half of it.
constexpr int64_t kBlockLdsBytes = 160 * 1024 - 256;
constexpr int64_t kBlockMaxKeys = 1024;  // 32 bits of key pairs

template <int kD>
constexpr int64_t block_lds_bytes(int64_t n_k) {
  return (n_k + 31) / 32 * 32 * (4 * kD + 4);
}

template <typename T, typename OutT, int kD, int kWaves>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(kD <= 64 ? 4 : 2))) void
rbf_block_kernel(Problem p, int32_t splits, int32_t blocks_per_split, int32_t first_plane) {
  using Ops = MfmaOps<T>;
  using Qk = typename Ops::Qk;
  constexpr int kCB = 1;  // query blocks a wave takes at a time (see above)
  constexpr int kThreads = 64 * kWaves;
  constexpr int kChunks = kD / 8;       // 16-byte chunks of a row
  constexpr int kKSteps = kD / 32;      // 32-deep steps of S^T
  constexpr int kDTiles = kD / 16;
  constexpr int kRowBytes = 2 * kD;
  constexpr int kRowsPerSpan = 256 / kRowBytes;  // rows of one span of the banks
  constexpr int kStage = 4;                      // slots a thread has in flight
  constexpr uint32_t kOutSize = sizeof(OutT);
  constexpr bool kBf16 = __is_same(T, __bf16);
  constexpr float kSumLo = kBf16 ? 0x1p-32f : 0x1p-3f;
  constexpr float kSumHi = kBf16 ? 0x1p32f : 0x1p15f;

  extern __shared__ __align__(16) unsigned char lds[];
  __shared__ uint32_t live_pairs;  // bit kp: key pair kp has a key that counts
  __shared__ uint32_t any_live;    // with a bias: some key is not masked

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15;
  const int grp = lane >> 4;
  const int32_t n_q = static_cast<int32_t>(p.Nq);
  const int32_t n_k = static_cast<int32_t>(p.Nk);
  const int32_t pairs = (n_k + 31) / 32;
  const bool has_bias = p.bias != nullptr;
  const int32_t bias_esize = p.bias_dtype == VECTRA_F32 ? 4 : 2;
  const uint32_t q_row_bytes = static_cast<uint32_t>(p.sq[2]) * 2u;
  const uint32_t k_row_bytes = static_cast<uint32_t>(p.sk[2]) * 2u;
  const uint32_t v_row_bytes = static_cast<uint32_t>(p.sv[2]) * 2u;
  const uint32_t o_row = static_cast<uint32_t>(p.so[2]);
  const uint32_t o_dim = static_cast<uint32_t>(p.so[3]);
  constexpr int64_t kOutAlign = 16 / kOutSize;
  const bool out_vec = p.so[3] == 1 && p.so[2] % kOutAlign == 0 && p.so[1] % kOutAlign == 0 && p.so[0] % kOutAlign == 0 &&
                       (reinterpret_cast<uintptr_t>(p.out) & 15u) == 0;

  // XCD-local order: workgroups go round-robin over the 8 XCDs, and a
  // plane's workgroups and a batch entry's heads run on one.
  const int32_t items = static_cast<int32_t>(gridDim.x);
  int32_t item = static_cast<int32_t>(blockIdx.x);
  if (items % 8 == 0) item = (item & 7) * (items / 8) + (item >> 3);
  const int32_t plane = static_cast<int32_t>(fast_div(static_cast<uint32_t>(item), p.nq_mul, p.nq_shift));
  const int32_t split = item - plane * splits;
  const int32_t bh = first_plane + plane;
  const int32_t b = static_cast<int32_t>(fast_div(static_cast<uint32_t>(bh), p.h_mul, p.h_shift));
  const int32_t h = bh - b * static_cast<int32_t>(p.H);
  const int32_t q_blocks = (n_q + 15) / 16;
  const int32_t first_block = split * blocks_per_split;
  const int32_t end_block = min(first_block + blocks_per_split, q_blocks);

  unsigned char* kl = lds;
  unsigned char* vl = lds + pairs * 32 * kRowBytes;
  float* cl = reinterpret_cast<float*>(lds + 2 * pairs * 32 * kRowBytes);
  // Byte offset of chunk `chunk` of row `row` in K or V.
  auto at = [](int row, int chunk) { return row * kRowBytes + ((chunk ^ ((row / kRowsPerSpan) & (kChunks - 1))) * 16); };

  if (tid == 0) live_pairs = any_live = 0u;
  const float coef = 2.f * kLog2e * load_any(p.scale, b * p.ssb + h * p.ssh, p.scale_dtype);
  __syncthreads();

  // ---- Stage the plane: kStage slots (a 16-byte chunk of K and of V) per
  // thread at a time, every load of them issued first.  Rows past Nk read
  // zeros (buffer loads end at the plane's last row; where rows overlap they
  // read its own rows) and are stored as zeros.
  {
    const char* kp = static_cast<const char*>(p.k) + (b * p.sk[0] + h * p.sk[1]) * 2;
    const char* vp = static_cast<const char*>(p.v) + (b * p.sv[0] + h * p.sv[1]) * 2;
    const auto k_rsrc = plane_rsrc(kp, static_cast<uint32_t>(n_k - 1) * k_row_bytes + kD * 2);
    const auto v_rsrc = plane_rsrc(vp, static_cast<uint32_t>(n_k - 1) * v_row_bytes + kD * 2);
    const char* bp = static_cast<const char*>(p.bias) + (b * p.sbb + h * p.sbh) * bias_esize;
    const uint32_t misalign = base_misalign(bp);
    const int chunk = tid % kChunks;
    const int slots = pairs * 32 * kChunks;
    for (int slot0 = tid; slot0 < slots; slot0 += kStage * kThreads) {
      uint4 ks[kStage], vs[kStage];
      uint32_t bias_word[kStage];
#pragma unroll
      for (int s = 0; s < kStage; ++s) {
        const int key = (slot0 + s * kThreads) / kChunks;
        const uint32_t row = static_cast<uint32_t>(min(key, n_k - 1));
        ks[s] = load16_buf(k_rsrc, row * k_row_bytes + chunk * 16u);
        vs[s] = load16_buf(v_rsrc, row * v_row_bytes + chunk * 16u);
        if (has_bias)
          bias_word[s] = load_raw_scalar32(bp, misalign, row * static_cast<uint32_t>(p.sbn), p.bias_dtype).word;
      }
#pragma unroll
      for (int s = 0; s < kStage; ++s) {
        const int slot = slot0 + s * kThreads;  // wave-uniform bound: whole waves of slots
        if (slot >= slots) break;
        const int key = slot / kChunks;
        const bool in = key < n_k;
        const float sq = reduce_low<kChunks>(dot_chunk<T>(ks[s], ks[s], 0.f), OpSum());
        float bias = 0.f;
        bool unmasked = in;
        if (has_bias) {
          const uint32_t bytes =
              static_cast<uint32_t>(min(key, n_k - 1)) * static_cast<uint32_t>(p.sbn) * bias_esize + misalign;
          bias = decode_raw_scalar(RawScalar{bias_word[s], (bytes & 2u) * 8u}, p.bias_dtype) * kLog2e;
          unmasked = in && !(bias == -INFINITY && __builtin_isfinite(sq));
        }
        const uint64_t live = __builtin_amdgcn_ballot_w64(unmasked);
        const uint64_t counts = live | __builtin_amdgcn_ballot_w64(in && !finite_chunk<T>(vs[s]));
        if (lane == 0) {
          if (counts != 0) atomicOr(&live_pairs, 1u << (key / 32));
          if (live != 0) any_live = 1u;
        }
        if (!in) ks[s] = vs[s] = make_uint4(0, 0, 0, 0);
        *reinterpret_cast<uint4*>(kl + at(key, chunk)) = ks[s];
        *reinterpret_cast<uint4*>(vl + at(key, chunk)) = vs[s];
        if (chunk == 0) cl[key] = in ? fmaf(-0.5f * coef, sq, bias) : -INFINITY;
      }
    }
  }
  __syncthreads();
  const uint32_t live = __builtin_amdgcn_readfirstlane(live_pairs);
  const bool plane_live = __builtin_amdgcn_readfirstlane(any_live) != 0;
  const bool plain = !has_bias && coef >= 0.f;

  // ---- The wave's query blocks.
  const uint32_t one = Ops::kOnePair;
  const Qk ones8 = __builtin_bit_cast(Qk, make_uint4(one, one, one, one));
  const char* qp = static_cast<const char*>(p.q) + (b * p.sq[0] + h * p.sq[1]) * 2;
  char* out_plane = static_cast<char*>(p.out) + (b * p.so[0] + h * p.so[1]) * static_cast<int64_t>(kOutSize);
  for (int32_t block = first_block + wave * kCB; block < end_block; block += kWaves * kCB) {
    uint4 qf[kCB][kKSteps];
    float q_half[kCB];
#pragma unroll
    for (int cb = 0; cb < kCB; ++cb) {
      // Rows past Nq read row Nq - 1 and are not stored.
      const uint32_t row = static_cast<uint32_t>(min((block + cb) * 16 + col, n_q - 1));
#pragma unroll
      for (int ks = 0; ks < kKSteps; ++ks)
        qf[cb][ks] = load16(qp + row * q_row_bytes + static_cast<uint32_t>(64 * ks + 16 * grp));
    }
#pragma unroll
    for (int cb = 0; cb < kCB; ++cb) {
      float sq = 0.f;
#pragma unroll
      for (int ks = 0; ks < kKSteps; ++ks) sq = dot_chunk<T>(qf[cb][ks], qf[cb][ks], sq);
      q_half[cb] = -0.5f * allreduce_bit32(allreduce_bit16(sq, OpSum()), OpSum());
    }

    // The logits (in log2 units) of key pair kp: lane (query col, group g)
    // gets keys 32 kp + 16 hb + 4 g + r.
    auto logits = [&](int kp, float (&x)[kCB][2][4]) __attribute__((always_inline)) {
      f32x4 s[kCB][2];
#pragma unroll
      for (int hb = 0; hb < 2; ++hb) {
#pragma unroll
        for (int ks = 0; ks < kKSteps; ++ks) {
          const Qk a = *reinterpret_cast<const Qk*>(kl + at(32 * kp + 16 * hb + col, 4 * ks + grp));
#pragma unroll
          for (int cb = 0; cb < kCB; ++cb)
            s[cb][hb] = Ops::qk(a, __builtin_bit_cast(Qk, qf[cb][ks]),
                                ks == 0 ? f32x4{q_half[cb], q_half[cb], q_half[cb], q_half[cb]} : s[cb][hb]);
        }
      }
#pragma unroll
      for (int hb = 0; hb < 2; ++hb) {
        const float4 c = *reinterpret_cast<const float4*>(cl + 32 * kp + 16 * hb + 4 * grp);
#pragma unroll
        for (int cb = 0; cb < kCB; ++cb) {
          x[cb][hb][0] = fmaf(coef, s[cb][hb][0], c.x);
          x[cb][hb][1] = fmaf(coef, s[cb][hb][1], c.y);
          x[cb][hb][2] = fmaf(coef, s[cb][hb][2], c.z);
          x[cb][hb][3] = fmaf(coef, s[cb][hb][3], c.w);
        }
      }
    };
    // Each query's largest logit over the given pairs; 0 where none is live
    // (the row then ends as NaN, or its sum leaves the range).
    float shift[kCB];
    auto largest = [&](uint32_t mask) __attribute__((always_inline)) {
#pragma unroll
      for (int cb = 0; cb < kCB; ++cb) shift[cb] = -INFINITY;
      for (; mask != 0; mask &= mask - 1) {
        float x[kCB][2][4];
        logits(__builtin_ctz(mask), x);
#pragma unroll
        for (int cb = 0; cb < kCB; ++cb)
#pragma unroll
          for (int hb = 0; hb < 2; ++hb)
            shift[cb] = fmaxf(shift[cb], fmaxf(fmaxf(x[cb][hb][0], x[cb][hb][1]), fmaxf(x[cb][hb][2], x[cb][hb][3])));
      }
#pragma unroll
      for (int cb = 0; cb < kCB; ++cb) {
        const float m = allreduce_bit32(allreduce_bit16(shift[cb], OpMax()), OpMax());
        shift[cb] = m == -INFINITY ? 0.f : m;
      }
    };

    f32x4 acc[kCB][kDTiles];
    f32x4 total[kCB];  // every row of the product with ones: the weight sum of the lane's query
#pragma unroll
    for (int cb = 0; cb < kCB; ++cb) shift[cb] = 0.f;
    uint32_t max_pairs = plain ? 0u : (live & (0u - live));  // pairs the shift is taken over
    while (true) {
      if (max_pairs != 0) largest(max_pairs);
#pragma unroll
      for (int cb = 0; cb < kCB; ++cb) {
        total[cb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < kDTiles; ++u) acc[cb][u] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      for (uint32_t mask = live; mask != 0; mask &= mask - 1) {
        const int kp = __builtin_ctz(mask);
        float x[kCB][2][4];
        logits(kp, x);
        Qk p_hi[kCB], p_lo[kCB];
#pragma unroll
        for (int cb = 0; cb < kCB; ++cb) {
          uint32_t hi[4], lo[4];
#pragma unroll
          for (int hb = 0; hb < 2; ++hb) {
            float w[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) w[r] = __builtin_amdgcn_exp2f(x[cb][hb][r] - shift[cb]);
            Ops::split2(w[0], w[1], hi[2 * hb], lo[2 * hb]);
            Ops::split2(w[2], w[3], hi[2 * hb + 1], lo[2 * hb + 1]);
          }
          p_hi[cb] = __builtin_bit_cast(Qk, make_uint4(hi[0], hi[1], hi[2], hi[3]));
          p_lo[cb] = __builtin_bit_cast(Qk, make_uint4(lo[0], lo[1], lo[2], lo[3]));
          total[cb] = Ops::qk(ones8, p_hi[cb], total[cb]);
          total[cb] = Ops::qk(ones8, p_lo[cb], total[cb]);
        }
#pragma unroll
        for (int u = 0; u < kDTiles; ++u) {
          // A operand of O^T (see rbf_tile_kernel): lane i of a 16-lane group
          // addresses key row 32kp + 4g + i / 4 (+16), dims 16u + 4 (i % 4).
          const int row = 32 * kp + 4 * grp + col / 4;
          const int chunk = 2 * u + (col % 4) / 2;
          const int half = (col & 1) * 8;
          const uint2 a0 = lds_read_tr16(vl + at(row, chunk) + half);
          const uint2 a1 = lds_read_tr16(vl + at(row + 16, chunk) + half);
          const Qk a = __builtin_bit_cast(Qk, make_uint4(a0.x, a0.y, a1.x, a1.y));
#pragma unroll
          for (int cb = 0; cb < kCB; ++cb) {
            acc[cb][u] = Ops::qk(a, p_hi[cb], acc[cb][u]);
            acc[cb][u] = Ops::qk(a, p_lo[cb], acc[cb][u]);
          }
        }
      }
      bool off = false;
#pragma unroll
      for (int cb = 0; cb < kCB; ++cb) {
        off = off || !(total[cb][0] >= kSumLo && (plain || total[cb][0] <= kSumHi));
        if (!plain) {
#pragma unroll
          for (int u = 0; u < kDTiles; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r) off = off || !__builtin_isfinite(acc[cb][u][r]);
        }
      }
      // Once more with the exact maxima, unless that was this pass or no key
      // of the plane is live (every sum is 0 and every row NaN already).
      if (max_pairs == live || !plane_live || __builtin_amdgcn_ballot_w64(off) == 0) break;
      max_pairs = live;
    }

    // ---- Store; a fully masked row has sum 0 and ends as 0 * inf = NaN.
#pragma unroll
    for (int cb = 0; cb < kCB; ++cb) {
      const int32_t q_row = (block + cb) * 16 + col;
      if (block + cb >= end_block) continue;
      const float inv = __builtin_amdgcn_rcpf(total[cb][0]);
      const uint32_t row_off = static_cast<uint32_t>(q_row) * o_row;
      if constexpr (kOutSize == 2) {
        if (out_vec) {
          // One swap between lane groups 2m and 2m + 1 leaves each lane 8
          // adjacent dims (rbf_plane_kernel): 16-byte non-temporal stores.
          const uint32_t t = static_cast<uint32_t>(((grp & 1) << 1) | (grp >> 1));
#pragma unroll
          for (int j = 0; j < kDTiles / 2; ++j) {
            uint32_t w[2][2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              w[u][0] = pack2<OutT>(acc[cb][2 * j + u][0] * inv, acc[cb][2 * j + u][1] * inv);
              w[u][1] = pack2<OutT>(acc[cb][2 * j + u][2] * inv, acc[cb][2 * j + u][3] * inv);
            }
            const auto s0 = __builtin_amdgcn_permlane16_swap(w[0][0], w[1][0], false, false);
            const auto s1 = __builtin_amdgcn_permlane16_swap(w[0][1], w[1][1], false, false);
            if (q_row < n_q)
              __builtin_nontemporal_store(u32x4{s0[0], s1[0], s0[1], s1[1]},
                                          reinterpret_cast<u32x4*>(out_plane + (row_off + 32u * j + 8u * t) * 2u));
          }
          continue;
        }
      }
      if (q_row >= n_q) continue;
#pragma unroll
      for (int u = 0; u < kDTiles; ++u) {
        const uint32_t off = (row_off + static_cast<uint32_t>(16 * u + 4 * grp) * o_dim) * kOutSize;
        const float y[4] = {acc[cb][u][0] * inv, acc[cb][u][1] * inv, acc[cb][u][2] * inv, acc[cb][u][3] * inv};
        if constexpr (kOutSize == 4) {
          if (out_vec) {
            *reinterpret_cast<float4*>(out_plane + off) = make_float4(y[0], y[1], y[2], y[3]);
            continue;
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
          *reinterpret_cast<OutT*>(out_plane + off + r * o_dim * kOutSize) = from_float<OutT>(y[r]);
      }
    }
  }
}

// ------------------------------------------------------------------- host

template <typename T, typename OutT, int kD, int kWaves>
hipError_t launch_block_k(Problem& p, int64_t splits, int64_t per_split, hipStream_t s) {
  Problem k = p;  // the kernel divides workgroups by the splits with the Nq slots
  make_fast_div(splits, &k.nq_mul, &k.nq_shift);
  int32_t n = static_cast<int32_t>(splits), per = static_cast<int32_t>(per_split), first = 0;
  void* args[] = {&k, &n, &per, &first};
  // A grid holds fewer than 2^32 threads: very many planes take several
  // launches (planes below 2^30: tile_supports).
  const int64_t planes = p.B * p.H, most = 0xffffffffLL / (64 * kWaves) / splits;
  for (int64_t plane = 0; plane < planes; plane += most) {
    const int64_t here = planes - plane < most ? planes - plane : most;
    first = static_cast<int32_t>(plane);
    const hipError_t err = hipLaunchKernel(reinterpret_cast<const void*>(&rbf_block_kernel<T, OutT, kD, kWaves>),
                                           dim3(static_cast<unsigned>(here * splits)), dim3(64 * kWaves), args,
                                           static_cast<size_t>(block_lds_bytes<kD>(p.Nk)), s);
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

// Waves per workgroup by its LDS, so that the CU's workgroups together hold
// about 16 waves, and as many workgroups per plane as fill the chip once
// (each stages the whole plane; a second round of workgroups costs more than
// longer ones), at most one per four query blocks.
// Measured with 4 / 8 / 16 waves, us: 512 planes of 257 x 257, 64 dims (75 KB)
// 30.1 / 24.9 / 28.1; 1,200 of 130 x 130, 128 dims (83 KB) 94 / 67 / 55; 800 of
// 400 x 400, 64 dims (108 KB) 134 / 87 / 78; 1,600 of 100 x 100, 64 dims (33 KB)
// 23.2 / 26.7 / -.  64 planes of 500 x 500 in 512 workgroups 22.3, in 256 14.9.
struct BlockShape {
  int waves;           // per workgroup
  int64_t resident;    // workgroups on the chip at once
  int64_t splits, per;  // workgroups per plane and query blocks of each
};

template <int kD>
BlockShape block_shape(const Problem& p) {
  BlockShape b;
  const int64_t planes = p.B * p.H, blocks = (p.Nq + 15) / 16;
  const int64_t lds = block_lds_bytes<kD>(p.Nk);
  b.waves = lds <= 40 * 1024 ? 4 : (lds <= 80 * 1024 ? 8 : 16);
  const int64_t by_lds = kBlockLdsBytes / lds, by_waves = 16 / b.waves;
  b.resident = (p.compute_units > 0 ? p.compute_units : 1) * (by_lds < by_waves ? by_lds : by_waves);
  b.splits = b.resident / planes;
  if (b.splits > (blocks + 3) / 4) b.splits = (blocks + 3) / 4;
  if (b.splits < 1) b.splits = 1;
  b.per = (blocks + b.splits - 1) / b.splits;
  b.splits = (blocks + b.per - 1) / b.per;
  return b;
}

// Whether planes whose keys fit LDS are better streamed by the tile kernel all
// the same: without a bias, from 256 keys (160 of 128 dims) and two of its
// items per CU on, by time.  In units of one query block of this kernel on a CU (0.9 us
// at 600 keys of 64 dims): a workgroup takes its blocks and 7 for the staging,
// an item of the tile kernel 9.4 (128 rows of 32 dims), 24.6 (256 of 64) or
// 12.3 (128 of 128), and the fullest CU decides.  Here and streamed, us: 300
// planes of 700 x 600 x 64 (two workgroups on some CUs, 1.2 on average) 99 and
// 79, of 700 x 600 x 32 74 and 55, 1000 of 100 x 600 x 32 36 and 31; 256 of
// 512 x 512 x 64 41 and 43, 128 of 600 x 600 x 64 27 and 42, 256 of
// 600 x 288 x 128 44 and 55.  fp16 planes of 64 and 128 dims stay: the
// unshifted weights of rows far from their keys leave fp16's range and take the
// tile kernel three passes (300 planes of 700 x 350 x 64 65 and 103; at 32 dims
// rows lie nearer, 1000 of 100 x 1000 x 32 71 and 43).  From 1,024 keys on the
// tile kernel weighs by fp16: not here.
template <typename T, int kD>
bool block_streams(const Problem& p, int64_t most_keys) {
  if (!__is_same(T, __bf16) && kD != 32) return false;
  if (p.bias != nullptr || p.Nk < (kD == 128 ? 160 : 256) || p.Nk >= most_keys) return false;
  const BlockShape b = block_shape<kD>(p);
  const int64_t planes = p.B * p.H, units = p.compute_units > 0 ? p.compute_units : 1;
  constexpr int64_t kRows = kD == 64 ? 256 : 128;
  constexpr double kItem = kD == 32 ? 9.4 : (kD == 64 ? 24.6 : 12.3);
  const int64_t items = (planes * ((p.Nq + kRows - 1) / kRows) + units - 1) / units;
  const int64_t staged = (planes * b.splits + units - 1) / units;
  return items >= 2 && kItem * static_cast<double>(items) < static_cast<double>(staged * (7 + b.per));
}

template <typename T, typename OutT, int kD>
hipError_t launch_block_d(Problem& p, hipStream_t s) {
  const BlockShape b = block_shape<kD>(p);
  const int waves = b.waves;
  const int64_t splits = b.splits, per = b.per;
  if (waves == 16) return launch_block_k<T, OutT, kD, 16>(p, splits, per, s);
  if (waves == 8) return launch_block_k<T, OutT, kD, 8>(p, splits, per, s);
  return launch_block_k<T, OutT, kD, 4>(p, splits, per, s);
}

}  // namespace vectra
