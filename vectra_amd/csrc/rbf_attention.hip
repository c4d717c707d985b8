// Fused RBF attention for MI355X (gfx950 / CDNA4, wave64).
//
//   out[b,h,i,:] = sum_j softmax_j(-scale[b,h] * max(|q_i|^2 + |k_j|^2 - 2 q_i.k_j, 0)
//                                  + key_bias[b,h,j]) * v[b,h,j,:]
//
// Semantics follow the reference operator (kernels/vectra_kernels/
// spatial_rbf_attention.py:47-174 and custom_ops.py:52-72):
//  * distances by the Euclidean expansion with a clamp at zero (:137);
//  * logits -scale*d plus the key bias; without a bias only keys < Nk count
//    (:139-150);
//  * an online softmax whose running maximum is replaced by 0 while it is
//    still -inf, so a row whose keys are all masked ends as 0/0 = NaN, as
//    eager softmax gives (:152-157);
//  * fp32 accumulation throughout, the result divided by the running sum and
//    converted once to the output dtype (:168-174).
// Unlike the reference kernel, the attention weights are never rounded to
// the input dtype before the value product: P.V accumulates in fp32.
//
// Kernels in this file:
//  * rbf_stream_kernel  -- few query rows per (b,h) plane (the serving shape:
//    one subject query against tens of comparables).  HBM-bound: each wave
//    owns one query row, streams the plane's K and V once with coalesced
//    128-bit loads straight into registers and reduces with DPP.
//  * rbf_split_kernel   -- the same for more than one key tile: the waves of a
//    workgroup share a row's key axis.
//  * rbf_generic_kernel -- any strides, head dims and alignments.
//  * rbf_mfma_kernel (rbf_mfma.hip) -- query tiles on bf16/fp16 MFMA.

#include "rbf_common.h"
#include "rbf_kernels.h"

namespace vectra {

// ------------------------------------------------------------------------
// Stream kernel.
//
// Layout: a 64-key tile of K is 64 rows of D = kChunks * Vec<T> elements.
// Lane l holds chunk (l % kChunks) of key rows  p * (64 / kChunks) + l / kChunks
// for the kChunks passes p, so each pass is one fully coalesced 1 KiB wave
// load.  V is held the same way (requires Dv == D), so a lane owns the value
// chunk of exactly the keys whose weights it computed and P.V needs no
// shuffle until the final reduction.
//
// Scheduling: one key tile per row (Nk <= 64; longer key axes take the split
// kernel below).  Where a wave takes several rows, it has the next one in
// flight while it reduces the current one, so the softmax and P.V arithmetic
// of one row overlaps the HBM stream of the next.  Every load of a row (K, V,
// the key bias, q and the coefficient) is issued together; rows past Nk are
// loaded from row Nk - 1 (always in bounds) and masked afterwards, so no load
// is behind a branch.  Per-lane addresses are 32-bit offsets from
// wave-uniform bases.
// ------------------------------------------------------------------------

// Sums kVec accumulators per lane over the row-group lane bits (kChunks ..
// 32) of the stream layout.  Lane bits 32 and 16 use butterfly steps: a
// permlane swap of the value pair (a_i, a_{i+n/2}) hands each half of the
// wave the partner's copy of the half it keeps, so one swap and one add
// halve the values per lane.  The remaining row-group bits (below 16) are
// all-reduced with DPP.  On return res[0 .. kVec/4) are the finished sums of
// elements first_e .. first_e + kVec/4 of the lane's chunk.
template <int kChunks, int kVec>
__device__ __forceinline__ void reduce_rows_butterfly(const float* acc, float* res, int& first_e) {
  const int lane = threadIdx.x & (kWave - 1);
  constexpr int kHalf = kVec / 2, kQuarter = kVec / 4;
  float half[kHalf];
#pragma unroll
  for (int i = 0; i < kHalf; ++i) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[i]),
                                                    __float_as_uint(acc[i + kHalf]), false, false);
    half[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);  // lanes < 32: a_i, else a_{i+n/2}
  }
#pragma unroll
  for (int i = 0; i < kQuarter; ++i) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(half[i]),
                                                    __float_as_uint(half[i + kQuarter]), false, false);
    res[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  first_e = ((lane & 32) ? kHalf : 0) + ((lane & 16) ? kQuarter : 0);
  if constexpr (kChunks < 16) {
#pragma unroll
    for (int i = 0; i < kQuarter; ++i) {
      float x = res[i];
      if constexpr (kChunks <= 1) x += dpp<0xB1>(x);
      if constexpr (kChunks <= 2) x += dpp<0x4E>(x);
      if constexpr (kChunks <= 4) {
        x += dpp<0x124>(x);
        x += dpp<0x128>(x);
      } else {
        x += dpp<0x128>(x);
      }
      res[i] = x;
    }
  }
}

template <int kPasses>
struct StreamSlot {
  uint4 k[kPasses];
  uint4 v[kPasses];
  uint32_t bias[kPasses];  // aligned words holding the key biases
  uint32_t bias_misalign;  // address & 3 of the row's bias plane (wave-uniform)
  uint4 q;
  RawScalar scale;
};

struct RowCoords {
  int32_t b, h, i;
};

__device__ __forceinline__ RowCoords row_coords(int32_t row, const Problem& p) {
  RowCoords c;
  const int32_t bh = static_cast<int32_t>(fast_div(row, p.nq_mul, p.nq_shift));
  c.i = row - bh * static_cast<int32_t>(p.Nq);
  c.b = static_cast<int32_t>(fast_div(bh, p.h_mul, p.h_shift));
  c.h = bh - c.b * static_cast<int32_t>(p.H);
  return c;
}

template <typename T, typename OutT, int kChunks, int kRows>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void rbf_stream_kernel(Problem p) {
  // The wave takes rows wave * kRows .. + kRows - 1, each one key tile
  // (Nk <= 64), in a fully unrolled pipeline with no loop and no branch
  // around a load, so the compiler can wait for exactly the loads each step
  // needs.  Rows past the end are clamped to the last row: the duplicate
  // wave recomputes that row and stores the same bytes.
  constexpr int kVec = Vec<T>::kN;
  constexpr int kRowsPerPass = kWave / kChunks;
  constexpr int kPasses = kChunks;  // kPasses * kRowsPerPass == 64 keys
  using Slot = StreamSlot<kPasses>;

  // Every argument read below, loaded in one batch (measured at the serving
  // shape: 12.4 -> 12.0 us back to back, 12.9 -> 12.65 us per isolated launch).
  args_in_sgprs(p.q, p.k, p.v, p.out, p.scale, p.bias, p.scale_dtype, p.bias_dtype, p.H, p.Nq, p.Nk);
  args_in_sgprs(p.sq[0], p.sq[1], p.sq[2], p.sk[0], p.sk[1], p.sk[2], p.sv[0], p.sv[1], p.sv[2]);
  args_in_sgprs(p.so[0], p.so[1], p.so[2], p.ssb, p.ssh, p.sbb, p.sbh, p.sbn, p.total_rows);
  args_in_sgprs(p.grid_waves, p.nq_mul, p.nq_shift, p.h_mul, p.h_shift);
  const int lane = threadIdx.x & (kWave - 1);
  const int32_t wave_id =
      static_cast<int32_t>(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int32_t total_rows = static_cast<int32_t>(p.total_rows);
  // No barriers below: early exit is safe.
  if (wave_id * kRows >= total_rows) return;

  const int32_t n_waves = p.grid_waves;
  const int32_t n_k = static_cast<int32_t>(p.Nk);
  const int chunk = lane % kChunks;
  const int group = lane / kChunks;
  const uint32_t chunk_bytes = chunk * 16u;
  const uint32_t k_row_bytes = static_cast<uint32_t>(p.sk[2]) * sizeof(T);
  const uint32_t v_row_bytes = static_cast<uint32_t>(p.sv[2]) * sizeof(T);
  const bool has_bias = p.bias != nullptr;
  const int32_t bias_esize = p.bias_dtype == VECTRA_F32 ? 4 : 2;

  if (n_k == 0) {  // softmax over no keys contributes nothing (eager gives 0)
    for (int32_t row = wave_id; row < total_rows; row += n_waves) {
      const RowCoords c = row_coords(row, p);
      float zero[kVec];
#pragma unroll
      for (int e = 0; e < kVec; ++e) zero[e] = 0.f;
      if (group == 0)
        store_chunk<OutT, kVec>(static_cast<OutT*>(p.out) + c.b * p.so[0] + c.h * p.so[1] +
                                    c.i * p.so[2] + chunk * kVec,
                                zero);
    }
    return;
  }

  // Per-lane byte offsets of the keys inside a (b, h) plane.  They are the
  // same for every row, so they are computed once: issuing the next row's
  // loads then only changes wave-uniform base addresses.
  struct Offsets {
    uint32_t k[kPasses], v[kPasses], bias[kPasses];
  };
  Offsets o;
#pragma unroll
  for (int s = 0; s < kPasses; ++s) {
    const int32_t j = s * kRowsPerPass + group;
    const uint32_t key = static_cast<uint32_t>(j < n_k - 1 ? j : n_k - 1);
    o.k[s] = key * k_row_bytes + chunk_bytes;
    o.v[s] = key * v_row_bytes + chunk_bytes;
    o.bias[s] = key * static_cast<uint32_t>(p.sbn);
  }

  // Issues every load of a row into `slot`.
  auto issue = [&](Slot& slot, int32_t row) {
    const RowCoords c = row_coords(row, p);
    const char* kp = reinterpret_cast<const char*>(p.k) + (c.b * p.sk[0] + c.h * p.sk[1]) * sizeof(T);
    const char* vp = reinterpret_cast<const char*>(p.v) + (c.b * p.sv[0] + c.h * p.sv[1]) * sizeof(T);
    // Issue order is use order: vector loads complete in order, so q, the
    // coefficient and the biases go first and K before V; the scores are
    // then computed while V is still arriving, and only the value product
    // waits for the last bytes.
    const char* qp = reinterpret_cast<const char*>(p.q) +
                     (c.b * p.sq[0] + c.h * p.sq[1] + c.i * p.sq[2]) * sizeof(T);
    slot.q = load16(qp + chunk_bytes);
    slot.scale = load_raw_scalar(p.scale, c.b * p.ssb + c.h * p.ssh, p.scale_dtype);
    if (has_bias) {
      const char* bp = reinterpret_cast<const char*>(p.bias) +
                       (c.b * p.sbb + c.h * p.sbh) * bias_esize;
      slot.bias_misalign = base_misalign(bp);
#pragma unroll
      for (int s = 0; s < kPasses; ++s)
        slot.bias[s] = load_raw_scalar32(bp, slot.bias_misalign, o.bias[s], p.bias_dtype).word;
    }
#pragma unroll
    for (int s = 0; s < kPasses; ++s) slot.k[s] = load16_stream(kp + o.k[s]);
#pragma unroll
    for (int s = 0; s < kPasses; ++s) slot.v[s] = load16_stream(vp + o.v[s]);
    // Nothing that waits for a load may be scheduled among them (a wait for
    // q or a bias there would hold back the V loads by a memory latency).
    __builtin_amdgcn_sched_barrier(0);
  };

  // Reduces the row held in `slot`.
  auto consume = [&](const Slot& slot, int32_t row) {
    const uint4 q_raw = slot.q;
    const float q_norm = reduce_low<kChunks>(dot_chunk<T>(q_raw, q_raw, 0.f), OpSum());
    const float neg_scale = -decode_raw_scalar(slot.scale, p.scale_dtype);
    float acc[kVec];
#pragma unroll
    for (int e = 0; e < kVec; ++e) acc[e] = 0.f;
    float logit[kPasses];
    bool live[kPasses];
    float row_max = -INFINITY;
#pragma unroll
    for (int s = 0; s < kPasses; ++s) {
      const int32_t j = s * kRowsPerPass + group;
      live[s] = j < n_k;
      const float dot = reduce_low<kChunks>(dot_chunk<T>(q_raw, slot.k[s], 0.f), OpSum());
      const float k_norm = reduce_low<kChunks>(dot_chunk<T>(slot.k[s], slot.k[s], 0.f), OpSum());
      const float dist = clamp_distance((q_norm + k_norm) - 2.f * dot);
      float x = neg_scale * dist;
      if (has_bias) {
        // Position of a 2-byte bias inside its word, from the key index
        // (the same arithmetic as the load).
        const uint32_t key = static_cast<uint32_t>(j < n_k - 1 ? j : n_k - 1);
        const uint32_t bytes = key * static_cast<uint32_t>(p.sbn) * bias_esize + slot.bias_misalign;
        x += decode_raw_scalar(RawScalar{slot.bias[s], (bytes & 2u) * 8u}, p.bias_dtype);
      }
      x = live[s] ? x : -INFINITY;
      logit[s] = x;
      row_max = fmaxf(row_max, x);
    }
    row_max = reduce_high<kChunks>(row_max, OpMax());
    const float safe_max = row_max == -INFINITY ? 0.f : row_max;
    float row_sum = 0.f;
    // Rows past Nk do not exist: their (clamped) values must not reach the
    // sum even as 0 * inf, so a tile with such rows zeroes them.
    const bool ragged = kWave > n_k;
#pragma unroll
    for (int s = 0; s < kPasses; ++s) {
      const float w = __builtin_amdgcn_exp2f((logit[s] - safe_max) * kLog2e);
      row_sum += w;
      uint4 vr = slot.v[s];
      if (ragged && !live[s]) vr = make_uint4(0, 0, 0, 0);
      float vf[kVec];
      unpack<T>(vr, vf);
#pragma unroll
      for (int e = 0; e < kVec; ++e) acc[e] = fmaf(w, vf[e], acc[e]);
    }
    // Each weight is replicated over the kChunks lanes of its key row; sum
    // over row groups only.
    row_sum = reduce_high<kChunks>(row_sum, OpSum());
    // Sum the accumulators over row groups; lane `lane` ends with
    // kVec / 4 finished values of its chunk, starting at element `first_e`.
    constexpr int kOut = kVec / 4;
    float res[kOut];
    int first_e;
    reduce_rows_butterfly<kChunks, kVec>(acc, res, first_e);
    // A row whose keys are all masked has row_sum 0: 0 * inf = NaN, as eager.
    const float inv = __builtin_amdgcn_rcpf(row_sum);
#pragma unroll
    for (int e = 0; e < kOut; ++e) res[e] *= inv;
    // Row groups below lane bit 16 hold copies; one of them stores.
    if ((lane & (16 - kChunks)) == 0) {
      const RowCoords c = row_coords(row, p);
      store_small<OutT, kOut>(static_cast<OutT*>(p.out) + c.b * p.so[0] + c.h * p.so[1] +
                                  c.i * p.so[2] + chunk * kVec + first_e,
                              res);
    }
  };

  Slot slots[2];
  auto row_at = [&](int r) {
    const int32_t row = wave_id * kRows + r;
    return row < total_rows ? row : total_rows - 1;
  };
  issue(slots[0], row_at(0));
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    if (r + 1 < kRows) issue(slots[(r + 1) & 1], row_at(r + 1));
    consume(slots[r & 1], row_at(r));
  }
}

// ------------------------------------------------------------------------
// Split kernel: few query rows over key axes of more than one 64-key tile.
//
// W waves (a power of two up to 16) own one query row and take its key tiles
// in turn, so a call with few rows still has W waves per row streaming.  A
// tile is kSplitPasses passes of the stream layout: lane l holds chunk
// l % kChunks of key row l / kChunks of each pass (one coalesced 1 KiB wave
// load), V in the same layout.  Each lane group of kChunks lanes keeps a
// softmax of its own over the keys it sees (maximum, sum, value
// accumulators), so the loop reduces nothing across groups: one merge over
// the wave's groups and one over the row's waves (through LDS) end the row.
//
// Bound: HBM (K and V once each).  Two passes per tile and one tile in
// flight per wave keep 58 registers, eight waves per SIMD, whose loads cover
// each other's latency; a second tile in flight (87 registers, five waves)
// and four passes (85) were no faster, and eight passes spilled.  Measured,
// bf16, 64 subjects x 8 heads x 1000 keys of 64 dims: 22.4 us, 5.9 TB/s (a
// plain read of the bytes: 20.3; 634 us before, on the generic kernel); 1024
// x 8 x 128 keys of 32 dims: 22.2 us (23.2 before, as a loop of the one-tile
// kernel), x 65 keys 13.5 (20.2).
// ------------------------------------------------------------------------

constexpr int kSplitPasses = 2;
constexpr int kSplitMaxWaves = 16;

template <typename T, typename OutT, int kChunks>
__global__ __launch_bounds__(kSplitMaxWaves * kWave) void rbf_split_kernel(Problem p) {
  constexpr int kVec = Vec<T>::kN;
  constexpr int kDim = kChunks * kVec;
  constexpr int kGroups = kWave / kChunks;      // key rows per pass
  constexpr int kKeys = kSplitPasses * kGroups;  // key rows per tile
  __shared__ float part_acc[kSplitMaxWaves][kDim];
  __shared__ float part_max[kSplitMaxWaves], part_sum[kSplitMaxWaves];

  args_in_sgprs(p.q, p.k, p.v, p.out, p.scale, p.bias, p.scale_dtype, p.bias_dtype, p.H, p.Nq, p.Nk);
  args_in_sgprs(p.sq[0], p.sq[1], p.sq[2], p.sk[0], p.sk[1], p.sk[2], p.sv[0], p.sv[1], p.sv[2]);
  args_in_sgprs(p.so[0], p.so[1], p.so[2], p.ssb, p.ssh, p.sbb, p.sbh, p.sbn, p.total_rows);
  args_in_sgprs(p.grid_waves, p.first_row, p.nq_mul, p.nq_shift, p.h_mul, p.h_shift);
  const int lane = threadIdx.x & (kWave - 1);
  const int slot_wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int log_waves = p.grid_waves;
  const int n_waves = 1 << log_waves;          // per row
  const int wave = slot_wave & (n_waves - 1);  // of the row
  // Workgroups are dispatched round-robin over the 8 XCDs: contiguous rows
  // (the queries of a plane) run on one XCD and share its L2.
  const int32_t total_rows = static_cast<int32_t>(p.total_rows);
  const int32_t per_xcd = static_cast<int32_t>(gridDim.x >> 3);
  const int32_t item = static_cast<int32_t>(blockIdx.x & 7) * per_xcd + static_cast<int32_t>(blockIdx.x >> 3);
  const int32_t rows_here = static_cast<int>(blockDim.x) >> (6 + log_waves);
  const int32_t first_row = p.first_row + item * rows_here;
  if (first_row >= total_rows) return;  // the whole workgroup, before any barrier
  // Waves past the last row repeat it (same bytes stored).
  const int32_t row_id = first_row + (slot_wave >> log_waves);
  const int32_t row = row_id < total_rows ? row_id : total_rows - 1;
  const RowCoords c = row_coords(row, p);

  const int32_t n_k = static_cast<int32_t>(p.Nk);
  const int chunk = lane % kChunks;
  const int group = lane / kChunks;
  const uint32_t chunk_bytes = chunk * 16u;
  const uint32_t k_row_bytes = static_cast<uint32_t>(p.sk[2]) * sizeof(T);
  const uint32_t v_row_bytes = static_cast<uint32_t>(p.sv[2]) * sizeof(T);
  const bool has_bias = p.bias != nullptr;
  const int32_t bias_esize = p.bias_dtype == VECTRA_F32 ? 4 : 2;
  const char* kp = reinterpret_cast<const char*>(p.k) + (c.b * p.sk[0] + c.h * p.sk[1]) * sizeof(T);
  const char* vp = reinterpret_cast<const char*>(p.v) + (c.b * p.sv[0] + c.h * p.sv[1]) * sizeof(T);
  const char* bp = reinterpret_cast<const char*>(p.bias) + (c.b * p.sbb + c.h * p.sbh) * bias_esize;
  const uint32_t bias_misalign = base_misalign(bp);
  const int32_t tiles = (n_k + kKeys - 1) / kKeys;

  struct Slot {
    uint4 k[kSplitPasses], v[kSplitPasses];
    uint32_t bias[kSplitPasses];
  };
  // Issues every load of a tile; rows past Nk read row Nk - 1 and are masked.
  auto issue = [&](Slot& slot, int32_t tile) {
    uint32_t key[kSplitPasses];
#pragma unroll
    for (int s = 0; s < kSplitPasses; ++s) {
      const int32_t j = tile * kKeys + s * kGroups + group;
      key[s] = static_cast<uint32_t>(j < n_k - 1 ? j : n_k - 1);
    }
    if (has_bias) {
#pragma unroll
      for (int s = 0; s < kSplitPasses; ++s)
        slot.bias[s] =
            load_raw_scalar32(bp, bias_misalign, key[s] * static_cast<uint32_t>(p.sbn), p.bias_dtype).word;
    }
#pragma unroll
    for (int s = 0; s < kSplitPasses; ++s) slot.k[s] = load16_stream(kp + (key[s] * k_row_bytes + chunk_bytes));
#pragma unroll
    for (int s = 0; s < kSplitPasses; ++s) slot.v[s] = load16_stream(vp + (key[s] * v_row_bytes + chunk_bytes));
    __builtin_amdgcn_sched_barrier(0);
  };

  Slot a;
  const uint4 q_raw =
      load16(reinterpret_cast<const char*>(p.q) + (c.b * p.sq[0] + c.h * p.sq[1] + c.i * p.sq[2]) * sizeof(T) +
             chunk_bytes);
  const RawScalar scale_raw = load_raw_scalar(p.scale, c.b * p.ssb + c.h * p.ssh, p.scale_dtype);
  // The row's tile order is rotated by a hash of its plane: where planes are a
  // power of two apart, waves that walk them in step from the first tile
  // would all be on the same few HBM channels (8192 rows of 256 keys: 41.9 us
  // rotated, 51.2 in order).  The rows of a plane walk it in one order and
  // meet its tiles in the caches (rotated row by row, 2000 planes of 3 rows x
  // 500 keys took 51.2 us in fp32 at 16 dims, now 38.3; of 15 rows x 300 at 64
  // dims 529 and 323).
  const uint32_t plane = static_cast<uint32_t>(c.b * p.H + c.h);
  const int32_t rotation = static_cast<int32_t>(__umulhi(plane * 0x9e3779b1u, tiles));
  auto rotated = [&](int32_t t) { return t + rotation < tiles ? t + rotation : t + rotation - tiles; };
  int32_t step = wave, tile = rotated(step);
  if (step < tiles) issue(a, tile);
  const float q_norm = reduce_low<kChunks>(dot_chunk<T>(q_raw, q_raw, 0.f), OpSum());
  const float neg_scale = -decode_raw_scalar(scale_raw, p.scale_dtype);

  // The lane group's softmax state.  Logits are subtracted before they are
  // scaled to log2 units: a bias of the type's lowest value would overflow
  // the other way round.
  float run_max = -INFINITY, run_sum = 0.f;
  float acc[kVec];
#pragma unroll
  for (int e = 0; e < kVec; ++e) acc[e] = 0.f;

  auto consume = [&](const Slot& slot, int32_t t) {
    const bool ragged = (t + 1) * kKeys > n_k;
    float logit[kSplitPasses];
    float tile_max = -INFINITY;
#pragma unroll
    for (int s = 0; s < kSplitPasses; ++s) {
      const int32_t j = t * kKeys + s * kGroups + group;
      const float dot = dot_chunk<T>(q_raw, slot.k[s], 0.f);
      const float k_norm = dot_chunk<T>(slot.k[s], slot.k[s], 0.f);
      const float part = reduce_low<kChunks>(fmaf(-2.f, dot, k_norm), OpSum());
      const float dist = clamp_distance(q_norm + part);
      float x = neg_scale * dist;
      if (has_bias) {
        const uint32_t key = static_cast<uint32_t>(j < n_k - 1 ? j : n_k - 1);
        const uint32_t bytes = key * static_cast<uint32_t>(p.sbn) * bias_esize + bias_misalign;
        x += decode_raw_scalar(RawScalar{slot.bias[s], (bytes & 2u) * 8u}, p.bias_dtype);
      }
      x = j < n_k ? x : -INFINITY;
      logit[s] = x;
      tile_max = fmaxf(tile_max, x);
    }
    const float new_max = fmaxf(run_max, tile_max);
    const float safe_max = new_max == -INFINITY ? 0.f : new_max;
    const float alpha = __builtin_amdgcn_exp2f((run_max - safe_max) * kLog2e);
    run_sum *= alpha;
#pragma unroll
    for (int e = 0; e < kVec; ++e) acc[e] *= alpha;
#pragma unroll
    for (int s = 0; s < kSplitPasses; ++s) {
      const float w = __builtin_amdgcn_exp2f((logit[s] - safe_max) * kLog2e);
      run_sum += w;
      uint4 vr = slot.v[s];
      // Rows past Nk do not exist: their (clamped) values must not reach the
      // sum even as 0 * inf.
      if (ragged && t * kKeys + s * kGroups + group >= n_k) vr = make_uint4(0, 0, 0, 0);
      float vf[kVec];
      unpack<T>(vr, vf);
#pragma unroll
      for (int e = 0; e < kVec; ++e) acc[e] = fmaf(w, vf[e], acc[e]);
    }
    run_max = new_max;
  };

  while (step < tiles) {
    consume(a, tile);
    step += n_waves;
    tile = rotated(step);
    if (step < tiles) issue(a, tile);
  }

  // Merge the wave's lane groups: a group without a live key weighs 0.
  const float wave_max = reduce_high<kChunks>(run_max, OpMax());
  const float mine = __builtin_amdgcn_exp2f((run_max - (wave_max == -INFINITY ? 0.f : wave_max)) * kLog2e);
  const float wave_sum = reduce_high<kChunks>(run_sum * mine, OpSum());
#pragma unroll
  for (int e = 0; e < kVec; ++e) acc[e] *= mine;
  constexpr int kOut = kChunks == 32 ? kVec / 2 : kVec / 4;
  float res[kOut];
  int first_e;
  if constexpr (kChunks == 32) {  // two key rows per pass: lane bit 32 only
#pragma unroll
    for (int i = 0; i < kOut; ++i) {
      const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[i]), __float_as_uint(acc[i + kOut]), false,
                                                      false);
      res[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    first_e = (lane & 32) ? kOut : 0;
  } else {
    reduce_rows_butterfly<kChunks, kVec>(acc, res, first_e);
  }
  OutT* out = static_cast<OutT*>(p.out) + c.b * p.so[0] + c.h * p.so[1] + c.i * p.so[2];
  // Row groups below lane bit 16 hold copies; one of them writes.
  const bool writer = kChunks >= 16 || (lane & (16 - kChunks)) == 0;
  if (n_waves == 1) {
    // A quotient, as the generic kernel has it (the reciprocal's rounding adds
    // one more).  A row whose keys are all masked is 0 / 0 = NaN, as eager.
#pragma unroll
    for (int i = 0; i < kOut; ++i) res[i] /= wave_sum;
    if (writer) store_small<OutT, kOut>(out + chunk * kVec + first_e, res);
    return;
  }
  if (writer) {
#pragma unroll
    for (int i = 0; i < kOut; ++i) part_acc[slot_wave][chunk * kVec + first_e + i] = res[i];
  }
  if (lane == 0) {
    part_max[slot_wave] = wave_max;
    part_sum[slot_wave] = wave_sum;
  }
  __syncthreads();
  const int w0 = slot_wave & -n_waves;  // the row's first wave
  const int d = static_cast<int>(threadIdx.x) - w0 * kWave;
  if (d < kDim) {
    float m = -INFINITY;
    for (int w = 0; w < n_waves; ++w) m = fmaxf(m, part_max[w0 + w]);
    const float safe = m == -INFINITY ? 0.f : m;
    float sum = 0.f, value = 0.f;
    for (int w = 0; w < n_waves; ++w) {
      const float f = __builtin_amdgcn_exp2f((part_max[w0 + w] - safe) * kLog2e);
      sum = fmaf(f, part_sum[w0 + w], sum);
      value = fmaf(f, part_acc[w0 + w][d], value);
    }
    out[d] = from_float<OutT>(value / sum);
  }
}

// ------------------------------------------------------------------------
// Generic kernel: one wave per (b, h, query row) and per 256-wide slice of
// the value dimension (blockIdx.y).  Scores: lane = key within a 64-key
// tile.  Value product: lane = value column, weights broadcast with
// readlane.  Handles any strides (including zero), any D and Dv.  Waves
// loop over rows with a grid stride, so the grid stays within HIP's
// per-dimension thread limit however many rows there are.
// ------------------------------------------------------------------------
template <typename T, typename OutT>
__device__ void generic_row(const Problem& p, int64_t row_id, int lane);

template <typename T, typename OutT>
__global__ __launch_bounds__(256) void rbf_generic_kernel(Problem p) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t stride = static_cast<int64_t>(gridDim.x) * 4;
  // Wave-uniform loop (no barriers inside).
  for (int64_t row_id = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6); row_id < p.total_rows;
       row_id += stride)
    generic_row<T, OutT>(p, row_id, lane);
}

template <typename T, typename OutT>
__device__ void generic_row(const Problem& p, int64_t row_id, int lane) {
  constexpr int kCols = 4;  // value columns per lane: 4 * 64 = 256 per slice
  const int64_t i = row_id % p.Nq;
  const int64_t bh = row_id / p.Nq;
  const int64_t h = bh % p.H;
  const int64_t b = bh / p.H;
  const int64_t dv0 = static_cast<int64_t>(blockIdx.y) * (kCols * kWave);

  const T* q_row = static_cast<const T*>(p.q) + b * p.sq[0] + h * p.sq[1] + i * p.sq[2];
  const T* k_plane = static_cast<const T*>(p.k) + b * p.sk[0] + h * p.sk[1];
  const T* v_plane = static_cast<const T*>(p.v) + b * p.sv[0] + h * p.sv[1];

  float q_norm = 0.f;
  for (int64_t d = lane; d < p.D; d += kWave) {
    const float x = to_float<T>(q_row[d * p.sq[3]]);
    q_norm += x * x;
  }
  q_norm = reduce_wave(q_norm, OpSum());

  const float neg_scale = -load_any(p.scale, b * p.ssb + h * p.ssh, p.scale_dtype);
  const bool has_bias = p.bias != nullptr;
  const int64_t bias_base = b * p.sbb + h * p.sbh;

  float run_max = -INFINITY, run_sum = 0.f;
  float acc[kCols];
#pragma unroll
  for (int c = 0; c < kCols; ++c) acc[c] = 0.f;

  for (int64_t j0 = 0; j0 < p.Nk; j0 += kWave) {
    const int64_t j = j0 + lane;
    const bool live = j < p.Nk;
    float logit = -INFINITY;
    if (live) {
      const T* k_row = k_plane + j * p.sk[2];
      float dot = 0.f, k_norm = 0.f;
      for (int64_t d = 0; d < p.D; ++d) {
        const float qd = to_float<T>(q_row[d * p.sq[3]]);
        const float kd = to_float<T>(k_row[d * p.sk[3]]);
        dot += qd * kd;
        k_norm += kd * kd;
      }
      const float dist = clamp_distance((q_norm + k_norm) - 2.f * dot);
      logit = neg_scale * dist;
      if (has_bias) logit += load_any(p.bias, bias_base + j * p.sbn, p.bias_dtype);
    }
    const float new_max = fmaxf(run_max, reduce_wave(logit, OpMax()));
    const float safe_max = new_max == -INFINITY ? 0.f : new_max;
    const float alpha = __builtin_amdgcn_exp2f((run_max - safe_max) * kLog2e);
    const float w = __builtin_amdgcn_exp2f((logit - safe_max) * kLog2e);
    run_sum = run_sum * alpha + reduce_wave(w, OpSum());
#pragma unroll
    for (int c = 0; c < kCols; ++c) acc[c] *= alpha;
    const int n_live = static_cast<int>(p.Nk - j0 < kWave ? p.Nk - j0 : kWave);
    for (int jj = 0; jj < n_live; ++jj) {
      const float wj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), jj));
      const T* v_row = v_plane + (j0 + jj) * p.sv[2];
#pragma unroll
      for (int c = 0; c < kCols; ++c) {
        const int64_t d = dv0 + c * kWave + lane;
        if (d < p.Dv) acc[c] += wj * to_float<T>(v_row[d * p.sv[3]]);
      }
    }
    run_max = new_max;
  }

  OutT* o = static_cast<OutT*>(p.out) + b * p.so[0] + h * p.so[1] + i * p.so[2];
#pragma unroll
  for (int c = 0; c < kCols; ++c) {
    const int64_t d = dv0 + c * kWave + lane;
    if (d < p.Dv) o[d * p.so[3]] = from_float<OutT>(p.Nk > 0 ? acc[c] / run_sum : 0.f);
  }
}

// Row norms |x_j|^2 in fp32 (norm_precompute.py:34-64): one thread per row.
struct NormArgs {
  const void* x;
  float* out;
  int64_t B, H, N, D;
  int64_t s[4];
};

// Threads loop over rows with a grid stride.
template <typename T>
__global__ __launch_bounds__(256) void squared_norms_kernel(NormArgs a) {
  const int64_t total = a.B * a.H * a.N;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t r = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; r < total; r += stride) {
    const int64_t n = r % a.N;
    const int64_t bh = r / a.N;
    const T* row = static_cast<const T*>(a.x) + (bh / a.H) * a.s[0] + (bh % a.H) * a.s[1] + n * a.s[2];
    float acc = 0.f;
    for (int64_t d = 0; d < a.D; ++d) {
      const float t = to_float<T>(row[d * a.s[3]]);
      acc += t * t;
    }
    a.out[r] = acc;
  }
}

// ------------------------------------------------------------------------
// Launch helpers (host).
// ------------------------------------------------------------------------

static hipError_t launch(const void* fn, dim3 grid, dim3 block, Problem& p, hipStream_t s) {
  void* args[] = {&p};
  return hipLaunchKernel(fn, grid, block, args, 0, s);
}

template <typename T, typename OutT, int kChunks, int kRows>
static hipError_t launch_stream_k(Problem& p, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>((p.grid_waves + 3) / 4));
  return launch(reinterpret_cast<const void*>(&rbf_stream_kernel<T, OutT, kChunks, kRows>), grid,
                dim3(256), p, s);
}

// Waves per row: enough for 8 waves per CU over all rows (two per SIMD; from
// there on more waves per row only add merges: 2048 rows of 65-400 keys ran
// 0-50% slower with two to eight), at most one per key tile.  Measured with 1
// / 2 / 4 / 8 / 16 waves: 8 rows of 2048 keys 98.7 / 48.6 / 23.3 / 14.7 /
// 12.4 us, 512 rows of 1000 keys 54.5 / 31.2 / 22.3 / 22.4 / 22.6 us, 8192
// rows of 65 keys 13.5 / 14.0 / 17.3 / 29.5 us.
template <typename T, typename OutT, int kChunks>
static hipError_t launch_split(Problem& p, hipStream_t s) {
  constexpr int kKeys = kSplitPasses * (kWave / kChunks);
  const int64_t tiles = (p.Nk + kKeys - 1) / kKeys;
  const int64_t slots = static_cast<int64_t>(p.compute_units) * 8;
  int log_waves = 0;
  while ((1 << log_waves) < kSplitMaxWaves && (2 << log_waves) <= tiles && (p.total_rows << log_waves) < slots)
    ++log_waves;
  const int rows_here = log_waves < 2 ? 4 >> log_waves : 1;
  p.grid_waves = log_waves;
  // A grid holds fewer than 2^32 threads, so very many rows (of one wave
  // each) take several launches.
  constexpr int64_t kMaxRows = int64_t{1} << 25;
  for (int64_t row = 0; row < p.total_rows; row += kMaxRows) {
    const int64_t rows = p.total_rows - row < kMaxRows ? p.total_rows - row : kMaxRows;
    const int64_t items = (rows + rows_here - 1) / rows_here;
    p.first_row = static_cast<int32_t>(row);
    const dim3 grid(static_cast<unsigned>((items + 7) / 8 * 8));
    const hipError_t err = launch(reinterpret_cast<const void*>(&rbf_split_kernel<T, OutT, kChunks>), grid,
                                  dim3(static_cast<unsigned>(rows_here << (log_waves + 6))), p, s);
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

// Rows per wave for one-tile rows: about `budget` waves, at most kMaxRows
// rows each (the register footprint of two slots bounds it for wide heads).
template <typename T, typename OutT, int kChunks, int kMaxRows>
static hipError_t launch_stream_c(Problem& p, hipStream_t s) {
  if (p.Nk > kWave) return launch_split<T, OutT, kChunks>(p, s);
  const int64_t budget = p.grid_waves;
  const int64_t rows = p.total_rows;
  int rows_per_wave = rows > 2 * budget ? 4 : (rows > budget ? 2 : 1);
  if (rows_per_wave > kMaxRows) rows_per_wave = kMaxRows;
  p.grid_waves = static_cast<int32_t>((rows + rows_per_wave - 1) / rows_per_wave);
  if (kMaxRows >= 4 && rows_per_wave == 4) return launch_stream_k<T, OutT, kChunks, (kMaxRows >= 4 ? 4 : 1)>(p, s);
  if (kMaxRows >= 2 && rows_per_wave == 2) return launch_stream_k<T, OutT, kChunks, (kMaxRows >= 2 ? 2 : 1)>(p, s);
  return launch_stream_k<T, OutT, kChunks, 1>(p, s);
}

// p.grid_waves holds the persistent wave budget on entry; it is replaced by
// the number of waves launched.
template <typename T, typename OutT>
static hipError_t launch_stream_t(Problem& p, int chunks, hipStream_t s) {
  switch (chunks) {
    case 2: return launch_stream_c<T, OutT, 2, 4>(p, s);
    case 4: return launch_stream_c<T, OutT, 4, 4>(p, s);
    case 8: return launch_stream_c<T, OutT, 8, 4>(p, s);
    case 16: return launch_stream_c<T, OutT, 16, 1>(p, s);
    case 32:  // 128-dim fp32 heads: any key count (a 64-key tile would spill)
      if constexpr (sizeof(T) == 4) return launch_split<T, OutT, 32>(p, s);
      return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
}

// Workgroups of the grid-stride kernels: at most this many (of 256 threads).
constexpr int64_t kMaxGridStrideBlocks = int64_t{1} << 20;

template <typename T, typename OutT>
static hipError_t launch_generic_t(Problem& p, hipStream_t s) {
  const int64_t blocks = (p.total_rows + 3) / 4;
  const int64_t slices = (p.Dv + 255) / 256;
  if (slices > kMaxGenericSlices) return hipErrorInvalidValue;  // the host rejects these first
  const dim3 grid(static_cast<unsigned>(blocks < kMaxGridStrideBlocks ? blocks : kMaxGridStrideBlocks),
                  static_cast<unsigned>(slices));
  return launch(reinterpret_cast<const void*>(&rbf_generic_kernel<T, OutT>), grid, dim3(256), p, s);
}

// Dispatch on (input dtype, output dtype).
template <template <typename, typename> class F, typename... A>
static hipError_t by_dtype(int in_dt, int out_dt, A&&... a) {
#define VECTRA_CASE(IN_ENUM, IN_T)                                             \
  if (in_dt == IN_ENUM) {                                                      \
    if (out_dt == VECTRA_F32) return F<IN_T, float>::run(a...);                \
    if (out_dt == VECTRA_F16) return F<IN_T, _Float16>::run(a...);             \
    if (out_dt == VECTRA_BF16) return F<IN_T, __bf16>::run(a...);              \
  }
  VECTRA_CASE(VECTRA_F32, float)
  VECTRA_CASE(VECTRA_F16, _Float16)
  VECTRA_CASE(VECTRA_BF16, __bf16)
#undef VECTRA_CASE
  return hipErrorInvalidValue;
}

template <typename T, typename OutT>
struct GenericLauncher {
  static hipError_t run(Problem& p, hipStream_t s) { return launch_generic_t<T, OutT>(p, s); }
};

hipError_t launch_stream(Problem& p, int in_dt, int out_dt, int chunks, hipStream_t s) {
  // Output in the input dtype (the operator) or fp32 (parity harnesses).
  switch (in_dt) {
    case VECTRA_BF16:
      return out_dt == VECTRA_F32 ? launch_stream_t<__bf16, float>(p, chunks, s)
                                  : launch_stream_t<__bf16, __bf16>(p, chunks, s);
    case VECTRA_F16:
      return out_dt == VECTRA_F32 ? launch_stream_t<_Float16, float>(p, chunks, s)
                                  : launch_stream_t<_Float16, _Float16>(p, chunks, s);
    default:
      return launch_stream_t<float, float>(p, chunks, s);
  }
}

hipError_t launch_generic(Problem& p, int in_dt, int out_dt, hipStream_t s) {
  return by_dtype<GenericLauncher>(in_dt, out_dt, p, s);
}

hipError_t launch_squared_norms(const void* x, int dtype, int64_t B, int64_t H, int64_t N,
                                int64_t D, const int64_t* st, float* out, hipStream_t s) {
  NormArgs a{x, out, B, H, N, D, {st[0], st[1], st[2], st[3]}};
  const int64_t blocks = (B * H * N + 255) / 256;
  const dim3 grid(static_cast<unsigned>(blocks < kMaxGridStrideBlocks ? blocks : kMaxGridStrideBlocks));
  void* args[] = {&a};
  const void* fn = nullptr;
  switch (dtype) {
    case VECTRA_F32: fn = reinterpret_cast<const void*>(&squared_norms_kernel<float>); break;
    case VECTRA_F16: fn = reinterpret_cast<const void*>(&squared_norms_kernel<_Float16>); break;
    case VECTRA_BF16: fn = reinterpret_cast<const void*>(&squared_norms_kernel<__bf16>); break;
    default: return hipErrorInvalidValue;
  }
  return hipLaunchKernel(fn, grid, dim3(256), args, 0, s);
}

}  // namespace vectra
