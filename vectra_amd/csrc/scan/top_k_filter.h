// Filtered k-nearest search for several queries over many candidates: the
// matrix cores bound every distance, and only candidates whose bound lets
// them be among the k nearest get the reference's own arithmetic.  Included
// by scan.hip (which holds the shared types and the C ABI).
//
// With q^ and r^ the query and row rounded to bf16 (relative error at most
// 2^-8 an element), |q|, |r| the norms and u the rounding of every 32-bit sum
// involved, the reference's distance d lies in
//
//   |q|^2 + |r|^2 - 2 q^.r^  -+  (c1 |q||r| + c2 (|q|^2 + |r|^2)),
//   c1 = 2 (2^-7 + 2^-16 + dim 2^-22),   c2 = (dim + 36) 2^-22
//
// (Cauchy-Schwarz on the element errors; c2 covers the sums of the norms, of
// the matrix product and of the reference's own order, with room).  Queries
// that lie together, far from the origin for their spread, are taken from a
// centre, as are the rows: a shift changes no distance, but the norms above it.
// The rounding of q - c and r - c moves the distance of the pair by at most
// 2^-22 (|q - c|^2 + |r - c|^2), which is in c2.  Four launches:
//
//  1. top_k_bound_kernel<..., true>: over a sample of the candidates, the
//     smallest upper end of every group of candidates;
//  2. top_k_limit_kernel: per query, a value at or just above the k-th
//     smallest of the groups' minima.  k different candidates lie at or below
//     it, so it is at or above the k-th smallest distance;
//  3. top_k_bound_kernel<..., false>: every candidate; those whose lower end is
//     not above the limit are computed exactly, and the ones at or below
//     the limit go into the workgroup's short list of the query;
//  4. top_k_merge_kernel: per query, the k smallest keys of the lists.  A list
//     that runs over (ties, loose bounds) keeps its smallest keys, so what it
//     left out is no nearer than the last of them: its workgroup's candidates
//     are scanned again only where that key is below the k-th found.
//
// The results are those of scan_top_k_kernel, bit for bit: every returned
// distance is the reference's arithmetic, and a candidate is dropped only
// where its distance is provably above the k-th.  A NaN or an overflow in a
// row or a query makes its bounds NaN, which pass the filter.
//
// Bound: HBM (the rows once, plus the sample) for few queries, the exact
// computation of the surviving pairs and four launches beyond.  An exact
// distance costs 3 vector operations per dimension and its fold; the bound
// costs a matrix instruction per 16 queries, 16 rows and 32 dimensions.
// Measured, 64 queries over 200,000 rows of 128, k = 100: 57.6 us (launches
// 11, 6.5, 30 and 9 us; the rows alone take 16 us at a plain read's rate)
// against 1,889 us with one workgroup per query; 1,024 queries over 12,500
// rows 87 against 307 us; 8 over 500,000 rows of 64, k = 50, 49 against 643.
#pragma once

constexpr int kFilterQueries = 64;      // queries of a workgroup: four 16-query tiles
constexpr int kFilterWaves = 4;
constexpr int kFilterThreads = kFilterWaves * kWaveLanes;
constexpr int kFilterTile = 16;         // candidates of a wave's step
constexpr int kFilterCap = 16;          // keys of a (workgroup, query) list
// Survivors a wave collects: it computes them when more than kFilterDrain
// wait, and a step may add every pair of its tile.
constexpr int kFilterDrain = 64;
constexpr int kFilterQueue = kFilterDrain + kFilterTile * kFilterQueries;
constexpr int kFilterMaxGroups = 4096;  // groups of the sample
constexpr int kFilterMaxDim = 256;      // query fragments: 32 KiB of LDS
constexpr int kFilterMaxK = 512;
constexpr int kFilterMaxWorkgroups = 1024;  // of the filter launch, per query block

struct TopKFilter {
  TopK t;
  float* minima;     // [query blocks][groups][64]
  float* limit;      // [query blocks][64]
  uint32_t* centred;  // [query blocks]: whether the block's queries and the rows are taken from a centre
  float* centres;     // [query blocks][kFilterMaxDim]
  uint32_t* counts;  // [query blocks][workgroups][64]; above kFilterCap: ran over
  uint64_t* lists;   // [query blocks][workgroups][64][kFilterCap]; of one that ran over, its smallest keys
  int64_t num_queries;
  int32_t tiles;         // 16-candidate tiles of the call
  int32_t workgroups;    // of the filter launch, per query block
  int32_t sample_waves;  // waves of the sample launch, per query block
  int32_t sample_tiles;  // tiles of each of them
  int32_t sample_step;   // one tile in this many is in the sample
  int32_t group_cols;    // groups per sample wave: 1 or 4
};

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T, typename Op>
__device__ __forceinline__ T wave_fold(T x, Op op) {
#pragma unroll
  for (int s = 1; s < kWaveLanes; s <<= 1) x = op(x, __shfl_xor(x, s));
  return x;
}

template <typename C>
__device__ __forceinline__ float dpp_min(float x, C) {
  const float y = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), C::value, 0xf, 0xf, false));
  return fminf(x, y);
}

template <typename C>
__device__ __forceinline__ float dpp_add(float x, C) {
  return x + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), C::value, 0xf, 0xf, false));
}

// Sums over the four 16-lane rows of a wave, in every lane.
__device__ __forceinline__ float fold_rows(float x) {
  auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(s[0]) + __uint_as_float(s[1]);
  s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

// A key in LDS that other waves change meanwhile.
__device__ __forceinline__ uint64_t shared_key(const uint64_t* key) {
  return __hip_atomic_load(key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Puts `key` into a full list of kFilterCap keys in LDS in place of its largest,
// for each 16-lane group with `left` (the lanes of a group hold a slot each);
// other waves insert at the same time.  A slot that still reads as empty
// (kNoKey) has been given to a wave that is about to write it: look again.
// Written slots only ever fall, so a key found no smaller than every slot, or
// replaced as the largest, is no smaller than any key the list ends with;
// `worst` is such a bound, above which no look at the slots is needed.
//
// The whole wave runs this and each of its rounds: conditions are computed
// without branches (&, unconditional loads), as lanes that the compiler takes
// around a load could otherwise reach a ballot apart from the rest.
__device__ __forceinline__ void list_replace(uint64_t* list, uint64_t* worst, uint64_t key, bool left, int lane,
                                             int wave_lane) {
  static_assert(kFilterCap == kLanes, "a lane per slot");
  typedef unsigned long long Word;
  const int group_bit = wave_lane & ~(kLanes - 1);
  // (`worst` is told of lists that have run over only: what it keeps out is not counted.)
  const bool tells = left & (lane == 0);
  do {
    const uint64_t slot = shared_key(list + lane);
    uint64_t largest = slot;
    auto fold = [&](auto s_tag) {
      const uint64_t other = lane_xor<decltype(s_tag)::value>(largest, wave_lane);
      largest = other > largest ? other : largest;
    };
    fold(std::integral_constant<int, 1>{});
    fold(std::integral_constant<int, 2>{});
    fold(std::integral_constant<int, 4>{});
    fold(std::integral_constant<int, 8>{});
    const bool whole = largest != kNoKey;
    left = left & (key < largest);
    const bool placing = left & whole;
    // The first lane whose slot is the largest.
    const uint64_t holders = (__ballot(placing & (slot == largest)) >> group_bit) & 0xffffu;
    const bool mine = placing & (((holders >> lane) & 1) != 0) & ((holders & ((uint64_t{1} << lane) - 1)) == 0);
    bool put = false;
    if (mine) put = atomicCAS(reinterpret_cast<Word*>(list) + lane, static_cast<Word>(largest), static_cast<Word>(key)) == largest;
    if (tells & whole) atomicMin(reinterpret_cast<Word*>(worst), static_cast<Word>(largest));
    left = left & (((__ballot(put) >> group_bit) & 0xffffu) == 0);
  } while (__ballot(left) != 0);
}

// The exact distance of kN (query, row) pairs of this 16-lane group, in the
// row scan's order; lane 0 of the group holds the results.
template <int kN>
__device__ __forceinline__ void exact_distances(const float* const (&query)[kN], const float* const (&row)[kN],
                                                int dim, int lane, float (&sum)[kN]) {
  const int full = dim - dim % kLanes;
  const int tail = dim - full;
  float acc[kN];
#pragma unroll
  for (int n = 0; n < kN; ++n) acc[n] = 0.f;
  int i = 0;
  for (; i + 4 * kLanes <= full; i += 4 * kLanes) {
    float q[kN][4], r[kN][4];
#pragma unroll
    for (int n = 0; n < kN; ++n)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        r[n][u] = row[n][i + kLanes * u + lane];
        q[n][u] = query[n][i + kLanes * u + lane];
      }
#pragma unroll
    for (int n = 0; n < kN; ++n)
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[n] = acc[n] + term<VECTRA_SCAN_L2_SQUARED>(q[n][u], r[n][u]);
  }
  for (; i < full; i += kLanes) {
#pragma unroll
    for (int n = 0; n < kN; ++n)
      acc[n] = acc[n] + term<VECTRA_SCAN_L2_SQUARED>(query[n][i + lane], row[n][i + lane]);
  }
#pragma unroll
  for (int n = 0; n < kN; ++n) {
    sum[n] = reduce_lanes(acc[n]);
    if (tail > 0) {
      float t = 0.f;
      if (lane < tail) t = term<VECTRA_SCAN_L2_SQUARED>(query[n][full + lane], row[n][full + lane]);
      for (int e = 0; e < tail; ++e) sum[n] = sum[n] + __shfl(t, e, kLanes);
    }
  }
}

// kSample: launch 1, else launch 3.  kChunks: 32-dimension chunks of a row
// loaded together (a step: 16 candidates x 32 kChunks dimensions).  kTiles:
// 16-query tiles computed (1 where the call has no more than 16 queries).
// Requires dim % 4 == 0 and 16-byte-aligned rows; grid (workgroups, query
// blocks).
template <bool kIds, int kChunks, int kTiles, bool kSample>
__global__ __launch_bounds__(kFilterThreads, kSample ? 4 : 3) void top_k_bound_kernel(TopKFilter p) {
  // Query fragments, [16-query tile][chunk][lane]: the A operand of a product
  // as one 16-byte read per lane.
  extern __shared__ __align__(16) uint8_t dynamic_lds[];
  bf16x8* qfrag = reinterpret_cast<bf16x8*>(dynamic_lds);
  __shared__ float qnorm[kFilterQueries];
  __shared__ __align__(16) float qa[kFilterQueries], qc[kFilterQueries];
  __shared__ float qlimit[kFilterQueries];
  __shared__ uint32_t fill[kFilterQueries];
  __shared__ __align__(16) float centre[kFilterMaxDim];
  __shared__ uint64_t worst[kSample ? 1 : kFilterQueries];
  __shared__ uint64_t list[kSample ? 1 : kFilterQueries][kSample ? 1 : kFilterCap];
  __shared__ uint32_t queue[kSample ? 1 : kFilterWaves][kSample ? 1 : kFilterQueue];

  const int tid = static_cast<int>(threadIdx.x);
  const int lane = tid & (kWaveLanes - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWaveLanes);
  const int col = lane & 15;  // the candidate of a tile this lane holds
  const int grp = lane >> 4;  // ... its dimensions 8 grp .. + 7 of a chunk, and queries 4 grp .. + 3 of a product
  const int dim = p.t.dim;
  const int chunks = (dim + 31) / 32;
  const int slabs = (chunks + kChunks - 1) / kChunks;
  const int padded = slabs * kChunks;
  const int64_t q0 = static_cast<int64_t>(blockIdx.y) * kFilterQueries;
  const int nq = static_cast<int>(p.num_queries - q0 < kFilterQueries ? p.num_queries - q0 : kFilterQueries);

  // ---- The block's queries: bf16 fragments, norms, limits.  A thread takes
  // eight dimensions of a query, eight adjacent lanes 64 of them.
  const bool whole = p.t.query_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(p.t.queries) & 15) == 0;
  const int items = kTiles * 16 * padded * 4;
  bool centred = false;
  // Eight dimensions of a query: its fragment, and its norm's part.
  auto stage = [&](int q, int d8, float (&x)[8]) {
    if (centred) {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] -= centre[8 * d8 + e];
    }
    bf16x8 f;
    float n = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      f[e] = static_cast<__bf16>(x[e]);
      n = fmaf(x[e], x[e], n);
    }
    qfrag[((q / 16) * padded + d8 / 4) * kWaveLanes + (q & 15) + 16 * (d8 & 3)] = f;
    n = dpp_add(n, std::integral_constant<int, 0xB1>{});
    n = dpp_add(n, std::integral_constant<int, 0x4E>{});
    n = dpp_add(n, std::integral_constant<int, 0x141>{});  // row_half_mirror: the other four of eight
    if ((tid & 7) == 0) atomicAdd(&qnorm[q], n);
  };
  // The sample finds out whether to take a centre, and the filter is told.
  if constexpr (!kSample) {
    centred = p.centred[blockIdx.y] != 0;
    if (centred && tid < padded * 32) centre[tid] = p.centres[blockIdx.y * kFilterMaxDim + tid];
  }
#pragma unroll 1
  while (true) {
    if (tid < kFilterQueries) qnorm[tid] = 0.f;
    __syncthreads();
    if (whole) {
      // Loads of four items in flight (all items are whole eights of lanes).
      constexpr int kAhead = 4;
#pragma unroll 1
      for (int first = tid; first < items; first += kAhead * kFilterThreads) {
        f32x4 part[kAhead][2];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
          const int item = first + u * kFilterThreads < items ? first + u * kFilterThreads : first;
          const int q = item / (padded * 4);
          const int d = 8 * (item - q * (padded * 4));
          const float* src = p.t.queries + (q0 + (q < nq ? q : nq - 1)) * p.t.query_stride;
#pragma unroll
          for (int h = 0; h < 2; ++h) part[u][h] = *reinterpret_cast<const f32x4*>(src + (d + 4 * h < dim ? d + 4 * h : 0));
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
          const int item = first + u * kFilterThreads;
          if (item >= items) break;
          const int q = item / (padded * 4);
          const int d8 = item - q * (padded * 4);
          float x[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] = 8 * d8 + (e & 4) < dim ? part[u][e / 4][e % 4] : 0.f;
          stage(q, d8, x);
        }
      }
    } else {
#pragma unroll 1
      for (int item = tid; item < items; item += kFilterThreads) {
        const int q = item / (padded * 4);
        const int d8 = item - q * (padded * 4);  // dimensions 8 d8 .. + 7
        const float* src = p.t.queries + (q0 + (q < nq ? q : nq - 1)) * p.t.query_stride;
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = 8 * d8 + e < dim ? src[8 * d8 + e] : 0.f;
        stage(q, d8, x);
      }
    }
    __syncthreads();
    if (!kSample || centred) break;
    // The first m (at most 16) queries lie together where their mean's square
    // is over three quarters of the mean of their squares (a shift of 1.7
    // deviations an element): the sum of their products with each other
    // against that of their squares.  A NaN is not over it.  Every workgroup of
    // the query block computes the same bits.  256 queries x 50,000 x 96, k = 10,
    // bounded from the origin and from the centre, us (exact search 540): no
    // shift 54 and 61, 2 deviations 63 and 62, 4 272 and 62, 8 1,193 and 61.
    const int m = nq < 16 ? nq : 16;
    f32x4 gram = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int c = 0; c < padded; ++c)
      gram = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qfrag[c * kWaveLanes + lane], qfrag[c * kWaveLanes + lane], gram, 0, 0, 0);
    float over = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 4 * grp + r;
      const float g = row == col ? gram[r] * (1.f - 0.75f * static_cast<float>(m)) : gram[r];
      over += row < m && col < m ? g : 0.f;
    }
    over = dpp_add(over, std::integral_constant<int, 0xB1>{});
    over = dpp_add(over, std::integral_constant<int, 0x4E>{});
    over = dpp_add(over, std::integral_constant<int, 0x141>{});
    over = dpp_add(over, std::integral_constant<int, 0x140>{});  // row_mirror
    over = fold_rows(over);
    centred = __builtin_amdgcn_readfirstlane(over > 0.f) != 0;
    if (!centred) break;
    if (tid < padded * 32) {
      float sum = 0.f;
      if (tid < dim)
        for (int q = 0; q < m; ++q) sum += p.t.queries[(q0 + q) * p.t.query_stride + tid];
      centre[tid] = sum / static_cast<float>(m);
    }
    // (The loop's first barrier lies between the centre and its use, and
    // between the products above and the new fragments.)
  }
  if constexpr (kSample) {
    if (blockIdx.x == 0) {
      if (tid == 0) p.centred[blockIdx.y] = centred ? 1u : 0u;
      if (centred && tid < padded * 32) p.centres[blockIdx.y * kFilterMaxDim + tid] = centre[tid];
    }
  }
  const float c1 = 2.f * (0x1p-7f + 0x1p-16f + static_cast<float>(dim) * 0x1p-22f);
  const float c2 = static_cast<float>(dim + 36) * 0x1p-22f;
  if (tid < kFilterQueries) {
    const float n = qnorm[tid], length = sqrtf(n);
    if constexpr (kSample) {
      qa[tid] = n * (1.f + c2) + 1e-30f;
      qc[tid] = c1 * length;
    } else {
      const float limit = p.limit[blockIdx.y * kFilterQueries + tid];
      qlimit[tid] = limit;
      // Kept: 2 q^.r^ + c1 |q||r| - (1 - c2) |r|^2  >=  (1 - c2) |q|^2 - limit, halved.
      qa[tid] = tid < nq ? 0.5f * (n * (1.f - c2) - limit - 1e-30f) : INFINITY;
      qc[tid] = 0.5f * c1 * length;
      fill[tid] = 0u;
      worst[tid] = kNoKey;
    }
  }
  if constexpr (!kSample) {
    for (int s = tid; s < kFilterQueries * kFilterCap; s += kFilterThreads) list[s / kFilterCap][s % kFilterCap] = kNoKey;
  }
  __syncthreads();

  // ---- The wave's tiles.
  const int gw = static_cast<int>(blockIdx.x) * kFilterWaves + wave;
  const int all_waves = kSample ? p.sample_waves : p.workgroups * kFilterWaves;
  const int n_tiles = kSample ? (gw < p.sample_waves ? p.sample_tiles : 0)
                              : (gw < p.tiles ? (p.tiles - 1 - gw) / all_waves + 1 : 0);
  auto tile_at = [&](int i) -> int64_t {
    const int64_t n = gw + static_cast<int64_t>(i) * all_waves;
    return kSample ? n * p.sample_step : n;
  };
  // The id of this lane's candidate of tile i (requested a step ahead).
  auto load_id = [&](int i) -> uint32_t {
    const int64_t cand = tile_at(i < n_tiles ? i : n_tiles - 1) * kFilterTile + col;
    if constexpr (kIds) return p.t.ids[cand < p.t.num_cand ? cand : 0];
    return 0u;
  };
  // The row of this lane's candidate of tile i (row 0 where there is none).
  auto row_at = [&](int i, uint32_t id, bool& ok) -> const float* {
    const int64_t cand = tile_at(i) * kFilterTile + col;
    ok = cand < p.t.num_cand;
    int64_t row = ok ? cand : 0;
    if constexpr (kIds) {
      ok = ok && static_cast<int64_t>(id) < p.t.num_rows;
      row = ok ? id : 0;
    }
    return p.t.rows + row * p.t.row_stride;
  };
  f32x4 x[kChunks][2];  // this lane's part of a step's rows
  auto load = [&](const float* r, int slab, int c) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // Past the last dimension: the row's first floats, zeroed at use.
      const int d = (slab * kChunks + c) * 32 + 8 * grp + 4 * h;
      x[c][h] = *reinterpret_cast<const f32x4*>(r + (d < dim ? d : 0));
    }
  };

  f32x4 acc[kTiles];
  float norm = 0.f;
  float best[kTiles][4];  // sample: the smallest upper ends so far
#pragma unroll
  for (int t = 0; t < kTiles; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) best[t][r] = INFINITY;
  int queued = 0;  // survivors in the wave's queue (wave-uniform)

  // Fills slot `pos` of query q's list.
  auto put_key = [&](int q, uint32_t pos, uint64_t key) {
    __hip_atomic_store(&list[kSample ? 0 : q][kSample ? 0 : pos], key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };

  // Computes the queued pairs exactly and lists those at or below the limit.
  auto drain = [&]() {
    constexpr int kPairs = 4;
    __builtin_amdgcn_wave_barrier();
    for (int e0 = 0; e0 < queued; e0 += 4 * kPairs) {
      const float* query[kPairs];
      const float* row[kPairs];
      uint32_t node[kPairs];
      int q[kPairs];
#pragma unroll
      for (int n = 0; n < kPairs; ++n) {
        const int e = e0 + n * 4 + grp;
        const uint32_t entry = queue[kSample ? 0 : wave][e < queued ? e : 0];
        q[n] = static_cast<int>(entry & 63u);
        const int64_t cand = tile_at(static_cast<int>(entry >> 10)) * kFilterTile + ((entry >> 6) & 15u);
        node[n] = static_cast<uint32_t>(cand);
        if constexpr (kIds) node[n] = p.t.ids[cand];
        query[n] = p.t.queries + (q0 + (q[n] < nq ? q[n] : 0)) * p.t.query_stride;
        row[n] = p.t.rows + static_cast<int64_t>(node[n]) * p.t.row_stride;
      }
      float sum[kPairs];
      exact_distances<kPairs>(query, row, dim, col, sum);
      // Into the lists (fill counts the keys offered): a slot of the key's own,
      // or, where the list is full, the largest key's.
      bool want[kPairs];
      uint32_t pos[kPairs];
#pragma unroll
      for (int n = 0; n < kPairs; ++n) {
        want[n] = (col == 0) & (e0 + n * 4 + grp < queued) & (q[n] < nq) & !(sum[n] > qlimit[q[n]]);
        pos[n] = kFilterCap;
        if (want[n]) pos[n] = atomicAdd(&fill[q[n]], 1u);
      }
      bool full = false;
#pragma unroll
      for (int n = 0; n < kPairs; ++n) {
        if (pos[n] < static_cast<uint32_t>(kFilterCap)) put_key(q[n], pos[n], nearest_key(sum[n], node[n]));
        want[n] = want[n] & (pos[n] >= static_cast<uint32_t>(kFilterCap));
        full = full | want[n];
      }
      if (__ballot(full) == 0) continue;
#pragma unroll
      for (int n = 0; n < kPairs; ++n) {
        const uint64_t key = nearest_key(sum[n], node[n]);
        uint64_t* bound = &worst[kSample ? 0 : q[n]];
        const bool left = want[n] & (key < shared_key(bound));
        if (__ballot(left) == 0) continue;
        list_replace(list[kSample ? 0 : q[n]], bound, __shfl(key, 0, kLanes), __shfl(static_cast<int>(left), 0, kLanes) != 0,
                     col, lane);
      }
    }
    queued = 0;
    __builtin_amdgcn_wave_barrier();
  };

  // The bounds of a tile whose products are complete.
  auto finish = [&](int i, bool ok) {
    // |r|^2 of the lane's candidate: its four lane groups hold a part each.
    const float rn = fold_rows(norm);
    const float length = sqrtf(rn);
    if constexpr (kSample) {
      const float rb = rn * (1.f + c2);
#pragma unroll
      for (int t = 0; t < kTiles; ++t) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(&qa[16 * t + 4 * grp]);
        const f32x4 c = *reinterpret_cast<const f32x4*>(&qc[16 * t + 4 * grp]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float upper = fmaf(-2.f, acc[t][r], fmaf(c[r], length, a[r] + rb));
          best[t][r] = fminf(best[t][r], ok ? upper : INFINITY);  // a NaN is left out
        }
      }
    } else {
      const float rb = 0.5f * (1.f - c2) * rn;
      const uint64_t exists = __ballot(ok);
#pragma unroll
      for (int t = 0; t < kTiles; ++t) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(&qa[16 * t + 4 * grp]);
        const f32x4 c = *reinterpret_cast<const f32x4*>(&qc[16 * t + 4 * grp]);
        uint64_t keep[4];
        int kept = 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          // Queries past the block's last have an infinite bound to reach (a
          // NaN still passes: drain() leaves them out by number).
          keep[r] = __ballot(!(fmaf(c[r], length, acc[t][r]) - rb < a[r])) & exists;
          kept += __popcll(keep[r]);
        }
        if (kept == 0) continue;
        int base = queued;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if ((keep[r] >> lane) & 1) {
            const int at = base + __popcll(keep[r] & ((uint64_t{1} << lane) - 1));
            queue[kSample ? 0 : wave][at] = (static_cast<uint32_t>(i) << 10) | (static_cast<uint32_t>(col) << 6) |
                                            static_cast<uint32_t>(16 * t + 4 * grp + r);
          }
          base += __popcll(keep[r]);
        }
        queued = base;
      }
    }
  };

  // Steps (tile, slab).  A chunk's registers take the next step's rows as
  // soon as the chunk is converted, so a whole step is in flight while one is
  // computed; with ids, the next tile's are requested a step before that.
  if (n_tiles > 0) {
    uint32_t id = load_id(0);
    bool ok;
    const float* row = row_at(0, id, ok);
#pragma unroll
    for (int c = 0; c < kChunks; ++c) load(row, 0, c);
    if (slabs == 1) id = load_id(1);
    int i = 0, slab = 0;
    while (true) {
      const int next_slab = slab + 1 == slabs ? 0 : slab + 1;
      const int next_i = next_slab == 0 ? i + 1 : i;
      const bool more = next_i < n_tiles;
      // (The last step loads its own rows again.)
      bool next_ok = ok;
      if (more && next_slab == 0) row = row_at(next_i, id, next_ok);
      const int load_slab = more ? next_slab : slab;
      if (next_slab + 1 == slabs) id = load_id(next_i + 1);
      if (slab == 0) {
        norm = 0.f;
#pragma unroll
        for (int t = 0; t < kTiles; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      const bool partial = (slab + 1) * kChunks * 32 > dim;
#pragma unroll
      for (int c = 0; c < kChunks; ++c) {
        bf16x8 f;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int d = (slab * kChunks + c) * 32 + 8 * grp + 4 * h;
          f32x4 v = x[c][h];
          if (centred) v -= *reinterpret_cast<const f32x4*>(&centre[d]);
          if (partial && d >= dim) v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            f[4 * h + e] = static_cast<__bf16>(v[e]);
            norm = fmaf(v[e], v[e], norm);
          }
        }
        load(row, load_slab, c);
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
          const bf16x8 a = qfrag[(t * padded + slab * kChunks + c) * kWaveLanes + lane];
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, f, acc[t], 0, 0, 0);
        }
      }
      if (next_slab == 0) finish(i, ok);
      if constexpr (!kSample) {
        if (queued > kFilterDrain || (!more && queued > 0)) drain();
      }
      if (!more) break;
      ok = next_ok;
      i = next_i;
      slab = next_slab;
    }
  }

  if constexpr (kSample) {
    if (gw >= p.sample_waves) return;
    // One minimum per query over the wave's 16 candidate columns, or per four.
    const int cols = p.group_cols;
    const int64_t groups = static_cast<int64_t>(p.sample_waves) * cols;
    float* out = p.minima + static_cast<int64_t>(blockIdx.y) * groups * kFilterQueries;
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
      f32x4 m;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float x = best[t][r];
        x = dpp_min(x, std::integral_constant<int, 0xB1>{});
        x = dpp_min(x, std::integral_constant<int, 0x4E>{});
        if (cols == 1) {
          x = dpp_min(x, std::integral_constant<int, 0x141>{});  // row_half_mirror
          x = dpp_min(x, std::integral_constant<int, 0x140>{});  // row_mirror
        }
        m[r] = x;
      }
      if (cols == 1 ? col == 0 : (col & 3) == 0)
        *reinterpret_cast<f32x4*>(out + (static_cast<int64_t>(gw) * cols + col / 4) * kFilterQueries + 16 * t +
                                  4 * grp) = m;
    }
  } else {
    __syncthreads();
    const int64_t at = (static_cast<int64_t>(blockIdx.y) * p.workgroups + blockIdx.x) * kFilterQueries;
    if (tid < kFilterQueries) p.counts[at + tid] = fill[tid];
    for (int s = tid; s < kFilterQueries * kFilterCap; s += kFilterThreads) {
      const int q = s / kFilterCap, e = s % kFilterCap;
      if (e < static_cast<int>(fill[q])) p.lists[(at + q) * kFilterCap + e] = list[kSample ? 0 : q][kSample ? 0 : e];
    }
  }
}

// Launch 2: a limit at or above the k-th smallest of a query's group minima,
// one wave per query, four queries of a block per workgroup.
template <int kPer>  // groups per lane: 64 kPer is at least the groups
__global__ __launch_bounds__(kFilterThreads) void top_k_limit_kernel(TopKFilter p) {
  const int lane = static_cast<int>(threadIdx.x) & (kWaveLanes - 1);
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWaveLanes);
  const int q = static_cast<int>(blockIdx.x) * kFilterWaves + wave;
  const int groups = p.sample_waves * p.group_cols;
  const float* in = p.minima + static_cast<int64_t>(blockIdx.y) * groups * kFilterQueries + q;
  // Bits mapped so that unsigned order is float order; +inf past the groups.
  uint32_t v[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int at = i * kWaveLanes + lane;
    const uint32_t b = __float_as_uint(at < groups ? in[static_cast<int64_t>(at) * kFilterQueries] : INFINITY);
    v[i] = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
  }
  uint32_t lo = 0xffffffffu, hi = 0u;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const uint32_t w = i * kWaveLanes + lane < groups ? v[i] : 0u;
    lo = lo < v[i] ? lo : v[i];
    hi = hi > w ? hi : w;
  }
  lo = wave_fold(lo, [](uint32_t a, uint32_t b) { return a < b ? a : b; });
  hi = wave_fold(hi, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
  // At least k minima are at or below hi, throughout; 14 halvings leave it
  // within 2^-14 of the minima's range of the k-th.
  for (int step = 0; step < 14 && lo < hi; ++step) {
    const uint32_t mid = lo + (hi - lo) / 2;
    int n = 0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) n += __popcll(__ballot(v[i] <= mid));
    if (n >= p.t.k) hi = mid;
    else lo = mid + 1;
  }
  if (lane == 0)
    p.limit[blockIdx.y * kFilterQueries + q] =
        __uint_as_float((hi & 0x80000000u) ? (hi & 0x7fffffffu) : ~hi);
}

// Sorts keys[0 .. n) ascending as sort_keys does, padded to at least 64 keys,
// with 64-key runs sorted in the lanes of a wave and the last six
// strides of every longer run there too: a barrier for each stride of 64 keys
// or more and one per run length, 14 for 1,024 keys where sort_keys has 55.
template <int kSortThreads>
__device__ __forceinline__ void sort_keys_by_wave(uint64_t* keys, int n, int tid) {
  int size = kWaveLanes;
  while (size < n) size <<= 1;
  for (int i = n + tid; i < size; i += kSortThreads) keys[i] = kNoKey;
  __syncthreads();
  const int lane = tid & (kWaveLanes - 1);
  for (int i = tid; i < size; i += kSortThreads) {
    // Runs alternate in direction; a descending one is the ascending sort of
    // the complements.
    const uint64_t flip = size > kWaveLanes && (i & kWaveLanes) ? ~uint64_t{0} : 0;
    keys[i] = wave_sort(keys[i] ^ flip, lane) ^ flip;
  }
  __syncthreads();
  for (int span = 2 * kWaveLanes; span <= size; span <<= 1) {
    for (int stride = span >> 1; stride >= kWaveLanes; stride >>= 1) {
      for (int t = tid; t < size / 2; t += kSortThreads) {
        const int i = 2 * t - (t & (stride - 1));
        const uint64_t a = keys[i], b = keys[i + stride];
        if ((a > b) == ((i & span) == 0)) {
          keys[i] = b;
          keys[i + stride] = a;
        }
      }
      __syncthreads();
    }
    for (int i = tid; i < size; i += kSortThreads) {
      const uint64_t flip = span < size && (i & span) ? ~uint64_t{0} : 0;
      keys[i] = bitonic_merge<kWaveLanes, kWaveLanes / 2>(keys[i] ^ flip, lane) ^ flip;
    }
    __syncthreads();
  }
}

// Launch 4: one workgroup per query gathers the keys of its lists and sorts
// them (in pieces where they exceed the LDS buffer).
template <bool kIds, int kMergeThreads>
__global__ __launch_bounds__(kMergeThreads) void top_k_merge_kernel(TopKFilter p) {
  __shared__ uint64_t keys[kTopKKeys];  // the k best so far (none at first), then new ones
  __shared__ uint32_t fill, over_count, equal;
  __shared__ uint32_t over[kFilterMaxWorkgroups];  // workgroups whose list ran over ...
  __shared__ uint64_t over_last[kFilterMaxWorkgroups];  // ... and their lists' largest keys
  const int tid = static_cast<int>(threadIdx.x);
  const int64_t query = blockIdx.x;
  const int64_t block = query / kFilterQueries;
  const int q = static_cast<int>(query - block * kFilterQueries);
  const int k = p.t.k;
  uint32_t held = 0;  // 0, or k once keys have been merged
  if (tid == 0) fill = over_count = 0u;
  __syncthreads();

  for (int first = 0; first < p.workgroups; first += kMergeThreads) {
    const int w = first + tid;
    const int64_t at = (block * p.workgroups + w) * kFilterQueries + q;
    uint32_t n = w < p.workgroups ? p.counts[at] : 0u;
    if (n > static_cast<uint32_t>(kFilterCap)) {
      n = kFilterCap;
      uint64_t last = 0;
      for (uint32_t s = 0; s < n; ++s) {
        const uint64_t x = p.lists[at * kFilterCap + s];
        last = x > last ? x : last;
      }
      const uint32_t o = atomicAdd(&over_count, 1u);
      over[o] = static_cast<uint32_t>(w);
      over_last[o] = last;
    }
    bool pending = n > 0;
    while (true) {
      if (pending) {
        const uint32_t pos = atomicAdd(&fill, n);
        const uint32_t room = kTopKKeys - held;
        pending = pos + n > room;
        // A list that does not fit waits for the merge; the slots it took
        // inside the buffer stay empty.
        for (uint32_t s = 0; s < n && pos + s < room; ++s)
          keys[held + pos + s] = pending ? kNoKey : p.lists[at * kFilterCap + s];
      }
      __syncthreads();
      const bool full = fill > kTopKKeys - held;
      __syncthreads();
      if (!full) break;
      sort_keys_by_wave<kMergeThreads>(keys, kTopKKeys, tid);
      held = static_cast<uint32_t>(k);
      if (tid == 0) fill = 0u;
      __syncthreads();
    }
  }
  {
    const int n = static_cast<int>(held + fill);
    __syncthreads();
    for (int i = n + tid; i < k; i += kMergeThreads) keys[i] = kNoKey;
    sort_keys_by_wave<kMergeThreads>(keys, n, tid);
    if (tid == 0) fill = 0u;
    __syncthreads();
  }

  // Workgroups whose list ran over with its largest key below the k-th found:
  // their candidates once more, the keys above that largest (and, of those
  // equal to it, the ones the list left out), kMergeThreads / 4 at a time: a
  // 16-lane group computes four.
  const int n_over = static_cast<int>(over_count);
  const int lane = tid & (kLanes - 1);
  const int group = tid / kLanes;
  constexpr int kStripes = kMergeThreads / kFilterThreads;  // of 64 candidates
  const float* qrow = p.t.queries + query * p.t.query_stride;
  for (int o = 0; o < n_over; ++o) {
    const uint64_t last = over_last[o];
    if (last >= keys[k - 1]) continue;  // uniform: the keys were sorted behind a barrier
    const int64_t w = over[o];
    const uint64_t* held_keys = p.lists + ((block * p.workgroups + w) * kFilterQueries + q) * kFilterCap;
    uint32_t last_held = 0;
    for (int e = 0; e < kFilterCap; ++e) last_held += held_keys[e] == last;
    if (tid == 0) equal = 0u;
    __syncthreads();
    for (int64_t first = w * 64; first < p.t.num_cand; first += static_cast<int64_t>(p.workgroups) * 64 * kStripes) {
      const float* query4[4];
      const float* row4[4];
      uint32_t node[4];
      bool ok[4];
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const int64_t cand = first + static_cast<int64_t>(group / 16) * p.workgroups * 64 + (group & 15) * 4 + n;
        ok[n] = cand < p.t.num_cand;
        node[n] = ok[n] ? static_cast<uint32_t>(cand) : 0u;
        if constexpr (kIds) {
          node[n] = ok[n] ? p.t.ids[cand] : 0u;
          ok[n] = ok[n] && static_cast<int64_t>(node[n]) < p.t.num_rows;
          if (!ok[n]) node[n] = 0u;
        }
        query4[n] = qrow;
        row4[n] = p.t.rows + static_cast<int64_t>(node[n]) * p.t.row_stride;
      }
      float sum[4];
      exact_distances<4>(query4, row4, p.t.dim, lane, sum);
      const uint64_t kth = keys[k - 1];
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        if (ok[n] && lane == 0) {
          const uint64_t key = nearest_key(sum[n], node[n]);
          if (key < kth && (key > last || (key == last && atomicAdd(&equal, 1u) >= last_held)))
            keys[k + atomicAdd(&fill, 1u)] = key;
        }
      }
      __syncthreads();
      const int n = static_cast<int>(fill);
      __syncthreads();
      if (n + 64 * kStripes > kTopKKeys - k || (n > 0 && kth == kNoKey)) {
        sort_keys_by_wave<kMergeThreads>(keys, k + n, tid);
        if (tid == 0) fill = 0u;
        __syncthreads();
      }
    }
    const int n = static_cast<int>(fill);
    __syncthreads();
    if (n > 0) {
      sort_keys_by_wave<kMergeThreads>(keys, k + n, tid);
      if (tid == 0) fill = 0u;
      __syncthreads();
    }
  }
  for (int r = tid; r < k; r += kMergeThreads) {
    const uint64_t key = keys[r];
    const int64_t off = query * p.t.out_stride + r;
    p.t.distances[off] = key == kNoKey ? INFINITY : key_distance(key);
    p.t.nodes[off] = key == kNoKey ? VECTRA_SCAN_NO_NODE : static_cast<uint32_t>(key);
  }
}
