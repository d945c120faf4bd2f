// Rows that need most of their vocabulary in rank order: sampling from the whole vocabulary (k <= 1 with p >= 1).
// (Nuclei of p < 1 stay with the candidate lists of nucleus_stream_kernel: routed through here 64 x 128256 rows with
// nuclei of 4000 tokens took 84 us per step instead of 41.)
//
// The reference sorts such a row, adds the exponentials of all of it one after the other and draws from the result.
// One workgroup per row (exact_rows_kernel) spends 0.55 ms on that however few rows there are: its sort moves every
// key three times at the memory rate of a single CU, and its sums run over 128 K exponentials in one workgroup.  Here
// every step but the last is spread over the GPU, in five launches (16 x 128256 fp16: 557 -> 59 us per
// step on the same rows again and 66 on rows that come from memory: 4.7 + 4.7 + 11.5 + 21.6 + 20 us by a trace; every
// one of them is a chain of dependent phases of a few barriers each, no launch moves more than 33 MB).  Rows whose token
// alone is asked for need no order: for p = 1 a launch behind 2 picks it from the histogram (wide_pick_kernel), one launch does
// 3 and 4 for the rows it gives back (wide_rest_kernel), 0.3 % of such rows, and 5 finishes these.
//   1. wide_max:     the maximum of every chunk of kWideChunk logits.
//   2. wide_count:   a histogram per chunk over kWideBuckets buckets, linear in the score below the row's maximum down
//                    to the depth past which no element can lie inside the kept set.
//   3. wide_scatter: every workgroup scans the row's histograms, gives its chunk's keys their places, bucket by
//                    bucket, in the row's key buffer, and the first chunk's cuts the list into tiles of whole buckets
//                    (kWideTile keys and at most one bucket more).
//   4. wide_rank:    a workgroup per tile sorts it in LDS (a counting sort with buckets linear between the tile's own
//                    extremes), writes (exponential, id) entries in rank order, and composes the tile's step record
//                    for the exact sequential sum under the binade the double sums of the tiles before it predict (a
//                    look-back at sums that lower workgroup indices of the same launch publish, as in
//                    seqsum_exp_step).
//   5. wide_finish:  a workgroup per row walks the records (the exact sum behind every tile), searches the one tile
//                    in which the stop of FindNucleus can lie, and draws from the double sums of the tiles.
// Elements of equal score need not be told apart before the draw: a run of ties weighs the same in any order.  Runs
// of ties (bf16 logits have hundreds to thousands per value, the more the further their bulk lies from zero) stay in
// arrival order, also across the tiles they are cut into, and the id of the drawn rank is taken from the run the draw
// falls into.  A call that asks for the kept ids has its ties ordered by wide_rank.  A bucket of several scores too
// large for a tile (a flat row, or one whose bulk is narrow) is cut between ranks its tiles select (wide_gather_cut).
// A row this does not fit (a maximum that is not finite, a stop beyond the listed elements, more than kWideSelectMax keys
// of several scores in one bucket) is finished by the exact path inside wide_finish.
#pragma once
#include "sample_stream.h"
#include "seqsum_exp_step.h"
#include "token_pick.h"
#include "seq_walk.h"

namespace ms {

constexpr int kWideBlock = 1024;
constexpr int kWidePer = kWideChunk / kWideBlock;  // logits per thread
constexpr int kWideRankBlock = 512;
static_assert(kWideTile + kWideBucketMax <= kSegElems, "a tile fits the segment its step record describes");

// Rows of this kind: every element counts, whatever k says (k <= 1) and however large p is.
__device__ __forceinline__ bool wide_row(mi355x_sample_params prm) { return prm.k <= 1 && !(prm.p < 1.0f); }

// How far below the maximum (in score units) the list reaches: an element past ln V + 18 exponent units below the
// maximum satisfies the stop of FindNucleus for p = 1, (V - i - 1) * e_i < prefix * 2^-25, wherever it ranks, so the
// stop lies at or before the first such element (which follows the list, wide_best).
__device__ __forceinline__ float wide_depth(mi355x_sample_params prm, int vocab) {
  return (logf(static_cast<float>(vocab)) + 18.0f) * prm.temperature;
}

// Which row, and which of its `per_row` shares of the work, a workgroup has.  Workgroups go round-robin over the eight
// XCDs; all shares of a row get indices of one remainder, so what they hand over -- every launch reads what the one
// before it wrote, scattered all over the row's buffers -- stays in one L2 (scattered from all XCDs, the keys' 8-byte
// writes would reach memory one partial line each).  Rows past the last have no work.
struct WideShare {
  int row, item;
};
__device__ __forceinline__ WideShare wide_share(int per_row) {
  const int xcd = static_cast<int>(blockIdx.x) & 7, slot = static_cast<int>(blockIdx.x) >> 3;
  return WideShare{xcd + 8 * (slot / per_row), slot % per_row};
}

// The logits of thread t of BLOCK in a chunk, in loads of 16 bytes; ids past the vocabulary are NaN.
template <typename InT, int BLOCK = kWideBlock>
__device__ __forceinline__ void wide_load(const InT* row, int V, int chunk, float (&v)[kWideChunk / BLOCK]) {
  constexpr int VEC = 16 / static_cast<int>(sizeof(InT));
#pragma unroll
  for (int j = 0; j < kWideChunk / BLOCK / VEC; ++j) {
    const int i0 = chunk * kWideChunk + (j * BLOCK + static_cast<int>(threadIdx.x)) * VEC;
    if (i0 + VEC <= V) {
      if constexpr (VEC == 4) {
        const v4f_any q = *reinterpret_cast<const v4f_any*>(row + i0);
        v[j * 4] = q.x, v[j * 4 + 1] = q.y, v[j * 4 + 2] = q.z, v[j * 4 + 3] = q.w;
      } else {
        const v4u q = *reinterpret_cast<const v4u_any*>(row + i0);
        if constexpr (__is_same(InT, uint16_t)) widen_half8(q, &v[j * 8]);
        else widen_bf16x8(q, &v[j * 8]);
      }
    } else {
#pragma unroll
      for (int c = 0; c < VEC; ++c) v[j * VEC + c] = i0 + c < V ? load_one<InT>(row, i0 + c) : __uint_as_float(0x7fc00000u);
    }
  }
}
// The same loads, not widened yet (a chunk past the last one: the last one's), for the launch that has several chunks on their way.
// (The others through these as well: 16 x 5000 fp16 24.6 -> 25.2 us a step, 64 x 128256 bf16 64.8 -> 65.9, 256 x 5000 bf16 28.3 -> 29.3.)
template <typename InT>
struct WideRaw {
  static constexpr int kVec = 16 / static_cast<int>(sizeof(InT)), kLoads = kWidePer / kVec;
  v4u q[kLoads];
  __device__ __forceinline__ void load(const InT* row, int V, int chunks, int chunk) {
    const int c = chunk < chunks ? chunk : chunks - 1;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int i0 = c * kWideChunk + (j * kWideBlock + static_cast<int>(threadIdx.x)) * kVec;
      q[j] = *reinterpret_cast<const v4u_any*>(row + (i0 + kVec <= V ? i0 : V - kVec));  // (the row's end: shifted below)
    }
  }
  // Value e of the chunk, NaN past the end of the row.
  __device__ __forceinline__ void widen(int V, int chunk, float (&v)[kWidePer]) const {
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      if constexpr (kVec == 4) {
#pragma unroll
        for (int c = 0; c < 4; ++c) v[j * 4 + c] = __uint_as_float(q[j][c]);
      } else if constexpr (__is_same(InT, uint16_t)) {
        widen_half8(q[j], &v[j * 8]);
      } else {
        widen_bf16x8(q[j], &v[j * 8]);
      }
    }
    if ((chunk + 1) * kWideChunk > V) {  // (the row's last chunk: a group that crosses the end holds the row's last values)
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        const int i0 = chunk * kWideChunk + (j * kWideBlock + static_cast<int>(threadIdx.x)) * kVec;
        if (i0 + kVec > V) {
          const int past = i0 + kVec - V;  // value c of the group came as value c + past
          float w[kVec];
#pragma unroll
          for (int c = 0; c < kVec; ++c) {
            w[c] = __uint_as_float(0x7fc00000u);
#pragma unroll
            for (int d = 0; d < kVec; ++d) w[c] = d == c + past ? v[j * kVec + d] : w[c];
          }
#pragma unroll
          for (int c = 0; c < kVec; ++c) v[j * kVec + c] = w[c];
        }
      }
    }
  }
};
template <typename InT, int BLOCK = kWideBlock>
__device__ __forceinline__ int wide_index(int chunk, int e) {
  constexpr int VEC = 16 / static_cast<int>(sizeof(InT));
  return chunk * kWideChunk + ((e / VEC) * BLOCK + static_cast<int>(threadIdx.x)) * VEC + e % VEC;
}

// The row's maximum as the chunks left it (0xffffffff where the row is not one for this path).
__device__ __forceinline__ uint32_t wide_row_max(const SampleArgs& a, const WideArgs& w, int row) {
  const int lane = lane_id();
  uint32_t m = 0u;
  for (int c = lane; c < w.chunks; c += 64) {
    const uint32_t k = a.chunk_max[static_cast<size_t>(row) * w.chunks + c];
    m = k > m ? k : m;
  }
  m = wave_max<uint32_t>(m);
  return (m <= order_key(-1e30f) || m >= order_key(1e30f)) ? 0xffffffffu : m;
}

template <typename InT, bool INLINE>
__global__ __launch_bounds__(kWideBlock) void wide_max_kernel(const SampleArgs a, const typename WideTable<INLINE>::type, const WideArgs w) {
  __shared__ uint32_t red[16];
  const WideShare mine = wide_share(w.chunks);
  const int chunk = mine.item, row = mine.row, tid = threadIdx.x;
  if (blockIdx.x == 0 && tid == 0) *w.rest.sorted = *w.rest.exact = 0u;
  if (row >= a.rows || !wide_row(row_params<INLINE>(a, row))) return;
  float v[kWidePer];
  wide_load<InT>(static_cast<const InT*>(row_start<INLINE>(a, row, sizeof(InT))), a.vocab, chunk, v);
  // (this launch is the first of its sequence: it also marks the sums of the row's tiles as not written, and none of its chunks as
  // scattered by wide_rest)
  if (chunk == 0) {
    for (int t = tid; t < w.max_tiles; t += kWideBlock) store_sum_bits(w.tile_sum + static_cast<size_t>(row) * w.max_tiles + t, kSumNotReady);
    if (tid == 0) {
      w.best_below[row] = 0;
      w.rest.scattered[row * kRestStride] = w.rest.gave_up[row] = 0u;
    }
  }
  float m = -__builtin_inff();
#pragma unroll
  for (int e = 0; e < kWidePer; ++e) m = fmaxf(m, v[e]);
  const uint32_t k = block_max<uint32_t>(order_key(m), red, false);
  if (tid == 0) a.chunk_max[static_cast<size_t>(row) * w.chunks + chunk] = k;
}

// What one workgroup writes and others of the same launch read (HANDED) goes past the caches of the CUs and the XCDs in both
// directions; what the next launch reads need not.  (Plain stores and loads, with the caches written back by every chunk's workgroup and
// invalidated by every tile's: wide_rest of 64 x 128256 rows 33 us longer, of 256 x 32064 34.)
template <bool HANDED, typename T>
__device__ __forceinline__ void wide_put(T* p, T v) {
  if constexpr (HANDED) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = v;
}
template <bool HANDED, typename T>
__device__ __forceinline__ T wide_get(const T* p) {
  if constexpr (HANDED) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else return *p;
}
template <bool HANDED>
__device__ __forceinline__ void wide_put(uint2* p, uint2 v) {
  wide_put<HANDED>(reinterpret_cast<u64*>(p), static_cast<u64>(v.x) | (static_cast<u64>(v.y) << 32));
}
template <bool HANDED>
__device__ __forceinline__ uint2 wide_get(const uint2* p) {
  const u64 v = wide_get<HANDED>(reinterpret_cast<const u64*>(p));
  return make_uint2(static_cast<uint32_t>(v), static_cast<uint32_t>(v >> 32));
}

// Bucket of a score: a non-increasing function of it (every operation is monotone), kWideBuckets and up for what lies
// past the depth and for NaN.
struct WideBuckets {
  float top, scale;
  __device__ __forceinline__ WideBuckets(float max_score, float depth) : top(max_score), scale(static_cast<float>(kWideBuckets) / depth) {}
  __device__ __forceinline__ uint32_t operator()(float x) const {
    const float b = (top - x) * scale;
    return b < static_cast<float>(kWideBuckets) ? static_cast<uint32_t>(b) : static_cast<uint32_t>(kWideBuckets);
  }
};

// The masses of a row's buckets lie behind the counts, chunk by chunk; the first one of a chunk that has a NaN is negative.
__device__ __forceinline__ double2* wide_masses(const SampleArgs& a, const WideArgs& w, int row) {
  return reinterpret_cast<double2*>(a.big + static_cast<size_t>(row) * a.big_stride + static_cast<size_t>(w.chunks) * (kWideBlock / 2));
}

// (Eight waves a SIMD: two workgroups a CU.  With 66 registers instead of 64 it was one: 256 x 128256 fp16, all launches, 158.7 -> 132.3 us,
// 64 x 201088 104.5 -> 94.3, 64 x 128256 55.3 -> 50.6; 16 rows as before.)
template <typename InT, bool INLINE>
__global__ __launch_bounds__(kWideBlock, 8) void wide_count_kernel(const SampleArgs a, const typename WideTable<INLINE>::type, const WideArgs w) {
  __shared__ uint32_t hist[kWideBuckets + 1];
  __shared__ double mass[kWideBuckets];
  __shared__ uint64_t exp_tab[32];
  __shared__ int has_nan;
  const WideShare mine = wide_share(w.chunks);
  const int chunk = mine.item, row = mine.row, tid = threadIdx.x;
  if (row >= a.rows) return;
  const mi355x_sample_params prm = row_params<INLINE>(a, row);
  if (!wide_row(prm)) return;
  const uint32_t rmax = wide_row_max(a, w, row);
  if (rmax == 0xffffffffu) return;
  float v[kWidePer];
  wide_load<InT>(static_cast<const InT*>(row_start<INLINE>(a, row, sizeof(InT))), a.vocab, chunk, v);
  for (int b = tid; b <= kWideBuckets; b += kWideBlock) hist[b] = 0u;
  const bool pick = w.pick != 0 && prm.p == 1.0f;
  if (pick) {
    mass[tid] = mass[tid + kWideBlock] = 0.0;
    if (tid < 32) exp_tab[tid] = em::exp2_tab(static_cast<uint32_t>(tid));
    if (tid == 0) has_nan = 0;
  }
  __syncthreads();
  const WideBuckets bucket_of(key_to_float(rmax), wide_depth(prm, a.vocab));
  if (pick) {
    const float top = key_to_float(rmax), inv_temp = 1.0f / prm.temperature;
    const uint64_t* const tab = exp_tab;
    float ex[kWidePer];
#pragma unroll
    for (int e = 0; e < kWidePer; ++e) ex[e] = em::expf_in_range((v[e] - top) * inv_temp, [=](uint32_t i) { return tab[i]; });
#pragma unroll
    for (int e = 0; e < kWidePer; ++e) {
      const uint32_t b = bucket_of(v[e]);
      if (b < static_cast<uint32_t>(kWideBuckets)) {
        atomicAdd(&hist[b], 1u);
        __hip_atomic_fetch_add(&mass[b], static_cast<double>(ex[e]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      } else if (v[e] != v[e] && wide_index<InT>(chunk, e) < a.vocab) {
        has_nan = 1;
      }
    }
  } else {
#pragma unroll
    for (int e = 0; e < kWidePer; ++e) {
      const uint32_t b = bucket_of(v[e]);
      if (b < static_cast<uint32_t>(kWideBuckets)) atomicAdd(&hist[b], 1u);
    }
  }
  __syncthreads();
  // two buckets a thread, packed: a chunk holds at most kWideChunk keys
  static_assert(kWideBuckets == 2 * kWideBlock && kWideChunk < 1 << 16, "a pair of buckets per thread, of 16 bits each");
  uint32_t* out = reinterpret_cast<uint32_t*>(a.big + static_cast<size_t>(row) * a.big_stride) + static_cast<size_t>(chunk) * kWideBlock;
  out[tid] = hist[2 * tid] | (hist[2 * tid + 1] << 16);
  if (pick) {
    double2* const masses = wide_masses(a, w, row) + static_cast<size_t>(chunk) * kWideBlock;
    masses[tid] = make_double2(tid == 0 && has_nan ? -mass[0] : mass[2 * tid], mass[2 * tid + 1]);
  }
}

// The token of a row of p = 1 whose kept set nobody asks for, without ordering the row (see token_pick.h).  The search
// stops where (V - i - 1) e_i is half a unit of the running sum or less, so whatever it keeps past there weighs less than
// 2^-24 of the sum, and the draw is decided by the histogram of masses and the keys of the bucket it points into -- unless
// a share lies closer to u than what the reference's roundings may move it by (u (1 - u) 2^-23) and that rest: 0.1 to 0.3 %
// of rows of 128256 and 201088 logits, which go the long way behind this.  (Masses as whole numbers of 2^-43, whose rounding
// such rows of a few heavy tokens notice: twice as many.)  One workgroup per row: it adds the chunks' histograms up,
// finds the bucket and looks the row through once more for its keys.  A trace of 16 x 128256 fp16: 3.2 (maximum) + 7.1
// (counts and masses, 4.8 without these) + 19.2 us and what wide_rest and wide_finish take to find nothing to do; steps, with three
// launches in their place, 62.9 -> 35.1 us, 64 x 128256 fp16 142 -> 58, 1 x 128256 fp32 50 -> 29, 24 x 201088 bf16 129 -> 51.  A compare of every logit with the two
// buckets and a load of four chunks at a time instead of eight ahead: 23.0 us for this launch.
template <typename InT, bool INLINE>
__global__ __launch_bounds__(kWideBlock) void wide_pick_kernel(const SampleArgs a, const typename WideTable<INLINE>::type, const WideArgs w) {
  extern __shared__ u64 lds_keys[];
  PickShared& sh = *reinterpret_cast<PickShared*>(lds_keys + kPickRoom);
  __shared__ uint64_t exp_tab[32];
  __shared__ uint32_t wave_counts[16];
  static_assert(kPickBlock == kWideBlock && kPickRoom * sizeof(u64) + sizeof(PickShared) <= kFinishLds, "the pick's room");
  const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, V = a.vocab;
  const mi355x_sample_params prm = row_params<INLINE>(a, row);
  if (!wide_row(prm)) return;
  const uint32_t rmax = wide_row_max(a, w, row);
  // (rows to be sorted are listed from the front, those of the exact path from the back)
  auto give_back = [&](bool exact) {
    const uint32_t i = atomicAdd(exact ? w.rest.exact : w.rest.sorted, 1u);
    w.rest.rows[exact ? static_cast<uint32_t>(a.rows) - 1u - i : i] = static_cast<uint32_t>(row);
    atomicAdd(a.fallback_rows + 3, 1u);
  };
  if (rmax == 0xffffffffu || !(prm.p == 1.0f)) {
    if (tid == 0) give_back(rmax == 0xffffffffu);
    return;
  }
  // The first of the row's chunks are requested now: they are looked through last.
  constexpr int kAhead = WideRaw<InT>::kLoads == 1 ? 8 : 4;
  const InT* const x = static_cast<const InT*>(row_start<INLINE>(a, row, sizeof(InT)));
  WideRaw<InT> raw[kAhead];
#pragma unroll
  for (int c = 0; c < kAhead; ++c) raw[c].load(x, V, w.chunks, c);
  // the thread's two buckets in the whole row
  double m0 = 0.0, m1 = 0.0;
  uint32_t n_own = 0u, n_first = 0u;
  bool nan = false;
  const double2* const masses = wide_masses(a, w, row) + tid;
  const uint32_t* const counts = reinterpret_cast<const uint32_t*>(a.big + static_cast<size_t>(row) * a.big_stride) + tid;
  for (int c0 = 0; c0 < w.chunks; c0 += 8) {
    double2 m[8];
    uint32_t n[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      m[c] = c0 + c < w.chunks ? masses[static_cast<size_t>(c0 + c) * kWideBlock] : make_double2(0.0, 0.0);
      n[c] = c0 + c < w.chunks ? counts[static_cast<size_t>(c0 + c) * kWideBlock] : 0u;
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      nan |= signbit(m[c].x);
      m0 += fabs(m[c].x);
      m1 += m[c].y;
      n_first += n[c] & 0xffffu;
      n_own += (n[c] & 0xffffu) + (n[c] >> 16);
    }
  }
  TokenPick::clear(sh);
  if (tid < 32) exp_tab[tid] = em::exp2_tab(static_cast<uint32_t>(tid));
  const double inc = wave_prefix_sum<double>(m0 + m1);
  const uint32_t n_inc = wave_prefix_sum<uint32_t>(n_own);
  if (lane == 63) {
    sh.sums[wave] = em::as_u64(inc);
    wave_counts[wave] = n_inc;
  }
  if (__syncthreads_or(nan)) {  // (one that is kept makes all weights NaN: the long way)
    if (tid == 0) give_back(false);
    return;
  }
  const double ws = wave_prefix_sum<double>(lane < 16 ? em::as_double(sh.sums[lane]) : 0.0);
  const uint32_t wn = wave_prefix_sum<uint32_t>(lane < 16 ? wave_counts[lane] : 0u);
  const double before = (wave > 0 ? wave_read_lane(ws, wave - 1) : 0.0) + (inc - (m0 + m1)), total = wave_read_lane(ws, 15);
  const uint32_t n_before = (wave > 0 ? wave_read_lane(wn, wave - 1) : 0u) + n_inc - n_own;
  const double u = a.uniforms[row];
  // the first bucket in which the search may stop: up to it, (V - i - 1) e_i exceeds half a unit of any running sum
  const WideBuckets bucket_of(key_to_float(rmax), wide_depth(prm, V));
  const float step = 1.0f / (prm.temperature * bucket_of.scale);
  const float rest = static_cast<float>(total) * 5.97e-8f * (1.02f + static_cast<float>(V) * 6.1e-8f);
  auto may_stop = [&](uint32_t n, int bucket_end) { return !(static_cast<float>(V - static_cast<int>(n)) * __expf(-step * static_cast<float>(bucket_end)) > rest); };
  const bool stop0 = may_stop(n_before + n_first, 2 * tid + 1), stop1 = may_stop(n_before + n_own, 2 * tid + 2);
  u64 kept_bits = em::as_u64(stop0 ? before : before + m0), stop_bucket = static_cast<u64>(stop0 ? 2 * tid : 2 * tid + 1);
  int at, at_again;
  block_firsts(stop0 || stop1, kept_bits, at, stop0 || stop1, stop_bucket, at_again, sh.firsts[0]);
  const double kept_lo = at == kIntMax ? total : em::as_double(kept_bits);
  if (at == kIntMax) stop_bucket = kWideBuckets;
  // (what follows the listed elements: two of them at most, each under e^-18 / V)
  const double kept_hi = total + 4e-8 / static_cast<double>(V);
  const double guard = kept_hi * (u * (1.0 - u) * 1.21e-7 + 16.0 * 1.2e-16 * static_cast<double>(V) + 1e-11);
  const double t_lo = u * kept_lo - guard, t_hi = u * kept_hi + guard;
  // the buckets the draw may fall into
  const double mid = before + m0, upto = mid + m1;
  const bool lo_first = m0 != 0.0 && mid >= t_lo, hi_first = m0 != 0.0 && mid >= t_hi;
  // (which of the two it is takes the lowest bit of the mass in front of it)
  u64 front = (em::as_u64(lo_first ? before : mid) & ~1ull) | (lo_first ? 0u : 1u), hi_second = hi_first ? 0u : 1u;
  int d_lo, d_hi;
  block_firsts(m0 + m1 != 0.0 && upto >= t_lo, front, d_lo, m0 + m1 != 0.0 && upto >= t_hi, hi_second, d_hi, sh.firsts[1]);
  const uint32_t bucket_lo = 2u * static_cast<uint32_t>(d_lo) + static_cast<uint32_t>(front & 1u);
  const uint32_t bucket_hi = 2u * static_cast<uint32_t>(d_hi) + static_cast<uint32_t>(hi_second);
  bool ok = d_lo != kIntMax && d_hi != kIntMax && bucket_hi < stop_bucket;
  uint32_t id = kNoPick;
  if (ok) {
    // their keys
    u64* const list = lds_keys + kPickHits * (kPickBlock / 64);
    // (A score of these buckets lies within `reach` of their middle; one in a few thousand that does is not of them.)
    const float middle = key_to_float(rmax) - 0.5f * static_cast<float>(bucket_lo + bucket_hi + 1u) / bucket_of.scale;
    const float reach = 0.505f * static_cast<float>(bucket_hi - bucket_lo + 1u) / bucket_of.scale + 1e-5f * (fabsf(middle) + fabsf(key_to_float(rmax)));
    for (int c0 = 0; c0 < w.chunks; c0 += kAhead) {
#pragma unroll
      for (int c = 0; c < kAhead; ++c) {
        if (c0 + c < w.chunks) {
          float v[kWidePer];
          raw[c].widen(V, c0 + c, v);
          bool near = false;
#pragma unroll
          for (int e = 0; e < kWidePer; ++e) near |= fabsf(v[e] - middle) <= reach;
          if (near) {
#pragma unroll
            for (int e = 0; e < kWidePer; ++e) {
              if (fabsf(v[e] - middle) <= reach && bucket_of(v[e]) - bucket_lo <= bucket_hi - bucket_lo) {
                const uint32_t i = atomicAdd(&sh.n_list, 1u);
                if (i < static_cast<uint32_t>(kPickList)) list[i] = make_key64(order_key(v[e]), static_cast<uint32_t>(wide_index<InT>(c0 + c, e)));
              }
            }
          }
        }
        raw[c].load(x, V, w.chunks, c0 + c + kAhead);
      }
    }
    if (tid == 0) {
      sh.token = kNoPick;
      sh.tie_rank = -1;
      sh.stop_lo = sh.stop_hi = V - 1;  // (all of the buckets' elements are kept)
      sh.kept_lo = kept_lo;
      sh.kept_hi = kept_hi;
    }
    __syncthreads();
    const int n_list = static_cast<int>(sh.n_list);
    ok = n_list > 0 && n_list <= kPickList;
    if (ok) {
      TokenPick pick(sh, lds_keys, exp_tab, rmax, 0u, prm, V, u, static_cast<uint32_t>(n_list));
      pick.scale = bucket_of.scale;
      pick.sub_from[1] = static_cast<float>(bucket_lo);
      pick.sub_scale[1] = static_cast<float>(kPickSubs - 1) / static_cast<float>(bucket_hi - bucket_lo + 1u);
      pick.base = em::as_double(front);
      pick.draw_before = 0;
      for (int i = tid; i < n_list; i += kWideBlock) {
        const uint32_t okey = key64_okey(list[i]);
        const float score = key_to_float(okey);
        pick.refine(1, pick.sub_of(1, score), pick.exp_of(score), okey);
      }
      __syncthreads();
      if (wave == 0) {
        u64 sum[TokenPick::kSubPer];
        const u64 run = pick.scan_subs(1, 0, sum);
        pick.resolve_draw(sum, run, n_list);
      }
      id = pick.resolved(n_list);
    }
  }
  if (tid == 0) {
    if (id != kNoPick) {
      *row_outputs(a, row).token = static_cast<int32_t>(id);
      atomicAdd(a.fallback_rows, 1u);  // (a row of the exact path, spread over the GPU)
    } else {
      give_back(false);
    }
  }
}

// The keys go to LDS in bucket order first and from there to memory, so that neighbouring lanes write neighbouring
// places (eight keys a bucket and chunk at 128256 logits).  Written straight from the registers every lane's 8 bytes
// are a line of their own: 8.3 of the 17.9 us the launch took at 16 x 128256.  ROOM: the keys LDS has room for; a chunk of more goes
// through it in several parts.
template <int BLOCK, int ROOM>
struct WideScatterShared {
  u64 keys[ROOM];
  uint32_t place[kWideBuckets];  // the bucket's next place among the chunk's keys
  uint32_t shift[kWideBuckets];  // what takes a place among these to one in the row's buffer
  uint32_t wave_sums[BLOCK / 64], wave_own[BLOCK / 64];
  u64 red64[BLOCK / 64];
};
template <typename InT, bool INLINE, bool HANDED, int BLOCK, int ROOM>
__device__ __forceinline__ void wide_scatter_chunk(const SampleArgs& a, const WideArgs& w, int row, int chunk, mi355x_sample_params prm, WideScatterShared<BLOCK, ROOM>& sh) {
  constexpr int kElems = kWideChunk / BLOCK;
  constexpr int kWords = kWideBlock / BLOCK;  // of two buckets each, a thread
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  WideRow* const info = w.rows + row;
  const uint32_t rmax = wide_row_max(a, w, row);
  if (rmax == 0xffffffffu) {
    if (chunk == 0 && tid == 0) *info = WideRow{0u, 0u, kWideDeclined, 0.0f};
    return;
  }
  float v[kElems];
  wide_load<InT, BLOCK>(static_cast<const InT*>(row_start<INLINE>(a, row, sizeof(InT))), a.vocab, chunk, v);
  // the thread's buckets: keys in the whole row, in the chunks before this one, and in this one
  uint32_t all[2 * kWords], before[2 * kWords], own[2 * kWords];
#pragma unroll
  for (int b = 0; b < 2 * kWords; ++b) all[b] = before[b] = own[b] = 0u;
  const uint32_t* h = reinterpret_cast<const uint32_t*>(a.big + static_cast<size_t>(row) * a.big_stride) + tid * kWords;
  for (int c0 = 0; c0 < w.chunks; c0 += 8) {
    uint32_t pair[8][kWords];
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int q = 0; q < kWords; ++q) pair[c][q] = c0 + c < w.chunks ? h[static_cast<size_t>(c0 + c) * kWideBlock + q] : 0u;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
#pragma unroll
      for (int q = 0; q < kWords; ++q) {
        const uint32_t n0 = pair[c][q] & 0xffffu, n1 = pair[c][q] >> 16;
        all[2 * q] += n0;
        all[2 * q + 1] += n1;
        if (c0 + c < chunk) {
          before[2 * q] += n0;
          before[2 * q + 1] += n1;
        }
        if (c0 + c == chunk) {
          own[2 * q] = n0;
          own[2 * q + 1] = n1;
        }
      }
    }
  }
  uint32_t all_sum = 0u, own_sum = 0u;
#pragma unroll
  for (int b = 0; b < 2 * kWords; ++b) {
    all_sum += all[b];
    own_sum += own[b];
  }
  const uint32_t inc = wave_prefix_sum<uint32_t>(all_sum), own_inc = wave_prefix_sum<uint32_t>(own_sum);
  if (lane == 63) {
    sh.wave_sums[wave] = inc;
    sh.wave_own[wave] = own_inc;
  }
  __syncthreads();
  const uint32_t ws = wave_prefix_sum<uint32_t>(lane < BLOCK / 64 ? sh.wave_sums[lane] : 0u), wo = wave_prefix_sum<uint32_t>(lane < BLOCK / 64 ? sh.wave_own[lane] : 0u);
  const uint32_t n = wave_read_lane(ws, BLOCK / 64 - 1), n_own = wave_read_lane(wo, BLOCK / 64 - 1);
  const uint32_t start = (wave > 0 ? wave_read_lane(ws, wave - 1) : 0u) + inc - all_sum;
  {
    uint32_t at = start, here = (wave > 0 ? wave_read_lane(wo, wave - 1) : 0u) + own_inc - own_sum;
#pragma unroll
    for (int b = 0; b < 2 * kWords; ++b) {
      sh.place[2 * kWords * tid + b] = here;
      sh.shift[2 * kWords * tid + b] = at + before[b] - here;
      at += all[b];
      here += own[b];
    }
  }
  if (chunk == 0) {
    // Tile t begins with the first bucket that starts at or after t * kWideTile: a bucket's start and the one before
    // it enclose the multiples it is the first after.  (The first bucket starts tile 0; an empty tile begins where
    // the next one does.)  A bucket of more than kWideBucketMax keys is cut at the multiples themselves, and the cut
    // remembers the bucket.
    uint32_t* const tile = w.tile_start + static_cast<size_t>(row) * (w.max_tiles + 1);
    uint2* const cut = w.cut_bucket + static_cast<size_t>(row) * (w.max_tiles + 1);
    auto enclose = [&](uint32_t prev, uint32_t at) {
      for (uint32_t t = prev / kWideTile + 1u; t <= at / kWideTile; ++t) {
        const bool inside = at - prev > static_cast<uint32_t>(kWideBucketMax) && t * kWideTile < at;
        wide_put<HANDED>(tile + t, inside ? t * kWideTile : at);
        wide_put<HANDED>(cut + t, inside ? make_uint2(prev, at) : make_uint2(0u, 0u));
      }
    };
    if (tid == 0) {
      wide_put<HANDED>(tile, 0u);
      wide_put<HANDED>(cut, make_uint2(0u, 0u));
    }
    uint32_t at = start;
#pragma unroll
    for (int b = 0; b < 2 * kWords; ++b) {  // (the start after the last bucket's is n)
      enclose(at, at + all[b]);
      at += all[b];
    }
    const uint32_t tiles = (n + kWideTile - 1u) / kWideTile;
    if (tid == 0) {
      if (n % kWideTile != 0u) {  // (where n is a multiple itself, it is enclosed above)
        wide_put<HANDED>(tile + tiles, n);
        wide_put<HANDED>(cut + tiles, make_uint2(0u, 0u));
      }
      wide_put<HANDED>(&info->n, n);
      wide_put<HANDED>(&info->tiles, tiles);
      wide_put<HANDED>(&info->declined, 0u);
      wide_put<HANDED>(&info->top, key_to_float(rmax));
    }
  }
  __syncthreads();
  const WideBuckets bucket_of(key_to_float(rmax), wide_depth(prm, a.vocab));
  u64* const keys = a.big2 + static_cast<size_t>(row) * a.big_stride;
  u64 below = 0;
  constexpr uint32_t kLeftOut = 0xffffffffu;
  uint32_t place[kElems];
#pragma unroll
  for (int e = 0; e < kElems; ++e) {
    const uint32_t b = bucket_of(v[e]);
    place[e] = kLeftOut;
    if (b < static_cast<uint32_t>(kWideBuckets)) {
      place[e] = atomicAdd(&sh.place[b], 1u);
    } else if (v[e] == v[e]) {
      const u64 k = make_key64(order_key(v[e]), static_cast<uint32_t>(wide_index<InT, BLOCK>(chunk, e)));
      below = k > below ? k : below;
    }
  }
#pragma unroll
  for (uint32_t from = 0u; from < static_cast<uint32_t>(kWideChunk); from += ROOM) {
    if (from != 0u) {
      if (n_own <= from) break;
      __syncthreads();
    }
#pragma unroll
    for (int e = 0; e < kElems; ++e)
      if (place[e] - from < static_cast<uint32_t>(ROOM))
        sh.keys[place[e] - from] = make_key64(order_key(v[e]), static_cast<uint32_t>(wide_index<InT, BLOCK>(chunk, e)));
    if (from == 0u) {
      below = block_max<u64>(below, sh.red64, false);  // (its barrier: the keys are in their places)
      if (tid == 0 && below != 0) atomicMax(reinterpret_cast<unsigned long long*>(w.best_below + row), static_cast<unsigned long long>(below));
    } else {
      __syncthreads();
    }
#pragma unroll
    for (int e = 0; e < ROOM / BLOCK; ++e) {
      const uint32_t p = static_cast<uint32_t>(e * BLOCK + tid);
      if (from + p < n_own) {
        const u64 k = sh.keys[p];
        wide_put<HANDED>(keys + (from + p + sh.shift[bucket_of(key_to_float(key64_okey(k)))]), k);
      }
    }
  }
}

typedef WideScatterShared<kWideBlock, kWideChunk> WideScatterWhole;
template <typename InT, bool INLINE>
__global__ __launch_bounds__(kWideBlock) void wide_scatter_kernel(const SampleArgs a, const typename WideTable<INLINE>::type, const WideArgs w) {
  extern __shared__ u64 lds_keys[];
  const WideShare mine = wide_share(w.chunks);
  if (mine.row >= a.rows) return;
  const mi355x_sample_params prm = row_params<INLINE>(a, mine.row);
  if (!wide_row(prm)) return;
  wide_scatter_chunk<InT, INLINE, false, kWideBlock, kWideChunk>(a, w, mine.row, mine.item, prm, *reinterpret_cast<WideScatterWhole*>(lds_keys));
}

constexpr int kWideSubBuckets = 4096;

struct WideRankShared {  // 50 KB: three workgroups a CU
  static constexpr int kWaves = kWideRankBlock / 64;
  union {
    u64 keys[kSegElems];                  // by bucket, then in rank order with the exponentials in the score half
    uint32_t first_key[kWideSubBuckets];  // while the keys are counted: the score of the first key of a bucket
  };
  uint32_t start[kWideSubBuckets + 1];
  uint32_t mixed[kWideSubBuckets / 32];  // buckets that hold more than one score
  uint64_t exp_tab[32];
  uint32_t red[kWaves], red2[kWaves];
  double dred[kWaves];
  Step wave_tot[kWaves];
  u64 low[kWaves], high[kWaves];  // a cut bucket's extremes
  uint32_t pick[2], fill;  // the selection's digit and the rank inside it; the next free place in keys
};

// The key of rank r (from 0, best first) among the m distinct keys at src, whose lowest and highest are given: a
// selection by twelve bits at a time below the bits all keys share.  (Two or three passes over the bucket: its keys
// differ in the lower bits of their scores, or in their ids alone.)  Ends with a barrier.
__device__ __forceinline__ u64 wide_select_key(const u64* src, uint32_t m, uint32_t r, u64 lowest, u64 highest, WideRankShared& sh) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int kDigitBits = 12, kPer = (1 << kDigitBits) / kWideRankBlock;
  static_assert(1 << kDigitBits == kWideSubBuckets, "the counts take the sub-buckets' place");
  int open = 64 - __clzll(static_cast<long long>(lowest ^ highest));  // bits still to be decided
  u64 prefix = open < 64 ? highest >> open : 0;
  while (open > 0) {
    const int take = open < kDigitBits ? open : kDigitBits, above = open;
    open -= take;
    for (int d = tid; d < kWideSubBuckets; d += kWideRankBlock) sh.start[d] = 0u;
    __syncthreads();
#pragma unroll 4
    for (uint32_t i = tid; i < m; i += kWideRankBlock) {
      const u64 k = src[i];
      if ((above < 64 ? k >> above : 0) == prefix) atomicAdd(&sh.start[(k >> open) & ((1u << take) - 1u)], 1u);
    }
    __syncthreads();
    uint32_t cnt[kPer], local = 0u;  // the highest digits belong to the first thread
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      cnt[j] = sh.start[kWideSubBuckets - 1 - (tid * kPer + j)];
      local += cnt[j];
    }
    const uint32_t inc = wave_prefix_sum<uint32_t>(local);
    if (lane == 63) sh.red[wave] = inc;
    __syncthreads();
    const uint32_t ws = wave_prefix_sum<uint32_t>(lane < kWideRankBlock / 64 ? sh.red[lane] : 0u);
    uint32_t before = (wave > 0 ? wave_read_lane(ws, wave - 1) : 0u) + inc - local;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      if (r >= before && r < before + cnt[j]) {
        sh.pick[0] = static_cast<uint32_t>(kWideSubBuckets - 1 - (tid * kPer + j));
        sh.pick[1] = r - before;
      }
      before += cnt[j];
    }
    __syncthreads();
    prefix = (prefix << take) | sh.pick[0];
    r = sh.pick[1];
  }
  return prefix;
}

// The keys of tile [first, first + n) of the row's list, in any order, in sh.keys, where one of its ends cuts a bucket
// (head / tail: the buckets its two ends lie inside, or zeros).  The keys of a cut bucket lie in the list in the order
// of arrival.  Where they all have one score, and nobody asks for the order of ties, any share of them will do: the one
// at the tile's own places.  Otherwise the tile takes the keys whose ranks are its places, between two keys that it
// selects from the bucket: every tile of the bucket reads all of it, 5.5 us per 1000 keys.  False, for one tile of the
// bucket at least, where that would be more than kWideSelectMax keys (a bulk of nearly one score far from outliers, a
// temperature of 40 spreads, kept ids of as many ties): the row is given back.  (Largest bucket 29 K keys: 64 x 201088
// fp32 rows of sigma 1 at T = 25 take 1014 us a step against 1154 on the exact path, 24 x 128256 at T = 40 368 against
// 602, one 208 against 537; with all of a row in one or two buckets 24 x 128256 took 1400 to 1800 against 620 to 930.)
constexpr uint32_t kWideSelectMax = 32768;
__device__ __forceinline__ bool wide_gather_cut(const u64* list, uint32_t first, uint32_t n, uint2 head, uint2 tail, bool order_ties,
                                                WideRankShared& sh) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t end = first + n;
  uint32_t done = first;  // the tile's places up to here have their keys
#pragma unroll 1
  for (int side = 0; side < 2; ++side) {  // (loops, so that the passes over a bucket are compiled once)
    const uint2 bucket = side == 0 ? head : tail;
    if (bucket.y == 0u || (side == 1 && bucket.x < done)) continue;  // (a tile inside one bucket has its only share already)
    const uint32_t from = side == 0 ? first : bucket.x, to = bucket.y < end ? bucket.y : end;
    for (uint32_t i = done + tid; i < from; i += kWideRankBlock) sh.keys[i - first] = list[i];  // the buckets between the two
    done = to;
    const u64* const src = list + bucket.x;
    const uint32_t m = bucket.y - bucket.x;
    if (m > kWideSelectMax) {  // (all of its tiles together see whether it has one score)
      int differs = order_ties ? 1 : 0;
      const uint32_t score = key64_okey(src[0]);
      for (uint32_t i = from + tid; i < to && !order_ties; i += kWideRankBlock) {
        const u64 k = list[i];
        sh.keys[i - first] = k;
        differs |= key64_okey(k) != score ? 1 : 0;
      }
      if (__syncthreads_or(differs)) return false;
      continue;
    }
    u64 highest = 0, below = 0;  // (below: complement of the lowest)
#pragma unroll 4
    for (uint32_t i = tid; i < m; i += kWideRankBlock) {
      const u64 k = src[i];
      highest = k > highest ? k : highest;
      below = ~k > below ? ~k : below;
    }
    highest = wave_max<u64>(highest);
    below = wave_max<u64>(below);
    if (lane == 0) {
      sh.high[wave] = highest;
      sh.low[wave] = below;
    }
    if (tid == 0) sh.fill = from - first;
    __syncthreads();
    highest = row16_max<u64>(lane < kWideRankBlock / 64 ? sh.high[lane] : 0);
    const u64 lowest = ~row16_max<u64>(lane < kWideRankBlock / 64 ? sh.low[lane] : 0);
    if (!order_ties && key64_okey(lowest) == key64_okey(highest)) {
      for (uint32_t i = from + tid; i < to; i += kWideRankBlock) sh.keys[i - first] = list[i];
    } else {
      u64 best = highest, last = lowest;
#pragma unroll 1
      for (int e = 0; e < 2; ++e) {
        if (e == 0 ? from == bucket.x : to == bucket.y) continue;
        const u64 key = wide_select_key(src, m, (e == 0 ? from : to - 1u) - bucket.x, lowest, highest, sh);
        if (e == 0) best = key;
        else last = key;
      }
      for (uint32_t i = tid; i < m; i += kWideRankBlock) {
        const u64 k = src[i];
        if (k <= best && k >= last) sh.keys[atomicAdd(&sh.fill, 1u)] = k;
      }
    }
    __syncthreads();
  }
  for (uint32_t i = done + tid; i < end; i += kWideRankBlock) sh.keys[i - first] = list[i];
  __syncthreads();
  return true;
}

// Sub-buckets that have to be ranked are, by comparing the keys of each, unless one holds more than this: then the tile
// is sorted by a network.  (Kept sets of 16 x 128256 bf16 rows, in order: by the network from 129 keys on and by pairs
// 190 and 188 us a step for runs of up to 270 ties, 195 and 202 for runs of up to 400, 208 and 594 for runs of 1600.)
constexpr uint32_t kWideRankCap = 256;

template <bool HANDED>
__device__ __forceinline__ void wide_rank_tile(const SampleArgs& a, const WideArgs& w, int row, int t, mi355x_sample_params prm, WideRankShared& sh) {
  constexpr int kPerThread = kSegElems / kWideRankBlock;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const WideRow* const of_row = w.rows + row;
  const WideRow info{wide_get<HANDED>(&of_row->n), wide_get<HANDED>(&of_row->tiles), wide_get<HANDED>(&of_row->declined), wide_get<HANDED>(&of_row->top)};
  if (info.declined == kWideDeclined || static_cast<uint32_t>(t) >= info.tiles) return;
  const uint32_t* const tile = w.tile_start + static_cast<size_t>(row) * (w.max_tiles + 1) + t;
  const uint32_t first = wide_get<HANDED>(tile), n = wide_get<HANDED>(tile + 1) - first;
  const u64* const keys = a.big2 + static_cast<size_t>(row) * a.big_stride;
  const uint2* const cut = w.cut_bucket + static_cast<size_t>(row) * (w.max_tiles + 1) + t;
  const uint2 head = wide_get<HANDED>(cut), tail = wide_get<HANDED>(cut + 1);
  const bool order_ties = a.kept_ids != nullptr;
  const u64* const src = keys + first;
  u64 k[kPerThread];
#pragma unroll
  for (int r = 0; r < kPerThread; ++r) {
    const uint32_t i = static_cast<uint32_t>(r * kWideRankBlock + tid);
    k[r] = i < n ? wide_get<HANDED>(src + i) : 0;
  }
  for (int b = tid; b <= kWideSubBuckets; b += kWideRankBlock) sh.start[b] = 0u;
  if (tid < kWideSubBuckets / 32) sh.mixed[tid] = 0u;
  if (tid >= 64 && tid < 96) sh.exp_tab[tid - 64] = em::exp2_tab(static_cast<uint32_t>(tid - 64));
  if (__builtin_expect((head.y | tail.y) != 0u, 0)) {  // (its code lies behind the kernel's: in line it makes every row's launch 0.7 us longer)
    // (A cut bucket's keys are read by all of its tiles, several times each: from the XCD's cache, once a wave has invalidated it.)
    if (HANDED && tid == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    __syncthreads();  // (the gather uses the table as well)
    if (!wide_gather_cut(keys, first, n, head, tail, order_ties, sh)) {
      if (tid == 0) {
        w.rows[row].declined = kWideGivenBack;
        store_sum_bits(w.tile_sum + static_cast<size_t>(row) * w.max_tiles + t, 0ull);  // (other tiles of the row wait for one)
      }
      return;
    }
#pragma unroll
    for (int r = 0; r < kPerThread; ++r) {
      const uint32_t i = static_cast<uint32_t>(r * kWideRankBlock + tid);
      k[r] = i < n ? sh.keys[i] : 0;
    }
    for (int b = tid; b <= kWideSubBuckets; b += kWideRankBlock) sh.start[b] = 0u;
  }
  uint32_t hi = 0u, lo = 0xffffffffu;
#pragma unroll
  for (int r = 0; r < kPerThread; ++r) {
    const uint32_t o = key64_okey(k[r]);
    hi = o > hi ? o : hi;
    if (k[r] != 0) lo = o < lo ? o : lo;
  }
  hi = wave_max<uint32_t>(hi);
  lo = wave_min_u32(lo);
  if (lane == 0) {
    sh.red[wave] = hi;
    sh.red2[wave] = lo;
  }
  __syncthreads();
  hi = row16_max<uint32_t>(lane < kWideRankBlock / 64 ? sh.red[lane] : 0u);
  lo = ~row16_max<uint32_t>(lane < kWideRankBlock / 64 ? ~sh.red2[lane] : 0u);
  const float top = key_to_float(hi), span = top - key_to_float(lo);
  const float scale = span > 0.0f ? static_cast<float>(kWideSubBuckets) / span : 0.0f;
  auto bucket_of = [=](u64 key) {
    float bf = (top - key_to_float(key64_okey(key))) * scale;
    bf = bf < static_cast<float>(kWideSubBuckets - 1) ? bf : static_cast<float>(kWideSubBuckets - 1);
    return bf > 0.0f ? static_cast<uint32_t>(bf) : 0u;
  };
  uint32_t slot[kPerThread];
#pragma unroll
  for (int r = 0; r < kPerThread; ++r) {
    if (k[r] != 0) {
      const uint32_t b = bucket_of(k[r]);
      slot[r] = atomicAdd(&sh.start[b], 1u);
      if (slot[r] == 0u) sh.first_key[b] = key64_okey(k[r]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kPerThread; ++r) {
    if (k[r] != 0 && slot[r] != 0u) {
      const uint32_t b = bucket_of(k[r]);
      if (sh.first_key[b] != key64_okey(k[r])) atomicOr(&sh.mixed[b >> 5], 1u << (b & 31u));
    }
  }
  bool crowded;  // some bucket holds more than kWideRankCap keys
  {  // the buckets' first places: eight consecutive buckets per thread
    constexpr int kPer = kWideSubBuckets / kWideRankBlock;
    constexpr uint32_t kCrowded = 1u << 31;
    uint32_t cnt[kPer], local = 0u, most = 0u;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      cnt[i] = sh.start[tid * kPer + i];
      local += cnt[i];
      most = cnt[i] > most ? cnt[i] : most;
    }
    const uint32_t inc = wave_prefix_sum<uint32_t>(local);
    const bool crowded_wave = __ballot(most > kWideRankCap) != 0;
    if (lane == 63) sh.red[wave] = inc | (crowded_wave ? kCrowded : 0u);
    __syncthreads();
    const uint32_t of_wave = lane < kWideRankBlock / 64 ? sh.red[lane] : 0u;
    crowded = __ballot((of_wave & kCrowded) != 0u) != 0;
    const uint32_t ws = wave_prefix_sum<uint32_t>(of_wave & ~kCrowded);
    uint32_t c = (wave > 0 ? wave_read_lane(ws, wave - 1) : 0u) + inc - local;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      sh.start[tid * kPer + i] = c;
      c += cnt[i];
    }
    if (tid == kWideRankBlock - 1) sh.start[kWideSubBuckets] = c;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kPerThread; ++r)
    if (k[r] != 0) sh.keys[sh.start[bucket_of(k[r])] + slot[r]] = k[r];
  __syncthreads();
  // Ranks, place by place (the lanes of a wave then look at the same few buckets).  A bucket of one score is in order
  // as it lies unless the ids are asked for; so are its exponentials.
  auto must_rank = [&](uint32_t b) { return order_ties || ((sh.mixed[b >> 5] >> (b & 31u)) & 1u); };
  bool by_network = false;
  if (__builtin_expect(crowded, 0)) {
    int too_full = 0;
#pragma unroll
    for (int r = 0; r < kPerThread; ++r) {
      const uint32_t p = static_cast<uint32_t>(r * kWideRankBlock + tid);
      if (p < n) {
        const uint32_t b = bucket_of(sh.keys[p]);
        if (sh.start[b + 1u] - sh.start[b] > kWideRankCap && must_rank(b)) too_full = 1;
      } else {
        sh.keys[p] = 0;
      }
    }
    by_network = __syncthreads_or(too_full) != 0;
    if (by_network) block_sort_desc(sh.keys, kSegElems);
  }
  uint32_t fin[kPerThread];
#pragma unroll
  for (int r = 0; r < kPerThread; ++r) {
    const uint32_t p = static_cast<uint32_t>(r * kWideRankBlock + tid);
    k[r] = 0;
    fin[r] = p;
    if (p < n) {
      k[r] = sh.keys[p];
      const uint32_t b = bucket_of(k[r]);
      const uint32_t s0 = sh.start[b], s1 = sh.start[b + 1u];
      if (s1 - s0 > 1u && !by_network && must_rank(b)) {
        uint32_t rank = 0u;
        for (uint32_t j = s0; j < s1; ++j) rank += sh.keys[j] > k[r] ? 1u : 0u;
        fin[r] = s0 + rank;
      }
    }
  }
  __syncthreads();
  const float inv_temp = 1.0f / prm.temperature;
  const uint64_t* const tab = sh.exp_tab;
  auto lds_tab = [=](uint32_t i) { return tab[i]; };
  double part = 0.0;
#pragma unroll
  for (int r = 0; r < kPerThread; ++r) {
    const float e = k[r] != 0 ? em::expf_core((key_to_float(key64_okey(k[r])) - info.top) * inv_temp, lds_tab) : 0.0f;
    part += static_cast<double>(e);
    sh.keys[exp_slot(fin[r])] = (static_cast<u64>(__float_as_uint(e)) << 32) | (k[r] & 0xffffffffull);  // (zeros past the tile's end)
  }
  part = wave_sum<double>(part);
  if (lane == 0) sh.dred[wave] = part;
  __syncthreads();
  const double own = wave_read_lane(row_scan_add(lane < kWideRankBlock / 64 ? sh.dred[lane] : 0.0), kWideRankBlock / 64 - 1);
  double* const sums = w.tile_sum + static_cast<size_t>(row) * w.max_tiles;
  if (tid == 0) store_sum_bits(sums + t, static_cast<unsigned long long>(__double_as_longlong(own)));
  u64* const dst = a.big + static_cast<size_t>(row) * a.big_stride + first;
#pragma unroll
  for (int r = 0; r < kPerThread; ++r) {
    const uint32_t p = static_cast<uint32_t>(r * kWideRankBlock + tid);
    if (p < n) dst[p] = sh.keys[exp_slot(p)];
  }
  // the exact sum's step record, as in seqsum_exp_step_body: the sums of the tiles before this one tell the binade
  double before = 0.0;
  bool gave_up = false;
  for (int s = tid; s < t; s += kWideRankBlock) {
    unsigned long long bits = load_sum_bits(sums + s);
    for (int spins = 0; bits == kSumNotReady && spins < a.poll_limit; ++spins) {
      __builtin_amdgcn_s_sleep(1);
      bits = load_sum_bits(sums + s);
    }
    if (bits == kSumNotReady) gave_up = true;
    else before += __longlong_as_double(static_cast<long long>(bits));
  }
  gave_up = __syncthreads_or(gave_up ? 1 : 0) != 0;
  before = wave_sum<double>(before);
  if (lane == 0) sh.dred[wave] = before;
  __syncthreads();
  before = wave_read_lane(row_scan_add(lane < kWideRankBlock / 64 ? sh.dred[lane] : 0.0), kWideRankBlock / 64 - 1);
  const size_t rec_at = static_cast<size_t>(row) * w.max_tiles + t;
  int4* const rec = w.tile_step + rec_at;
  if (gave_up) {
    if (tid < kSegSubs) w.sub_se[rec_at * kSegSubs + tid] = -1;
    if (tid == 0) {
      *rec = make_int4(0, 0, -2, 0);
      atomicAdd(a.fallback_rows + 2, 1u);
    }
    return;
  }
  float ev[kPerThread];
#pragma unroll
  for (int j = 0; j < kPerThread; ++j)
    ev[j] = __uint_as_float(static_cast<uint32_t>(sh.keys[exp_slot(static_cast<uint32_t>(tid * kPerThread + j))] >> 32));
  const float lo_f = __double2float_rd(before * (1.0 - seq_drift(static_cast<int>(first))));
  const float hi_f = __double2float_ru((before + own) * (1.0 + seq_drift(static_cast<int>(first + n))));
  const int se = seq_decompose(lo_f).se;
  const bool known = lo_f > 0.0f && hi_f < 3.0e38f && seq_decompose(hi_f).se == se;
  if (!known) {
    // powers of two may fall inside the tile: records per part of 64 elements, eight lanes each
    constexpr int kPartLanes = kWalkPart / kPerThread;
    static_assert(kPartLanes == 8 && kSegSubs * kPartLanes == kWideRankBlock, "a part is eight lanes");
    double mine = 0.0;
#pragma unroll
    for (int j = 0; j < kPerThread; ++j) mine += static_cast<double>(ev[j]);
    mine += __longlong_as_double(static_cast<long long>(lane_xor64<1>(static_cast<u64>(__double_as_longlong(mine)))));
    mine += __longlong_as_double(static_cast<long long>(lane_xor64<2>(static_cast<u64>(__double_as_longlong(mine)))));
    mine += __longlong_as_double(static_cast<long long>(lane_xor64<4>(static_cast<u64>(__double_as_longlong(mine)))));
    const int part_i = tid / kPartLanes;
    const double upto = wave_prefix_sum<double>((lane & (kPartLanes - 1)) == 0 ? mine : 0.0);
    __syncthreads();
    if (lane == 63) sh.dred[wave] = upto;
    __syncthreads();
    double start = before + upto - mine;
    for (int w = 0; w < wave; ++w) start += sh.dred[w];
    const int p_first = static_cast<int>(first) + part_i * kWalkPart;
    const float plo = __double2float_rd(start * (1.0 - seq_drift(p_first)));
    const float phi = __double2float_ru((start + mine) * (1.0 + seq_drift(p_first + kWalkPart)));
    int pse = seq_decompose(plo).se;
    const int pse_end = seq_decompose(phi).se;
    if (!(plo > 0.0f && phi < 3.0e38f && pse_end <= pse + 1)) pse = -1;  // the walk adds this part itself
    Step lo_step{0u, 0u}, hi_step{0u, 0u};
    if (pse >= 0) {
      lo_step = seq_compose_run(ev, kPerThread, pse);
      hi_step = seq_compose_run(ev, kPerThread, pse + 1);
    }
    lo_step = oct_scan_steps(lo_step);
    hi_step = oct_scan_steps(hi_step);
    if ((lane & (kPartLanes - 1)) == kPartLanes - 1) {
      const size_t at = rec_at * kSegSubs + part_i;
      w.sub_step[at] = make_int4(static_cast<int>(lo_step.d0), static_cast<int>(lo_step.d1), static_cast<int>(hi_step.d0),
                                      static_cast<int>(hi_step.d1));
      w.sub_se[at] = pse >= 0 && pse_end != pse ? pse | kPartMayCross : pse;
    }
    if (tid == 0) *rec = make_int4(0, 0, -2, 0);
    return;
  }
  const Step inc = wave_scan_steps(seq_compose_run(ev, kPerThread, se));
  if (lane == 63) sh.wave_tot[wave] = inc;
  __syncthreads();
  if (tid == 0) {
    Step s = sh.wave_tot[0];
    for (int w = 1; w < kWideRankBlock / 64; ++w) s = step_compose(s, sh.wave_tot[w]);
    *rec = make_int4(static_cast<int>(s.d0), static_cast<int>(s.d1), se, 0);
  }
}

template <bool INLINE>
__global__ __launch_bounds__(kWideRankBlock) void wide_rank_kernel(const SampleArgs a, const typename WideTable<INLINE>::type, const WideArgs w) {
  __shared__ WideRankShared sh;
  const WideShare mine = wide_share(w.max_tiles);
  if (mine.row >= a.rows) return;
  const mi355x_sample_params prm = row_params<INLINE>(a, mine.row);
  if (!wide_row(prm)) return;
  wide_rank_tile<false>(a, w, mine.row, mine.item, prm, sh);
}

// The tiles of a row as the walk reads them.
struct WideSegments {
  int segs;
  const int4* seg_step;
  const int4* sub_step;
  const int* sub_se;
  const u64* list;             // (exponential, ~id) entries in rank order
  const uint32_t* tile_start;  // LDS
  __device__ __forceinline__ int first(int sg) const { return static_cast<int>(tile_start[sg]); }
  __device__ __forceinline__ int count(int sg) const { return static_cast<int>(tile_start[sg + 1] - tile_start[sg]); }
  __device__ __forceinline__ float value(int i) const { return __uint_as_float(static_cast<uint32_t>(list[i] >> 32)); }
  __device__ __forceinline__ float load(int i) const { return value(i); }
  __device__ __forceinline__ float value_of(float loaded) const { return loaded; }
};

struct WideFinishShared {
  WalkShared walk;
  uint32_t tile_start[kWideMaxTiles + 1];
  uint2 cut_bucket[kWideMaxTiles + 1];
  float ends[kWideMaxTiles];       // the exact sequential sum behind every tile
  double weight[kWideMaxTiles];    // a tile's share of the kept weight ...
  double upto[kWideMaxTiles];      // ... and the shares of all tiles up to it
  u64 ties[kTiePairs];
  uint32_t tie_table[kTieTable];
};
static_assert(sizeof(WideFinishShared) <= kFinishLds, "the finish runs in the finish kernels' LDS");

// First position whose cumulative weight reaches u times the total, for weights w(0 .. keep) that the caller has
// summed per tile into sh.weight[0 .. used) (double).  A comparison within `band` of the total decides nothing:
// returns -1.  The last position's value is forced to one, as std::discrete_distribution forces it.
template <typename W>
__device__ __forceinline__ int wide_draw(W w, int keep, int used, double u, double band, WideFinishShared& sh, SeqShared& seqsh) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (wave == 0) {
    constexpr int kPer = kWideMaxTiles / 64;
    double s[kPer], loc = 0.0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      loc += lane * kPer + i < used ? sh.weight[lane * kPer + i] : 0.0;
      s[i] = loc;
    }
    const double before = wave_scan_add(loc) - loc;
#pragma unroll
    for (int i = 0; i < kPer; ++i) sh.upto[lane * kPer + i] = before + s[i];
  }
  __syncthreads();
  const double total = sh.upto[used - 1];
  const double target = u * total, guard = band * total;
  // the tile the target falls into, the last one if none reaches it
  int lo = 0, hi = used - 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (sh.upto[mid] >= target) hi = mid;
    else lo = mid + 1;
  }
  const int first = static_cast<int>(sh.tile_start[lo]);
  const int end = keep < static_cast<int>(sh.tile_start[lo + 1]) || lo == used - 1 ? keep : static_cast<int>(sh.tile_start[lo + 1]);
  const double base = lo > 0 ? sh.upto[lo - 1] : 0.0;
  int risky = (lo > 0 && fabs(base - target) <= guard) ? 1 : 0, found = kIntMax;
  constexpr int kPer = 5;  // a tile and the entry that may follow the last one
  static_assert(kPer * kFinishBlock > kSegElems, "a tile in one window");
  double pv[kPer], loc = 0.0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int i = first + tid * kPer + j;
    pv[j] = i < end ? w(i) : 0.0;
    loc += pv[j];
  }
  const double inc = wave_scan_add(loc);
  if (lane == 63) seqsh.dscan[wave] = inc;
  __syncthreads();
  const double ws = row_scan_add(lane < 16 ? seqsh.dscan[lane] : 0.0);
  double run = base + (wave > 0 ? wave_read_lane(ws, wave - 1) : 0.0) + (inc - loc);
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int i = first + tid * kPer + j;
    run += pv[j];
    if (i < end) {
      if (i != keep - 1 && fabs(run - target) <= guard) risky = 1;
      if ((i == keep - 1 || run >= target) && i < found) found = i;
    }
  }
  int calm = risky ? 0 : 1;
  block_min2(found, calm, seqsh);
  return calm == 0 || found == kIntMax ? -1 : found;
}

// Id of the element of rank `pos`, one of the entries run_lo .. run_lo + run of the list.  (A call of its own: inlined
// into the finish, which seldom needs it, it made every row's 1 us longer.)
__device__ __noinline__ uint32_t wide_tie_id(const u64* list, int run_lo, int run, int pos, const void* row0, int dtype, uint32_t* table) {
  const RowPtr<AnyDtype> lrow(row0, dtype);
  auto whole_key = [=](int i) {
    const uint32_t id = key64_index(list[i]);
    return make_key64(order_key(lrow[id]), id);
  };
  return block_tie_id(run, pos - run_lo, key64_okey(whole_key(pos)), [=](int i) { return whole_key(run_lo + i); }, table);
}

// The position the reference's own operations end on (block_discrete_draw's replay), run by one wave: the additions are one
// chain in the reference's order, the loads, conversions and quotients of 64 weights at a time lie beside it.  (One lane
// that loads, divides and adds in turn: 13.4 -> 1.57 ms for 128256 elements, 21.2 -> 2.4 for 201088, 0.90 -> 0.16 for 8000: 6 ns
// an element and pass.)
__device__ __noinline__ int wide_replay(const u64* list, int listed, float e_below, float scale, int keep, double u) {
  const int lane = lane_id();
  auto weight = [=](int i) {
    const float e = i < listed ? __uint_as_float(static_cast<uint32_t>(list[i < keep ? i : 0] >> 32)) : e_below;
    return i < keep ? e * scale : 0.0f;  // (what is added behind the last weight changes nothing)
  };
  double sum = 0.0;
  float w = weight(lane);
  for (int i0 = 0; i0 < keep; i0 += 64) {
    const double x = static_cast<double>(w);
    w = weight(i0 + 64 + lane);
#pragma unroll
    for (int l = 0; l < 64; ++l) sum += wave_read_lane(x, l);
  }
  double cp = 0.0;
  w = weight(lane);
  for (int i0 = 0; i0 < keep; i0 += 64) {
    const double x = static_cast<double>(w) / sum, start = cp;
    w = weight(i0 + 64 + lane);
#pragma unroll
    for (int l = 0; l < 64; ++l) cp += wave_read_lane(x, l);
    if (cp >= u) {  // one of these, or the last one, whose value is forced to one
      cp = start;
      for (int l = 0; l < 64 && i0 + l < keep - 1; ++l) {
        cp += wave_read_lane(x, l);
        if (cp >= u) return i0 + l;
      }
    }
  }
  return keep - 1;
}

// Runs by the whole workgroup; false: the row needs the exact path.
template <bool INLINE>
__device__ __forceinline__ bool wide_finish_row(const SampleArgs& a, const WideArgs& w, int row, mi355x_sample_params prm, WideFinishShared& sh, SeqShared& seqsh) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, V = a.vocab;
  const WideRow info = w.rows[row];
  if (info.declined != 0u || info.n == 0u) return false;
  const int n = static_cast<int>(info.n), tiles = static_cast<int>(info.tiles);
  const size_t rbase = static_cast<size_t>(row) * w.max_tiles;
  for (int t = tid; t <= tiles; t += kFinishBlock) {
    sh.tile_start[t] = w.tile_start[static_cast<size_t>(row) * (w.max_tiles + 1) + t];
    sh.cut_bucket[t] = w.cut_bucket[static_cast<size_t>(row) * (w.max_tiles + 1) + t];
  }
  for (int t = tid; t < tiles; t += kFinishBlock) sh.weight[t] = w.tile_sum[rbase + t];
  const u64 below = w.best_below[row];  // the best element past the list; it follows the list's last
  const u64* const list = a.big + static_cast<size_t>(row) * a.big_stride;
  const double u = a.uniforms[row];
  __syncthreads();
  const WideSegments segments{tiles, w.tile_step + rbase, w.sub_step + rbase * kSegSubs, w.sub_se + rbase * kSegSubs, list, sh.tile_start};
  walk_segments<true>(segments, sh.walk, sh.ends);
  __syncthreads();
  const float inv_temp = 1.0f / prm.temperature;
  const int limit = n + (below != 0 ? 1 : 0);
  const float e_below = below != 0 ? em::expf_exact((key_to_float(key64_okey(below)) - info.top) * inv_temp) : 0.0f;
  auto exps = [=](int i) { return i < n ? __uint_as_float(static_cast<uint32_t>(list[i] >> 32)) : e_below; };
  // the first tile the stop of FindNucleus may lie in: it lies in none whose last element misses it by a margin
  const float p = prm.p;
  const StopAtNucleus stop{p, V, 0};
  int first_tile = tiles;
  for (int t = tid; t < tiles; t += kFinishBlock) {
    const int last = static_cast<int>(sh.tile_start[t + 1]) - 1;
    const bool empty = sh.tile_start[t] == sh.tile_start[t + 1];
    if (!empty && !stop.nowhere_in_run_ending(sh.ends[t], exps(last), last) && t < first_tile) first_tile = t;
  }
  int dummy = kIntMax;
  block_min2(first_tile, dummy, seqsh);
  int base = first_tile < tiles ? static_cast<int>(sh.tile_start[first_tile]) : n;
  float prefix = first_tile > 0 ? sh.ends[first_tile - 1] : 0.0f;
  int keep;
  for (;;) {  // (the batches of the reference's search: see block_sample_epilogue)
    const int b = base;
    int si;
    prefix = block_seq_sum<8>(prefix, limit - b, [=](int i) { return exps(i + b); }, StopAtNucleus{p, V, b}, &si, seqsh, nullptr, b == 0 ? kEpiHead : 0);
    if (si < 0) {
      if (limit != V) return false;
      keep = V;
      break;
    }
    keep = b + si + 1;
    const bool batch_end = keep >= 16 && (keep & (keep - 1)) == 0 && ((__ffs(keep) - 1) & 1) == 0;
    if (!batch_end || keep >= V) break;
    if (keep >= limit) return false;
    base = keep;
  }
  const float scale = prefix > 0.0f ? 1.0f / prefix : 0.0f;
  // Where the draw falls.  The reference's weights are q_i = e_i * scale, rounded to fp32; the common factor cancels
  // and the roundings move no cumulative share by more than 2^-23, so unless the target lies within 1.3e-7 of the total
  // of a cumulative value, the exponentials' own double sums decide.  Otherwise the weights themselves are summed.
  int used = 0;  // tiles that hold kept entries
  {
    int lo = 0, hi = tiles - 1;
    while (lo < hi) {  // the tile of entry keep - 1 (the last one for the entry that follows the list)
      const int mid = (lo + hi) >> 1;
      if (static_cast<int>(sh.tile_start[mid + 1]) >= keep) hi = mid;
      else lo = mid + 1;
    }
    used = lo + 1;
  }
  int pos = 0;
  if (keep >= 2) {
    {  // the last of these tiles counts only as far as it is kept
      double part = 0.0;
      for (int i = static_cast<int>(sh.tile_start[used - 1]) + tid; i < keep; i += kFinishBlock) part += static_cast<double>(exps(i));
      part = wave_sum<double>(part);
      if (lane == 0) seqsh.dred[wave] = part;
      __syncthreads();
      if (tid == 0) {
        double s = 0.0;
        for (int w = 0; w < kFinishBlock / 64; ++w) s += seqsh.dred[w];
        sh.weight[used - 1] = s;
      }
      __syncthreads();
    }
    pos = wide_draw([=](int i) { return static_cast<double>(exps(i)); }, keep, used, u, 1.3e-7, sh, seqsh);
    if (pos < 0) {
      for (int t = wave; t < used; t += kFinishBlock / 64) {
        const int end = t == used - 1 ? keep : static_cast<int>(sh.tile_start[t + 1]);
        double s = 0.0;
#pragma unroll 4
        for (int i = static_cast<int>(sh.tile_start[t]) + lane; i < end; i += 64) s += static_cast<double>(exps(i) * scale);
        s = wave_sum<double>(s);
        if (lane == 0) sh.weight[t] = s;
      }
      __syncthreads();
      // The reference's sum and its cumulative value have `keep` roundings of 2^-53 each at most, the quotients one; here every
      // value comes from a tree of fewer than 256.  (A band of 16 keep of them takes seven times as many rows the long way, 5.8e-5 of
      // those of 128256 elements and 1.4e-4 of 201088: 0.8 and 3 us a row and step at what that took.  24 x 201088 bf16, 24 inputs of
      // which one has such a row: 1858 -> 51 us.)
      pos = wide_draw([=](int i) { return static_cast<double>(exps(i) * scale); }, keep, used, u, (2.25 * keep + 512.0) * 1.1102230246251565e-16, sh, seqsh);
      if (pos < 0) {
        if (wave == 0) {
          const int p = wide_replay(list, n, e_below, scale, keep, u);
          if (lane == 0) seqsh.bcast_i = p;
        }
        __syncthreads();
        pos = seqsh.bcast_i;
        __syncthreads();
      }
    }
  }
  const RowOutputs out = row_outputs(a, row);
  if (out.kept_count && tid == 0) *out.kept_count = keep;
  if (out.kept_ids) {
    const int kept = keep < out.kept_capacity ? keep : out.kept_capacity;
    const int lim = out.pad ? out.kept_capacity : kept;
    for (int i = tid; i < lim; i += kFinishBlock) {
      const bool in = i < kept;
      out.kept_ids[i] = in ? static_cast<int32_t>(key64_index(i < n ? list[i] : below)) : -1;
      if (out.kept_probs) out.kept_probs[i] = in ? exps(i) * scale : 0.0f;
    }
  }
  if (pos >= n) {
    if (tid == 0) *out.token = static_cast<int32_t>(key64_index(below));
    return true;
  }
  // Unless the order of ties was asked for, entries of one exponential may be ties in the order of arrival, within a tile
  // and, in a bucket that is cut, over all of its tiles: the id of the drawn rank is taken from all of these.
  if (out.kept_ids) {
    if (tid == 0) *out.token = static_cast<int32_t>(key64_index(list[pos]));
    return true;
  }
  int lo = 0, hi = tiles - 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (static_cast<int>(sh.tile_start[mid + 1]) > pos) hi = mid;
    else lo = mid + 1;
  }
  const uint2 head = sh.cut_bucket[lo], tail = sh.cut_bucket[lo + 1];
  int run_lo, run;  // the entries to choose from: as many before the first of them as elements rank before them all
  if (static_cast<int>(head.y) > pos) {
    run_lo = static_cast<int>(head.x);
    run = static_cast<int>(head.y - head.x);
  } else if (tail.y != 0u && static_cast<int>(tail.x) <= pos) {
    run_lo = static_cast<int>(tail.x);
    run = static_cast<int>(tail.y - tail.x);
  } else {
    const uint32_t mine = static_cast<uint32_t>(list[pos] >> 32);
    const int t0 = static_cast<int>(sh.tile_start[lo]), t1 = static_cast<int>(sh.tile_start[lo + 1]);
    int run_hi = kIntMax;  // minus the run's last entry
    run_lo = kIntMax;
    for (int i = t0 + tid; i < t1; i += kFinishBlock) {
      if (static_cast<uint32_t>(list[i] >> 32) == mine) {
        run_lo = i < run_lo ? i : run_lo;
        run_hi = -i < run_hi ? -i : run_hi;
      }
    }
    block_min2(run_lo, run_hi, seqsh);
    run = -run_hi - run_lo + 1;
  }
  if (run == 1) {
    if (tid == 0) *out.token = static_cast<int32_t>(key64_index(list[pos]));
    return true;
  }
  const void* const row0 = row_start<INLINE>(a, row, dtype_bytes(a.dtype));
  if (run > kTiePairs) {
    const uint32_t id = wide_tie_id(list, run_lo, run, pos, row0, a.dtype, sh.tie_table);
    if (tid == 0) *out.token = static_cast<int32_t>(id);
    return true;
  }
  const RowPtr<AnyDtype> lrow(row0, a.dtype);
  if (tid < run) {
    const uint32_t id = key64_index(list[run_lo + tid]);
    sh.ties[tid] = make_key64(order_key(lrow[id]), id);
  }
  __syncthreads();
  if (tid < run) {
    const u64 k = sh.ties[tid];
    int rank = 0;
    for (int j = 0; j < run; ++j) rank += sh.ties[j] > k ? 1 : 0;
    if (rank == pos - run_lo) *out.token = static_cast<int32_t>(key64_index(k));
  }
  return true;
}

struct WideFinishReds {
  SeqShared seq;
  uint32_t red32[16];
  u64 red64[16];
};
template <bool INLINE>
__device__ __forceinline__ void wide_finish_or_sort(const SampleArgs& a, const WideArgs& w, int row, mi355x_sample_params prm, bool exact, u64* lds, WideFinishReds& reds) {
  if (!exact && wide_finish_row<INLINE>(a, w, row, prm, *reinterpret_cast<WideFinishShared*>(lds), reds.seq)) {
    if (threadIdx.x == 0) atomicAdd(a.fallback_rows, 1u);  // (a row of the exact path, spread over the GPU)
    return;
  }
  __syncthreads();
  general_row<AnyDtype, SortWithTile, 8>(a, row, row_start<INLINE>(a, row, dtype_bytes(a.dtype)), prm, a.big + static_cast<size_t>(row) * a.big_stride, reds.seq,
                                         SortWithTile{a.big2 + static_cast<size_t>(row) * a.big_stride, lds, reds.red32, reds.red64});
}

template <bool INLINE>
__global__ __launch_bounds__(kFinishBlock) void wide_finish_kernel(const SampleArgs a, const typename WideTable<INLINE>::type, const WideArgs w) {
  extern __shared__ u64 lds_keys[];
  __shared__ WideFinishReds reds;
  int row = blockIdx.x;
  bool exact = false;
  if (w.pick != 0) {  // a row that the pick has given back
    const uint32_t sorted = *w.rest.sorted, i = blockIdx.x;
    if (i >= sorted + *w.rest.exact) return;
    exact = i >= sorted;
    row = static_cast<int>(__builtin_amdgcn_readfirstlane(w.rest.rows[exact ? static_cast<uint32_t>(a.rows) - 1u - (i - sorted) : i]));
    exact |= w.rest.gave_up[row] != 0u;
  }
  const mi355x_sample_params prm = row_params<INLINE>(a, row);
  if (!wide_row(prm)) return;
  wide_finish_or_sort<INLINE>(a, w, row, prm, exact, lds_keys, reds);
}

// What wide_scatter and wide_rank do, in one launch, for the rows that wide_pick has listed: seldom any, and then two launches that find
// nothing to do are all there is to pay, not three.  Both parts are workgroups of 512 threads of which three fit a CU (a chunk's keys go
// through LDS in two halves), in front the chunks of all listed rows, behind them their tiles, a row's all with indices of one remainder
// (see wide_share).  A tile waits for its row's chunks, whose workgroups have started before its own and wait for nothing; a wait that
// gives up leaves the row to the exact path, in the launch behind this one.  The polls are rare and a row's count has a line of memory to
// itself: 500 waiting workgroups that polled sixteen counts in one line every 0.1 us took the launch from 40 to 60 us.
// us a step, three launches behind the pick -> this one and the finish: no row given back 1 x 128256 fp32 29.3 -> 28.0, 16 x 128256 fp16
// 37.3 -> 33.9, 64 x 128256 57.6 -> 48.1, 256 x 32064 fp32 54.8 -> 46.3; one row of one given back 83.9 -> 88.9; a NaN in every row
// 16 x 128256 fp32 85.7 -> 92.8, 64 x 128256 174 -> 162, 256 x 32064 163 -> 156; near-flat rows 16 x 128256 766 -> 781, 64 x 128256
// 1166 -> 1171, 256 x 32064 425 -> 386.  The worst of 70 such batches: four rows of 128256 with open draws, 87.8 -> 100.5.
// (All in one launch of a workgroup a CU, the finish with it, is 2 to 4 us faster where nothing is given back, and up to 1.75 times as
// slow in batches of which every row is: 64 x 128256 with a NaN in each 304, near-flat 1390, 256 x 32064 286 and 604.)
constexpr int kWideRestRoom = kWideChunk / 2;
template <typename InT, bool INLINE>
__global__ __launch_bounds__(kWideRankBlock, 6) void wide_rest_kernel(const SampleArgs a, const typename WideTable<INLINE>::type, const WideArgs w) {
  __shared__ union {
    WideScatterShared<kWideRankBlock, kWideRestRoom> scatter;
    WideRankShared rank;
  } sh;
  __shared__ bool all_there;
  static_assert(3 * (sizeof(sh) + 1280) <= 160 * 1024, "three workgroups a CU");
  const int sorted = static_cast<int>(*w.rest.sorted);
  const int xcd = static_cast<int>(blockIdx.x) & 7, slot = static_cast<int>(blockIdx.x) >> 3;
  if (xcd >= sorted) return;
  const int rows = (sorted - xcd + 7) >> 3, of_chunks = rows * w.chunks;  // of the listed rows whose work has these indices
  if (slot >= of_chunks + rows * w.max_tiles) return;
  const bool ranks = slot >= of_chunks;
  const int at = ranks ? slot - of_chunks : slot, per_row = ranks ? w.max_tiles : w.chunks, i = xcd + 8 * (at / per_row), item = at % per_row;
  const int row = static_cast<int>(__builtin_amdgcn_readfirstlane(w.rest.rows[i]));
  const mi355x_sample_params prm = row_params<INLINE>(a, row);
  uint32_t* const scattered = w.rest.scattered + row * kRestStride;
  if (!ranks) {
    wide_scatter_chunk<InT, INLINE, true, kWideRankBlock, kWideRestRoom>(a, w, row, item, prm, sh.scatter);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every wave's own stores are done
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_fetch_add(scattered, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  if (threadIdx.x == 0) {
    const uint32_t chunks = static_cast<uint32_t>(w.chunks);
    uint32_t n = __hip_atomic_load(scattered, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int polls = 0; n < chunks && polls < a.poll_limit; ++polls) {
      __builtin_amdgcn_s_sleep(8);
      n = __hip_atomic_load(scattered, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    all_there = n >= chunks;
    if (n < chunks) {
      w.rest.gave_up[row] = 1u;
      store_sum_bits(w.tile_sum + static_cast<size_t>(row) * w.max_tiles + item, 0ull);  // (other tiles of the row wait for one)
      atomicAdd(a.fallback_rows + 2, 1u);
    }
  }
  __syncthreads();
  if (!all_there) return;
  wide_rank_tile<true>(a, w, row, item, prm, sh.rank);
}

template <bool INLINE>
hipError_t launch_wide(const SampleArgs& a, const typename WideTable<INLINE>::type& table, const WideArgs& w, hipStream_t stream) {
  const int rows8 = (a.rows + 7) & ~7;  // (see wide_share)
  const dim3 grid(w.chunks * rows8), block(kWideBlock);
  auto passes = [&](auto elt) {
    typedef decltype(elt) InT;
    hipLaunchKernelGGL((wide_max_kernel<InT, INLINE>), grid, block, 0, stream, a, table, w);
    hipLaunchKernelGGL((wide_count_kernel<InT, INLINE>), grid, block, 0, stream, a, table, w);
    if (w.pick != 0) {
      hipLaunchKernelGGL((wide_pick_kernel<InT, INLINE>), dim3(a.rows), block, kFinishLds, stream, a, table, w);
      hipLaunchKernelGGL((wide_rest_kernel<InT, INLINE>), dim3((w.chunks + w.max_tiles) * rows8), dim3(kWideRankBlock), 0, stream, a, table, w);
    } else {
      hipLaunchKernelGGL((wide_scatter_kernel<InT, INLINE>), grid, block, sizeof(WideScatterWhole), stream, a, table, w);
    }
  };
  if (a.dtype == MI355X_F16) passes(uint16_t{});
  else if (a.dtype == MI355X_BF16) passes(bf16_t{});
  else passes(float{});
  if (w.pick == 0) hipLaunchKernelGGL(wide_rank_kernel<INLINE>, dim3(w.max_tiles * rows8), dim3(kWideRankBlock), 0, stream, a, table, w);
  hipLaunchKernelGGL(wide_finish_kernel<INLINE>, dim3(a.rows), dim3(kFinishBlock), kFinishLds, stream, a, table, w);
  return hipGetLastError();
}

}  // namespace ms
