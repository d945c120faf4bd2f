// The launch that sums a segment's exponentials and composes its step record (see seqsum_kernels.hip), as a template so
// that a caller can give the workgroups something to do while they wait for the earlier segments' sums.
#pragma once
#include "kernels.h"
#include "block_seq.h"
#include "seg_io.h"
#include "wave_select.h"

namespace ms {

// Every wave for itself: the maxima are few and in the cache, a reduction over the block would be two barriers.
__device__ __forceinline__ float row_max_of_segments(const SeqSumArgs& a, int row) {
  uint32_t m = 0u;
  for (int s = lane_id(); s < a.segs; s += 64) {
    const uint32_t k = a.seg_max[static_cast<size_t>(row) * a.segs + s];
    m = k > m ? k : m;
  }
  return key_to_float(wave_max<uint32_t>(m));
}

// expf of N arguments a lane, none of them above 88 (or else its result is not used); reached by whole waves.  Below
// -103.98 the results are zeros, as expf_in_range's are from there down to -600, so a NaN is all that needs expf's special
// cases, and the wave looks for one once: N chains of a dozen double-precision operations and a look-up then run side by
// side, where a branch per argument kept them one behind the other.
template <int N, typename Tab>
__device__ __forceinline__ void wave_expf(const float (&x)[N], Tab tab, float (&out)[N]) {
  bool nan = false;
#pragma unroll
  for (int e = 0; e < N; ++e) nan |= x[e] != x[e];
  if (__builtin_expect(__ballot(nan) == 0ull, 1)) {
#pragma unroll
    for (int e = 0; e < N; ++e) out[e] = em::expf_in_range(fmaxf(x[e], -600.0f), tab);
  } else {
#pragma unroll 1
    for (int e = 0; e < N; ++e) out[e] = em::expf_core(x[e], tab);
  }
}

// A segment sum that has not been written yet: all bits set, a NaN no sum can be (sums of exponentials are
// finite, and a NaN that came in through the logits keeps zeros in its low bits when widened to double).  The
// buffer holds this value everywhere between launches: the walk puts it back.
constexpr unsigned long long kSumNotReady = ~0ull;

__device__ __forceinline__ unsigned long long load_sum_bits(const double* p) {
  return __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_sum_bits(double* p, unsigned long long bits) {
  __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Expected relative distance between the float the reference holds after adding `count` non-negative
// terms one by one and their exact sum: roundings mostly cancel, so it grows like sqrt(count) * 2^-24
// (the worst case grows like count * 2^-24).  Only an estimate is needed: a segment classified on a
// wrong estimate fails the walk's check and is scanned.
__device__ __forceinline__ double seq_drift(int count) {
  return (8.0 * sqrt(static_cast<double>(count)) + 8.0) * 6.0e-8;
}

// Steps 2 and 3 in one launch.  A segment's workgroup computes its exponentials and publishes their double sum;
// then it waits for the sums of the row's earlier segments, which earlier workgroups of the same launch publish
// (workgroups start in index order and a row's segments are consecutive indices, so whatever a workgroup waits for
// is running or done), and goes on with its step record from the exponentials it still holds.  A wait that gives
// up only costs time: the segment is recorded as one whose parts the walk adds element by element.
//
// `between(v, seg, row)` runs, in all threads, after the sum is out and before the earlier sums are needed: work
// on the segment's elements v (as loaded: zeros past the end of the row) that would otherwise wait for a launch of
// its own.
// Bound by the chain from the loads over the exponentials, the exchange of the sums and the composition to the record, with a
// third of the time spent issuing vector instructions (two thirds with the lists of the beam search): exponentials side by side (wave_expf) and a thread's sixteen elements in a row, so that
// neither a transposition through LDS nor a copy of the exponentials in memory is needed (the walk computes the few it
// looks at once more, and takes 1 us longer), took the launch from 12.3 to 8.7 us at 16 x 151936 fp32 (9.7 MB, in the cache by
// then), with the lists of the beam search from 20.4 to 17.1 at 32 x 151936 fp16 and from 11.4 to 8.9 at 8 x 51865.
//
// FULL: the segment lies inside the row (all but a row's last segment do), so nothing has to ask where the row ends.
// `Shared` is what it needs of LDS (declared once, by the kernel, for both forms of the body).
struct NothingBetween {
  struct Shared {};
  template <bool FULL>
  __device__ __forceinline__ void run(Shared&, const float (&)[kSegPer], int, int) const {}
};

struct ExpStepShared {
  double dred[4];
  unsigned long long before;  // the sum of the segments before this one; kSumNotReady: the wait for one gave up
  uint64_t exp_tab[32];  // the table of expf in LDS: a lookup per element from constant memory is a gather
  Step wave_tot[4];
  double wave_parts[4];
};

template <typename InT, typename Between, bool FULL>
__device__ __forceinline__ void seqsum_exp_step_body(const SeqSumArgs& a, const Between& between, ExpStepShared& sh,
                                                     typename Between::Shared& between_sh) {
  double* const dred = sh.dred;
  uint64_t* const exp_tab = sh.exp_tab;
  Step* const wave_tot = sh.wave_tot;
  double* const wave_parts = sh.wave_parts;
  const int seg = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const InT* x = static_cast<const InT*>(a.x) + static_cast<size_t>(row) * a.row_stride;
  // (a thread has sixteen elements in a row: the composition below takes them in order)
  float v[kSegPer];
  seg_load_run<InT>(x, FULL ? (seg + 1) * kSegElems : a.vocab, seg, 0.0f, v);
  if (tid < 32) exp_tab[tid] = em::exp2_tab(static_cast<uint32_t>(tid));
  const float max_score = row_max_of_segments(a, row);
  if (seg == 0 && tid == 0) a.out_max[row] = max_score;
  __syncthreads();  // (the table)
  const uint64_t* const tab = exp_tab;
  auto lds_tab = [=](uint32_t i) { return tab[i]; };
  const int first = seg * kSegElems;
  float ev[kSegPer];  // zeros past the end of the row
  {
    float arg[kSegPer];
#pragma unroll
    for (int e = 0; e < kSegPer; ++e) arg[e] = (v[e] - max_score) * a.inv_temp;
    wave_expf(arg, lds_tab, ev);
  }
  double part = 0.0;
#pragma unroll
  for (int e = 0; e < kSegPer; ++e) {
    if (!FULL && seg_run_index(seg, e) >= a.vocab) ev[e] = 0.0f;
    part += static_cast<double>(ev[e]);
  }
  const double own_part = part;
  part = wave_sum<double>(part);
  if (lane == 0) dred[wave] = part;
  __syncthreads();
  const double own = (dred[0] + dred[1]) + (dred[2] + dred[3]);
  double* sums = a.seg_sum + static_cast<size_t>(row) * a.segs;
  if (tid == 0) store_sum_bits(sums + seg, static_cast<unsigned long long>(__double_as_longlong(own)));
  between.template run<FULL>(between_sh, v, seg, row);
  // the sums of the segments before this one: the first wave's to wait for
  if (wave == 0) {
    double upto = 0.0;
    bool gave_up = false;
    for (int sg = lane; sg < seg; sg += 64) {
      unsigned long long bits = load_sum_bits(sums + sg);
      for (int spins = 0; bits == kSumNotReady && spins < a.poll_limit; ++spins) {
        __builtin_amdgcn_s_sleep(1);
        bits = load_sum_bits(sums + sg);
      }
      if (bits == kSumNotReady) gave_up = true;
      else upto += __longlong_as_double(static_cast<long long>(bits));
    }
    upto = wave_sum<double>(upto);
    gave_up = __ballot(gave_up) != 0ull;
    if (lane == 0) sh.before = gave_up ? kSumNotReady : static_cast<unsigned long long>(__double_as_longlong(upto));
  }
  __syncthreads();
  const double before = __longlong_as_double(static_cast<long long>(sh.before));
  const bool gave_up = sh.before == kSumNotReady;
  const int n = FULL ? kSegElems : a.vocab - first;
  int4* rec = a.seg_step + static_cast<size_t>(row) * a.segs + seg;
  if (gave_up) {
    if (tid < kSegSubs) a.sub_se[(static_cast<size_t>(row) * a.segs + seg) * kSegSubs + tid] = -1;
    if (tid == 0) {
      *rec = make_int4(0, 0, -2, 0);
      atomicAdd(a.gave_up, 1u);
    }
    return;
  }
  const double lo = before * (1.0 - seq_drift(first));
  const double hi = (before + own) * (1.0 + seq_drift(first + n));
  const float lo_f = __double2float_rd(lo), hi_f = __double2float_ru(hi);
  const int se = seq_decompose(lo_f).se;
  const bool known = lo_f > 0.0f && hi_f < 3.0e38f && seq_decompose(hi_f).se == se;
  if (!known) {
    // Powers of two may fall inside the segment.  Each of its 64-element parts (four lanes of sixteen elements)
    // estimates the binade the sum has where the part begins, from the double sums of the parts before it, and
    // gets a composed step under that binade and one under the next: the walk applies the one that matches the
    // sum it holds, and adds a part element by element where the sum leaves its binade inside the part or the
    // estimate was wrong.
    constexpr int kPart = kSegElems / kSegSubs;
    static_assert(kPart == 4 * kSegPer && kSegBlock == kSegSubs * 4, "a part is four lanes");
    double mine = own_part;
    mine += __longlong_as_double(static_cast<long long>(lane_xor64<1>(static_cast<u64>(__double_as_longlong(mine)))));
    mine += __longlong_as_double(static_cast<long long>(lane_xor64<2>(static_cast<u64>(__double_as_longlong(mine)))));
    // (all four lanes of a part hold its sum)
    const int part_i = tid >> 2;
    // the sum of the parts before this one: a prefix over the wave's sixteen parts and the totals of the waves before
    const double upto = wave_prefix_sum<double>((lane & 3) == 0 ? mine : 0.0);
    if (lane == 63) wave_parts[wave] = upto;
    __syncthreads();
    double start = before;
    for (int w = 0; w < wave; ++w) start += wave_parts[w];
    start += upto - mine;
    const int p_first = first + part_i * kPart;
    const float plo = __double2float_rd(start * (1.0 - seq_drift(p_first)));
    const float phi = __double2float_ru((start + mine) * (1.0 + seq_drift(p_first + kPart)));
    int pse = seq_decompose(plo).se;
    const int pse_end = seq_decompose(phi).se;
    if (!(plo > 0.0f && phi < 3.0e38f && pse_end <= pse + 1)) pse = -1;  // the walk adds this part itself
    Step lo_step{0u, 0u}, hi_step{0u, 0u};
    if (pse >= 0) {
      lo_step = seq_compose_run(ev, kSegPer, pse);
      hi_step = seq_compose_run(ev, kSegPer, pse + 1);
    }
    lo_step = quad_scan_steps(lo_step);
    hi_step = quad_scan_steps(hi_step);
    if ((lane & 3) == 3) {
      const size_t at = (static_cast<size_t>(row) * a.segs + seg) * kSegSubs + part_i;
      a.sub_step[at] = make_int4(static_cast<int>(lo_step.d0), static_cast<int>(lo_step.d1), static_cast<int>(hi_step.d0),
                                 static_cast<int>(hi_step.d1));
      a.sub_se[at] = pse >= 0 && pse_end != pse ? pse | kPartMayCross : pse;
    }
    if (tid == 0) *rec = make_int4(0, 0, -2, 0);
    return;
  }
  const Step agg = seq_compose_run(ev, kSegPer, se);
  const Step inc = wave_scan_steps(agg);
  if (lane == 63) wave_tot[wave] = inc;
  __syncthreads();
  if (tid == 0) {
    Step t = wave_tot[0];
    for (int w = 1; w < 4; ++w) t = step_compose(t, wave_tot[w]);
    *rec = make_int4(static_cast<int>(t.d0), static_cast<int>(t.d1), se, 0);
  }
}

template <typename InT, typename Between>
__global__ __launch_bounds__(kSegBlock) void seqsum_exp_step_kernel(const SeqSumArgs a, const Between between) {
  __shared__ ExpStepShared sh;
  __shared__ typename Between::Shared between_sh;
  if ((static_cast<int>(blockIdx.x) + 1) * kSegElems <= a.vocab)
    seqsum_exp_step_body<InT, Between, true>(a, between, sh, between_sh);
  else
    seqsum_exp_step_body<InT, Between, false>(a, between, sh, between_sh);
}

}  // namespace ms
