// The walk through a row's step records (see seqsum_kernels.hip for how the records come about): a device function
// shared by the kernels that need a long row's exact sequential sum.
#pragma once
#include "kernels.h"
#include "block_seq.h"

namespace ms {

// ---- the walk: one wave per row walks, fifteen more prepare its way ------------------------------------
// Steps compose associatively as long as the sum stays in one binade, so the walking wave does not visit the
// segments one by one: lane l takes the record of segment seg + l, the compositions over lanes are scanned, and
// every lane checks whether the sum would still be inside the binade after its segment.  All lanes before the
// first one that fails are exact; the failing segment is handled through the records of its 64 parts in the same
// way, a part that fails is added element by element (a chain of lane-shifted float additions), and the wave goes
// on behind it with the binade the sum then has.
//
// Which records compose with which is known before the sum is: a record says for which binade it holds, so the
// lanes fall into runs of equal binade, and the composition of a run from its first lane up to every lane of it
// (a scan that starts afresh at every run) does not depend on the sum.  The workgroup's other waves prepare
// these scans -- one wave for the segments' records, one per segment whose parts are needed -- and fetch the
// elements of the parts that will most likely be added one by one, all at the same time; the walking wave then
// only applies a prepared composition to the sum it holds wherever it stands at the first lane of a run in the
// binade the run expects, and falls back to a scan of its own anywhere else.
constexpr Step kStepIdentity{0u, 0u};
constexpr Step kStepLeaves{kStepSat, kStepSat};  // composed with anything, it still says "left the binade"
constexpr int kWalkSpecials = 16;                 // segments per group of 64 whose part records are cached in LDS
constexpr int kWalkWaves = 16;

// Applies the steps f (one per lane; identity below `from`, kStepLeaves where no valid record exists) to the sum
// s in lane order and returns the number of leading lanes from `from` on, below `limit`, whose results are exact;
// s becomes the sum behind the last of them.
__device__ __forceinline__ int wave_apply_steps(float& s, Step f, int from, int limit) {
  const int lane = lane_id();
  const SeqState st = seq_decompose(s);
  const Step p = wave_scan_steps(f);
  const uint32_t n2 = step_apply(st.n, p);
  const unsigned long long bad = __ballot(lane >= from && lane < limit && n2 >= kMantLimit);
  const int stop = bad != 0ull ? __ffsll(static_cast<long long>(bad)) - 1 : limit;
  if (stop > from) s = seq_recompose(wave_read_lane(n2, stop - 1), st.se);
  return stop;
}

// A prepared run: `run` composes the steps from lane `head` up to this lane; `se` is the binade they hold for
// (negative: none).  Applied to the sum s standing at lane `from`: the number of leading lanes from `from` on that
// are exact (from itself if the run does not start there or expects another binade); s moves behind them.
// *same_run: the lane it stopped at belongs to the run too, so the sum leaves the binade inside that lane's share.
__device__ __forceinline__ int wave_apply_run(float& s, uint2 run, int head, int se, int from, int limit, bool* same_run) {
  const int lane = lane_id();
  const SeqState st = seq_decompose(s);
  const uint32_t n2 = step_apply(st.n, Step{run.x, run.y});
  const bool mine = lane >= from && lane < limit && head == from && se == st.se;
  const unsigned long long in_run = __ballot(mine);
  const unsigned long long not_good = ~__ballot(mine && n2 < kMantLimit) & (~0ull << from);
  const int stop = not_good != 0ull ? __ffsll(static_cast<long long>(not_good)) - 1 : 64;
  if (stop > from) s = seq_recompose(wave_read_lane(n2, stop - 1), st.se);
  *same_run = stop < 64 && ((in_run >> stop) & 1ull) != 0ull;
  return stop;
}

// Scan of steps that starts afresh at every lane whose `se` differs from the lane's below (and at every lane
// without a valid step): the composition from the run's first lane up to each lane, and that first lane.
__device__ __forceinline__ void wave_prepare_runs(Step st, int se, uint2* run, int* head) {
  const int lane = lane_id();
  const int below = dpp_from_below_or<0x138, 0xf, int>(-4, se);  // wave_shr:1; lane 0 sees a value no lane holds
  int h = (lane == 0 || se < 0 || se != below) ? lane : -1;
  wave_segscan_steps(st, h);
  *run = make_uint2(st.d0, st.d1);
  *head = h;
}

constexpr int kWalkAhead = 8;  // parts per cached segment whose elements are fetched ahead into LDS


constexpr int kWalkPart = 64;  // elements of a part: one round of the addition chain
static_assert(kSegSubs == 64 && kSegElems == kSegSubs * kWalkPart, "one part per lane");

struct WalkShared {
  int4 part_rec[kWalkSpecials][kSegSubs];
  int part_se[kWalkSpecials][kSegSubs];
  uint2 part_run[kWalkSpecials][kSegSubs];
  unsigned char part_head[kWalkSpecials][kSegSubs];
  float ahead[kWalkSpecials][kWalkAhead][kWalkPart];
  int ahead_part[kWalkSpecials][kWalkAhead];
  uint2 seg_run[64];
  int seg_head[64];
};

// A row in segments of equal length (all but the last): segment sg starts at element sg * kSegElems.
struct EvenSegments {
  int segs, length;
  const int4* seg_step;  // this row's records, see SeqSumArgs
  const int4* sub_step;
  const int* sub_se;
  const float* e;
  __device__ __forceinline__ int first(int sg) const { return sg * kSegElems; }
  __device__ __forceinline__ int count(int sg) const { return length - sg * kSegElems < kSegElems ? length - sg * kSegElems : kSegElems; }
  __device__ __forceinline__ float value(int i) const { return e[i]; }
};

// The exact sequential sum of a row's elements, by a workgroup of kWalkWaves waves (every thread calls; the result is
// the first wave's).  ENDS: the walking wave also leaves the sum behind every segment in ends[segment].
template <bool ENDS, typename Row>
__device__ __forceinline__ float walk_segments(const Row& a, WalkShared& sh, float* ends) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float s = 0.0f;
  for (int g0 = 0; g0 < a.segs; g0 += 64) {  // groups of 64 segments, one per lane
    const int g_n = a.segs - g0 < 64 ? a.segs - g0 : 64;
    const int4 r = lane < g_n ? a.seg_step[g0 + lane] : make_int4(0, 0, -3, 0);
    const unsigned long long special = __ballot(lane < g_n && r.z == -2);
    const int n_special = __popcll(special) < kWalkSpecials ? __popcll(special) : kWalkSpecials;
    __syncthreads();  // the walk through the previous group is over
    // task 0: the runs of the segments' records; task 1 + slot: the parts of the slot-th segment that has part
    // records -- its runs and the elements of the parts that will most likely be added one by one (those whose
    // estimated binade differs from the next part's, and those without an estimate)
    for (int task = wave; task <= n_special; task += kWalkWaves) {
      if (task == 0) {
        uint2 run;
        int head;
        wave_prepare_runs(r.z >= 0 ? Step{static_cast<uint32_t>(r.x), static_cast<uint32_t>(r.y)} : kStepLeaves, r.z, &run,
                          &head);
        sh.seg_run[lane] = run;
        sh.seg_head[lane] = head;
        continue;
      }
      const int slot = task - 1;
      unsigned long long left = special;
      for (int i = 0; i < slot; ++i) left &= left - 1ull;
      const int sg = __ffsll(static_cast<long long>(left)) - 1;
      const size_t at = static_cast<size_t>(g0 + sg) * kSegSubs;
      const int sg_first = a.first(g0 + sg), sg_end = sg_first + a.count(g0 + sg);
      const int4 q = a.sub_step[at + lane];
      const int pse = a.sub_se[at + lane];
      sh.part_rec[slot][lane] = q;
      sh.part_se[slot][lane] = pse;
      const int next_se = static_cast<int>(__builtin_amdgcn_update_dpp(0u, static_cast<uint32_t>(pse), 0x130, 0xf, 0xf, false));  // wave_shl:1: the lane above
      unsigned long long want = __ballot(pse < 0 || (lane < 63 && next_se != pse));
      int pp[kWalkAhead];
      float val[kWalkAhead];
#pragma unroll
      for (int c = 0; c < kWalkAhead; ++c) {
        pp[c] = -1;
        val[c] = 0.0f;
        if (want != 0ull) {
          pp[c] = __ffsll(static_cast<long long>(want)) - 1;
          want &= want - 1ull;
          const int idx = sg_first + pp[c] * kWalkPart + lane;
          if (idx < sg_end) val[c] = a.value(idx);
        }
      }
      uint2 run;
      int head;
      wave_prepare_runs(pse >= 0 ? Step{static_cast<uint32_t>(q.x), static_cast<uint32_t>(q.y)} : kStepLeaves, pse, &run, &head);
      sh.part_run[slot][lane] = run;
      sh.part_head[slot][lane] = static_cast<unsigned char>(head);
#pragma unroll
      for (int c = 0; c < kWalkAhead; ++c) {
        if (lane == 0) sh.ahead_part[slot][c] = pp[c];
        if (pp[c] >= 0) sh.ahead[slot][c][lane] = val[c];
      }
    }
    __syncthreads();
    if (wave != 0) continue;
    const uint2 s_run = sh.seg_run[lane];
    const int s_head = sh.seg_head[lane];
    int seg = 0;  // inside the group
    while (seg < g_n) {
      bool same_run;
      // the prepared run of whole segments, if one starts here in the binade the sum is in now
      const SeqState at_seg = seq_decompose(s);
      const int ahead_seg = wave_apply_run(s, s_run, s_head, r.z, seg, g_n, &same_run);
      if (ahead_seg > seg) {
        if (ENDS && lane >= seg && lane < ahead_seg)
          ends[g0 + lane] = seq_recompose(step_apply(at_seg.n, Step{s_run.x, s_run.y}), at_seg.se);
        seg = ahead_seg;
        continue;
      }
      const int z = wave_read_lane(r.z, seg);
      if (z != -2) {
        // a segment with a record of its own that the prepared runs did not take: the scan from here
        const int se = seq_decompose(s).se;
        const Step f = lane < seg ? kStepIdentity : (r.z == se ? Step{static_cast<uint32_t>(r.x), static_cast<uint32_t>(r.y)} : kStepLeaves);
        // (where every segment's end is asked for, one segment at a time: this case is rare)
        const int next = wave_apply_steps(s, f, seg, ENDS ? seg + 1 : g_n);
        if (next > seg) {
          if (ENDS && lane == 0) ends[g0 + seg] = s;
          seg = next;
          continue;
        }
      }
      // segment `seg` part by part
      const int first = a.first(g0 + seg), n = a.count(g0 + seg);
      const int n_parts = (n + kWalkPart - 1) / kWalkPart;
      const int slot = __popcll(special & ((1ull << seg) - 1ull));
      const bool cached = z == -2 && slot < kWalkSpecials;
      int4 q = make_int4(0, 0, 0, 0);
      int pse = -1;
      uint2 p_run = make_uint2(0u, 0u);
      int p_head = -1;
      if (cached) {
        q = sh.part_rec[slot][lane];
        pse = sh.part_se[slot][lane];
        p_run = sh.part_run[slot][lane];
        p_head = sh.part_head[slot][lane];
      } else if (z == -2) {
        q = a.sub_step[static_cast<size_t>(g0 + seg) * kSegSubs + lane];
        pse = a.sub_se[static_cast<size_t>(g0 + seg) * kSegSubs + lane];
      }
      int part = 0;
      while (part < n_parts) {
        // the prepared run of parts, if one starts here in the binade the sum is in now; where it ends inside
        // its own run, the sum leaves the binade in that part
        const int ahead_part_n = wave_apply_run(s, p_run, p_head, pse, part, n_parts, &same_run);
        if (ahead_part_n > part) {
          part = ahead_part_n;
          if (part >= n_parts) break;
          if (!same_run) continue;
        } else {
          const int pe = seq_decompose(s).se;
          Step pf = kStepLeaves;
          if (lane < part) pf = kStepIdentity;
          else if (pse >= 0 && pse == pe) pf = Step{static_cast<uint32_t>(q.x), static_cast<uint32_t>(q.y)};
          else if (pse >= 0 && pse + 1 == pe) pf = Step{static_cast<uint32_t>(q.z), static_cast<uint32_t>(q.w)};
          part = wave_apply_steps(s, pf, part, n_parts);
          if (part >= n_parts) break;
        }
        // this part's elements one by one, from LDS where they were fetched ahead
        const int np = n - part * kWalkPart < kWalkPart ? n - part * kWalkPart : kWalkPart;
        const int from = first + part * kWalkPart;
        int hit = -1;
        if (cached) {
#pragma unroll
          for (int c = 0; c < kWalkAhead; ++c)
            if (sh.ahead_part[slot][c] == part) hit = c;
        }
        const float x = hit >= 0 ? sh.ahead[slot][hit][lane] : (lane < np ? a.value(from + lane) : 0.0f);
        s = wave_read_lane(wave_serial_prefix(lane == 0 ? s + x : x, 64), 63);
        ++part;
      }
      if (ENDS && lane == 0) ends[g0 + seg] = s;
      ++seg;
    }
  }
  return s;
}

}  // namespace ms
