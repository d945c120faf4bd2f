// The walk through a row's step records (see seqsum_kernels.hip for how the records come about): a device function
// shared by the kernels that need a long row's exact sequential sum.
#pragma once
#include "kernels.h"
#include "block_seq.h"

namespace ms {

// Steps compose associatively as long as the sum stays in one binade, and where it leaves one is known in advance up
// to the few parts of 64 elements in which the estimate of the running sum straddles a power of two (kPartMayCross),
// or nothing is known about it (a negative binade: the row's first part, whose sums change binade every few
// additions).  These parts are the row's events, ten to thirty of them; everything between two events is one composed
// step, whatever its length.  So the workgroup prepares, all at the same time,
//   * for every segment that has part records, the compositions of the parts before, between and behind its events,
//     and from those and the records of the other segments one composition ahead of every event of the row;
//   * for every event and each of its 64 elements l, the composition of all that lies between the event before and
//     element l, under the event's lower binade, and of all its elements behind l, under the next one.
// The first wave then goes from event to event with the sum it holds: every lane takes the sum in front of its element,
// adds the element for real and goes on to the end of the part as if the binade were left right there; the first lane
// whose addition does leave it has the sum behind the event.  About thirty instructions an event: the wave is alone on
// its SIMD by then and issues one every ten cycles.
// Every application is checked against the binade the step holds for, which makes the result exact whatever the
// estimates were.  An event that turns out otherwise is added element by element; where a composition between events
// holds for another binade than the sum is in, the group of segments is walked by walk_group_checked.
// (The walk as one wave that scanned part records wherever it stood took 12.7 us of the 18.4 us this launch took at
// 16 x 151936, most of it chains of 64 additions for the parts that leave a binade.)
constexpr Step kStepIdentity{0u, 0u};
constexpr Step kStepLeaves{kStepSat, kStepSat};  // composed with anything, it still says "left the binade"
constexpr int kWalkWaves = 16;
constexpr int kWalkSpecials = kWalkWaves;  // segments with part records per group of 64 segments, a wave each
constexpr int kWalkEvents = 40;            // events per group
constexpr int kWalkPart = 64;              // elements of a part
static_assert(kSegSubs == 64 && kSegElems == kSegSubs * kWalkPart, "one part per lane");

struct WalkShared {
  uint2 upto[kWalkEvents][kWalkPart];    // [l]: `before` and the steps of elements 0 .. l - 1 under the event's lower binade
  uint2 behind[kWalkEvents][kWalkPart];  // [l]: the steps of elements l + 1 .. 63 under the next one
  float x[kWalkEvents][kWalkPart];
  uint2 all[kWalkEvents];                // the steps of all elements under the next binade
  uint2 before[kWalkEvents];             // everything between the event before and this one
  int2 event[kWalkEvents];               // lower binade (-1: to be added element by element), binade `before` holds for (-1: any)
  int first[kWalkEvents], count[kWalkEvents];  // the part's elements
  int led;                               // events at the row's start that are added up already ...
  float lead;                            // ... to this
  float after[kWalkEvents];              // the sum behind the event (ENDS)
  uint2 tail[kWalkSpecials];             // per segment with part records: everything behind its last event ...
  int tail_se[kWalkSpecials];            // ... the binade that holds for
  int events_of[kWalkSpecials];
};

// A row in segments of equal length (all but the last): segment sg starts at element sg * kSegElems.  Its elements are the
// exponentials of x, computed once more for the few parts that the walk looks into: written out by the launch
// that sums them they were as many bytes as the row, for one part in fifty.
template <typename InT>
struct EvenSegments {
  int segs, length;
  const int4* seg_step;  // this row's records, see SeqSumArgs
  const int4* sub_step;
  const int* sub_se;
  const InT* x;
  float max_score, inv_temp;
  const uint64_t* exp_tab;  // LDS
  __device__ __forceinline__ int first(int sg) const { return sg * kSegElems; }
  __device__ __forceinline__ int count(int sg) const { return length - sg * kSegElems < kSegElems ? length - sg * kSegElems : kSegElems; }
  __device__ __forceinline__ float load(int i) const { return load_one<InT>(x, i); }
  __device__ __forceinline__ float value_of(float loaded) const {
    const uint64_t* const tab = exp_tab;
    return em::expf_core((loaded - max_score) * inv_temp, [=](uint32_t k) { return tab[k]; });
  }
  __device__ __forceinline__ float value(int i) const { return value_of(load(i)); }
};

__device__ __forceinline__ Step step_from_below_or(Step none, Step x) {  // wave_shr:1, `none` into lane 0
  Step y;
  y.d0 = dpp_from_below_or<0x138, 0xf, uint32_t>(none.d0, x.d0);
  y.d1 = dpp_from_below_or<0x138, 0xf, uint32_t>(none.d1, x.d1);
  return y;
}

// Inclusive scan of compositions in which the lane's own step comes first and the lanes below it follow.
__device__ __forceinline__ Step wave_scan_steps_backwards(Step x) {
  x = step_compose(x, step_from_below<0x111, 0xf>(x));  // row_shr:1
  x = step_compose(x, step_from_below<0x112, 0xf>(x));  // row_shr:2
  x = step_compose(x, step_from_below<0x114, 0xf>(x));  // row_shr:4
  x = step_compose(x, step_from_below<0x118, 0xf>(x));  // row_shr:8
  x = step_compose(x, step_from_below<0x142, 0xa>(x));  // row_bcast:15 into rows 1 and 3
  x = step_compose(x, step_from_below<0x143, 0xc>(x));  // row_bcast:31 into rows 2 and 3
  return x;
}

// The additions of a wave's 64 values to s, one by one.
__device__ __forceinline__ float wave_add_chain(float s, float x) {
  return wave_read_lane(wave_serial_prefix(lane_id() == 0 ? s + x : x, 64), 63);
}

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

// One wave walks segments g0 .. g0 + g_n - 1 with scans of its own wherever it stands, and adds element by element what
// leaves the binade it is in: right for any records (r: the lane's segment record), at about ten times the cost.
// ends, when not null: the sum behind every segment.
template <typename Row>
__device__ __forceinline__ float walk_group_checked(const Row& a, float s, int g0, int g_n, int4 r, float* ends) {
  const int lane = lane_id();
  int seg = 0;  // inside the group
  while (seg < g_n) {
    const int z = wave_read_lane(r.z, seg);
    if (z != -2) {
      const int se = seq_decompose(s).se;
      const Step f = lane < seg ? kStepIdentity : (r.z == se ? Step{static_cast<uint32_t>(r.x), static_cast<uint32_t>(r.y)} : kStepLeaves);
      const int next = wave_apply_steps(s, f, seg, ends != nullptr ? seg + 1 : g_n);
      if (next > seg) {
        if (ends != nullptr && lane == 0) ends[g0 + seg] = s;
        seg = next;
        continue;
      }
    }
    const int first = a.first(g0 + seg), n = a.count(g0 + seg);
    const int n_parts = (n + kWalkPart - 1) / kWalkPart;
    int4 q = make_int4(0, 0, 0, 0);
    int pse = -1;
    if (z == -2) {
      q = a.sub_step[static_cast<size_t>(g0 + seg) * kSegSubs + lane];
      pse = a.sub_se[static_cast<size_t>(g0 + seg) * kSegSubs + lane];
      if (pse >= 0) pse &= kPartMayCross - 1;
    }
    int part = 0;
    while (part < n_parts) {
      const int pe = seq_decompose(s).se;
      Step pf = kStepLeaves;
      if (lane < part) pf = kStepIdentity;
      else if (pse >= 0 && pse == pe) pf = Step{static_cast<uint32_t>(q.x), static_cast<uint32_t>(q.y)};
      else if (pse >= 0 && pse + 1 == pe) pf = Step{static_cast<uint32_t>(q.z), static_cast<uint32_t>(q.w)};
      part = wave_apply_steps(s, pf, part, n_parts);
      if (part >= n_parts) break;
      const int np = n - part * kWalkPart < kWalkPart ? n - part * kWalkPart : kWalkPart;
      s = wave_add_chain(s, lane < np ? a.value(first + part * kWalkPart + lane) : 0.0f);
      ++part;
    }
    if (ends != nullptr && lane == 0) ends[g0 + seg] = s;
    ++seg;
  }
  return s;
}

// The exact sequential sum of a row's elements, by a workgroup of kWalkWaves waves (every thread calls; the result is
// the first wave's).  ENDS: the sum behind every segment goes to ends[segment].
template <bool ENDS, typename Row>
__device__ __forceinline__ float walk_segments(const Row& a, WalkShared& sh, float* ends) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float s = 0.0f;
  for (int g0 = 0; g0 < a.segs; g0 += 64) {  // groups of 64 segments, one per lane
    const int g_n = a.segs - g0 < 64 ? a.segs - g0 : 64;
    const int4 r = lane < g_n ? a.seg_step[g0 + lane] : make_int4(0, 0, -3, 0);
    const unsigned long long special = __ballot(lane < g_n && r.z == -2);
    const int n_special = __popcll(special);
    __syncthreads();  // the walk through the previous group is over
    // Wave w takes the w-th segment that has part records, a part per lane.
    int4 q = make_int4(0, 0, 0, 0);
    int pse = -1, sg = 0, n_parts = 0;
    unsigned long long events = 0ull;
    const bool has_segment = wave < n_special && n_special <= kWalkSpecials;
    if (has_segment) {
      unsigned long long left = special;
      for (int i = 0; i < wave; ++i) left &= left - 1ull;
      sg = g0 + __ffsll(static_cast<long long>(left)) - 1;
      q = a.sub_step[static_cast<size_t>(sg) * kSegSubs + lane];
      pse = a.sub_se[static_cast<size_t>(sg) * kSegSubs + lane];
      n_parts = (a.count(sg) + kWalkPart - 1) / kWalkPart;
      events = __ballot(lane < n_parts && (pse < 0 || (pse & kPartMayCross)));
      if (pse >= 0) pse &= kPartMayCross - 1;
    }
    if (lane == 0) sh.events_of[wave] = __popcll(events);
    __syncthreads();
    const int in_segment = sh.events_of[lane & (kWalkWaves - 1)];
    const int upto = wave_prefix_sum<int>(lane < kWalkWaves ? in_segment : 0);
    const int total = wave_read_lane(upto, 63);
    const bool fits = total <= kWalkEvents && n_special <= kWalkSpecials;
    if (fits && has_segment) {
      const int base = wave_read_lane(upto, wave) - wave_read_lane(in_segment, wave);
      const bool is_event = (events >> lane) & 1ull, real = lane < n_parts;
      // the compositions of the parts behind an event, up to every lane; a part under another binade than the one
      // below it in the same run makes the run useless (and the walk finds out)
      const int se_below = dpp_from_below_or<0x138, 0xf, int>(-1, is_event || !real ? -1 : pse);
      const bool starts = lane == 0 || ((events >> (lane - 1)) & 1ull) || is_event;
      Step f = is_event || !real ? kStepIdentity : Step{static_cast<uint32_t>(q.x), static_cast<uint32_t>(q.y)};
      if (real && !is_event && !starts && se_below != pse) f = kStepLeaves;
      int h = starts ? lane : -1;
      wave_segscan_steps(f, h);
      const Step ahead = step_from_below_or(kStepIdentity, f);
      if (is_event) {
        const int e = base + __popcll(events & ((1ull << lane) - 1ull));
        sh.before[e] = make_uint2(ahead.d0, ahead.d1);
        sh.event[e] = make_int2(pse, se_below);
        sh.first[e] = a.first(sg) + lane * kWalkPart;
        sh.count[e] = a.count(sg) - lane * kWalkPart < kWalkPart ? a.count(sg) - lane * kWalkPart : kWalkPart;
      }
      if (lane == 63) sh.tail[wave] = make_uint2(f.d0, f.d1);
      // (the last part is an event: nothing is behind it)
      const int last_se = n_parts > 0 && !((events >> (n_parts - 1)) & 1ull) ? wave_read_lane(pse, n_parts - 1) : -1;
      if (lane == 0) sh.tail_se[wave] = last_se;
    }
    __syncthreads();
    // Every event's elements and their compositions, an event per wave in turn; the first wave, meanwhile, composes
    // the segments between the events.
    Step seg_upto = kStepIdentity;  // wave 0: everything from the last event at or before this lane's segment to its end
    int seg_upto_se = -1, events_upto = 0;
    if (fits) {
      if (wave == 0) {
        const int slot = __popcll(special & ((1ull << lane) - 1ull));
        const bool is_special = (special >> lane) & 1ull;
        const int mine = is_special ? sh.events_of[slot] : 0;
        Step f = kStepIdentity;
        int se = -1;
        if (is_special) {
          f = Step{sh.tail[slot].x, sh.tail[slot].y};
          se = sh.tail_se[slot];
          if (mine == 0 && se < 0) f = kStepLeaves;  // (a segment of no parts: it would hide its neighbours' binades from each other)
        } else if (r.z >= 0) {
          f = Step{static_cast<uint32_t>(r.x), static_cast<uint32_t>(r.y)};
          se = r.z;
        }
        const bool starts = lane == 0 || mine > 0;
        const int se_below = dpp_from_below_or<0x138, 0xf, int>(-1, se);
        if (!starts && se >= 0 && se_below >= 0 && se != se_below) f = kStepLeaves;
        int h = starts ? lane : -1;
        wave_segscan_steps(f, h);
        const Step ahead = step_from_below_or(kStepIdentity, f);
        events_upto = wave_prefix_sum<int>(mine);
        if (mine > 0) {  // the segment's first event: what its own segment has before it, behind all that
          const int e = events_upto - mine;
          int2 ev = sh.event[e];
          Step own{sh.before[e].x, sh.before[e].y};
          if (ev.y >= 0 && se_below >= 0 && ev.y != se_below) own = kStepLeaves;
          const Step both = step_compose(ahead, own);
          sh.before[e] = make_uint2(both.d0, both.d1);
          if (ev.y < 0) ev.y = se_below;
          sh.event[e] = ev;
        }
        seg_upto = f;
        seg_upto_se = se;
      }
    }
    // (an event's second word and what lies before it are still wave 0's to rewrite: they are used behind the barrier)
    constexpr int kPerWave = (kWalkEvents + kWalkWaves - 1) / kWalkWaves;
    Step in_front[kPerWave];
    float loaded[kPerWave];  // (all of the wave's loads before the first is used)
#pragma unroll
    for (int i = 0; i < kPerWave; ++i) {
      const int e = wave + i * kWalkWaves;
      loaded[i] = 0.0f;
      if (fits && e < total && lane < sh.count[e]) loaded[i] = a.load(sh.first[e] + lane);
    }
#pragma unroll
    for (int i = 0; i < kPerWave; ++i) {
      const int e = wave + i * kWalkWaves;
      in_front[i] = kStepIdentity;
      if (fits && e < total) {
        const float x = lane < sh.count[e] ? a.value_of(loaded[i]) : 0.0f;
        sh.x[e][lane] = x;
        const int se = sh.event[e].x;
        if (se >= 0) {
          const float back = __shfl(x, 63 - lane, 64);
          in_front[i] = step_from_below_or(kStepIdentity, wave_scan_steps(seq_make_step(x, se)));
          const Step b = wave_scan_steps_backwards(seq_make_step(back, se + 1));  // lane l: elements 63 - l .. 63
          if (lane < 63) sh.behind[e][62 - lane] = make_uint2(b.d0, b.d1);
          else sh.all[e] = make_uint2(b.d0, b.d1);
          if (lane == 63) sh.behind[e][63] = make_uint2(0u, 0u);
        }
      }
    }
    // A row starts with parts whose sums change binade every few additions: one wave adds those up meanwhile.
    if (wave == kWalkWaves - 1 && g0 == 0) {
      int e = 0;
      float sum = 0.0f;
      auto leads = [&](int e) { return fits && e < total && sh.event[e].x < 0 && sh.first[e] == e * kWalkPart; };
      auto load_part = [&](int e) { return leads(e) && lane < sh.count[e] ? a.load(e * kWalkPart + lane) : 0.0f; };
      float next = load_part(0);
      for (; leads(e); ++e) {
        const float mine = next;
        next = load_part(e + 1);  // (on its way while these are added)
        sum = wave_add_chain(sum, lane < sh.count[e] ? a.value_of(mine) : 0.0f);
        if (ENDS && lane == 0) sh.after[e] = sum;
      }
      if (lane == 0) {
        sh.led = e;
        sh.lead = sum;
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPerWave; ++i) {
      const int e = wave + i * kWalkWaves;
      if (fits && e < total) {
        const int2 ev = sh.event[e];
        const Step both = ev.y >= 0 && ev.y != ev.x ? kStepLeaves : step_compose(Step{sh.before[e].x, sh.before[e].y}, in_front[i]);
        sh.upto[e][lane] = make_uint2(both.d0, both.d1);
      }
    }
    __syncthreads();
    if (wave != 0) continue;
    const float s_start = s;
    bool good = fits;
    if (fits) {
      // what the next event needs is read while the current one is worked on
      uint2 upto_l = make_uint2(0u, 0u), behind_l = upto_l;
      int2 ev = make_int2(-1, -1);
      float x = 0.0f;
      auto fetch = [&](int e) __attribute__((always_inline)) {
        ev = sh.event[e];
        upto_l = sh.upto[e][lane];
        behind_l = sh.behind[e][lane];
        x = sh.x[e][lane];
      };
      const int e0 = g0 == 0 ? wave_read_lane(sh.led, 0) : 0;
      if (e0 > 0) s = wave_read_lane(sh.lead, 0);
      if (e0 < total) fetch(e0);
      for (int e = e0; e < total; ++e) {
        const uint2 c_upto = upto_l, c_behind = behind_l;
        const int2 c_ev = ev;
        const float c_x = x;
        fetch(e + 1 < total ? e + 1 : e);
        // One branch: where the sum is not in the event's lower binade no lane is right, and where no addition leaves
        // it the last lane has the sum.
        const SeqState st = seq_decompose(s);
        const uint32_t n = step_apply(st.n, Step{c_upto.x, c_upto.y});  // in front of the lane's element
        const float with = seq_recompose(n, c_ev.x) + c_x;
        const SeqState next = seq_decompose(with);
        const uint32_t n2 = step_apply(next.n, Step{c_behind.x, c_behind.y});
        const bool leaves = n >= kMantLimit || next.se != c_ev.x;
        const bool right = st.se == c_ev.x && n < kMantLimit && (next.se == c_ev.x || (next.se == c_ev.x + 1 && n2 < kMantLimit));
        const unsigned long long gone = __ballot(leaves), rights = __ballot(right);
        const int j = gone != 0ull ? __ffsll(static_cast<long long>(gone)) - 1 : 63;
        if ((rights >> j) & 1ull) {
          s = wave_read_lane(leaves ? seq_recompose(n2, c_ev.x + 1) : with, j);
        } else {
          const int c_se = __builtin_amdgcn_readfirstlane(c_ev.x), c_before_se = __builtin_amdgcn_readfirstlane(c_ev.y);
          const uint2 before = sh.before[e];
          uint32_t n = st.n;
          if (c_before_se >= 0) {
            n = step_apply(n, Step{before.x, before.y});
            good = c_before_se == st.se && n < kMantLimit;
            if (!good) break;
          }
          const uint2 all = sh.all[e];
          const uint32_t n_all = step_apply(n, Step{all.x, all.y});
          if (c_se >= 0 && st.se == c_se + 1 && n_all < kMantLimit) s = seq_recompose(n_all, st.se);
          else s = wave_add_chain(seq_recompose(n, st.se), c_x);
        }
        if (ENDS && lane == 0) sh.after[e] = s;
      }
      if (good) {
        // the sum behind every segment, from the last event before its end
        const float from = ENDS ? (events_upto > 0 ? sh.after[events_upto - 1] : s_start) : s;
        const SeqState st = seq_decompose(from);
        const uint32_t n = step_apply(st.n, seg_upto);
        const bool fine = (seg_upto_se < 0 && seg_upto.d0 == 0u && seg_upto.d1 == 0u) || (seg_upto_se == st.se && n < kMantLimit);
        const bool counts = ENDS ? lane < g_n : lane == g_n - 1;
        good = __ballot(counts && !fine) == 0ull;
        const float at_end = seg_upto_se < 0 ? from : seq_recompose(n, st.se);
        if (good) {
          if (ENDS && lane < g_n) ends[g0 + lane] = at_end;
          s = wave_read_lane(at_end, g_n - 1);
        }
      }
    }
    if (!good) s = walk_group_checked(a, s_start, g0, g_n, r, ENDS ? ends : nullptr);
  }
  return s;
}

}  // namespace ms
