// The token of a nucleus row (k <= 1, 0 < p < 1) whose kept set nobody asks for, without sorting the row.
//
// Which token a draw lands on takes the order of the elements at two places only: around the stop of FindNucleus and
// around the draw's target.  So the candidates' exponentials go into a histogram of masses over buckets that are linear
// in the score, a scan of it says which bucket or two hold the stop and which the target, and a second look at the
// candidates spreads those buckets over finer ones, where one wave finds the stop and another the token.  What the
// reference computes in fp32 in sequence is bounded:
//
//  * Its running sum s_i differs from the exact sum S_i of the exponentials by its roundings.  While the sum is in the
//    binade of unit U, adding e moves it by e/U rounded to an integer, whatever its value is -- unless e/U lies half way
//    between two, where the sum's parity decides.  The second look adds these roundings up (R), so s_i = S_i + R up to
//    U for each tie and U/2 for each element of a bucket in which the sum may change its binade: a few dozen units, where
//    the roundings' bound alone would be n/2 of them and leave the stop of a long nucleus open.
//  * The stop test s_i >= p * (s_i + (V - i - 1) * e_i) is off by its own three roundings.
//  * The weights of the draw are the exponentials times one factor, rounded: a share x moves by at most
//    x (1 - x) 2^-23.
//
// Where these bounds leave more than one token, the row is given back (kNoPick) and the caller sorts it: 0.02 to 0.1 % of
// rows of 3000 to 10000 candidates, most of them for the last of the three.
//
// One workgroup per row is bound by vector issue and by the phases between its barriers.  Sorting 7000 candidates took three
// passes over them, an exponential each, and two exact sums; picking takes two looks and eight barriers.  Finish kernels:
// 32 x 151936 bf16, p = 0.9: 27.3 -> 22.6 us (2.9 until the lists are there, 1.3 to move candidates together, 2.6 to count
// them, 4.4 for find(), 3 for the second look, 5 for resolve()), 48 x 50257 fp16 in several modes: 42.5 -> 26.6;
// 256 x 201088 fp32 under a mask of 5 %: 59.2 -> 50.5 a step, of which the gather is 35.  64 x 128256 fp32 N(0, 5^2): 40.0 ->
// 33.5 a step; 8 x 201088 bf16, T = 0.7, whose ties the sort gave to the exact path: 1530 -> 60.
#pragma once
#include "block_seq.h"

namespace ms {

constexpr uint32_t kNoPick = 0xffffffffu;
constexpr int kPickBlock = 1024;
constexpr int kPickBuckets = kPickBlock;  // a bucket per thread
constexpr int kPickSubs = 512;            // finer buckets of each of the two places, eight per lane of a wave
constexpr int kPickHits = 512;            // keys of those buckets a wave may meet
constexpr int kPickList = 8192;           // keys the draw's may hold
constexpr int kPickRoom = kPickHits * kPickBlock / 64 + kPickList;

struct PickShared {
  u64 table[kPickBuckets + 1];  // candidates << shift | mass; then 1 / U of the running sum in a bucket, as a float, or 0
                            // where the sum may change its binade
  struct Sub {
    u64 sum[kPickSubs];  // as in table
    uint32_t tag_max[kPickSubs], tag_min[kPickSubs];  // of the elements: exponentials (as bits), order keys of the scores
  } sub[2];  // of the stop, of the draw
  float sub_rounding[kPickSubs];  // of the stop: what adding the elements rounds by
  struct Firsts {
    int a[16], b[16];
    u64 va[16], vb[16];
  } firsts[2];
  u64 sums[16];
  uint32_t below[16];
  float rounding[16], slack[16];
  uint32_t n_list;
  int stop_lo, stop_hi;
  double kept_lo, kept_hi;
  uint32_t token;
  int tie_rank;
  uint32_t tie_okey;
  u64 last[64];  // the keys of the finer bucket the draw falls into
};
static_assert(kTieTable * sizeof(uint32_t) <= sizeof(PickShared::table), "the ties' table lies over the buckets'");

// The first threads of the block that satisfy a and b, each with what it says beside it (kIntMax: none does).  One
// barrier; the caller alternates between two `sh`.
__device__ __forceinline__ void block_firsts(bool a, u64& va, int& first_a, bool b, u64& vb, int& first_b, PickShared::Firsts& sh) {
  const int lane = lane_id(), wave = threadIdx.x >> 6;
  const int la = first_lane(__ballot(a)), lb = first_lane(__ballot(b));
  if (lane == la) sh.va[wave] = va;
  if (lane == lb) sh.vb[wave] = vb;
  if (lane == 0) {
    sh.a[wave] = la;
    sh.b[wave] = lb;
  }
  __syncthreads();
  const int xa = lane < 16 ? sh.a[lane] : -1, xb = lane < 16 ? sh.b[lane] : -1;
  const int wa = first_lane(__ballot(xa >= 0)), wb = first_lane(__ballot(xb >= 0));
  first_a = wa < 0 ? kIntMax : wa * 64 + wave_read_lane(xa, wa & 15);
  first_b = wb < 0 ? kIntMax : wb * 64 + wave_read_lane(xb, wb & 15);
  va = sh.va[wa & 15];
  vb = sh.vb[wb & 15];
}

// One row, one workgroup of kPickBlock threads.  Use: clear() | barrier | count() every candidate, any order | find() |
// gather() every candidate | resolve().
struct TokenPick {
  PickShared& sh;
  u64* const hits;  // LDS, kPickRoom words free from find() on: the keys of the two places that the wave has met ...
  u64* const list;  // ... and all those of the draw's
  const uint64_t* const exp_tab;  // LDS: em::exp2_tab
  const mi355x_sample_params prm;
  const int V;
  const double u;
  const float top;
  float scale;  // bucket = (top - score) * scale, within 0 .. kPickBuckets - 1
  const float inv_temp;
  const int shift;  // of the counts in a word; the mass below them has `frac` fractional bits
  const int frac;
  const double quant;  // what the masses' rounding may amount to

  // what find() leaves behind: the buckets of the stop and of the draw, and the (count, mass) in front of them
  int stop_lo, stop_hi, draw_lo, draw_hi;
  u64 stop_before, stop_end, draw_before;  // (stop_end: in front of stop_hi, whose first element is the last that may be the stop)
  double mass_end;  // the mass up to that element at most
  float e_end, e_end_low;  // its exponential at most and at least
  bool ends_in_zero = false;  // it is the first one of no weight
  float sub_from[2], sub_scale[2];
  double base = 0.0;  // mass in front of what the words count
  // the thread's share
  float rounding = 0.0f, slack = 0.0f;
  int n_hits = 0;  // the wave's

  // Whether picking is worth a try for one of `rows` rows of n candidates each: what it leaves open grows with the nucleus
  // twice, in the shares a draw may meet and in the roundings of a bucket in which the running sum changes its binade, and
  // one row that has to be sorted after all makes the launch longer by the sort.  Given back: 0.02 to 0.1 % of rows of 3000
  // to 13000 candidates, 1 to 3 % of flatter ones (16 x 128256 fp32 N(0, 3^2), T = 0.8, p = 0.9: 1.0 %, 48 us picked and 63
  // sorted; N(0, 4^2), p = 0.95: 1.7 %, 48 and 87), 6 % of N(0, 3^2), T = 1 (68 and 135: the line), 37 % of the 110000
  // candidates of N(0, 2^2) (105 and 252).
  __device__ static __forceinline__ bool worth_it(int rows, uint32_t n) {
    return static_cast<float>(rows) * static_cast<float>(n) * static_cast<float>(n) < 4e10f;
  }

  // rtop, thr: order keys of the row's maximum and of the lowest candidate; n: at least the number of candidates,
  // 1 <= n < 2^20 (they and the element below them take b bits, the mass at most b before its point)
  __device__ __forceinline__ TokenPick(PickShared& sh_, u64* room, const uint64_t* exp_tab_, uint32_t rtop, uint32_t thr, mi355x_sample_params prm_, int V_,
                                       double u_, uint32_t n)
      : sh(sh_), hits(room + (threadIdx.x >> 6) * kPickHits), list(room + kPickHits * (kPickBlock / 64)), exp_tab(exp_tab_), prm(prm_), V(V_), u(u_), top(key_to_float(rtop)),
        scale(rtop > thr ? static_cast<float>(kPickBuckets) / (key_to_float(rtop) - key_to_float(thr)) : 0.0f), inv_temp(1.0f / prm_.temperature),
        shift(__clz(static_cast<int>(n + 1u)) + 32), frac(2 * __clz(static_cast<int>(n + 1u)) < 44 ? 2 * __clz(static_cast<int>(n + 1u)) : 44),
        quant(static_cast<double>(n) * ldexp(0.5, -frac)) {}

  __device__ static __forceinline__ void clear(PickShared& sh) {
    const int t = threadIdx.x;
    sh.table[t] = 0;
    if (t == 0) sh.table[kPickBuckets] = 0;
    sh.sub[t / kPickSubs].sum[t % kPickSubs] = 0;
    sh.sub[t / kPickSubs].tag_max[t % kPickSubs] = 0u;
    sh.sub[t / kPickSubs].tag_min[t % kPickSubs] = 0xffffffffu;
    if (t < kPickSubs) sh.sub_rounding[t] = 0.0f;
    if (t == 0) sh.n_list = 0u;
  }

  __device__ __forceinline__ float exp_of(float score) const {
    const uint64_t* const tab = exp_tab;
    return em::expf_in_range((score - top) * inv_temp, [=](uint32_t i) { return tab[i]; });
  }
  __device__ __forceinline__ int bucket_of(float score) const {
    const float b = (top - score) * scale;
    return static_cast<int>(b < static_cast<float>(kPickBuckets - 1) ? b : static_cast<float>(kPickBuckets - 1));
  }
  // The word that counts one element of exponential e (at most 1): its mass is rounded to 2^-frac by adding it to 2^52.
  __device__ __forceinline__ u64 word_of(float e) const {
    return em::as_u64(fma(static_cast<double>(e), ldexp(1.0, frac), 0x1p52)) - em::as_u64(0x1p52) + (1ull << shift);
  }
  __device__ __forceinline__ double mass_of(u64 x) const { return ldexp(static_cast<double>(x & ((1ull << shift) - 1ull)), -frac); }
  __device__ __forceinline__ int count_of(u64 x) const { return static_cast<int>(x >> shift); }

  __device__ __forceinline__ void count(float score, float e) const {
    atomicAdd(reinterpret_cast<unsigned long long*>(&sh.table[bucket_of(score)]), static_cast<unsigned long long>(word_of(e)));
  }

  // How far G = S (1 - p) - p T, T = (V - i - 1) e, may be from what decides the reference's test, when its running sum
  // is off by at most `eps`.
  __device__ __forceinline__ double stop_error(double s, double t, double eps) const {
    return (1.0 - static_cast<double>(prm.p)) * (eps + quant) + 6.03e-8 * static_cast<double>(prm.p) * (2.0 * s + 3.0 * t);
  }
  __device__ __forceinline__ double draw_guard(double kept, double n) const {
    return kept * (u * (1.0 - u) * 1.21e-7 + 16.0 * 1.2e-16 * n + 1e-11) + 2.0 * quant;
  }
  // Half the unit of a running sum of c elements near s.
  __device__ __forceinline__ float half_unit(double s, int c) const {
    const uint32_t field = __float_as_uint(static_cast<float>(s * (1.0 + static_cast<double>(c + 4) * 6.0e-8))) >> 23;
    return __uint_as_float((field - 24u) << 23);
  }

  // below: the highest score this thread knows of an element that is no candidate (-inf: of none); zero_below: elements of
  // no weight follow these.  False (for every
  // thread): no stop for certain, or the draw may fall behind the candidates.
  __device__ __forceinline__ bool find(float below, bool zero_below = false) {
    const int t = threadIdx.x, lane = lane_id(), wave = t >> 6;
    const float step = scale > 0.0f ? inv_temp / scale : 0.0f;  // exponent per bucket
    const uint32_t best_below = wave_max<uint32_t>(order_key(below));
    if (lane == 0) sh.below[wave] = best_below;
    __syncthreads();  // (and every candidate is counted)
    const u64 own = sh.table[t];
    const u64 inc = wave_prefix_sum<u64>(own);
    if (lane == 63) sh.sums[wave] = inc;
    __syncthreads();
    u64 waves = lane < 16 ? sh.sums[lane] : 0;
    waves += dpp_from_below_or<0x111, 0xf, u64>(0, waves);
    waves += dpp_from_below_or<0x112, 0xf, u64>(0, waves);
    waves += dpp_from_below_or<0x114, 0xf, u64>(0, waves);
    waves += dpp_from_below_or<0x118, 0xf, u64>(0, waves);
    const u64 all = wave_read_lane(waves, 15);
    const u64 before = (wave > 0 ? wave_read_lane(waves, wave - 1) : 0) + inc - own, upto = before + own;
    // G never decreases along the row.  stop_lo: the first bucket that may hold the stop, stop_hi: the first one at whose
    // first element the search stops for certain.  An exponential of bucket b lies between exp(-(b + 1) step) and
    // exp(-b step); 2^-9 of every term is to spare, for these and for the fp32 arithmetic here, and what the running sum
    // and the test may be off by comes on top (2^-24 of the sum for each element, see stop_error).
    bool may = false, sure = false;
    if (own != 0) {
      const float rest = 1.0f - prm.p, s0 = static_cast<float>(mass_of(before)), s1 = static_cast<float>(mass_of(upto));
      const float c0 = static_cast<float>(count_of(before)), c1 = static_cast<float>(count_of(upto));
      const float tail_end = (static_cast<float>(V) - c1) * __expf(-step * static_cast<float>(t + 1)) * prm.p;
      const float tail_top = (static_cast<float>(V) - c0) * __expf(-step * static_cast<float>(t)) * prm.p;
      const float drift = (c1 + 4.0f) * 6.1e-8f, test = 3e-7f * s1, slop = static_cast<float>(quant);
      may = !(s1 * rest * (1.002f + drift) + test + slop < tail_end * 0.998f);
      sure = s0 * rest * (0.998f - drift) - test - slop > tail_top * 1.002f;
      const uint32_t from = __float_as_uint(s0 * (1.0f - drift - 3e-7f)) >> 23, to = __float_as_uint(s1 * (1.0f + drift + 3e-7f)) >> 23;
      reinterpret_cast<float*>(sh.table)[2 * t] = from == to ? __uint_as_float((277u - from) << 23) : 0.0f;  // sums of exponent field f: U = 2^(f - 150)
      if (from != to) slack = static_cast<float>(count_of(own)) * __uint_as_float((to - 24u) << 23);  // half a unit each
    }
    u64 v_lo = before, v_hi = before;
    block_firsts(may, v_lo, stop_lo, sure, v_hi, stop_hi, sh.firsts[0]);
    stop_before = stop_lo == kIntMax ? all : v_lo;  // (kIntMax: the element below the candidates alone)
    if (t >= stop_hi) slack = 0.0f;
    stop_end = stop_hi == kIntMax ? all : v_hi;
    e_end = __expf(-step * static_cast<float>(stop_hi)) * 1.001f;
    e_end_low = __expf(-step * (static_cast<float>(stop_hi) + 1.0f)) * 0.999f;
    float e_below = 0.0f;
    if (stop_hi == kIntMax) {  // the candidates may end before the nucleus does
      const uint32_t okey = row16_max<uint32_t>(lane < 16 ? sh.below[lane] : 0u);
      if (okey > order_key(-1e30f)) {
        // (Nothing says how far below it lies, exp_of is for what a candidate can be: from -104 on a zero, which leaves the stop open.)
        const float score = key_to_float(okey);
        e_below = (score - top) * inv_temp > -103.9f ? exp_of(score) : 0.0f;
      } else if (zero_below) ends_in_zero = true;  // (there at the latest: nothing of weight follows)
      else if (count_of(all) != V) return false;
      e_end = e_below;
      e_end_low = 0.0f;
    }
    mass_end = mass_of(stop_end) + static_cast<double>(e_end);
    // the buckets the draw's target may fall into
    const double guard = draw_guard(mass_end, static_cast<double>(count_of(all) + 1));
    const u64 t_lo = word_mass(u * mass_of(stop_before) - guard), t_hi = word_mass(u * mass_end + guard) + 1, mass = upto & ((1ull << shift) - 1ull);
    u64 v_d = before, v_unused = 0;
    block_firsts(own != 0 && mass >= t_lo, v_d, draw_lo, own != 0 && mass >= t_hi, v_unused, draw_hi, sh.firsts[1]);
    draw_before = v_d;
    if (draw_hi == kIntMax) return false;
    auto spread = [&](int place, int from, int to) {  // (buckets from .. to - 1; the last finer one is that of the element below the candidates)
      sub_from[place] = static_cast<float>(from);
      sub_scale[place] = static_cast<float>(kPickSubs - 1) / static_cast<float>((to < kPickBuckets ? to : kPickBuckets) - from);
    };
    spread(0, stop_lo, stop_hi);
    spread(1, draw_lo, draw_hi + 1);
    if (t == 0 && e_below != 0.0f) refine(0, kPickSubs - 1, e_below, __float_as_uint(e_below));
    return true;
  }
  // A mass as the words hold it, rounded down (0 for less than nothing).
  __device__ __forceinline__ u64 word_mass(double x) const { return x > 0.0 ? static_cast<u64>(ldexp(x, frac)) : 0; }

  __device__ __forceinline__ void refine(int place, int at, float e, uint32_t tag) const {
    PickShared::Sub& s = sh.sub[place];
    atomicAdd(reinterpret_cast<unsigned long long*>(&s.sum[at]), static_cast<unsigned long long>(word_of(e)));
    atomicMax(&s.tag_max[at], tag);
    atomicMin(&s.tag_min[at], tag);
  }
  // The finer bucket of a score in one of the place's buckets (a monotone map, as bucket_of is).
  __device__ __forceinline__ int sub_of(int place, float score) const {
    const float x = ((top - score) * scale - sub_from[place]) * sub_scale[place];
    return static_cast<int>(x < static_cast<float>(kPickSubs - 2) ? fmaxf(x, 0.0f) : static_cast<float>(kPickSubs - 2));
  }
  __device__ __forceinline__ void append(u64 key) const {
    const uint32_t at = atomicAdd(&sh.n_list, 1u);
    if (at < static_cast<uint32_t>(kPickList)) list[at] = key;
  }

  // What rounding e to a whole number of units (of 1 / per_unit) adds; a tie to the even one, but the sum's parity may ask
  // for the other: `open` grows by a unit.  Where the binade is not known the factor is 0, and so is all of this.
  __device__ __forceinline__ float rounding_of(float e, float per_unit, float& open) const {
    const float x = e * per_unit, r = __builtin_rintf(x) - x;
    const float unit = __uint_as_float(0x7f000000u - __float_as_uint(per_unit));
    open += fabsf(r) == 0.5f ? unit : 0.0f;
    return r * unit;
  }

  // The second look at N candidates (raw: score bits, complement of the id; e: the exponential).  Reached by whole waves;
  // have: the lane has one.  A wave puts its keys of the two places aside: one in twenty or fewer is of them, but nearly
  // every wave has one at each call, and would run through what is to be done for it.
  template <int N>
  __device__ __forceinline__ void gather(const bool (&have)[N], const u64 (&raw)[N], const float (&e)[N]) {
    int b[N];
    float per_unit[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      b[i] = bucket_of(__uint_as_float(static_cast<uint32_t>(raw[i] >> 32)));
      b[i] = have[i] ? b[i] : kPickBuckets;  // (whose place behind the table holds no factor that is used)
      per_unit[i] = reinterpret_cast<const float*>(sh.table)[2 * b[i]];
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      rounding += rounding_of(have[i] ? e[i] : 0.0f, b[i] < stop_lo ? per_unit[i] : 0.0f, slack);
      const bool hit = (b[i] >= stop_lo && b[i] < stop_hi) ||
                       static_cast<uint32_t>(b[i] - draw_lo) <= static_cast<uint32_t>(draw_hi - draw_lo);
      const u64 lanes = __ballot(hit && have[i]);
      if (lanes != 0) {
        const int at = static_cast<int>(__builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(lanes >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(lanes), n_hits)));
        if (hit && have[i] && at < kPickHits) hits[at] = raw[i];
        n_hits += static_cast<int>(__popcll(lanes));
      }
    }
  }
  // Once every candidate has been looked at twice.
  __device__ __forceinline__ void refine_hits() {
    const int n = n_hits < kPickHits ? n_hits : kPickHits;
    for (int i = lane_id(); i < n; i += 64) {
      const u64 raw = hits[i];
      const float score = __uint_as_float(static_cast<uint32_t>(raw >> 32)), e = exp_of(score);
      const int b = bucket_of(score);
      if (b >= stop_lo && b < stop_hi) {
        const int at = sub_of(0, score);
        refine(0, at, e, __float_as_uint(e));
        atomicAdd(&sh.sub_rounding[at], rounding_of(e, reinterpret_cast<const float*>(sh.table)[2 * b], slack));
      }
      if (b >= draw_lo && b <= draw_hi) {
        const uint32_t okey = order_key(score);
        refine(1, sub_of(1, score), e, okey);
        append((static_cast<u64>(okey) << 32) | (raw & 0xffffffffull));
      }
    }
    if (n_hits > kPickHits && lane_id() == 0) atomicAdd(&sh.n_list, static_cast<uint32_t>(kPickList) + 1u);  // (the row is given back)
  }

  // A wave's scan of a place's finer buckets: those of this lane and what lies in front of them.
  static constexpr int kSubPer = kPickSubs / 64;
  __device__ __forceinline__ u64 scan_subs(int place, u64 before, u64 (&sum)[kSubPer]) const {
    u64 local = 0;
#pragma unroll
    for (int i = 0; i < kSubPer; ++i) {
      sum[i] = sh.sub[place].sum[lane_id() * kSubPer + i];
      local += sum[i];
    }
    return before + wave_prefix_sum<u64>(local) - local;
  }

  // Wave 0: the first element the search may stop at and the first one it stops at for certain, with the mass kept.
  __device__ __forceinline__ void resolve_stop() const {
    const int lane = lane_id();
    const double p = static_cast<double>(prm.p), rest = 1.0 - p;
    const double off = static_cast<double>(wave_sum<float>(lane < 16 ? sh.rounding[lane] : 0.0f));
    const double open = static_cast<double>(wave_sum<float>(lane < 16 ? sh.slack[lane] : 0.0f)) * 1.0001;
    const PickShared::Sub& subs = sh.sub[0];
    const int first_at = count_of(stop_before);
    // (what the roundings leave open, their ties and binades, and what adding them up in fp32 may have lost)
    const double eps = open + static_cast<double>(half_unit(mass_end, first_at + 1)) * (1.0 + static_cast<double>(count_of(stop_end)) * 1e-5);
    // every lane's run of finer buckets first: where the stop cannot lie yet, where it has certainly been
    u64 sum[kSubPer];
    const u64 run = scan_subs(0, stop_before, sum);
    u64 end = run;
    uint32_t top_bits = 0u, low_bits = 0xffffffffu;
    float local = 0.0f;
#pragma unroll
    for (int i = 0; i < kSubPer; ++i) {
      end += sum[i];
      top_bits = max(top_bits, subs.tag_max[lane * kSubPer + i]);
      low_bits = min(low_bits, subs.tag_min[lane * kSubPer + i]);
      local += sh.sub_rounding[lane * kSubPer + i];
    }
    const double e_top = static_cast<double>(__uint_as_float(top_bits)), e_low = static_cast<double>(__uint_as_float(low_bits));
    const float off1 = wave_prefix_sum<float>(local);
    const int c0 = count_of(run), c1 = count_of(end);
    const double s0 = mass_of(run), s1 = mass_of(end);
    const double run_eps = eps + static_cast<double>(half_unit(mass_end, c1)) * static_cast<double>(c1 - c0);
    const double tail_top = static_cast<double>(V - c0 - 1) * e_top, tail_low = static_cast<double>(V - c1) * e_low;
    const bool any = end != run;
    const int first_may = first_lane(__ballot(any && !((s1 + off + off1) * rest - p * tail_low < -stop_error(s1, tail_low, run_eps))));
    const bool sure_run = any && (s0 + off + (off1 - local)) * rest - p * tail_top > stop_error(s1, tail_top, run_eps);
    int lo = kIntMax, hi = kIntMax;
    double s_lo = 0.0, s_hi = 0.0;
    if (first_may >= 0) {
      // A finer bucket a lane, from that run on.  Its j-th element, of an exponential e between the bucket's least and
      // largest: G_j = G_0 + j e, and what each of them rounds by.
      const int b = first_may * kSubPer + lane;
      const u64 mine = b < kPickSubs ? subs.sum[b] : 0;
      const u64 front = wave_read_lane(run, first_may) + wave_prefix_sum<u64>(mine) - mine;
      const float mine_off = b < kPickSubs ? sh.sub_rounding[b] : 0.0f;
      const double front_off = static_cast<double>(wave_read_lane(off1 - local, first_may) + wave_prefix_sum<float>(mine_off) - mine_off);
      if (mine != 0) {
        const int at = count_of(front), n = count_of(mine);
        const double s = mass_of(front);
        const double e_min = static_cast<double>(__uint_as_float(subs.tag_min[b])), e_max = static_cast<double>(__uint_as_float(subs.tag_max[b]));
        // (several exponentials: the roundings up to one of them are not known)
        const double each = e_min == e_max ? static_cast<double>(mine_off) / n : 0.0;
        const double open_here = e_min == e_max ? eps : eps + static_cast<double>(half_unit(mass_end, at + n)) * n;
        const double tail = static_cast<double>(V - at - 1), err = stop_error(s + n * e_max, tail * e_max, open_here);
        const double g0 = (s + off + front_off + each) * rest;
        const double j_may = ceil((-err - (g0 + e_max * rest - p * (tail * e_min))) / (e_max + each * rest));
        const double j_sure = ceil((err - (g0 + e_min * rest - p * (tail * e_max))) / (e_min + each * rest));
        if (j_may < static_cast<double>(n)) {
          const int j = j_may > 0.0 ? static_cast<int>(j_may) : 0;
          lo = at + j;
          s_lo = s + static_cast<double>(j + 1) * e_min;
        }
        if (j_sure < static_cast<double>(n)) {
          const int j = j_sure > 0.0 ? static_cast<int>(j_sure) : 0;
          hi = at + j;
          s_hi = s + static_cast<double>(j + 1) * e_max;
        }
      }
      // the runs behind those: the first element of one may be the stop, and of the first that says so certainly is
      if (lane >= first_may + 64 / kSubPer && any) {
        if (lo == kIntMax || c0 < lo) {
          lo = c0;
          s_lo = s0 + e_low;
        }
        if (sure_run && c0 < hi) {
          hi = c0;
          s_hi = s0 + e_top;
        }
      }
    }
    int w_lo = wave_min_i(lo), w_hi = wave_min_i(hi);
    if (stop_hi != kIntMax || ends_in_zero) {  // (the first element of that bucket at the latest)
      const int at = count_of(stop_end);
      if (w_hi == kIntMax) {
        w_hi = hi = at;
        s_hi = mass_end;
      }
      if (w_lo == kIntMax) {
        w_lo = lo = at;
        s_lo = mass_of(stop_end) + static_cast<double>(e_end_low);
      }
    }
    if (lo == w_lo) {
      sh.stop_lo = lo;
      sh.kept_lo = s_lo;
    }
    if (hi == w_hi) {
      sh.stop_hi = hi;
      sh.kept_hi = s_hi;
    }
  }

  // Wave 1: the token, once the kept mass is known (sum, run: its scan of the draw's finer buckets).
  __device__ __forceinline__ void resolve_draw(const u64 (&sum)[kSubPer], u64 run, int n_list) const {
    const int lane = lane_id();
    const int lo = sh.stop_lo, hi = sh.stop_hi;
    if (hi == kIntMax) return;
    // A stop on the last element of one of the reference's batches (16, 64, 256, ... elements) is missed
    // (src/sampling_distribution.h:166-181).  (For p = 1 the element it then goes on to has next to no weight.)
    bool batch_end = false;
    for (int end = 16; end <= hi + 1 && end < V && prm.p < 1.0f; end *= 4) batch_end = batch_end || end >= lo + 1;
    const double kept_hi = sh.kept_hi, guard = draw_guard(kept_hi, static_cast<double>(hi) + 1.0);
    const double t_lo = u * sh.kept_lo - guard, t_hi = u * kept_hi + guard;
    const u64 w_lo = word_mass(t_lo - base), w_hi = word_mass(t_hi - base) + 1, mask = (1ull << shift) - 1ull;
    // the finer bucket the target falls into
    int b_lo = kIntMax, b_hi = kIntMax;
    u64 front = 0;
#pragma unroll
    for (int i = 0; i < kSubPer; ++i) {
      const u64 next = run + sum[i];
      if (sum[i] != 0 && (next & mask) >= w_lo && b_lo == kIntMax) {
        b_lo = lane * kSubPer + i;
        front = run;
      }
      if (sum[i] != 0 && (next & mask) >= w_hi && b_hi == kIntMax) b_hi = lane * kSubPer + i;
      run = next;
    }
    const int sub = wave_min_i(b_lo), sub_sure = wave_min_i(b_hi);
    if (batch_end || sub != sub_sure || sub == kIntMax) return;  // (a boundary between two elements lies in reach)
    front = wave_read_lane(front, first_lane(__ballot(b_lo == sub)));
    const int n = count_of(sh.sub[1].sum[sub]), at = count_of(front);
    const double s = base + mass_of(front);
    const uint32_t okey = sh.sub[1].tag_min[sub];
    if (n > 64) {
      // If they are ties, which of them it is comes from their ids.
      const double e = static_cast<double>(exp_of(key_to_float(okey)));
      const double j_lo = fmax(ceil((t_lo - s) / e), 1.0), j_hi = fmax(ceil((t_hi - s) / e), 1.0);
      const bool sure = okey == sh.sub[1].tag_max[sub] && j_lo == j_hi && j_lo <= static_cast<double>(n);
      if (lane == 0 && sure && at + static_cast<int>(j_lo) - 1 <= lo) {
        sh.tie_okey = okey;
        sh.tie_rank = at - count_of(draw_before) + static_cast<int>(j_lo) - 1;
      }
      return;
    }
    // its keys, one a lane, in order
    int have = 0;
    for (int i = 0; i < n_list; i += 64) {
      const u64 k = i + lane < n_list ? list[i + lane] : 0;
      const bool in = k != 0 && sub_of(1, key_to_float(key64_okey(k))) == sub;
      const u64 hits = __ballot(in);
      if (in) sh.last[have + static_cast<int>(__popcll(hits & ((1ull << lane) - 1ull)))] = k;
      have += static_cast<int>(__popcll(hits));
    }
    u64 key = lane < have ? sh.last[lane] : 0;
    if (n > 1) key = wave_sort_desc_fast<u64>(key);
    const double upto = s + wave_prefix_sum<double>(key != 0 ? static_cast<double>(exp_of(key_to_float(key64_okey(key)))) : 0.0);
    const int first = first_lane(__ballot(key != 0 && upto >= t_lo)), sure = first_lane(__ballot(key != 0 && upto >= t_hi));
    if (first < 0 || first != sure || at + first > lo) return;
    if (lane == first) sh.token = key64_index(key);
  }

  // The row's token, the same for every thread; kNoPick: it takes the exact sums.
  __device__ __forceinline__ uint32_t resolve() {
    const int lane = lane_id(), wave = threadIdx.x >> 6;
    refine_hits();
    rounding = wave_sum<float>(rounding);
    slack = wave_sum<float>(slack);
    if (lane == 0) {
      sh.rounding[wave] = rounding;
      sh.slack[wave] = slack;
    }
    if (threadIdx.x == 0) {
      sh.token = kNoPick;
      sh.tie_rank = -1;
    }
    __syncthreads();  // (and the finer buckets are complete)
    const int n_list = static_cast<int>(sh.n_list);
    if (static_cast<uint32_t>(n_list) > static_cast<uint32_t>(kPickList)) return kNoPick;
    u64 sum[kSubPer], run = 0;
    if (wave == 0) resolve_stop();
    if (wave == 1) run = scan_subs(1, draw_before, sum);
    __syncthreads();
    if (wave == 1) resolve_draw(sum, run, n_list);
    return resolved(n_list);
  }
  // What resolve_draw has left behind.
  __device__ __forceinline__ uint32_t resolved(int n_list) const {
    __syncthreads();
    if (sh.tie_rank >= 0) {
      const u64* const keys = list;
      return block_tie_id(n_list, sh.tie_rank, sh.tie_okey, [=](int i) { return keys[i]; }, reinterpret_cast<uint32_t*>(sh.table));
    }
    return sh.token;
  }
};

}  // namespace ms
