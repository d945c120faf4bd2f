// Exact sequential-order sum of exp((x - max) / T) over long rows, spread over the whole GPU.
//
// The reference adds the exponentials of a row one by one into a float (LogSoftMax / Softmax,
// src/softmax.h:26-47); block_seq.h reproduces that with a scan of step functions, but one workgroup
// per row leaves most of the chip idle when there are few, long rows (beam search: 32 rows of 152K).
// Here a row is cut into segments of kSegElems elements and three launches share the work:
//   1. seqsum_max:      segment maxima.
//   2. seqsum_exp_step: e_i = expf((x_i - rowmax) * inv_T) (exact) and the segment's
//                       sum in double; then, from the double sums of the segments before it, a segment
//                       knows the binade its running sum will be in -- unless a power of two may fall
//                       inside it -- and composes the step functions of its elements under that binade
//                       into one (d0, d1) pair.
//   3. seqsum_walk:     one wave per row goes through the composed steps (seq_walk.h): each is applied after
//                       checking that the running sum really is in the assumed binade and stays in it
//                       (then the composition is exactly the sequential result).
// The check in step 3 makes the result independent of the estimate in step 2: a wrong guess only
// costs a scan.
#include "kernels.h"
#include "block_seq.h"
#include "seg_io.h"
#include "seqsum_exp_step.h"
#include "seq_walk.h"

namespace ms {

template <typename InT>
__global__ __launch_bounds__(kSegBlock) void seqsum_max_kernel(const SeqSumArgs a) {
  __shared__ uint32_t red[4];
  const int seg = blockIdx.x, row = blockIdx.y;
  const InT* x = static_cast<const InT*>(a.x) + static_cast<size_t>(row) * a.row_stride;
  float v[kSegPer];
  seg_load<InT>(x, a.vocab, seg, -__builtin_inff(), v);
  float fm = -__builtin_inff();
#pragma unroll
  for (int e = 0; e < kSegPer; ++e) fm = fmaxf(fm, v[e]);
  const uint32_t m = block_max<uint32_t>(order_key(fm), red);
  if (threadIdx.x == 0) {
    a.seg_max[static_cast<size_t>(row) * a.segs + seg] = m;
    // This launch comes first in every sequence: it marks the segment's sum as not written, so that the look-back
    // of the next launch never takes a sum left by an earlier call for this one's (the walk puts the mark back too,
    // but a sequence that was cut short after its second launch would otherwise leave finite sums behind).
    store_sum_bits(a.seg_sum + static_cast<size_t>(row) * a.segs + seg, kSumNotReady);
  }
}

// WAVES of a SIMD: 8 for more rows than CUs, two workgroups a CU, for which a wave may have 64 vector registers and 80 scalar ones.
// (softmax of 300 x 20000 fp32 45.6 -> 42.9 us, log-softmax 38.0 -> 36.7, 1000 x 17000 105.4 -> 102.0.)  It spills two registers then: where every
// row has a CU to itself the other kernel, of 68 and 88, is 0.4 to 1 us faster (log-softmax of 16 x 151936 27.5 against 28.2).
template <typename InT, int WAVES>
__global__ __launch_bounds__(64 * kWalkWaves, WAVES) void seqsum_walk_kernel(const SeqSumArgs a) {
  extern __shared__ u64 walk_lds[];
  __shared__ uint64_t exp_tab[32];
  WalkShared& sh = *reinterpret_cast<WalkShared*>(walk_lds);
  const int row = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const size_t rbase = static_cast<size_t>(row) * a.segs;
  if (threadIdx.x < 32) exp_tab[threadIdx.x] = em::exp2_tab(threadIdx.x);  // (barriers follow before it is used)
  const float max_score = a.out_max[row];  // (of the launch before this one)
  // (the row's segment sums have served: back to "not written" for the next launch)
  for (int sg = static_cast<int>(threadIdx.x) - 64; sg >= 0 && sg < a.segs; sg += 64 * (kWalkWaves - 1))
    store_sum_bits(a.seg_sum + rbase + sg, kSumNotReady);
  const EvenSegments<InT> segments{a.segs, a.vocab, a.seg_step + rbase, a.sub_step + rbase * kSegSubs, a.sub_se + rbase * kSegSubs,
                                   static_cast<const InT*>(a.x) + static_cast<size_t>(row) * a.row_stride, max_score, a.inv_temp, exp_tab};
  const float s = walk_segments<false>(segments, sh, nullptr);
  if (wave == 0 && lane == 0) a.out_sum[row] = s;
}

// Element-wise finish of Softmax / LogSoftMax (src/softmax.h:26-47) once a row's maximum and sum
// are known: log-softmax writes (x - max) * inv_T - log(sum); softmax writes e * (1 / sum), with e the
// exponential (left as is when the sum is zero).
template <bool LOG>
__global__ __launch_bounds__(kSegBlock) void softmax_apply_kernel(float* scores, int64_t row_stride, const SeqSumArgs a) {
  const int seg = blockIdx.x, row = blockIdx.y;
  float* x = scores + static_cast<size_t>(row) * row_stride;
  const float max_score = a.out_max[row], sum = a.out_sum[row];
  const float lse = LOG ? em::logf_exact(sum) : 0.0f;
  const float inv_sum = 1.0f / sum;
  // four elements per load and store (whatever the row's alignment), the loads of a thread under way together
  float v[kSegPer], r[kSegPer];
  seg_load<float>(x, a.vocab, seg, 0.0f, v);
  if constexpr (LOG) {
    // x - max is never -0 where it shows (see softmax_kernel): the maximum here lost the sign of its zero
#pragma unroll
    for (int e = 0; e < kSegPer; ++e) {
      const float d = v[e] - max_score;
      r[e] = (d == 0.0f ? 0.0f : d) * a.inv_temp - lse;
    }
  } else {
    __shared__ uint64_t exp_tab[32];
    if (threadIdx.x < 32) exp_tab[threadIdx.x] = em::exp2_tab(threadIdx.x);
    __syncthreads();
    const uint64_t* const tab = exp_tab;
#pragma unroll
    for (int e = 0; e < kSegPer; ++e) v[e] = (v[e] - max_score) * a.inv_temp;
    wave_expf(v, [=](uint32_t i) { return tab[i]; }, r);
#pragma unroll
    for (int e = 0; e < kSegPer; ++e) r[e] = sum > 0.0f ? r[e] * inv_sum : r[e];
  }
#pragma unroll
  for (int e0 = 0; e0 < kSegPer; e0 += 4) {
    const int i = seg_index<float>(seg, e0);
    if (i + 4 <= a.vocab) {
      v4f_any q;
      q.x = r[e0], q.y = r[e0 + 1], q.z = r[e0 + 2], q.w = r[e0 + 3];
      *reinterpret_cast<v4f_any*>(x + i) = q;
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (i + c < a.vocab) x[i + c] = r[e0 + c];
    }
  }
}

}  // namespace ms

extern "C" hipError_t ms_launch_seqsum_max(const ms::SeqSumArgs* a, int dtype, hipStream_t stream) {
  const dim3 grid(a->segs, a->rows), block(ms::kSegBlock);
  if (dtype == MI355X_F16) hipLaunchKernelGGL(ms::seqsum_max_kernel<uint16_t>, grid, block, 0, stream, *a);
  else if (dtype == MI355X_BF16) hipLaunchKernelGGL(ms::seqsum_max_kernel<ms::bf16_t>, grid, block, 0, stream, *a);
  else hipLaunchKernelGGL(ms::seqsum_max_kernel<float>, grid, block, 0, stream, *a);
  return hipGetLastError();
}

extern "C" hipError_t ms_launch_seqsum_walk(const ms::SeqSumArgs* a, int dtype, hipStream_t stream) {
  auto* f = dtype == MI355X_F16 ? ms::seqsum_walk_kernel<uint16_t, 4> : dtype == MI355X_BF16 ? ms::seqsum_walk_kernel<ms::bf16_t, 4> : ms::seqsum_walk_kernel<float, 4>;
  if (a->rows > ms::kCus)
    f = dtype == MI355X_F16 ? ms::seqsum_walk_kernel<uint16_t, 8> : dtype == MI355X_BF16 ? ms::seqsum_walk_kernel<ms::bf16_t, 8> : ms::seqsum_walk_kernel<float, 8>;
  hipLaunchKernelGGL(f, dim3(a->rows), dim3(64 * ms::kWalkWaves), sizeof(ms::WalkShared), stream, *a);
  return hipGetLastError();
}

extern "C" hipError_t ms_launch_seqsum(const ms::SeqSumArgs* a, int dtype, hipStream_t stream) {
  const dim3 grid(a->segs, a->rows), block(ms::kSegBlock);
  hipError_t e = ms_launch_seqsum_max(a, dtype, stream);
  if (e != hipSuccess) return e;
  const ms::NothingBetween nothing;
  if (dtype == MI355X_F16)
    hipLaunchKernelGGL((ms::seqsum_exp_step_kernel<uint16_t, ms::NothingBetween>), grid, block, 0, stream, *a, nothing);
  else if (dtype == MI355X_BF16)
    hipLaunchKernelGGL((ms::seqsum_exp_step_kernel<ms::bf16_t, ms::NothingBetween>), grid, block, 0, stream, *a, nothing);
  else
    hipLaunchKernelGGL((ms::seqsum_exp_step_kernel<float, ms::NothingBetween>), grid, block, 0, stream, *a, nothing);
  return ms_launch_seqsum_walk(a, dtype, stream);
}

extern "C" hipError_t ms_launch_softmax_apply(float* scores, int64_t row_stride, const ms::SeqSumArgs* a,
                                              int log_softmax, hipStream_t stream) {
  const dim3 grid(a->segs, a->rows), block(ms::kSegBlock);
  if (log_softmax)
    hipLaunchKernelGGL(ms::softmax_apply_kernel<true>, grid, block, 0, stream, scores, row_stride, *a);
  else
    hipLaunchKernelGGL(ms::softmax_apply_kernel<false>, grid, block, 0, stream, scores, row_stride, *a);
  return hipGetLastError();
}
