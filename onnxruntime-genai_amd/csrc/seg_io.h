// Segment-wise row access shared by the kernels that cut long rows into segments of kSegElems
// elements handled by 256-thread workgroups (exact sequential sums, beam-search candidates).
#pragma once
#include "kernels.h"
#include "device_utils.h"

namespace ms {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

constexpr int kSegBlock = 256;
constexpr int kSegPer = kSegElems / kSegBlock;  // 16 elements per thread

// Sixteen-byte groups of a segment: load j of thread t brings the VEC (4 fp32, 8 fp16 or bf16) consecutive ids from
// seg * kSegElems + group * VEC on; ids >= vocab yield `fill`.  Two ways to share them out:
// seg_load: group j * 256 + t, so that a wave's load is one run of memory;
// seg_load_run: group t * (16 / VEC) + j, the thread's sixteen ids in a row, for what needs them in order (a wave's loads
// then touch all the lines of its share, each load again, from the cache).
template <typename InT, bool RUN>
__device__ __forceinline__ void seg_load_groups(const InT* row, int vocab, int seg, float fill, float (&v)[kSegPer]) {
  constexpr int VEC = sizeof(InT) == 4 ? 4 : 8;
  constexpr int NV = kSegPer / VEC;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int t = static_cast<int>(threadIdx.x);
    const int i0 = seg * kSegElems + (RUN ? t * NV + j : j * kSegBlock + t) * VEC;
    if (i0 + VEC <= vocab) {
      if constexpr (VEC == 4) {
        const v4f_any q = *reinterpret_cast<const v4f_any*>(row + i0);
        v[j * 4] = q.x, v[j * 4 + 1] = q.y, v[j * 4 + 2] = q.z, v[j * 4 + 3] = q.w;
      } else {
        const v4u q = *reinterpret_cast<const v4u_any*>(row + i0);
        if constexpr (__is_same(InT, uint16_t)) {
          widen_half8(q, &v[j * 8]);  // the hardware conversion, redone by the bit formula where it differs
        } else {
          const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            v[j * 8 + 2 * c] = narrow_bits_to_float<InT>(w[c] & 0xffffu);
            v[j * 8 + 2 * c + 1] = narrow_bits_to_float<InT>(w[c] >> 16);
          }
        }
      }
    } else {
#pragma unroll
      for (int c = 0; c < VEC; ++c) v[j * VEC + c] = (i0 + c < vocab) ? load_one<InT>(row, i0 + c) : fill;
    }
  }
}
template <typename InT>
__device__ __forceinline__ void seg_load(const InT* row, int vocab, int seg, float fill, float (&v)[kSegPer]) {
  seg_load_groups<InT, false>(row, vocab, seg, fill, v);
}
template <typename InT>
__device__ __forceinline__ void seg_load_run(const InT* row, int vocab, int seg, float fill, float (&v)[kSegPer]) {
  seg_load_groups<InT, true>(row, vocab, seg, fill, v);
}

template <typename InT>
__device__ __forceinline__ int seg_index(int seg, int e) {
  constexpr int VEC = sizeof(InT) == 4 ? 4 : 8;
  return seg * kSegElems + ((e / VEC) * kSegBlock + static_cast<int>(threadIdx.x)) * VEC + e % VEC;
}
__device__ __forceinline__ int seg_run_index(int seg, int e) { return seg * kSegElems + static_cast<int>(threadIdx.x) * kSegPer + e; }

}  // namespace ms
