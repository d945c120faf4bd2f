// The streaming kernels of the sampling path for fp32 logits.
#include "sample_stream.h"

MS_STREAM_KERNELS(, float, MS_MANY_OF_LARGE_K)
