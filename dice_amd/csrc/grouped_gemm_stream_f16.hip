// The streaming expert GEMMs for fp16 activations and weights: the same source as
// the bf16 kernels (see the head of grouped_gemm_stream.hip).
#define DICE_STREAM_F16 1
#include "grouped_gemm_stream.hip"
