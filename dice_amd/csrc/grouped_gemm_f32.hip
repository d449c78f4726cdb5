// The permutation-addressed expert GEMMs for fp32 activations and weights on the
// fp32 MFMA, for what the split kernels (grouped_gemm_split.hip) do not take: more
// than 64 experts, source rows or an expert's weights of 2 GiB and more, a tiling that
// the tuning hook names.  The same source as the bf16 kernels with the element type, the
// k step and the inner loop switched (see the head of grouped_gemm_bf16.hip).
#define DICE_GEMM_F32 1
#include "grouped_gemm_bf16.hip"
