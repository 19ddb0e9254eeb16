// Prefill GEMM tiles of 256 weight rows x 256 tokens (gemm_wide in
// gemm_tile.h), in a code object of their own so that they compile beside
// the others.  Not for f32 X, whose words in flight would not fit the
// registers beside the 64 x 128 wave tiles.
#include "gemm_tile.h"

// name: cima_gemm_<fmt>_w256_<x type>_<y type>
#define WIDE_KERNEL(FN, D, XT, XN, YT, YN)                                                          \
    extern "C" __global__ __launch_bounds__(512, 2) void cima_gemm_##FN##_w256_##XN##_##YN(         \
        const void* x, const uint8_t* w, void* y, int m, int n, int k, int ldy, GemmExt ext) {     \
        gemm_wide<D, XT, YT, 2, 4, 4, 2>(x, w, y, m, n, k, ldy, ext);                               \
    }
#define WIDE_FMT(FN, D)                            \
    WIDE_KERNEL(FN, D, XT_F16, f16, XT_F32, f32)   \
    WIDE_KERNEL(FN, D, XT_BF16, bf16, XT_F32, f32) \
    WIDE_KERNEL(FN, D, XT_F16, f16, XT_F16, f16)   \
    WIDE_KERNEL(FN, D, XT_BF16, bf16, XT_F16, f16)

WIDE_FMT(q8_0, GG<DQ8_0>)
WIDE_FMT(q4_0, GG<DQ4_0>)
WIDE_FMT(q4_1, GG<DQ4_1>)
WIDE_FMT(q5_0, GG<DQ5_0>)
WIDE_FMT(q5_1, GG<DQ5_1>)
WIDE_FMT(q4_k, GG<DQ4_K>)
WIDE_FMT(q5_k, GG<DQ5_K>)
WIDE_FMT(q6_k, GG<DQ6_K>)
WIDE_FMT(iq4_xs, GG<DIQ4_XS>)
WIDE_FMT(nf4, DNF4)
WIDE_FMT(f16w, DF16)
