// One instantiation unit of the tall-tile GEMM kernels per bit width: the build
// compiles this file once per K with -DEXL3_K=K.
#include "exl3_tall_impl.h"

#ifndef EXL3_K
#error "build with -DEXL3_K=<bits>"
#endif

#define EXL3_CAT2(a, b) a##b
#define EXL3_CAT(a, b) EXL3_CAT2(a, b)

namespace exl3 {
int EXL3_CAT(tall_launch_K, EXL3_K)(int cb, int mt, const FatParams& p, int row_tiles, int splits, bool gu_fused, hipStream_t st) {
    return tall_launch_k<EXL3_K>(cb, mt, p, row_tiles, splits, gu_fused, st);
}
}  // namespace exl3
