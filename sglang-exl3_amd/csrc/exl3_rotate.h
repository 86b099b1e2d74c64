// Input rotation of a row batch: xr = fp16( H(x (.) suh) / sqrt(128) ) (feeds the
// k-split GEMV's pre-rotated mode and the MFMA GEMM).
#pragma once

#include "exl3_gemv_impl.h"

namespace exl3 {
namespace {

// blockIdx.y: the matrix whose suh applies; its rotated rows follow those of
// the matrix before.  rs (optional): the sum of each chunk's 128 rotated fp16
// values, [row][k/128] per matrix (the mul1 raw-entry GEMM's affine correction).
struct RotateSuh {
    const __half* suh[kMaxMats];
};

// Many chunks: a wave takes 8 chunks of 128 values, 8 lanes and 32 bytes a lane
// each (rotate_chunk).  One chunk a wave, 4 bytes a lane, is bound by its
// instruction count there: 1000 x 14336 bf16 19 -> 10.7 us (57 MB).
__global__ __launch_bounds__(256) void rotate_rows_kernel(const __half* x, RotateSuh suhs, __half* xr,
                                                          long long chunks, int k, int x_bf16, float* rs) {
    const int lane = threadIdx.x & 63;
    const long long chunk = ((long long)blockIdx.x * 4 + (threadIdx.x >> 6)) * 8 + (lane >> 3);
    const long long cc = chunk < chunks ? chunk : chunks - 1;  // whole waves stay active for the lane exchanges
    const int c = (int)((unsigned)cc % (unsigned)(k >> 7)) * 128 + (lane & 7) * 16;
    const RowChunk o = rotate_chunk(ld_chunk(gptr(x) + cc * 128 + (lane & 7) * 16),
                                    ld_chunk(gptr(suhs.suh[blockIdx.y]) + c), x_bf16, lane);
    float t = 0.f;
    if (rs) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t u = o.v[e >> 2][e & 3];
            const __half2 h = *reinterpret_cast<const __half2*>(&u);
            t += __low2float(h) + __high2float(h);
        }
        t += lane_xor<1>(t);
        t += lane_xor<2>(t);
        t += lane_xor<4>(t);
    }
    if (chunk >= chunks) return;
    EXL3_GLOBAL u32x4_t* dst = reinterpret_cast<EXL3_GLOBAL u32x4_t*>(
        gptr(xr) + ((size_t)blockIdx.y * chunks + chunk) * 128 + (lane & 7) * 16);
    dst[0] = o.v[0];
    dst[1] = o.v[1];
    if (rs && (lane & 7) == 0) gptr(rs)[(size_t)blockIdx.y * chunks + chunk] = t;
}

// Few chunks: one a wave, 2 values a lane, so that the launch's latency is one
// short chain on many CUs.
__global__ __launch_bounds__(256) void rotate_few_rows_kernel(const __half* x, RotateSuh suhs, __half* xr,
                                                              int chunks, int k, int x_bf16, float* rs) {
    const int chunk = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (chunk >= chunks) return;
    const int lane = threadIdx.x & 63;
    const int c = chunk % (k >> 7) * 128 + 2 * lane;
    const __half2 pr = __hmul2(x_h2(ld_h2(gptr(x) + (size_t)chunk * 128 + 2 * lane), x_bf16),
                               ld_h2(gptr(suhs.suh[blockIdx.y]) + c));
    float a = __low2float(pr), b = __high2float(pr);
    fwht128_pair_fast(a, b, lane);
    const __half2 o = h2_rn(a * kHadNorm, b * kHadNorm);
    const size_t at = (size_t)blockIdx.y * chunks + chunk;
    st_h2(gptr(xr) + at * 128 + 2 * lane, o);
    if (rs) {
        const float t = wave_sum(__low2float(o) + __high2float(o));
        if (lane == 0) gptr(rs)[at] = t;
    }
}

// Chunks (of all matrices) up to which one goes to each wave.  Whole gate/up call,
// k = 4096, n = 6144, K = 4 mul1, us, eight chunks a wave / one: 128 chunks (4 rows)
// 16.81 / 16.47, 512 17.96 / 17.82, 1024 23.37 / 22.97, 2048 28.33 / 27.78, 3072 34.57 /
// 34.42.  Env EXL3_ROTATE_FEW overrides.
constexpr int kRotateFewChunks = 3072;

inline int rotate_rows(const __half* x, const RotateSuh& suhs, int mats, __half* xr, int m, int k, int x_bf16,
                       float* rs, hipStream_t st, const char* what) {
    const long long chunks = (long long)m * (k / 128);
    if (chunks * mats <= env_int("EXL3_ROTATE_FEW", kRotateFewChunks))
        rotate_few_rows_kernel<<<dim3((unsigned)((chunks + 3) / 4), mats), 256, 0, st>>>(x, suhs, xr, (int)chunks, k,
                                                                                       x_bf16, rs);
    else
        rotate_rows_kernel<<<dim3((unsigned)((chunks + 31) / 32), mats), 256, 0, st>>>(x, suhs, xr, chunks, k, x_bf16,
                                                                                      rs);
    return launch_status(what);
}

}  // namespace
}  // namespace exl3
