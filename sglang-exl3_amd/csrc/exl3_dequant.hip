// exl3_dequant_trellis: whole-weight decode to fp16, bit-identical to the
// reference host dequant (csrc/bindings.cpp:15-100):
//   1. decode every tile with truncating fp16 rounding,
//   2. per 128x128 block: radix-2 FWHT of each row (strides 1..64), x norm,
//   3. FWHT of each column, then ((v * norm) * suh[r]) * svh[c] in fp32,
//   4. round to fp16 (nearest-even).
// One workgroup of 8 waves per 128x128 block, 32 values per thread in every
// phase.  The work is ~25 VALU ops per value, so the kernel keeps both FWHTs in
// registers: a lane holds 32 consecutive values of a row (column), lane bits 4
// and 5 the two top index bits, so strides 1..16 are register butterflies and
// strides 32 and 64 one permlane swap per two values, which leaves both
// operands of a butterfly in one lane.  Wave w decodes tile row w, i.e. the 16
// rows that it then transforms, so the first LDS turn (fp16, tile order to row
// order) needs no barrier; the second (fp32, rows to columns) needs one.  Both
// are XOR-swizzled by 16-byte chunk so that every access is conflict-free, and
// share 64 KB, so two workgroups fit a CU.
// k = 4096, n = 14336, K = 4, MCG: 135.2 -> 52.1 us (29 MB read, 117 MB
// written: 30 us at the rate of a large copy).
#include "exl3_common.h"
#include "exl3_decode.h"

namespace exl3 {
namespace {

constexpr int DQ_THREADS = 512;

// Unnormalised FWHT over 128 values: index bits 0..4 in the register index,
// bits 5 and 6 in lane bits 4 and 5.  On return register bit 4 is index bit 5,
// register bit 3 is index bit 6, lane bit 4 is index bit 4 and lane bit 5 is
// index bit 3.  Strides 1, 2, .., 64 in this order, each (x + y, x - y): the
// same fp32 operations as fwht128_pair_f.
__device__ __forceinline__ void fwht128_x32(float (&v)[32]) {
#pragma unroll
    for (int h = 1; h < 32; h <<= 1)
#pragma unroll
        for (int e = 0; e < 32; ++e)
            if (!(e & h)) {
                const float x = v[e], y = v[e | h];
                v[e] = x + y;
                v[e | h] = x - y;
            }
    // the swaps bring values (index bit 5 = 0) to the first and (= 1) to the second result
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[e]), __float_as_uint(v[e + 16]), false, false);
        const float x = __uint_as_float(s[0]), y = __uint_as_float(s[1]);
        v[e] = x + y;
        v[e + 16] = x - y;
    }
#pragma unroll
    for (int e = 0; e < 32; ++e)
        if (!(e & 8)) {
            const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[e]), __float_as_uint(v[e + 8]), false, false);
            const float x = __uint_as_float(s[0]), y = __uint_as_float(s[1]);
            v[e] = x + y;
            v[e + 8] = x - y;
        }
}

// LDS traffic between lanes of one wave: no reordering across this point.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Words (lo, hi) of lanes 2i and 2i + 1 -> the even lane gets both low halves,
// the odd lane both high halves (lane 2i's half in the low bits).
__device__ __forceinline__ uint32_t pair_transpose(uint32_t x, uint32_t sel) {
    const uint32_t y = (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xB1, 0xF, 0xF, false);  // lane ^ 1
    return __builtin_amdgcn_perm(y, x, sel);
}

template <int K, int CB>
__global__ __launch_bounds__(DQ_THREADS, 4) void dequant_kernel(const uint32_t* __restrict__ trellis,
                                                                const __half* __restrict__ suh,
                                                                const __half* __restrict__ svh,
                                                                __half* __restrict__ W, int n) {
#pragma clang fp contract(off)
    __shared__ __align__(16) unsigned char blk[128 * 512];
    __shared__ __align__(16) float sus[128];
    const int bn = blockIdx.x, bk = blockIdx.y;
    const int ntiles = n >> 4;
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const int odd = lane & 1;
    const uint32_t sel = odd ? 0x03020706u : 0x05040100u;
    if (tid < 128) sus[tid] = __half2float(suh[bk * 128 + tid]);
    const float sv = __half2float(svh[bn * 128 + 16 * w + (lane & 15)]);

    // 1. decode: lane (tn, q) of wave w takes group q of tile (w, tn).  Word
    // (c, h, p) holds rows 4h + kofs(2p), + 1 of column q + 8c; a pair of lanes
    // turns it into (row, two columns).  Row r, 16-byte chunk j of the wave's
    // 16 x 128 fp16 values sits at chunk j ^ r.
    {
        const int tn = lane >> 3, q = lane & 7;
        const uint32_t* tp = trellis + ((size_t)(bk * 8 + w) * ntiles + (bn * 8 + tn)) * (8 * K) + K * q;
        uint32_t buf[K + 1];
#pragma unroll
        for (int j = 0; j < K; ++j) buf[1 + j] = tp[j];
        buf[0] = (uint32_t)__builtin_amdgcn_ds_bpermute(((lane & ~7) | ((lane + 7) & 7)) << 2, (int)buf[K]);
        // The decode's fp16 arithmetic runs under round-toward-zero: an fp16 add
        // (mul1: fma) rounds the exact sum once, which is the reference's
        // truncation of the exact value (csrc/exl3_dequant.cuh:41-55) since every
        // codebook value is a normal number (at least 2^-13).  The operands tie
        // the mode changes to the arithmetic between them.
        asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 3" : "+v"(buf[0]));
#pragma unroll
        for (int j = 1; j <= K; ++j) asm volatile("" : "+v"(buf[j]));
        uint32_t frag[2][2][4];
        decode_group<K, CB, false, false, true>(buf, frag);
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int p = 0; p < 4; ++p) asm volatile("" : "+v"(frag[c][h][p]));
        asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 0" : "+v"(frag[1][1][3]));
        const uint32_t base = w * 8192 + odd * 256 + (((2 * tn) ^ odd) << 4) + (q >> 1) * 4;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const int k0 = 4 * h + kofs(2 * p);
                    *reinterpret_cast<uint32_t*>(blk + (base ^ (uint32_t)((c ^ k0) << 4)) + k0 * 256) =
                        pair_transpose(frag[c][h][p], sel);
                }
    }
    wave_lds_sync();

    float v[32];
    const int l16 = lane & 15, lj = lane >> 4;
    // 2. row pass: lane (r, j) takes columns 32j .. + 31 of row 16w + r
    {
        const uint32_t base = w * 8192 + l16 * 256 + (((4 * lj) ^ l16) << 4);
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const u32x4_t u = *reinterpret_cast<const u32x4_t*>(blk + (base ^ (uint32_t)(x << 4)));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[8 * x + 2 * e] = __half2float(__ushort_as_half((unsigned short)(u[e] & 0xffffu)));
                v[8 * x + 2 * e + 1] = __half2float(__ushort_as_half((unsigned short)(u[e] >> 16)));
            }
        }
        wave_lds_sync();
        fwht128_x32(v);
        // fp32 rows of 32 chunks: row R, chunk j at j ^ (R & 15) ^ (R bit 5) << 2 ^ (R bit 6) << 3
        const int lc = ((lane >> 5) << 1) | (((lane >> 4) & 1) << 2);
        const uint32_t ob = w * 8192 + l16 * 512 + ((lc ^ l16 ^ (((w >> 1) & 3) << 2)) << 4);
#pragma unroll
        for (int e = 0; e < 32; e += 4) {
            const int cc = ((e >> 2) & 1) | (((e >> 4) & 1) << 3) | (((e >> 3) & 1) << 4);
            *reinterpret_cast<float4*>(blk + (ob ^ (uint32_t)(cc << 4))) =
                make_float4(v[e] * kHadNorm, v[e + 1] * kHadNorm, v[e + 2] * kHadNorm, v[e + 3] * kHadNorm);
        }
    }
    __syncthreads();

    // 3. column pass: lane (c, j) takes rows 32j .. + 31 of column 16w + c
    {
        const int c = 16 * w + l16;
        const uint32_t base = lj * 32 * 512 + (((c >> 2) ^ (lj << 2)) << 4) + (c & 3) * 4;
#pragma unroll
        for (int t = 0; t < 32; ++t)
            v[t] = *reinterpret_cast<const float*>(blk + (base ^ (uint32_t)((t & 15) << 4)) + t * 512);
        fwht128_x32(v);
    }
    // 4. scales, fp16, and a pair of lanes turns (two rows, one column) into (row, two columns)
    const int rl = ((lane >> 5) << 3) | (((lane >> 4) & 1) << 4);
    __half* wp = W + (size_t)(bk * 128 + rl + odd) * (size_t)n + bn * 128 + 16 * w + (l16 & ~1);
#pragma unroll
    for (int e = 0; e < 32; e += 4) {
        const int rr = (e & 7) | (((e >> 4) & 1) << 5) | (((e >> 3) & 1) << 6);
        const float4 su = *reinterpret_cast<const float4*>(sus + rl + rr);
        const float s4[4] = {su.x, su.y, su.z, su.w};
#pragma unroll
        for (int h = 0; h < 4; h += 2) {
            const _Float16 lo = f16_rn(((v[e + h] * kHadNorm) * s4[h]) * sv);
            const _Float16 hi = f16_rn(((v[e + h + 1] * kHadNorm) * s4[h + 1]) * sv);
            const uint32_t o = (uint32_t)__builtin_bit_cast(unsigned short, lo) |
                               ((uint32_t)__builtin_bit_cast(unsigned short, hi) << 16);
            *reinterpret_cast<uint32_t*>(wp + (size_t)(rr + h) * (size_t)n) = pair_transpose(o, sel);
        }
    }
}

template <int K>
int launch_dequant_k(int cb, const uint32_t* t, const __half* su, const __half* sv, __half* W, int k, int n,
                     hipStream_t st) {
    dim3 grid(n / 128, k / 128);
    switch (cb) {
        case 0: dequant_kernel<K, 0><<<grid, DQ_THREADS, 0, st>>>(t, su, sv, W, n); break;
        case 1: dequant_kernel<K, 1><<<grid, DQ_THREADS, 0, st>>>(t, su, sv, W, n); break;
        default: dequant_kernel<K, 2><<<grid, DQ_THREADS, 0, st>>>(t, su, sv, W, n); break;
    }
    return launch_status("exl3_dequant_trellis launch");
}

}  // namespace
}  // namespace exl3

extern "C" int exl3_dequant_trellis(const int16_t* trellis, const uint16_t* suh, const uint16_t* svh,
                                    uint16_t* W, int k, int n, int K, int codebook, void* stream) {
    using namespace exl3;
    clear_error();
    EXL3_REQUIRE(trellis && suh && svh && W, "exl3_dequant_trellis: null pointer");
    EXL3_REQUIRE(k > 0 && n > 0 && k % 128 == 0 && n % 128 == 0,
                 "exl3_dequant_trellis: k=%d n=%d must be positive multiples of 128", k, n);
    EXL3_REQUIRE(K >= 1 && K <= 8, "exl3_dequant_trellis: K=%d outside 1..8", K);
    EXL3_REQUIRE(codebook >= 0 && codebook <= 2, "exl3_dequant_trellis: codebook=%d", codebook);
    EXL3_REQUIRE(aligned(trellis, 4) && aligned(W, 16), "exl3_dequant_trellis: misaligned pointer");
    const uint32_t* t = reinterpret_cast<const uint32_t*>(trellis);
    const __half* su = reinterpret_cast<const __half*>(suh);
    const __half* sv = reinterpret_cast<const __half*>(svh);
    __half* w = reinterpret_cast<__half*>(W);
    hipStream_t st = as_stream(stream);
    switch (K) {
        case 1: return launch_dequant_k<1>(codebook, t, su, sv, w, k, n, st);
        case 2: return launch_dequant_k<2>(codebook, t, su, sv, w, k, n, st);
        case 3: return launch_dequant_k<3>(codebook, t, su, sv, w, k, n, st);
        case 4: return launch_dequant_k<4>(codebook, t, su, sv, w, k, n, st);
        case 5: return launch_dequant_k<5>(codebook, t, su, sv, w, k, n, st);
        case 6: return launch_dequant_k<6>(codebook, t, su, sv, w, k, n, st);
        case 7: return launch_dequant_k<7>(codebook, t, su, sv, w, k, n, st);
        default: return launch_dequant_k<8>(codebook, t, su, sv, w, k, n, st);
    }
}
