// EXL3 GEMM for many rows on gfx950 MFMA, tall tiles.
//
// A workgroup of 4 waves owns up to MT (128 or 256) rows x 128 columns and a
// range of k; each wave decodes its own 32 columns into MFMA B fragments in
// registers and multiplies them with every staged row.  What bounds the
// many-row product is the decode's VALU time, which does not hide under the
// MFMAs on gfx950: per 64-k step a wave spends ~620 cycles on the decode and 16
// per MFMA, 4 MFMAs per 16 rows.  A 64-row tile therefore spends 70 % of its time
// on the decode, a 256-row tile 38 %.  Against the 256 x 256 tiles of
// fat_big_kernel the B fragments never go through LDS, a grid has twice the
// workgroups, and two (MT = 256) or four (128) of them share a CU, so one's
// decode, staging wait or epilogue runs beside another's MFMAs without a
// barrier between them.
//
// A (fp16 rows, rotated) is copied global -> LDS by the load unit itself
// (global_load_lds, 16 bytes per lane), one 64-k step ahead into the other of
// two buffers: no staging registers, which 128 accumulators leave no room for.
// LDS row r holds its 16-byte chunk c at slot c ^ (r & 7) ^ ((r >> 3) & 1), by
// choosing the source address per lane, so the fragment reads are
// conflict-free.  The copies are issued by inline asm that the compiler does
// not count; a step ends with an explicit wait that leaves only the last weight
// request in flight (weights are requested two steps ahead) and one barrier.
#pragma once

#include "exl3_fat_impl.h"

namespace exl3 {

constexpr int TL_THREADS = 256;
constexpr int TL_PASS_ROWS = 64;  // epilogue rows per LDS pass
constexpr int TL_CTS = 128 + 4;   // epilogue row stride (floats)

constexpr size_t tall_smem_bytes(int mt) {
    const size_t stage = 2 * (size_t)mt * 128, tile = (size_t)TL_PASS_ROWS * TL_CTS * sizeof(float);
    return stage > tile ? stage : tile;
}

// 16 bytes per lane from base + off (bytes) to LDS byte lds + 16 lane.  The
// caller waits (vmcnt) before a barrier and the reads.
__device__ __forceinline__ void copy_to_lds16(const EXL3_GLOBAL char* base, uint32_t off, uint32_t lds) {
    asm volatile(
        "s_mov_b32 m0, %2\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %0, %1" ::"v"(off),
        "s"(base), "s"(lds)
        : "memory", "m0");
}

// The k loop of one wave: `rows` rows (up to MT) x the wave's 32 columns over
// nsteps (even) 64-k steps.  tb: the wave's words of step 0; abase: row 0 of the
// tile at the split's first k; lds: the byte offset of the two A buffers in
// the workgroup's LDS, copied by SW waves, of which this is wave sw.
template <int K, int CB, int MT, int SW, bool RAW>
__device__ __forceinline__ void tall_loop(float4_t (&acc)[MT / 16][2], const EXL3_GLOBAL uint32_t* tb,
                                          size_t step_stride, int nsteps, const EXL3_GLOBAL char* abase, int k,
                                          int rows, unsigned char* smem, uint32_t lds, int sw, int lane) {
    constexpr int RB = MT / 16;
    constexpr int PF = MT == 128 ? 1 : 2;  // row blocks whose fragments are read ahead
    constexpr int GR = 8 * SW;             // rows copied by one instruction of each wave
    const int g = lane >> 4, i = lane & 15;
    const int prev_addr = ((lane & ~7) | ((lane + 7) & 7)) << 2;
    // A copies: wave w's j-th instruction of a step moves rows GR j + 8w .. + 7;
    // rows past the tile repeat its last row (never stored)
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem + lds;
    uint32_t aoff[MT / GR];
    const uint32_t achunk = 16u * (uint32_t)((lane & 7) ^ (lane >> 3) ^ (sw & 1));
#pragma unroll
    for (int j = 0; j < MT / GR; ++j)
        aoff[j] = (uint32_t)min(GR * j + 8 * sw + (lane >> 3), rows - 1) * (uint32_t)k * 2u + achunk;
    auto copy_a = [&](int step, int bufi) {
        const EXL3_GLOBAL char* src = abase + (size_t)step * 128;
#pragma unroll
        for (int j = 0; j < MT / GR; ++j)
            if (GR * j < rows) copy_to_lds16(src, aoff[j], lds0 + bufi * (MT * 128) + (GR * j + 8 * sw) * 128);
    };
    // A fragment reads: row 16 rb + i, logical chunk 2g + h
    uint32_t rd_off[2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
        rd_off[h] = lds + (uint32_t)i * 128u + 16u * (uint32_t)((2 * g + h) ^ (i & 7) ^ (i >> 3));

#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        acc[rb][0] = float4_t{0.f, 0.f, 0.f, 0.f};
        acc[rb][1] = float4_t{0.f, 0.f, 0.f, 0.f};
    }
    uint32_t wa[K], wb[K];  // the words of this step and of the next one
    copy_a(0, 0);
    load_words<K>(tb, wa);
    load_words<K>(tb + step_stride, wb);
    // Wait for everything but the last weight request, and pass the next step's
    // words through, so that the compiler adds no wait of its own behind the
    // copies.  A request is at least WL load instructions (of 16 bytes at most)
    // behind the step's copies, and all its words are used (after the loop, the
    // last two's), so WL operations left in flight are never a copy.  With one
    // for every K, each step of 5 to 8 bits waited for half of the request that it
    // had just made (gate/up, k = 4096, n = 14336, 17 rows, MCG, K = 6 / 8: 42.1 / 43.3 ->
    // 32.8 / 35.4 us).
    constexpr int WL = (K + 3) / 4;
    auto step_end = [&](uint32_t (&wn)[K]) {
#pragma unroll
        for (int j = 0; j < K; ++j) asm volatile("" : "+v"(wn[j]));
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(WL) : "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    step_end(wa);

    auto step_body = [&](int s, auto slot_c, uint32_t (&w)[K], uint32_t (&wn)[K]) {
        constexpr int SL = decltype(slot_c)::value;
        const unsigned char* ab = smem + SL * (MT * 128);
        half8_t A[PF + 1][2];
        auto read_a = [&](int rb) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
                A[rb % (PF + 1)][h] = *reinterpret_cast<const half8_t*>(ab + rd_off[h] + rb * 2048);
        };
        // LDS reads of this step go first: the previous word of each group, and
        // the first row blocks' fragments
        uint32_t buf[K + 1];
#pragma unroll
        for (int j = 0; j < K; ++j) buf[1 + j] = w[j];
        buf[0] = (uint32_t)__builtin_amdgcn_ds_bpermute(prev_addr, (int)buf[K]);
#pragma unroll
        for (int rb = 0; rb < PF; ++rb) read_a(rb);
        __builtin_amdgcn_sched_barrier(0);
        if (s + 1 < nsteps) copy_a(s + 1, SL ^ 1);
        uint32_t f[2][2][4];  // [column half][h][j]
        nat_decode<K, CB, RAW, true>(buf, f);
        load_words<K>(tb + (size_t)(s + 2 < nsteps ? s + 2 : nsteps - 1) * step_stride, w);
        // row blocks in groups of 32 rows (none past the tile); the fragments of
        // a block are read PF blocks ahead
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r2 = 0; r2 < RB / 2; ++r2)
            if (32 * r2 < rows) {
#pragma unroll
                for (int rb = 2 * r2; rb < 2 * r2 + 2; ++rb) {
                    if (rb + PF < RB) read_a(rb + PF);
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int c = 0; c < 2; ++c)
                            acc[rb][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                A[rb % (PF + 1)][h], *reinterpret_cast<const half8_t*>(f[c][h]), acc[rb][c], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        step_end(wn);
    };
    for (int s = 0; s < nsteps; s += 2) {  // an even number of steps
        step_body(s, std::integral_constant<int, 0>{}, wa, wb);
        step_body(s + 1, std::integral_constant<int, 1>{}, wb, wa);
    }
#pragma unroll
    for (int j = 0; j < K; ++j) asm volatile("" ::"v"(wa[j]), "v"(wb[j]));
}

template <int K, int CB, int MT, bool RAW>
__global__ __launch_bounds__(TL_THREADS, MT == 256 ? 2 : 4) void tall_kernel(FatParams p) {
    static_assert(!RAW || CB == 2, "raw entries: mul1");
    constexpr int RB = MT / 16;
    extern __shared__ __align__(16) unsigned char fat_smem[];

    const int bx = blockIdx.x, sidx = blockIdx.z;
    // gate/up mode: block bx is column block bx / 2 of the gate (even) or up
    // (odd) projection, and its partial tile goes to the finish launch
    const uint32_t* trel = (p.gu && (bx & 1)) ? p.trellis2 : p.trellis;
    const __half* svh_p = p.svh;
    const __half* arows = p.a;
    const float* rowsum = p.rowsum;
    int bxm = p.gu ? bx >> 1 : bx, nm = p.n;  // column block and width inside the matrix
    long long y0 = 0;                         // its output, rows ys apart
    int ys = p.n;
    int m0 = blockIdx.y * MT;
    int rows = min(MT, p.M - m0);
    if (p.gmode) {
        if ((int)blockIdx.y >= __builtin_amdgcn_readfirstlane(*gptr(p.ntiles))) return;
        const EXL3_GLOBAL FatTile* tl = gptr(p.tiles) + blockIdx.y;
        const int e = __builtin_amdgcn_readfirstlane(tl->e);
        m0 = __builtin_amdgcn_readfirstlane(tl->crow0);
        rows = __builtin_amdgcn_readfirstlane(tl->nrows);
        trel = reinterpret_cast<const uint32_t*>(gptr(p.tabs[6])[e]);  // down (gmode 3)
        svh_p = reinterpret_cast<const __half*>(gptr(p.tabs[8])[e]);
    } else if (p.mats.count > 1) {
        const MatRef r = mat_of_block(p.mats, bx);
        trel = r.trellis;
        svh_p = r.svh;
        bxm = bx - r.nb0;
        nm = r.n;
        y0 = r.y0;
        ys = r.ys;
        arows += (size_t)r.j * p.M * p.k;
        if constexpr (RAW) rowsum += (size_t)r.j * p.M * (p.k >> 7);
    }
    const int tid = threadIdx.x, lane = tid & 63;
    const int cw = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, i = lane & 15, q = i & 7;
    const int ntiles = nm >> 4;
    const int nsteps = p.ksteps;
    const int kt0 = sidx * nsteps * 4;
    const int nt = bxm * 8 + cw * 2 + (i >> 3);
    const EXL3_GLOBAL uint32_t* tb = gptr(trel) + ((size_t)(kt0 + g) * ntiles + nt) * (8 * K) + K * q;
    const size_t step_stride = (size_t)4 * ntiles * (8 * K);
    const EXL3_GLOBAL char* abase =
        reinterpret_cast<const EXL3_GLOBAL char*>(gptr(arows)) + ((size_t)m0 * p.k + (size_t)kt0 * 16) * 2;
    float4_t acc[RB][2];
    tall_loop<K, CB, MT, 4, RAW>(acc, tb, step_stride, nsteps, abase, p.k, rows, fat_smem, 0, cw, lane);

    // epilogue: passes of 64 rows through LDS; 8 lanes hold a row, 16
    // consecutive columns each (fwht128_x16)
    float* ct = reinterpret_cast<float*>(fat_smem);
    const int col = (lane & 7) * 16;
    const float hn = fwht_x16_norm(lane);
    float sv[16];
    {
        // svh is only 4-byte aligned by contract
        const EXL3_GLOBAL uint32_t* svp = reinterpret_cast<const EXL3_GLOBAL uint32_t*>(gptr(svh_p) + bxm * 128 + col);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t u = svp[e];
            sv[2 * e] = __half2float(__ushort_as_half((unsigned short)(u & 0xffffu)));
            sv[2 * e + 1] = __half2float(__ushort_as_half((unsigned short)(u >> 16)));
        }
    }
    const size_t rs = (size_t)p.M * 128;  // between splits
    float* const part = p.split_out ? p.partials + ((size_t)bx * gridDim.z + sidx) * rs + (size_t)m0 * 128 : nullptr;
#pragma unroll
    for (int pass = 0; pass < MT / TL_PASS_ROWS; ++pass) {
        if (pass * TL_PASS_ROWS >= rows) break;
        if (pass) __syncthreads();
#pragma unroll
        for (int rr = 0; rr < TL_PASS_ROWS / 16; ++rr)
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    ct[(rr * 16 + 4 * g + r) * TL_CTS + cw * 32 + (i >> 3) * 16 + (i & 7) + 8 * c] =
                        acc[pass * (TL_PASS_ROWS / 16) + rr][c][r];
        __syncthreads();
#pragma unroll
        for (int it = 0; it < TL_PASS_ROWS / 32; ++it) {
            const int lr = it * 32 + cw * 8 + (lane >> 3);
            const int row = pass * TL_PASS_ROWS + lr;
            if (pass * TL_PASS_ROWS + it * 32 + cw * 8 >= rows) break;
            float v[16];
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                const float4 t = *reinterpret_cast<const float4*>(ct + lr * TL_CTS + col + 4 * q4);
                v[4 * q4] = t.x;
                v[4 * q4 + 1] = t.y;
                v[4 * q4 + 2] = t.z;
                v[4 * q4 + 3] = t.w;
            }
            if (part) {  // fat_split_finish_kernel sums the splits and finishes
                if (row < rows)
#pragma unroll
                    for (int q4 = 0; q4 < 4; ++q4)
                        *reinterpret_cast<EXL3_GLOBAL u32x4_t*>(gptr(part) + (size_t)row * 128 + col + 4 * q4) =
                            *reinterpret_cast<const u32x4_t*>(v + 4 * q4);
                continue;
            }
            const int crow = m0 + (row < rows ? row : rows - 1);
            if constexpr (RAW) {
                const float* r = rowsum + (size_t)crow * (p.k >> 7) + (kt0 >> 3);
                float t = 0.f;
                for (int c = lane & 7; c < (nsteps >> 1); c += 8) t += gptr(r)[c];
                t += lane_xor<1>(t);
                t += lane_xor<2>(t);
                t += lane_xor<4>(t);
                raw_fix16(v, kMul1Bias * t);
            }
            fwht128_x16(v, lane);
#pragma unroll
            for (int e = 0; e < 16; ++e) v[e] = (v[e] * hn) * sv[e];
            uint32_t ow[8];
            size_t orow = (size_t)crow;
            if (p.gmode) orow = (size_t)gptr(p.rows_map)[crow];  // by (token, slot) entry
#pragma unroll
            for (int e = 0; e < 8; ++e) ow[e] = y_bits(h2_rn(v[2 * e], v[2 * e + 1]), p.y_bf16);
            if (row >= rows) continue;
            EXL3_GLOBAL uint32_t* o =
                reinterpret_cast<EXL3_GLOBAL uint32_t*>(gptr(p.out16) + y0 + orow * ys + bxm * 128 + col);
            if (p.out_vec) {
                reinterpret_cast<EXL3_GLOBAL u32x4_t*>(o)[0] = u32x4_t{ow[0], ow[1], ow[2], ow[3]};
                reinterpret_cast<EXL3_GLOBAL u32x4_t*>(o)[1] = u32x4_t{ow[4], ow[5], ow[6], ow[7]};
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = ow[e];
            }
        }
    }
}

// Gate and up of a 128-column block in one workgroup of 8 waves (waves 0-3
// gate, 4-7 up), so the SwiGLU runs on the accumulators: no partial tiles or
// fp32 gate rows through memory.  Dense (GRP = false): both halves read one
// staged A (the projections share their input rotation); p.out16 = the activation;
// tiles_x, tail_first, tail_tiles and tail_parts describe the linear grid.
// Grouped (MoE prefill): each half stages its own projection's rotated rows
// (p.a, then p.a + p.up_rows * k for up), the weights are the tile's expert's, and
// out16[crow] is the activation rotated for the down projection.
template <int MT, bool GRP>
constexpr size_t tall_gu_smem_bytes() {
    constexpr size_t stage = (GRP ? 4 : 2) * (size_t)MT * 128, tile = (size_t)TL_PASS_ROWS * (256 + 4) * sizeof(float);
    return stage > tile ? stage : tile;
}

template <int K, int CB, int MT, bool RAW, bool GRP>
__global__ __launch_bounds__(2 * TL_THREADS, MT == 256 ? 2 : 4) void tall_gu_kernel(FatParams p) {
    static_assert(!RAW || (CB == 2 && !GRP), "raw entries: mul1, dense");
    constexpr int RB = MT / 16, CTS = 256 + 4;
    extern __shared__ __align__(16) unsigned char fat_smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), up = wv >> 2, cw = wv & 3;
    const int g = lane >> 4, i = lane & 15, q = i & 7;
    const uint32_t* trel = up ? p.trellis2 : p.trellis;
    const __half *svg = p.svh, *svu = p.svh2, *dsuh = nullptr;
    const __half* arows = p.a;
    int bx = blockIdx.x, m0 = 0, rows = 0;
    if constexpr (!GRP) {
        // linear grid, column blocks fastest; the tiles from tail_first on run
        // as tail_parts workgroups of MT / tail_parts rows each
        int lin = blockIdx.x, part = 0, mt = MT;
        if (lin >= p.tail_first) {
            const int o = lin - p.tail_first, t = o / p.tail_parts;
            part = o - t * p.tail_parts;
            mt = MT / p.tail_parts;
            lin = p.tail_first + t;
        }
        const int by = __builtin_amdgcn_readfirstlane(lin / p.tiles_x);
        bx = __builtin_amdgcn_readfirstlane(lin - by * p.tiles_x);
        m0 = __builtin_amdgcn_readfirstlane(by * MT + part * mt);
        rows = __builtin_amdgcn_readfirstlane(min(mt, p.M - m0));
        if (rows <= 0) return;
    }
    if constexpr (GRP) {
        if ((int)blockIdx.y >= __builtin_amdgcn_readfirstlane(*gptr(p.ntiles))) return;
        const EXL3_GLOBAL FatTile* tl = gptr(p.tiles) + blockIdx.y;
        const int e = __builtin_amdgcn_readfirstlane(tl->e);
        m0 = __builtin_amdgcn_readfirstlane(tl->crow0);
        rows = __builtin_amdgcn_readfirstlane(tl->nrows);
        trel = reinterpret_cast<const uint32_t*>(gptr(p.tabs[up ? 3 : 0])[e]);
        svg = reinterpret_cast<const __half*>(gptr(p.tabs[2])[e]);
        svu = reinterpret_cast<const __half*>(gptr(p.tabs[5])[e]);
        dsuh = reinterpret_cast<const __half*>(gptr(p.tabs[7])[e]);
        if (up) arows += (size_t)p.up_rows * p.k;
    }
    const int ntiles = p.n >> 4;
    const int nt = bx * 8 + cw * 2 + (i >> 3);
    const EXL3_GLOBAL uint32_t* tb = gptr(trel) + ((size_t)g * ntiles + nt) * (8 * K) + K * q;
    const EXL3_GLOBAL char* abase = reinterpret_cast<const EXL3_GLOBAL char*>(gptr(arows)) + (size_t)m0 * p.k * 2;
    float4_t acc[RB][2];
    tall_loop<K, CB, MT, GRP ? 4 : 8, RAW>(acc, tb, (size_t)4 * ntiles * (8 * K), p.ksteps, abase, p.k, rows, fat_smem,
                                           GRP ? up * (2 * MT * 128) : 0, GRP ? cw : wv, lane);

    // passes of 64 rows through LDS, gate in the left and up in the right 128
    // columns; 8 rows per wave, 16 consecutive columns of both per lane
    float* ct = reinterpret_cast<float*>(fat_smem);
    const int col = (lane & 7) * 16, c0 = bx * 128 + col;
    const float hn = fwht_x16_norm(lane);
#pragma unroll
    for (int pass = 0; pass < MT / TL_PASS_ROWS; ++pass) {
        if (pass * TL_PASS_ROWS >= rows) break;
        if (pass) __syncthreads();
#pragma unroll
        for (int rr = 0; rr < TL_PASS_ROWS / 16; ++rr)
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    ct[(rr * 16 + 4 * g + r) * CTS + up * 128 + cw * 32 + (i >> 3) * 16 + (i & 7) + 8 * c] =
                        acc[pass * (TL_PASS_ROWS / 16) + rr][c][r];
        __syncthreads();
        if (pass * TL_PASS_ROWS + wv * 8 >= rows) continue;
        const int lr = wv * 8 + (lane >> 3), row = pass * TL_PASS_ROWS + lr;
        const int crow = m0 + (row < rows ? row : rows - 1);
        float gv[16], uv[16];
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
            *reinterpret_cast<float4*>(gv + 4 * q4) = *reinterpret_cast<const float4*>(ct + lr * CTS + col + 4 * q4);
            *reinterpret_cast<float4*>(uv + 4 * q4) = *reinterpret_cast<const float4*>(ct + lr * CTS + 128 + col + 4 * q4);
        }
        if constexpr (RAW) {
            const float sx = raw_row_bias(p, crow, 0, p.k >> 7, lane);
            raw_fix16(gv, sx);
            raw_fix16(uv, sx);
        }
        fwht128_x16(gv, lane);
        fwht128_x16(uv, lane);
        // svh and suh are only 4-byte aligned by contract
        const EXL3_GLOBAL uint32_t* sgp = reinterpret_cast<const EXL3_GLOBAL uint32_t*>(gptr(svg) + c0);
        const EXL3_GLOBAL uint32_t* sup = reinterpret_cast<const EXL3_GLOBAL uint32_t*>(gptr(svu) + c0);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            gv[e] = (gv[e] * hn) * __half2float(__ushort_as_half((unsigned short)(sgp[e >> 1] >> (16 * (e & 1)))));
            uv[e] = (uv[e] * hn) * __half2float(__ushort_as_half((unsigned short)(sup[e >> 1] >> (16 * (e & 1)))));
        }
        if (p.limit > 0.0f && p.limit < __builtin_huge_valf()) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                gv[e] = fminf(gv[e], p.limit);
                uv[e] = fminf(fmaxf(uv[e], -p.limit), p.limit);
            }
        }
        uint32_t ow[8];
        if constexpr (GRP) {
            // the activation in fp16, then the down projection's input rotation of this 128-wide chunk
            const EXL3_GLOBAL uint32_t* dsp = reinterpret_cast<const EXL3_GLOBAL uint32_t*>(gptr(dsuh) + c0);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t du = dsp[e];
                const __half2 pr = __hmul2(h2_rn(silu_f(gv[2 * e]) * uv[2 * e], silu_f(gv[2 * e + 1]) * uv[2 * e + 1]),
                                           *reinterpret_cast<const __half2*>(&du));
                gv[2 * e] = __low2float(pr);
                gv[2 * e + 1] = __high2float(pr);
            }
            fwht128_x16(gv, lane);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const __half2 o = h2_rn(gv[2 * e] * hn, gv[2 * e + 1] * hn);
                ow[e] = *reinterpret_cast<const uint32_t*>(&o);
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const __half2 o = h2_rn(silu_f(gv[2 * e]) * uv[2 * e], silu_f(gv[2 * e + 1]) * uv[2 * e + 1]);
                ow[e] = *reinterpret_cast<const uint32_t*>(&o);
            }
        }
        if (row >= rows) continue;
        EXL3_GLOBAL uint32_t* o = reinterpret_cast<EXL3_GLOBAL uint32_t*>(gptr(p.out16) + (size_t)crow * p.n + c0);
        if (p.out_vec) {
            reinterpret_cast<EXL3_GLOBAL u32x4_t*>(o)[0] = u32x4_t{ow[0], ow[1], ow[2], ow[3]};
            reinterpret_cast<EXL3_GLOBAL u32x4_t*>(o)[1] = u32x4_t{ow[4], ow[5], ow[6], ow[7]};
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = ow[e];
        }
    }
}

// Tiles of `mt` (128 or 256) rows.  gu_fused: tall_gu_kernel (dense with 256-row
// tiles, or grouped, p.gmode = 4, with 128), else tall_kernel: plain fp16 output,
// grouped down pass (p.gmode = 3), or partial tiles for
// fat_split_finish_kernel (p.split_out; always in gate/up mode).
template <int K>
int tall_launch_k(int cb, int mt, const FatParams& p, int row_tiles, int splits, bool gu_fused, hipStream_t st) {
#define EXL3_TALL_GO(FN, GRID, THREADS, SMEM)                                                          \
    {                                                                                                  \
        const void* fn = reinterpret_cast<const void*>(&FN);                                           \
        const int lrc = allow_dynamic_lds(fn, SMEM, "exl3 gemm (tall tiles)");                         \
        if (lrc) return lrc;                                                                           \
        FN<<<GRID, THREADS, SMEM, st>>>(p);                                                            \
        return launch_status("exl3 gemm (tall tiles) launch");                                         \
    }
#define EXL3_TALL_GU(CBV, MTV, RAWV, GRPV)                                                             \
    if (cb == CBV && mt == MTV && (p.rowsum != nullptr) == RAWV && (p.gmode != 0) == GRPV)             \
    EXL3_TALL_GO((tall_gu_kernel<K, CBV, MTV, RAWV, GRPV>),                                            \
                 GRPV ? dim3(p.n / 128, row_tiles) : dim3(p.tail_first + p.tail_tiles * p.tail_parts),         \
                 2 * TL_THREADS,                                                                       \
                 (tall_gu_smem_bytes<MTV, GRPV>()))
#define EXL3_TALL(CBV, MTV, RAWV)                                                                      \
    if (cb == CBV && mt == MTV && (p.rowsum != nullptr) == RAWV)                                       \
    EXL3_TALL_GO((tall_kernel<K, CBV, MTV, RAWV>), dim3((p.gu ? 2 : 1) * (p.n / 128), row_tiles, splits), TL_THREADS, \
                 tall_smem_bytes(MTV))
    if (gu_fused) {
        EXL3_TALL_GU(0, 256, false, false) EXL3_TALL_GU(1, 256, false, false)
        EXL3_TALL_GU(2, 256, false, false) EXL3_TALL_GU(2, 256, true, false)
        EXL3_TALL_GU(0, 128, false, true) EXL3_TALL_GU(1, 128, false, true) EXL3_TALL_GU(2, 128, false, true)
    } else {
        EXL3_TALL(0, 128, false) EXL3_TALL(1, 128, false) EXL3_TALL(2, 128, false) EXL3_TALL(2, 128, true)
        EXL3_TALL(0, 256, false) EXL3_TALL(1, 256, false) EXL3_TALL(2, 256, false) EXL3_TALL(2, 256, true)
    }
#undef EXL3_TALL
#undef EXL3_TALL_GU
#undef EXL3_TALL_GO
    set_error("exl3 gemm: no tall kernel for codebook %d tile rows %d", cb, mt);
    return EXL3_ERR_UNSUPPORTED;
}

// One instantiation unit per K (exl3_tall_inst.hip built with -DEXL3_K=K).
int tall_launch(int K, int cb, int mt, const FatParams& p, int row_tiles, int splits, bool gu_fused, hipStream_t st);

}  // namespace exl3
