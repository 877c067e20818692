#pragma once
// The integer-dot (dual) matvec of several tokens on the integer matrix cores with K split over a block's waves:
// matvec_kw8. The schedule is matvec_kw's (matvec_kw.hpp): 8 waves, each with its own 256-value stages of the block's
// rows, loaded a stage ahead into registers and passed through the wave's own LDS region to change lanes, no barrier
// until the partial sums meet; any number of tokens in one launch. The numerics are the integer-dot ones
// (matvec_i8.hip): the quantized activations' codes times the weights' codes in exact int32 sums per 32-value unit, then
// a d s in f32.
//
// v_mfma_i32_16x16x32_i8: A holds 16 tokens' q8 codes of a unit (lane l: token l % 16, values 8 (l / 16) .. + 7), B a
// 16-row group's codes (lane l: row l % 16, the same values), so lane l's sums are tokens 4 (l / 16) + i of row l % 16. The
// formats with a fixed code offset (Q4_0 -8, Q5_0 -16, Q6_K -32) enter as signed codes and need no offset term;
// Q6_K's two 16-value scale groups take two products, the other half's codes masked to zero, joined in integers by
// their int8 scales (exact, below 2^24). A unit's activation scales d reach the lanes of their tokens through LDS; the
// offset terms b (gs0 + gs1) of four units are one 16 x 16 x 4 f32 product.
//
// x's codes pass through LDS as the rows do: loaded straight into the A layout (8 bytes per lane, 16 rows apart) they took
// as long as the weights (K = 14336, N = 4096, Q4_K, 16 tokens: 25.3 us, 15.9 through LDS, 42.2 with the row-resident
// kernel; 31 tokens 27.8 / 21.2 / 80.7; quantization included). Bound: the latency of the few stages a wave has (two at
// K = 4096); the rows stream at 2.7 TB/s at the first size. Blocks of two token tiles and of four row tiles lost everywhere.
#include "matvec_i8.hpp"
#include "matvec_kw.hpp"

namespace slhip {

// The codes of unit u of a row's stage image as signed bytes, lane group g's eight.
template <int FMT>
__device__ __forceinline__ long kw8_codes(const uint8_t* row, int u, int g)
{
    uint2 c = i8_codes8<FMT>(reinterpret_cast<const uint32_t*>(row), u, g);
    constexpr uint32_t off = FMT == SLHIP_FMT_Q4_0 ? 0x08080808u : FMT == SLHIP_FMT_Q5_0 ? 0x10101010u
                             : FMT == SLHIP_FMT_Q6_K ? 0x20202020u : 0u;
    if constexpr (off != 0) {  // c - off per byte: (c + 128) - off cannot borrow, then the top bit flipped back
        c.x = ((c.x | 0x80808080u) - off) ^ 0x80808080u;
        c.y = ((c.y | 0x80808080u) - off) ^ 0x80808080u;
    }
    return static_cast<long>(__builtin_bit_cast(uint64_t, c));
}

template <int FMT, bool DUAL, int TN>
__global__ __launch_bounds__(64 * kKwWaves) __attribute__((amdgpu_waves_per_eu(2))) void matvec_kw8(I8Args a, int gy)
{
    using Geo = KwGeom<FMT>;
    constexpr int NM = DUAL ? 2 : 1;
    constexpr int G = NM * TN;             // 16-row groups: TN tiles of the first matrix, then the second
    constexpr int CH = 16 * TN * Geo::PR;  // 16-byte chunks of one matrix's rows per stage
    constexpr int NL = (CH + 63) / 64;     // loads per matrix
    constexpr bool K6 = FMT == SLHIP_FMT_Q6_K;
    constexpr bool MIN = FMT == SLHIP_FMT_Q4_K || FMT == SLHIP_FMT_Q5_K || FMT == SLHIP_FMT_Q4_1 || FMT == SLHIP_FMT_Q5_1;
    constexpr int WB = 16 * G * Geo::PITCH;  // a wave's stage image
    constexpr int DB = 8 * 16;               // a wave's activation scales of a stage: [unit][token]
    constexpr int XP = 256 + 16;             // a token's codes of a stage, at an odd number of 16-byte slots
    constexpr int RED = TN * NM * kKwWaves * 1024;
    constexpr int IMG = kKwWaves * WB + 16;  // + 16: word reads run past a row's end
    __shared__ __align__(16) uint8_t lds[IMG > RED ? IMG : RED];
    __shared__ __align__(16) uint8_t xim[kKwWaves][16 * XP];
    __shared__ __align__(16) float dsc[kKwWaves][DB], gsc[MIN ? kKwWaves : 1][MIN ? DB : 1];

    const int lane = threadIdx.x & 63;
    const int wave = wave_id();
    const int r = lane & 15, g = lane >> 4;
    // (block order as in matvec_kw: the token tiles of a row tile follow each other on one XCD)
    const int idx = static_cast<int>(blockIdx.x >> 3), rt = idx / gy;
    const int64_t n0 = (static_cast<int64_t>(rt) * 8 + (blockIdx.x & 7)) * (16 * TN);
    if (n0 >= a.N) return;  // block-uniform
    const int64_t t0 = a.t0 + static_cast<int64_t>(idx - rt * gy) * 16;

    const int ns = static_cast<int>(a.K >> 8);
    const int s0 = ns * wave / kKwWaves, s1 = ns * (wave + 1) / kKwWaves;
    uint8_t* img = lds + wave * WB;
    float* ds = dsc[wave];
    float* gs = gsc[MIN ? wave : 0];
    uint8_t* xi = xim[wave];

    f32x4_t acc[G][1];
#pragma unroll
    for (int m = 0; m < G; m++) acc[m][0] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    if (s0 < s1) {  // wave-uniform
        // chunk p = lane + 64 i of a matrix: row p / PR of the tile, chunk p % PR (past the end: the last chunk again)
        uint32_t src[NL], dst[NL];
#pragma unroll
        for (int i = 0; i < NL; i++) {
            int p = lane + 64 * i;
            p = p < CH ? p : CH - 1;
            const int rr = p / Geo::PR, c = p - rr * Geo::PR;
            const int64_t last = a.N - 1 - n0;
            const uint32_t row = static_cast<uint32_t>(rr < last ? rr : last);
            src[i] = row * static_cast<uint32_t>(a.wrow) + (c < Geo::PR - 1 ? 16 * c : Geo::RB - 16);
            dst[i] = static_cast<uint32_t>(rr * Geo::PITCH + 16 * c);
        }
        auto token = [&](int t) {
            const int64_t tok = t0 + t;
            return a.xq + (tok < a.T ? tok : a.T - 1) * (a.K + a.K / 2);
        };
        const uint8_t* xr[4];  // codes: tokens l / 16 + 4 i, chunk l % 16
        const uint8_t* sr[2];  // scales {d, gs0, gs1, 0}: tokens l / 8 + 8 i, unit l % 8
#pragma unroll
        for (int i = 0; i < 4; i++) xr[i] = token(g + 4 * i) + 16 * r;
#pragma unroll
        for (int i = 0; i < 2; i++) sr[i] = token((lane >> 3) + 8 * i) + a.K + 16 * (lane & 7);
        // the next stage's rows, codes and scales (vector types: arrays of HIP's own structs stay in scratch)
        uint4 w[NM][NL];
        u32x4 xn[4];
        f32x4_t sn[2];
        auto load = [&](int s) {
            const int64_t o = n0 * a.wrow + static_cast<int64_t>(s) * Geo::RB;
#pragma unroll
            for (int m = 0; m < NM; m++) {
                const char* base = (m ? a.wu : a.wg) + o;
#pragma unroll
                for (int i = 0; i < NL; i++) {
                    const u32x4_u2 v = *reinterpret_cast<const u32x4_u2*>(base + src[i]);
                    w[m][i] = make_uint4(v.x, v.y, v.z, v.w);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; i++) xn[i] = *reinterpret_cast<const u32x4*>(xr[i] + static_cast<int64_t>(s) * 256);
#pragma unroll
            for (int i = 0; i < 2; i++) sn[i] = *reinterpret_cast<const f32x4_t*>(sr[i] + static_cast<int64_t>(s) * 128);
        };
        load(s0);
        for (int s = s0; s < s1; s++) {
            wave_lds_sync();  // the previous stage's reads, by every lane, come first
#pragma unroll
            for (int m = 0; m < NM; m++)
#pragma unroll
                for (int i = 0; i < NL; i++)
                    *reinterpret_cast<uint4*>(img + m * (16 * TN * Geo::PITCH) + dst[i]) = w[m][i];
#pragma unroll
            for (int i = 0; i < 4; i++) *reinterpret_cast<u32x4*>(xi + (g + 4 * i) * XP + 16 * r) = xn[i];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int at = (lane & 7) * 16 + (lane >> 3) + 8 * i;
                ds[at] = sn[i][0];
                if constexpr (MIN) gs[at] = sn[i][1] + sn[i][2];
            }
            wave_lds_sync();
            __builtin_amdgcn_sched_barrier(0);
            if (s + 1 < s1) load(s + 1);  // (not the last stage again: dual Q4_K, K = 4096, N = 14336, T = 16 25.0 -> 23.7 us)
            __builtin_amdgcn_sched_barrier(0);
            KwScales<FMT> ks[G];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                long C[G];
                float a0[G];
                int h0[G], h1[G];  // Q6_K: the halves' scales
#pragma unroll
                for (int m = 0; m < G; m++) {
                    const uint8_t* row = img + (m * 16 + r) * Geo::PITCH;
                    if ((u & 3) == 0) ks[m].load(row, u >> 2);
                    C[m] = kw8_codes<FMT>(row, u, g);
                    if constexpr (K6) {
                        const uint32_t v = ((u & 2) ? ks[m].mn : ks[m].sc) >> (16 * (u & 1));
                        h0[m] = static_cast<int8_t>(v);
                        h1[m] = static_cast<int8_t>(v >> 8);
                        a0[m] = ks[m].d;
                    } else {
                        a0[m] = ks[m].scale(u, 0);
                    }
                }
                const long x = *reinterpret_cast<const long*>(xi + r * XP + 32 * u + 8 * g);
                const float4 d4 = *reinterpret_cast<const float4*>(ds + u * 16 + 4 * g);
                const float d[4] = {d4.x, d4.y, d4.z, d4.w};
                const i32x4_t z = {0, 0, 0, 0};
                i32x4_t S[G];
#pragma unroll
                for (int m = 0; m < G; m++) {
                    if constexpr (K6) {
                        const long c0 = g < 2 ? C[m] : 0, c1 = g < 2 ? 0 : C[m];
                        const i32x4_t S0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(x, c0, z, 0, 0, 0);
                        const i32x4_t S1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(x, c1, z, 0, 0, 0);
#pragma unroll
                        for (int i = 0; i < 4; i++) S[m][i] = __mul24(S0[i], h0[m]) + __mul24(S1[i], h1[m]);
                    } else {
                        S[m] = __builtin_amdgcn_mfma_i32_16x16x32_i8(x, C[m], z, 0, 0, 0);
                    }
                }
#pragma unroll
                for (int m = 0; m < G; m++) {
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        acc[m][0][i] = fmaf(__fmul_rn(a0[m], d[i]), static_cast<float>(S[m][i]), acc[m][0][i]);
                    asm volatile("" : "+v"(acc[m][0]));  // (nothing emitted: the multiply-adds stay here, as in matvec_kw)
                }
                if constexpr (MIN) {
                    if ((u & 3) == 3) {  // lane (r, g): token r's sum over unit g (A), row r's offset of unit g (B)
                        const float gs0 = gs[((u & 4) + g) * 16 + r];
#pragma unroll
                        for (int m = 0; m < G; m++)
                            acc[m][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(gs0, ks[m].min(g, 0), acc[m][0], 0, 0, 0);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);  // units in order: interleaved, their operands spill
            }
        }
    }
    reduce_store<DUAL, 1, TN>(a, acc, lds, wave, lane, n0, t0);
}

template <int FMT, bool DUAL, int TN>
int launch_kw8(I8Args a, hipStream_t st)
{
    const int64_t rows = ((a.N + 16 * TN - 1) / (16 * TN) + 7) / 8 * 8, toks = (a.T + 15) / 16;
    if (rows > kKwMaxBlocks) return SLHIP_ERR_UNSUPPORTED;
    const int64_t most = kKwMaxBlocks / rows;
    for (int64_t t = 0; t < toks; t += most) {
        const int64_t gy = toks - t < most ? toks - t : most;
        a.t0 = 16 * t;
        matvec_kw8<FMT, DUAL, TN><<<dim3(static_cast<unsigned>(rows * gy)), 64 * kKwWaves, 0, st>>>(a, static_cast<int>(gy));
        const int r = check_launch("matvec_kw8");
        if (r != SLHIP_OK) return r;
    }
    return SLHIP_OK;
}

// tn: the row tiles of a block of the plain form, 1 or (where the format takes it) 2.
template <int FMT>
int launch_kw8_fmt(const I8Args& a, bool dual, int tn, hipStream_t st)
{
    if (dual) return launch_kw8<FMT, true, 1>(a, st);
    if constexpr (kw8_two_tiles(FMT))
        if (tn == 2) return launch_kw8<FMT, false, 2>(a, st);
    return launch_kw8<FMT, false, 1>(a, st);
}

}  // namespace slhip
