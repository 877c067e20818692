#pragma once
// The (dual) product of many tokens with GGUF block-format weights (a prefill's MatMul on the float-rows numerics) on
// the bf16 matrix cores: matmul_tile. The same operands and arithmetic as matvec_kw (matvec_kw.hpp): exact x parts
// times exact codes, each lane scaling its own row.
//
// A block of 4 waves takes 64 tokens x 128 rows (of both matrices together for the dual form); a wave holds 4 x 2 output
// tiles. Against matvec_kw, whose waves each split x for themselves, the block shares x: it is split into its bf16
// parts once per block and 32 values and written to LDS in operand order (a fragment is 64 lanes x 16 bytes in a
// row, so neither the writes nor the reads conflict), two columns of 32 values ahead of the one in use, one barrier
// per column. The weights' stage images lie in one buffer, which the next stage, waiting in registers since the
// stage began, replaces after its last read; a column's codes are decoded while the previous one is multiplied.
// Sums are taken in two levels, a stage's and the stages', so that a long K adds no more rounding than the K split
// of matvec_kw does.
//
// What bounds it: issue, with two waves per SIMD (the vector unit is busy 51%, the matrix cores 39%; with bf16 x and weights at
// 192 blocks for 256 CUs, 13% each, it is waits) -- taking out of a copy of it the split of x, the scaling, the decoding
// or the minimum terms gives 33, 53, 58 or 35 us of 463, the matrix products 98 (Q4_K pair [14336, 4096], T = 512, f32 x,
// 1437 us as 16-token launches, 459 here: 0.79 PFLOP/s of bf16 products). 64 x 128 tiles by 4 waves measured best of
// the shapes tried (128 x 256 by 8 waves 473, 128 x 128 494, 32 x 64 per wave 463 - 495, 12 waves per CU 517 - 790
// spilling); interleaving the matrix and vector instructions by scheduling groups changed nothing. One level of sums
// would be 10% faster and twice as far from the exact result (4.5e-7 against 2.4e-7 of it).
#include "matvec_kw.hpp"

namespace slhip {

constexpr int kTileWaves = 4;
constexpr int kTileTokens = 64;

template <int FMT, bool DUAL, bool XF32>
__global__ __launch_bounds__(64 * kTileWaves) __attribute__((amdgpu_waves_per_eu(2, 2))) void matmul_tile(MatvecArgs a, int gy)
{
    using Geo = KwGeom<FMT>;
    constexpr int MT = kTileTokens / 16;           // token tiles
    constexpr int RT = 2;                          // 16-row tiles per wave, of both matrices together
    constexpr int NW = kTileWaves;
    constexpr int NM = DUAL ? 2 : 1;
    constexpr int RN = RT / NM;                    // 16-row tiles per wave and matrix
    constexpr int BM = kTileTokens;
    constexpr int BN = 16 * RN * NW;               // rows per block and matrix
    constexpr int NP = XF32 ? 3 : 1, NPX = NP + kKwXParts<FMT>;
    constexpr int SKB = Geo::SKB;
    constexpr int CH = NM * BN * Geo::PR;          // 16-byte chunks of a stage
    constexpr int NL = (CH + 64 * NW - 1) / (64 * NW);
    constexpr int FW = MT / NW;                    // x fragments (16 tokens x 32 values) per wave
    constexpr bool FOLD = FMT == SLHIP_FMT_Q2_K || FMT == SLHIP_FMT_Q3_K;
    constexpr bool K6 = FMT == SLHIP_FMT_Q6_K;
    constexpr bool Q2K = FMT == SLHIP_FMT_Q2_K;
    constexpr bool PLAIN = kKwPlain<FMT>;
    constexpr bool MIN = FMT == SLHIP_FMT_Q4_K || FMT == SLHIP_FMT_Q5_K || FMT == SLHIP_FMT_Q4_1 || FMT == SLHIP_FMT_Q5_1 || Q2K;
    constexpr int NX = MIN ? (Q2K ? 2 : 1) : 0;    // x sums kept per token and block
    constexpr int NCH = K6 ? 2 : 1;                // product chains per tile (Q6_K: one per value half)
    constexpr int NC = K6 ? 2 : Geo::NC;           // operand vectors per row and block
    constexpr int NB = 3;                          // x buffers
    __shared__ __align__(16) uint8_t img[NM * BN * Geo::PITCH + 16];  // + 16: word reads run past a row's end
    __shared__ __align__(16) uint4 xs[NB][MT][NPX][64];
    __shared__ float xsum[NX ? 8 : 1][NX ? NX : 1][NX ? BM : 1];  // of the last eight blocks

    const int lane = threadIdx.x & 63;
    const int wave = wave_id();
    const int r = lane & 15, g = lane >> 4;
    const int idx = static_cast<int>(blockIdx.x >> 3), rt = idx / gy;
    const int64_t n0 = (static_cast<int64_t>(rt) * 8 + (blockIdx.x & 7)) * BN;  // token tiles of a row tile on one XCD
    if (n0 >= a.N) return;  // block-uniform
    const int64_t t0 = a.t0 + static_cast<int64_t>(idx - rt * gy) * BM;
    const int ns = static_cast<int>(a.K / (32 * SKB));
    const int nk = SKB * ns;

    // chunk p = threadIdx + 256 i of a stage: row (of both matrices) and chunk (past the end: the last chunk again)
    auto chunk_row = [&](int i, int& c) {
        int p = static_cast<int>(threadIdx.x) + 64 * NW * i;
        if (CH % (64 * NW) != 0) p = p < CH ? p : CH - 1;
        const int rr = p / Geo::PR;
        c = p - rr * Geo::PR;
        return rr;
    };
    uint32_t src[NL];
    const int64_t mdiff = DUAL ? a.wu - a.wg : 0;
#pragma unroll
    for (int i = 0; i < NL; i++) {
        int c;
        const int rr = chunk_row(i, c);
        const int64_t last = a.N - 1 - n0;
        const int row = rr % BN < last ? rr % BN : static_cast<int>(last);
        src[i] = static_cast<uint32_t>(row) * static_cast<uint32_t>(a.wrow) + (c < Geo::PR - 1 ? 16 * c : Geo::RB - 16);
    }
    uint4 w[NL];
    auto load_w = [&](int s) {
        const char* base = a.wg + n0 * a.wrow + static_cast<int64_t>(s) * Geo::RB;
#pragma unroll
        for (int i = 0; i < NL; i++) {
            int c;
            const char* p = base + src[i];
            if (DUAL) p += chunk_row(i, c) >= BN ? mdiff : 0;
            const u32x4_u2 v = *reinterpret_cast<const u32x4_u2*>(p);
            w[i] = make_uint4(v.x, v.y, v.z, v.w);
        }
    };
    auto store_w = [&]() {
#pragma unroll
        for (int i = 0; i < NL; i++) {
            int c;
            const int rr = chunk_row(i, c);
            *reinterpret_cast<uint4*>(img + rr * Geo::PITCH + 16 * c) = w[i];
        }
    };
    // the wave's x fragments: token r of the fragment, values 8g .. 8g + 7
    struct X {
        float4 f[2];
        uint4 b;
    };
    X x[2][FW];
    const char* xp[FW];
#pragma unroll
    for (int f = 0; f < FW; f++) {
        int64_t tok = t0 + 16 * (wave + NW * f) + r;
        tok = tok < a.T ? tok : a.T - 1;
        xp[f] = static_cast<const char*>(a.x) + (tok * a.xs + 8 * g) * (XF32 ? 4 : 2);
    }
    auto load_x = [&](int k, int b) {  // block column k
        const int64_t o = static_cast<int64_t>(k < nk ? k : nk - 1) * (XF32 ? 128 : 64);
#pragma unroll
        for (int f = 0; f < FW; f++) {
            if constexpr (XF32) {
                x[b][f].f[0] = *reinterpret_cast<const float4*>(xp[f] + o);
                x[b][f].f[1] = *reinterpret_cast<const float4*>(xp[f] + o + 16);
            } else {
                x[b][f].b = *reinterpret_cast<const uint4*>(xp[f] + o);
            }
        }
    };
    uint4 xq[FW][NPX];  // the wave's split fragments of a block column, and their sums
    float xps[FW];
    auto split_x = [&](int f, int b) {
        float v[8];
        xps[f] = 0.0f;
        if constexpr (XF32) {
            const float4 p = x[b][f].f[0], q = x[b][f].f[1];
            v[0] = p.x; v[1] = p.y; v[2] = p.z; v[3] = p.w;
            v[4] = q.x; v[5] = q.y; v[6] = q.z; v[7] = q.w;
            xps[f] = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
            split3_finite(v, xq[f][0], xq[f][1 % NP], xq[f][2 % NP]);
        } else {
            xq[f][0] = x[b][f].b;
            if constexpr (MIN) {
                Vec<SLHIP_BF16>::unpack(x[b][f].b, v);
                xps[f] = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
            }
        }
    };
    auto store_x = [&](int k, int buf, int b) {  // block column k's parts and sums into LDS
#pragma unroll
        for (int f = 0; f < FW; f++) {
            const int fi = wave + NW * f;
            if constexpr (XF32) {
                // a non-finite x has no remainders (inf - inf): the guarded split, where some lane's sum is not finite
                if (__builtin_amdgcn_ballot_w64(!(fabsf(xps[f]) <= 3.4028235e38f)) != 0) {
                    const float4 p = x[b][f].f[0], q = x[b][f].f[1];
                    const float v[8] = {p.x, p.y, p.z, p.w, q.x, q.y, q.z, q.w};
                    split3(v, xq[f][0], xq[f][1 % NP], xq[f][2 % NP]);
                }
            }
#pragma unroll
            for (int p = 0; p < NP; p++) xs[buf][fi][p][lane] = xq[f][p];
            if constexpr (NPX > NP) xs[buf][fi][NP][lane] = finite_bf16(xq[f][0]);
            if constexpr (MIN) {
                const float p01 = xps[f] + __shfl_xor(xps[f], 16);
                const float other = __shfl_xor(p01, 32);
                if constexpr (Q2K) {  // lane groups 0 and 1 hold the first half's sum, 2 and 3 the second's
                    if ((g & 1) == 0) xsum[k & 7][g >> 1][16 * fi + r] = p01;
                } else {
                    if (g == 0) xsum[k & 7][0][16 * fi + r] = p01 + other;
                }
            }
        }
    };

    // Two levels of sums: a stage's products, then the stages.
    f32x4_t acc[RT][MT], tot[RT][MT];
#pragma unroll
    for (int m = 0; m < RT; m++)
#pragma unroll
        for (int t = 0; t < MT; t++) acc[m][t] = tot[m][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    KwScales<FMT> ks[RT];
    uint4 C[2][RT][NC];
    float a0[2][RT][NCH], mn[2][RT][NX ? NX : 1];
    auto decode = [&](int u, int m) {  // block u of the stage, row group m
        const uint8_t* row = img + ((m / RN) * BN + (wave * RN + m % RN) * 16 + r) * Geo::PITCH;
        if constexpr (!PLAIN)
            if ((u & 3) == 0) {
                ks[m].load(row, u >> 2);
                if constexpr (MIN) {
#pragma unroll
                    for (int h = 0; h < NX; h++) mn[u >> 2][m][h] = ks[m].min(g, h);
                }
            }
        const int b = u & 1;
        a0[b][m][0] = 1.0f;
        uint4 v[Geo::NC];
        kw_codes<FMT>(row, u, g, a0[b][m][0], v);
        if constexpr (K6) {
            const uint32_t keep = g < 2 ? ~0u : 0u;
            C[b][m][0] = make_uint4(v[0].x & keep, v[0].y & keep, v[0].z & keep, v[0].w & keep);
            C[b][m][NC - 1] = make_uint4(v[0].x & ~keep, v[0].y & ~keep, v[0].z & ~keep, v[0].w & ~keep);
        } else {
#pragma unroll
            for (int c = 0; c < NC; c++) C[b][m][c] = v[c];
        }
        if constexpr (!FOLD && !PLAIN) {
#pragma unroll
            for (int h = 0; h < NCH; h++) a0[b][m][h] = ks[m].scale(u, h);
        }
    };

    load_x(0, 0);
    load_x(1, 1);
    load_w(0);
#pragma unroll
    for (int k = 0; k < 2; k++) {
#pragma unroll
        for (int f = 0; f < FW; f++) split_x(f, k);
        store_x(k, k, k);
        load_x(k + 2, k);
    }
    store_w();
    int buf = 0;  // the buffer of the current block column
    for (int s = 0; s < ns; s++) {
        load_w(s + 1 < ns ? s + 1 : s);
#pragma unroll
        for (int u = 0; u < SKB; u++) {
            const int k = SKB * s + u;
            __syncthreads();  // column k + 1's x (and, at u = 0, the stage) is in LDS; column k - 1 is no longer read
            const int b1 = buf == NB - 1 ? 0 : buf + 1, b2 = b1 == NB - 1 ? 0 : b1 + 1;
            if (u == 0) {
#pragma unroll
                for (int m = 0; m < RT; m++) decode(0, m);
            }
            uint4 P[2][NPX];
#pragma unroll
            for (int p = 0; p < NPX; p++) P[0][p] = xs[buf][0][p][lane];
            f32x4_t c[RT][NCH];
            auto scale = [&](int t) {  // the tile's products of this block times the rows' multipliers
                if constexpr (!PLAIN) {
#pragma unroll
                    for (int m = 0; m < RT; m++)
#pragma unroll
                        for (int h = 0; h < NCH; h++)
#pragma unroll
                            for (int i = 0; i < 4; i++)
                                acc[m][t][i] = u == 0 && h == 0 ? a0[u & 1][m][h] * c[m][h][i]
                                                                : fmaf(a0[u & 1][m][h], c[m][h][i], acc[m][t][i]);
                }
#pragma unroll
                for (int m = 0; m < RT; m++) asm volatile("" : "+v"(acc[m][t]));
            };
#pragma unroll
            for (int t = 0; t < MT; t++) {
                if (t + 1 < MT) {
#pragma unroll
                    for (int p = 0; p < NPX; p++) P[(t + 1) & 1][p] = xs[buf][t + 1][p][lane];
                }
                if (u + 1 < SKB && t < RT) decode(u + 1, t);
                if (t >= MT - FW) split_x(t - (MT - FW), u & 1);
#pragma unroll
                for (int p = 0; p < NP; p++)
#pragma unroll
                    for (int q = 0; q < (K6 ? 2 : kKwParts<FMT>); q++)
#pragma unroll
                        for (int m = 0; m < RT; m++) {
                            const f32x4_t z = {0.0f, 0.0f, 0.0f, 0.0f};
                            const int h = K6 ? q : 0;
                            const bool first = p == 0 && (K6 || q == 0);
                            f32x4_t& d = PLAIN ? acc[m][t] : c[m][h];
                            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(P[t & 1][kw_x<FMT>(NP, p, q)]), as_bf16x8(C[u & 1][m][kw_part<FMT>(p, q)]),
                                                                        first && (!PLAIN || u == 0) ? z : d, 0, 0, 0);
                        }
                scale(t);
                __builtin_amdgcn_sched_barrier(0);  // tiles in order: interleaved, their operands spill
            }
            if constexpr (MIN) {
                if ((u & 3) == 3) {  // lane (r, g): token r's sum over block g (A), row r's minimum of block g (B)
#pragma unroll
                    for (int h = 0; h < NX; h++)
#pragma unroll
                        for (int t = 0; t < MT; t++) {
                            const float xa = xsum[(u & 4) + g][h][16 * t + r];
#pragma unroll
                            for (int m = 0; m < RT; m++)
                                acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa, mn[u >> 2][m][h], acc[m][t], 0, 0, 0);
                        }
                }
            }
            if (u == SKB - 1) {
#pragma unroll
                for (int m = 0; m < RT; m++)
#pragma unroll
                    for (int t = 0; t < MT; t++) {
                        tot[m][t] += acc[m][t];
                        asm volatile("" : "+v"(tot[m][t]));
                    }
                store_w();  // (the image was last read for block SKB - 1, before this column's barrier)
            }
            if (k + 2 < nk) store_x(k + 2, b2, u & 1);
            load_x(k + 4, u & 1);
            buf = b1;
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int m = 0; m < RN; m++)
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                store_sum<DUAL>(a, t0 + 16 * t + 4 * g + i, n0 + 16 * (wave * RN + m) + r, tot[m][t][i],
                                DUAL ? tot[(m + RN) % RT][t][i] : 0.0f);
}

template <int FMT, bool DUAL, bool XF32>
int launch_tile(MatvecArgs a, hipStream_t st)
{
    constexpr int BM = kTileTokens, BN = 32 * kTileWaves / (DUAL ? 2 : 1);
    const int64_t rows = ((a.N + BN - 1) / BN + 7) / 8 * 8, toks = (a.T + BM - 1) / BM;
    if (rows > kKwMaxBlocks) return SLHIP_ERR_UNSUPPORTED;
    const int64_t most = kKwMaxBlocks / rows;
    for (int64_t t = 0; t < toks; t += most) {
        const int64_t gy = toks - t < most ? toks - t : most;
        a.t0 = BM * t;
        matmul_tile<FMT, DUAL, XF32>
            <<<dim3(static_cast<unsigned>(rows * gy)), 64 * kTileWaves, 0, st>>>(a, static_cast<int>(gy));
        const int r = check_launch("matmul_tile");
        if (r != SLHIP_OK) return r;
    }
    return SLHIP_OK;
}

template <int FMT>
int launch_tile_fmt(const MatvecArgs& a, bool dual, hipStream_t st)
{
    if (a.xt == SLHIP_F32) return dual ? launch_tile<FMT, true, true>(a, st) : launch_tile<FMT, false, true>(a, st);
    return dual ? launch_tile<FMT, true, false>(a, st) : launch_tile<FMT, false, false>(a, st);
}

}  // namespace slhip
