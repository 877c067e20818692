#pragma once
// The several-token (dual) matvec on GGUF block-format weights with f32 or bf16 activations (the float-rows
// numerics: the MatMul carries f32_activations, or its row count is outside the integer-dot rule), on the bf16
// matrix cores: matvec_kw. Any number of tokens, one launch.
//
// A block of 8 waves takes 16 MT tokens x TN 16-row tiles (gate/up pairs of tiles for the dual form) and splits
// K over its waves: a wave walks its own 256-value stages with nothing shared and no barrier until the partial
// sums meet in LDS at the end. A stage's rows come by 16-byte loads (consecutive lanes, consecutive chunks of a
// row) into registers, one stage ahead of the arithmetic, and pass through the wave's own LDS region only to
// change lanes: the loads of lane l are chunks of any row, the matrix cores want row l % 16. Loads, stores and
// waits are all the compiler's, which knows every register and every LDS byte involved.
//
// v_mfma_f32_16x16x32_bf16 multiplies the tokens' x (A: lane l holds token l % 16, values 8 (l / 16) .. + 7; f32 x
// as three bf16 parts h + m + l == x exactly, bf16 x as is) with a block's codes as exact bf16 (B: lane l holds
// row l % 16, the same values), so lane l's sums are tokens 4 (l / 16) + i of row l % 16: each lane decodes its
// own row's block scale once and applies it with one fma per output. Q6_K's two 16-value scale groups take two
// chains with the other half's codes masked to zero; Q2_K's and Q3_K's group scales are folded into the codes.
// Minimum terms (Q4_K / Q5_K -dmin mn sum(x), Q4_1 / Q5_1 +m sum(x), Q2_K -dmin m per half) of four blocks are one
// 16 x 16 x 4 f32 product (tokens x blocks . blocks x rows).
//
// Arithmetic against the reference (MatMulOp's f32 dot of dequantized rows): every product code x part is
// exact and the sums are f32, so the result is the f32 evaluation of sum(scale * code * x) + min terms in
// another order: within f32 accumulation of those terms.
//
// What bounds it: instruction issue (Q6_K K = 14336, N = 4096, T = 6: the vector unit is busy 79%, the matrix cores 16%), x's split
// above all, which is why the wider blocks (more 16-row groups per split) win as soon as they still fill the chip; the
// dispatch (matvec_kw.hip) picks the shape. Against the launch per 16 tokens that it replaces (the previous kernels,
// barriers per stage), K = 4096, f32 x, us: Q4_K N = 4096 12.8 -> 12.5 (T = 16), 51 -> 16 (T = 64), 102 -> 25 (T = 128);
// Q6_K K = 14336, N = 4096, T = 6 36.7 -> 29.6; bf16 K = 2880, N = 4096, T = 331, bf16 x 175 -> 30 (matmul_tile); f16
// (from the VALU kernel) N = 4096, T = 16 47 -> 13, T = 512 1454 -> 130.
#include "mq.hpp"

namespace slhip {

constexpr int kKwWaves = 8;
constexpr int64_t kKwMaxBlocks = int64_t{1} << 22;

// A stage is 256 values of a row: RB bytes in PR 16-byte chunks, the last chunk being the last 16 bytes (where RB
// is not a multiple of 16 it repeats the previous chunk's end, so that nothing past the row is read). In the
// image, chunk c sits at byte 16 c: bytes from TAIL on lie SHIFT further in. The pitch is an odd number of 16-byte
// slots, so that the 16 rows a wave reads at once spread over the LDS banks.
template <int FMT>
struct KwGeom {
    static constexpr int SKB = 8;  // 32-value blocks per stage
    static constexpr int NC = 1;   // operand vectors of a code
    static constexpr int RB = Fmt<FMT>::BB * (256 / Fmt<FMT>::BS);
    static constexpr int PR = (RB + 15) / 16;
    static constexpr int TAIL = 16 * (PR - 1);
    static constexpr int SHIFT = 16 * PR - RB;
    static constexpr int PITCH = 16 * (PR | 1);
};
// Unquantized weights: stages of 64 values; f16 values as two bf16 parts (11 significant bits: exact). A non-finite f16
// has no second part, and must meet only the first part of x (the others may be 0, and 0 inf is NaN), so C[2] is the
// first part without its non-finite values; likewise a non-finite x must not meet the second part (kw_x below).
template <>
struct KwGeom<SLHIP_FMT_BF16> {
    static constexpr int SKB = 2, NC = 1, RB = 128, PR = 8, TAIL = 112, SHIFT = 0, PITCH = 144;
};
template <>
struct KwGeom<SLHIP_FMT_F16> {
    static constexpr int SKB = 2, NC = 3, RB = 128, PR = 8, TAIL = 112, SHIFT = 0, PITCH = 144;
};
template <int FMT> constexpr int kKwParts = FMT == SLHIP_FMT_F16 ? 2 : 1;  // parts of a code in a product
// the vectors that part p of x and part c of a code take in their product
template <int FMT>
constexpr int kw_part(int p, int c)
{
    return FMT == SLHIP_FMT_F16 && p > 0 && c == 0 ? 2 : c;
}
template <int FMT>
constexpr int kw_x(int np, int p, int c)
{
    return FMT == SLHIP_FMT_F16 && p == 0 && c == 1 ? np : p;
}
template <int FMT> constexpr int kKwXParts = FMT == SLHIP_FMT_F16 ? 1 : 0;  // vectors of x beyond its parts
template <int FMT> constexpr bool kKwPlain = FMT == SLHIP_FMT_BF16 || FMT == SLHIP_FMT_F16;  // values, no scales

typedef uint32_t u32x4_u2 __attribute__((ext_vector_type(4), aligned(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

// Four bf16 pairs without their non-finite values.
__device__ __forceinline__ uint4 finite_bf16(const uint4& v)
{
    auto keep = [](uint32_t w) {
        const uint32_t lo = (w & 0x7F80u) == 0x7F80u ? 0u : 0xFFFFu, hi = (w & 0x7F800000u) == 0x7F800000u ? 0u : 0xFFFF0000u;
        return w & (lo | hi);
    };
    return make_uint4(keep(v.x), keep(v.y), keep(v.z), keep(v.w));
}

// Eight 4-bit codes in the bytes of lo, hi (0 .. 15) as four bf16 pairs. A byte n < 16 read as E4M3 is n 2^-9
// exactly (subnormals and the first binade share one step), so a scaled conversion gives two codes each.
__device__ __forceinline__ uint4 nibbles_bf16(uint32_t lo, uint32_t hi)
{
    auto two = [](bf16x2_t v) { return __builtin_bit_cast(uint32_t, v); };
    return make_uint4(two(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, false)),
                      two(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, true)),
                      two(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, false)),
                      two(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, true)));
}

// The multipliers of the four blocks u = 4h .. 4h + 3 of one row's stage image, prepared once per four blocks:
// scale(u) is the f32 multiplier of block u (of its value half hf for Q6_K), min(j, hf) the minimum coefficient
// of block 4h + j (j may differ between lanes).
template <int FMT>
struct KwScales {
    const uint8_t* row;
    int h;
    uint32_t sc, mn;
    float d, dm;

    __device__ __forceinline__ void load(const uint8_t* r, int half)
    {
        row = r;
        h = half;
        if constexpr (FMT == SLHIP_FMT_Q4_K || FMT == SLHIP_FMT_Q5_K) {
            const uint4 w = *reinterpret_cast<const uint4*>(r);  // {d, dmin, 12 bytes of 6-bit scales and minima}
            d = f16_lo(w.x);
            dm = f16_hi(w.x);
            sc = half ? (w.w & 0x0F0F0F0Fu) | ((w.y >> 2) & 0x30303030u) : w.y & 0x3F3F3F3Fu;
            mn = half ? ((w.w >> 4) & 0x0F0F0F0Fu) | ((w.z >> 2) & 0x30303030u) : w.z & 0x3F3F3F3Fu;
        } else if constexpr (FMT == SLHIP_FMT_Q6_K) {
            d = static_cast<float>(*reinterpret_cast<const _Float16*>(r + 208 + KwGeom<FMT>::SHIFT));
            const uint2 w = *reinterpret_cast<const uint2*>(r + 192 + 8 * half);  // two int8 scales per block
            sc = w.x;
            mn = w.y;
        } else if constexpr (FMT == SLHIP_FMT_Q2_K) {
            d = static_cast<float>(*reinterpret_cast<const _Float16*>(r + 80 + KwGeom<FMT>::SHIFT));
            dm = static_cast<float>(*reinterpret_cast<const _Float16*>(r + 82 + KwGeom<FMT>::SHIFT));
        }
    }
    // the multiplier of block u (compile-time) and its value half hf (Q6_K)
    __device__ __forceinline__ float scale(int u, int hf) const
    {
        if constexpr (FMT == SLHIP_FMT_Q4_K || FMT == SLHIP_FMT_Q5_K)
            return __fmul_rn(d, static_cast<float>((sc >> (8 * (u & 3))) & 0xFFu));
        else if constexpr (FMT == SLHIP_FMT_Q6_K) {
            const uint32_t w = (u & 2) ? mn : sc;
            return __fmul_rn(d, static_cast<float>(static_cast<int8_t>(w >> (16 * (u & 1) + 8 * hf))));
        } else
            return static_cast<float>(*reinterpret_cast<const _Float16*>(row + u * Fmt<FMT>::BB));
    }
    // the minimum coefficient of block 4h + j, value half hf (Q2_K)
    __device__ __forceinline__ float min(int j, int hf) const
    {
        if constexpr (FMT == SLHIP_FMT_Q4_K || FMT == SLHIP_FMT_Q5_K)
            return -__fmul_rn(dm, static_cast<float>((mn >> (8 * j)) & 0xFFu));
        else if constexpr (FMT == SLHIP_FMT_Q2_K)
            return -__fmul_rn(dm, static_cast<float>(row[2 * (4 * h + j) + hf] >> 4));
        else
            return static_cast<float>(*reinterpret_cast<const _Float16*>(row + (4 * h + j) * Fmt<FMT>::BB + 2));
    }
};

// The codes of block u of a row image, lane group g's eight (values 8g .. 8g + 7), as exact bf16 (Q2_K / Q3_K: times
// their group's scale, the super-block's d in `d`).
template <int FMT>
__device__ __forceinline__ uint4 kw_codes1(const uint8_t* row, int u, int g, float& d)
{
    if constexpr (FMT == SLHIP_FMT_Q4_K) {
        const uint2 w = *reinterpret_cast<const uint2*>(row + 16 + 32 * (u >> 1) + 8 * g);
        const uint32_t sh = 4 * static_cast<uint32_t>(u & 1);
        return nibbles_bf16((w.x >> sh) & 0x0F0F0F0Fu, (w.y >> sh) & 0x0F0F0F0Fu);
    } else if constexpr (FMT == SLHIP_FMT_Q4_1) {
        const int o = u * Fmt<FMT>::BB + Fmt<FMT>::QS + 8 * (g & 1);  // 4-byte aligned: BB = 20
        const uint32_t* w = reinterpret_cast<const uint32_t*>(row + o);
        const uint32_t sh = 4 * static_cast<uint32_t>(g >> 1);
        return nibbles_bf16((w[0] >> sh) & 0x0F0F0F0Fu, (w[1] >> sh) & 0x0F0F0F0Fu);
    } else if constexpr (FMT == SLHIP_FMT_Q5_K) {
        return q4k_codes<true>(row, 0, u, g);
    } else if constexpr (FMT == SLHIP_FMT_Q6_K) {
        return q6k_codes(row, 0, u, g);
    } else if constexpr (FMT == SLHIP_FMT_Q2_K || FMT == SLHIP_FMT_Q3_K) {
        return q23k_codes_scaled<FMT == SLHIP_FMT_Q3_K>(row, 0, u, g, d, KwGeom<FMT>::SHIFT);
    } else {
        return mq_codes<FMT>(row, u * Fmt<FMT>::BB, g);
    }
}

// The same as the MFMA's NC operand vectors: one, or an f16 value's two bf16 parts hi + lo (a non-finite one keeps hi).
template <int FMT>
__device__ __forceinline__ void kw_codes(const uint8_t* row, int u, int g, float& d, uint4 (&C)[KwGeom<FMT>::NC])
{
    if constexpr (kKwPlain<FMT>) {
        const uint4 v = *reinterpret_cast<const uint4*>(row + 64 * u + 16 * g);
        if constexpr (FMT == SLHIP_FMT_F16) {
            float f[8];
            Vec<SLHIP_F16>::unpack(v, f);
            split2(f, C[0], C[1]);
            C[2] = finite_bf16(C[0]);
        } else {
            C[0] = v;
        }
    } else {
        C[0] = kw_codes1<FMT>(row, u, g, d);
    }
}

// acc[m][t] += one block's product: the token tile's x parts P (A) with the codes of G row groups (B), each lane's
// sums times its own row's multiplier (Q6_K: per value half).
template <int FMT, int NP, int G, int MT>
__device__ __forceinline__ void block_product(const uint4 (&P)[NP + kKwXParts<FMT>], const uint4 (&Cs)[G][KwGeom<FMT>::NC], const float (&a0)[G],
                                              const float (&a1)[G], int g, f32x4_t (&acc)[G][MT], int t)
{
    const f32x4_t z = {0.0f, 0.0f, 0.0f, 0.0f};
    uint4 C[G];
#pragma unroll
    for (int m = 0; m < G; m++) C[m] = Cs[m][0];
    if constexpr (kKwPlain<FMT>) {
        // (parts of one block first, then one addition to the running sum: adding each part to it rounds more often)
        f32x4_t d[G];
#pragma unroll
        for (int m = 0; m < G; m++) d[m] = z;
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int c = 0; c < kKwParts<FMT>; c++)
#pragma unroll
                for (int m = 0; m < G; m++)
                    d[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(P[kw_x<FMT>(NP, p, c)]),
                                                                   as_bf16x8(Cs[m][kw_part<FMT>(p, c)]), d[m], 0, 0, 0);
#pragma unroll
        for (int m = 0; m < G; m++) acc[m][t] += d[m];
    } else if constexpr (FMT == SLHIP_FMT_Q6_K) {
        const uint32_t keep = g < 2 ? ~0u : 0u;
#pragma unroll
        for (int m = 0; m < G; m++) {
            const uint4 C0 = make_uint4(C[m].x & keep, C[m].y & keep, C[m].z & keep, C[m].w & keep);
            const uint4 C1 = make_uint4(C[m].x & ~keep, C[m].y & ~keep, C[m].z & ~keep, C[m].w & ~keep);
            f32x4_t c0 = z, c1 = z;
#pragma unroll
            for (int p = 0; p < NP; p++) {
                c0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(P[p]), as_bf16x8(C0), c0, 0, 0, 0);
                c1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(P[p]), as_bf16x8(C1), c1, 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) acc[m][t][i] = fmaf(a1[m], c1[i], fmaf(a0[m], c0[i], acc[m][t][i]));
        }
    } else {
        f32x4_t c[G];
#pragma unroll
        for (int m = 0; m < G; m++) c[m] = z;
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int m = 0; m < G; m++)
                c[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(P[p]), as_bf16x8(C[m]), c[m], 0, 0, 0);
#pragma unroll
        for (int m = 0; m < G; m++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[m][t][i] = fmaf(a0[m], c[m][i], acc[m][t][i]);
    }    // (nothing emitted: keeps the multiply-adds here, before the next barrier or branch; sunk below it, the products
    // of every tile stay alive and spill)
#pragma unroll
    for (int m = 0; m < G; m++) asm volatile("" : "+v"(acc[m][t]));
}

// A lane's eight values of x as the MFMA's parts, and their sum.
__device__ __forceinline__ float x_parts(const float (&v)[8], uint4* P)
{
    const float ps = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    // the split's guard against non-finite x (whose remainders would be NaN) only when some lane's eight values
    // have a non-finite (or overflowing) sum: a wave-uniform test
    if (__builtin_amdgcn_ballot_w64(!(fabsf(ps) <= 3.4028235e38f)) == 0) split3_finite(v, P[0], P[1], P[2]);
    else split3(v, P[0], P[1], P[2]);
    return ps;
}

// y[t, n] from the finished sums of one output (gate and up for the dual form).
template <bool DUAL, class Args>
__device__ __forceinline__ void store_sum(const Args& a, int64_t t, int64_t n, float sg, float su)
{
    float out = sg;
    if (DUAL) {
        const float act = a.act == SLHIP_ACT_SILU        ? activate<SLHIP_ACT_SILU>(sg)
                          : a.act == SLHIP_ACT_GELU_TANH ? activate<SLHIP_ACT_GELU_TANH>(sg)
                                                         : activate<SLHIP_ACT_GELU_ERF>(sg);
        out = act * su;
    }
    if (t < a.T && n < a.N) {
        if (!DUAL && a.bias) out = out + a.bias[n];
        if (a.yt == SLHIP_F32)
            static_cast<float*>(a.y)[t * a.ys + n] = out;
        else
            static_cast<uint16_t*>(a.y)[t * a.ys + n] = static_cast<uint16_t>(f32_to_bf16_bits(out));
    }
}

// The waves' partial sums of a block's tiles meet in the (now idle) stage memory, up to 4 output tiles per round:
// [wave][tile][matrix][lane]; wave q finishes tile q of the round.
template <bool DUAL, int MT, int TN, int G, class Args>
__device__ __forceinline__ void reduce_store(const Args& a, const f32x4_t (&acc)[G][MT], uint8_t* lds, int wave, int lane,
                                             int64_t n0, int64_t t0)
{
    constexpr int NM = DUAL ? 2 : 1, UN = TN * MT, UR = UN < 4 ? UN : 4;
    const int r = lane & 15, g = lane >> 4;
    f32x4_t* red = reinterpret_cast<f32x4_t*>(lds);
#pragma unroll
    for (int q0 = 0; q0 < UN; q0 += UR) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < UR; q++)
#pragma unroll
            for (int m = 0; m < NM; m++)
                red[((wave * UR + q) * NM + m) * 64 + lane] = acc[m * TN + (q0 + q) / MT][(q0 + q) % MT];
        __syncthreads();
        if (wave < UR) {
            f32x4_t sg = red[(wave * NM) * 64 + lane], su = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            if (DUAL) su = red[(wave * NM + NM - 1) * 64 + lane];
#pragma unroll
            for (int v = 1; v < kKwWaves; v++) {
                sg += red[((v * UR + wave) * NM) * 64 + lane];
                if (DUAL) su += red[((v * UR + wave) * NM + NM - 1) * 64 + lane];
            }
            const int64_t n = n0 + 16 * ((q0 + wave) / MT) + r;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int64_t t = t0 + 16 * ((q0 + wave) % MT) + 4 * g + i;
                store_sum<DUAL>(a, t, n, sg[i], su[i]);
            }
        }
    }
}

template <int FMT, bool DUAL, bool XF32, int MT, int TN>
__global__ __launch_bounds__(64 * kKwWaves) __attribute__((amdgpu_waves_per_eu(2, 2))) void matvec_kw(MatvecArgs a, int gy)
{
    using Geo = KwGeom<FMT>;
    constexpr int NM = DUAL ? 2 : 1;
    constexpr int G = NM * TN;                         // 16-row groups: TN tiles of the first matrix, then the second
    constexpr int NP = XF32 ? 3 : 1;                   // bf16 parts of x
    constexpr int CH = 16 * TN * Geo::PR;              // 16-byte chunks of one matrix's rows per stage
    constexpr int NL = (CH + 63) / 64;                 // loads per matrix
    constexpr int SKB = Geo::SKB;
    constexpr int PD = MT == 4 ? 1 : MT == 2 || SKB == 2 ? 2 : 4;  // x blocks in flight ahead of the one in use: 8 (f32) or 4 registers each per token tile
    constexpr bool FOLD = FMT == SLHIP_FMT_Q2_K || FMT == SLHIP_FMT_Q3_K;
    constexpr bool K6 = FMT == SLHIP_FMT_Q6_K;
    constexpr bool Q2K = FMT == SLHIP_FMT_Q2_K;
    constexpr bool MIN = FMT == SLHIP_FMT_Q4_K || FMT == SLHIP_FMT_Q5_K || FMT == SLHIP_FMT_Q4_1 || FMT == SLHIP_FMT_Q5_1 || Q2K;
    constexpr int WB = 16 * G * Geo::PITCH;            // a wave's stage image
    constexpr int UN = TN * MT;                        // output tiles
    constexpr int UR = UN < 4 ? UN : 4;                // of them per reduction round
    constexpr int RED = UR * NM * kKwWaves * 1024;
    constexpr int LDS = kKwWaves * WB + 16 > RED ? kKwWaves * WB + 16 : RED;  // + 16: word reads run past a row's end
    __shared__ __align__(16) uint8_t lds[LDS];

    const int lane = threadIdx.x & 63;
    const int wave = wave_id();
    const int r = lane & 15, g = lane >> 4;
    // Consecutive blocks go to the 8 XCDs in turn; the token tiles of one row tile follow each other on one XCD, so
    // that its L2 serves the weights again.
    const int idx = static_cast<int>(blockIdx.x >> 3), rt = idx / gy;
    const int64_t n0 = (static_cast<int64_t>(rt) * 8 + (blockIdx.x & 7)) * (16 * TN);
    if (n0 >= a.N) return;  // block-uniform
    const int64_t t0 = a.t0 + static_cast<int64_t>(idx - rt * gy) * (16 * MT);

    const int ns = static_cast<int>(a.K / (32 * SKB));
    const int s0 = ns * wave / kKwWaves, s1 = ns * (wave + 1) / kKwWaves;
    uint8_t* img = lds + wave * WB;

    f32x4_t acc[G][MT];
#pragma unroll
    for (int m = 0; m < G; m++)
#pragma unroll
        for (int t = 0; t < MT; t++) acc[m][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

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
        uint4 w[NM][NL];
        auto load_w = [&](int s) {
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
        };
        struct X {
            float4 f[2];
            uint4 b;
        };
        X x[PD][MT];
        const char* xp[MT];
#pragma unroll
        for (int t = 0; t < MT; t++) {
            int64_t tok = t0 + 16 * t + r;
            tok = tok < a.T ? tok : a.T - 1;
            xp[t] = static_cast<const char*>(a.x) + (tok * a.xs + 8 * g) * (XF32 ? 4 : 2);
        }
        auto load_x = [&](uint32_t k, int b) {  // 32-value block k of the tokens' rows (unsigned: signed, the 4 x 4 blocks spill more)
#pragma unroll
            for (int t = 0; t < MT; t++) {
                if constexpr (XF32) {
                    const float4* p = reinterpret_cast<const float4*>(xp[t] + static_cast<uint64_t>(k) * 128);
                    x[b][t].f[0] = p[0];
                    x[b][t].f[1] = p[1];
                } else {
                    x[b][t].b = *reinterpret_cast<const uint4*>(xp[t] + static_cast<uint64_t>(k) * 64);
                }
            }
        };
        load_w(s0);
#pragma unroll
        for (int u = 0; u < PD; u++) load_x(s0 * SKB + u, u);

        for (int s = s0; s < s1; s++) {
            wave_lds_sync();  // the previous stage's reads, by every lane, come first
#pragma unroll
            for (int m = 0; m < NM; m++)
#pragma unroll
                for (int i = 0; i < NL; i++)
                    *reinterpret_cast<uint4*>(img + m * (16 * TN * Geo::PITCH) + dst[i]) = w[m][i];
            wave_lds_sync();
            const int sn = s + 1 < s1 ? s + 1 : s;  // (x: the last stage's blocks again)
            __builtin_amdgcn_sched_barrier(0);
            if (s + 1 < s1) load_w(sn);  // (two stages a wave at K = 4096: not the last one again; 14336 rows -1 to -6 %)
            __builtin_amdgcn_sched_barrier(0);
            KwScales<FMT> ks[G];
            float xs0[MT], xs1[MT];
#pragma unroll
            for (int u = 0; u < SKB; u++) {
                uint4 C[G][Geo::NC];
                float a0[G], a1[G];
#pragma unroll
                for (int m = 0; m < G; m++) {
                    const uint8_t* row = img + (m * 16 + r) * Geo::PITCH;
                    if constexpr (!kKwPlain<FMT>)
                        if ((u & 3) == 0) ks[m].load(row, u >> 2);
                    a0[m] = 1.0f;
                    kw_codes<FMT>(row, u, g, a0[m], C[m]);
                    if constexpr (!FOLD && !kKwPlain<FMT>) a0[m] = ks[m].scale(u, 0);
                    if constexpr (K6) a1[m] = ks[m].scale(u, 1);
                }
                X cur[MT];
#pragma unroll
                for (int t = 0; t < MT; t++) cur[t] = x[u % PD][t];
                load_x(u + PD < SKB ? s * SKB + u + PD : sn * SKB + u + PD - SKB, u % PD);
#pragma unroll
                for (int t = 0; t < MT; t++) {
                    uint4 P[NP + kKwXParts<FMT>];
                    float v[8];
                    float ps = 0.0f;
                    if constexpr (XF32) {
                        v[0] = cur[t].f[0].x; v[1] = cur[t].f[0].y; v[2] = cur[t].f[0].z; v[3] = cur[t].f[0].w;
                        v[4] = cur[t].f[1].x; v[5] = cur[t].f[1].y; v[6] = cur[t].f[1].z; v[7] = cur[t].f[1].w;
                        ps = x_parts(v, P);
                    } else {
                        P[0] = cur[t].b;
                        if constexpr (MIN) {
                            Vec<SLHIP_BF16>::unpack(cur[t].b, v);
                            ps = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
                        }
                    }
                    if constexpr (kKwXParts<FMT> != 0) P[NP] = finite_bf16(P[0]);
                    if constexpr (MIN) {  // lane group j keeps the token's sum over block 4h + j
                        const float p01 = ps + __shfl_xor(ps, 16);
                        const float other = __shfl_xor(p01, 32);
                        const bool mine = g == (u & 3);
                        if constexpr (Q2K) {  // per 16-value half: lane groups {0, 1} and {2, 3}
                            xs0[t] = (u & 3) == 0 || mine ? (g < 2 ? p01 : other) : xs0[t];
                            xs1[t] = (u & 3) == 0 || mine ? (g < 2 ? other : p01) : xs1[t];
                        } else {
                            xs0[t] = (u & 3) == 0 || mine ? p01 + other : xs0[t];
                        }
                    }
                    block_product<FMT, NP, G, MT>(P, C, a0, a1, g, acc, t);
                }
                if constexpr (MIN) {
                    if ((u & 3) == 3) {  // lane (r, g): token r's sum over block g (A), row r's minimum of block g (B)
#pragma unroll
                        for (int m = 0; m < G; m++) {
                            const float m0 = ks[m].min(g, 0);
#pragma unroll
                            for (int t = 0; t < MT; t++)
                                acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xs0[t], m0, acc[m][t], 0, 0, 0);
                            if constexpr (Q2K) {
                                const float m1 = ks[m].min(g, 1);
#pragma unroll
                                for (int t = 0; t < MT; t++)
                                    acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xs1[t], m1, acc[m][t], 0, 0, 0);
                            }
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);  // blocks in order: interleaved, their operands spill
            }
        }
    }

    reduce_store<DUAL, MT, TN>(a, acc, lds, wave, lane, n0, t0);
}

template <int FMT, bool DUAL, bool XF32, int MT, int TN>
int launch_kw(MatvecArgs a, hipStream_t st)
{
    // one launch, or several where row tiles x token tiles would pass the grid's limit of 2^32 threads
    const int64_t rows = ((a.N + 16 * TN - 1) / (16 * TN) + 7) / 8 * 8, toks = (a.T + 16 * MT - 1) / (16 * MT);
    if (rows > kKwMaxBlocks) return SLHIP_ERR_UNSUPPORTED;  // the VALU kernel's persistent grid takes any N
    const int64_t most = kKwMaxBlocks / rows;
    for (int64_t t = 0; t < toks; t += most) {
        const int64_t gy = toks - t < most ? toks - t : most;
        a.t0 = 16 * MT * t;
        matvec_kw<FMT, DUAL, XF32, MT, TN><<<dim3(static_cast<unsigned>(rows * gy)), 64 * kKwWaves, 0, st>>>(a, static_cast<int>(gy));
        const int r = check_launch("matvec_kw");
        if (r != SLHIP_OK) return r;
    }
    return SLHIP_OK;
}

template <int FMT, bool DUAL, bool XF32>
int launch_kw_shape(const MatvecArgs& a, int mt, int tn, hipStream_t st)
{
    if (mt == 1 && tn == 1) return launch_kw<FMT, DUAL, XF32, 1, 1>(a, st);
    if (mt == 1 && tn == 2) return launch_kw<FMT, DUAL, XF32, 1, 2>(a, st);
    if (mt == 2 && tn == 2) return launch_kw<FMT, DUAL, XF32, 2, 2>(a, st);
    if constexpr (!DUAL) {
        if (mt == 1 && tn == 4) return launch_kw<FMT, DUAL, XF32, 1, 4>(a, st);
        if (mt == 2 && tn == 4) return launch_kw<FMT, DUAL, XF32, 2, 4>(a, st);
        if (mt == 4 && tn == 4) return launch_kw<FMT, DUAL, XF32, 4, 4>(a, st);
    }
    return fail(SLHIP_ERR_INVALID, "internal: matvec_kw tiles %d x %d", mt, tn);
}

template <int FMT>
int launch_kw_fmt(const MatvecArgs& a, bool dual, int mt, int tn, hipStream_t st)
{
    if (a.xt == SLHIP_F32)
        return dual ? launch_kw_shape<FMT, true, true>(a, mt, tn, st) : launch_kw_shape<FMT, false, true>(a, mt, tn, st);
    return dual ? launch_kw_shape<FMT, true, false>(a, mt, tn, st) : launch_kw_shape<FMT, false, false>(a, mt, tn, st);
}

}  // namespace slhip
