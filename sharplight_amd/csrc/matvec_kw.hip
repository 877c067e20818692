// Dispatch of the several-token matvec on the matrix cores: matvec_kw (matvec_kw.hpp: K split over a block's waves) at
// one of its block shapes, or matmul_tile (matmul_tile.hpp) for products large enough to fill the chip with its tiles.
#include "mq.hpp"

namespace slhip {

int launch_kw_part0(int fmt, const MatvecArgs& a, bool dual, int mt, int tn, hipStream_t st);
int launch_kw_part1(int fmt, const MatvecArgs& a, bool dual, int mt, int tn, hipStream_t st);
int launch_kw_part2(int fmt, const MatvecArgs& a, bool dual, int mt, int tn, hipStream_t st);
int launch_kw_part3(int fmt, const MatvecArgs& a, bool dual, int mt, int tn, hipStream_t st);
int launch_kw_part4(int fmt, const MatvecArgs& a, bool dual, int mt, int tn, hipStream_t st);
int launch_kw_part5(int fmt, const MatvecArgs& a, bool dual, int mt, int tn, hipStream_t st);
int launch_tile_part0(int fmt, const MatvecArgs& a, bool dual, hipStream_t st);
int launch_tile_part1(int fmt, const MatvecArgs& a, bool dual, hipStream_t st);
int launch_tile_part2(int fmt, const MatvecArgs& a, bool dual, hipStream_t st);
int launch_tile_part3(int fmt, const MatvecArgs& a, bool dual, hipStream_t st);
int launch_tile_part4(int fmt, const MatvecArgs& a, bool dual, hipStream_t st);
int launch_tile_part5(int fmt, const MatvecArgs& a, bool dual, hipStream_t st);

// A block shape: 16 mt tokens x tn 16-row tiles of each matrix; mt = 0 for matmul_tile (64 tokens x 128 rows).
struct KwShape {
    int mt, tn;
};

// The time of one round of blocks over the chip (256 CUs, a block each; matmul_tile two) relative to the smallest f32
// shape, in hundredths, by 16-row groups per block (both matrices counted) and token tiles. A launch costs its rounds
// times that, which orders the shapes alike at every K. From sweeps at K = 4096 and 7680, N = 1024 .. 14336, T = 3 ..
// 512; at K = N = 4096, T = 512, Q4_K, f32 x: 342 us (1 x 1: 32 rounds) / 193 (1 x 2) / 121 (1 x 4) / 152 (2 x 2) / 94
// (2 x 4) / 98 (4 x 4) / 101 (tile); T = 64: 42 / 24 / 16 / 21 / 23 / 46 / 101.
struct KwCosts {
    int c11, c12, c14, c22, c24, c44, tile1, tile2;  // ctg: t token tiles, g row groups; tile1: up to 256 tiles
};

static KwCosts kw_costs(int fmt, int xt)
{
    const bool f32 = xt == SLHIP_F32;
    if (fmt == SLHIP_FMT_Q6_K || fmt == SLHIP_FMT_F16)  // two operand vectors per code
        return f32 ? KwCosts{122, 160, 265, 235, 385, 670, 1400, 1830} : KwCosts{88, 113, 183, 150, 230, 400, 900, 1200};
    if (fmt == SLHIP_FMT_BF16 && !f32) return {63, 76, 104, 117, 150, 238, 385, 540};
    return f32 ? KwCosts{105, 120, 170, 195, 250, 480, 1000, 1270} : KwCosts{62, 75, 107, 112, 150, 238, 620, 760};
}

static KwShape kw_shape(int fmt, const MatvecArgs& a, bool dual)
{
    const KwCosts c = kw_costs(fmt, a.xt);
    KwShape best{1, 1};
    double least = 0.0;
    auto rounds = [](int64_t blocks, int slots) { return static_cast<double>((blocks + slots - 1) / slots); };
    auto blocks = [&](int tokens, int rows) { return ((a.T + tokens - 1) / tokens) * ((a.N + rows - 1) / rows); };
    auto offer = [&](int mt, int tn, double cost) {
        if (least == 0.0 || cost < least) {
            least = cost;
            best = {mt, tn};
        }
    };
    offer(1, 1, rounds(blocks(16, 16), 256) * (dual ? c.c12 : c.c11));
    offer(1, 2, rounds(blocks(16, 32), 256) * (dual ? c.c14 : c.c12));
    if (!dual) offer(1, 4, rounds(blocks(16, 64), 256) * c.c14);
    offer(2, 2, rounds(blocks(32, 32), 256) * (dual ? c.c24 : c.c22));
    if (!dual) offer(2, 4, rounds(blocks(32, 64), 256) * c.c24);
    if (!dual) offer(4, 4, rounds(blocks(64, 64), 256) * c.c44);
    const int64_t tiles = blocks(64, dual ? 64 : 128);
    offer(0, 0, tiles <= 256 ? c.tile1 : rounds(tiles, 512) * c.tile2);
    return best;
}

static int run_rows(int fmt, const MatvecArgs& a, bool dual, hipStream_t st)
{
    const KwShape s = kw_shape(fmt, a, dual);
    auto launch = [&](auto kw, auto tile) { return s.mt ? kw(fmt, a, dual, s.mt, s.tn, st) : tile(fmt, a, dual, st); };
    switch (fmt) {
    case SLHIP_FMT_Q4_K:
    case SLHIP_FMT_Q5_K: return launch(launch_kw_part0, launch_tile_part0);
    case SLHIP_FMT_Q6_K:
    case SLHIP_FMT_Q8_0: return launch(launch_kw_part1, launch_tile_part1);
    case SLHIP_FMT_Q4_0:
    case SLHIP_FMT_Q4_1: return launch(launch_kw_part2, launch_tile_part2);
    case SLHIP_FMT_Q5_0:
    case SLHIP_FMT_Q5_1: return launch(launch_kw_part3, launch_tile_part3);
    case SLHIP_FMT_Q2_K:
    case SLHIP_FMT_Q3_K: return launch(launch_kw_part4, launch_tile_part4);
    case SLHIP_FMT_BF16:
    case SLHIP_FMT_F16: return launch(launch_kw_part5, launch_tile_part5);
    default: return SLHIP_ERR_UNSUPPORTED;
    }
}

// y = x . W^T (or the dual form) for any number of tokens: K a multiple of 256 (block formats) or 64 (bf16, f16).
// SLHIP_ERR_UNSUPPORTED where a launch would pass the grid's size.
int run_kw(int fmt, const MatvecArgs& a, bool dual, hipStream_t st)
{
    // A lane addresses its block's rows (up to 128) by 32-bit offsets: longer rows go in slices of N whose rows those reach.
    const int64_t reach = UINT32_MAX / a.wrow > 0 ? UINT32_MAX / a.wrow : 1;
    if (reach >= 128 || a.N <= reach) return run_rows(fmt, a, dual, st);
    for (int64_t n = 0; n < a.N; n += reach) {
        MatvecArgs b = a;
        b.N = a.N - n < reach ? a.N - n : reach;
        b.wg += n * a.wrow;
        if (dual) b.wu += n * a.wrow;
        b.y = static_cast<char*>(a.y) + n * (a.yt == SLHIP_F32 ? 4 : 2);
        if (a.bias) b.bias += n;
        const int r = run_rows(fmt, b, dual, st);
        if (r != SLHIP_OK) return r;
    }
    return SLHIP_OK;
}

}  // namespace slhip
