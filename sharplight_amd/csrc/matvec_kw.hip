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

// The time of one round of blocks over the chip (a block on each CU; matmul_tile two) relative to the smallest f32
// shape, in hundredths, by 16-row groups per block (both matrices counted) and token tiles. A launch costs its rounds
// times that, which orders the shapes alike at every K. From sweeps at K = 4096 and 7680, N = 1024 .. 14336, T = 3 ..
// 512; at K = N = 4096, T = 512, Q4_K, f32 x: 342 us (1 x 1: 32 rounds) / 193 (1 x 2) / 121 (1 x 4) / 152 (2 x 2) / 94
// (2 x 4) / 98 (4 x 4) / 101 (tile); T = 64: 42 / 24 / 16 / 21 / 23 / 46 / 101.
struct KwCosts {
    int c11, c12, c14, c22, c24, c44, tile1, tile2;  // ctg: t token tiles, g row groups; tile1: up to a tile a CU
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
    const int cus = device_cus();
    offer(1, 1, rounds(blocks(16, 16), cus) * (dual ? c.c12 : c.c11));
    offer(1, 2, rounds(blocks(16, 32), cus) * (dual ? c.c14 : c.c12));
    if (!dual) offer(1, 4, rounds(blocks(16, 64), cus) * c.c14);
    offer(2, 2, rounds(blocks(32, 32), cus) * (dual ? c.c24 : c.c22));
    if (!dual) offer(2, 4, rounds(blocks(32, 64), cus) * c.c24);
    if (!dual) offer(4, 4, rounds(blocks(64, 64), cus) * c.c44);
    const int64_t tiles = blocks(64, dual ? 64 : 128);
    offer(0, 0, tiles <= cus ? c.tile1 : rounds(tiles, 2 * cus) * c.tile2);
    return best;
}

// Times of a call of up to 16 tokens at K = 4096, in tenths of a microsecond: of matvec_kw per round of its blocks by their
// 16-row groups (the first three shapes of KwCosts; pairs begin at two) and per two 16-row tiles a CU, and of
// matvec_mq2 per round of a block a CU, per two blocks a CU and per 16 tokens of those.
struct FewCosts {
    int kw[3], kw_rows;
    int round, rows, token;
};

// Fitted to both kernels' times at K = 2048 .. 8192, N = 2048 .. 40960, T = 3, 8, 16 (weights from HBM).
static FewCosts few_costs(int fmt, bool f32, bool dual)
{
    auto pick = [&](FewCosts a, FewCosts b, FewCosts c, FewCosts d) { return f32 ? (dual ? b : a) : dual ? d : c; };
    switch (fmt) {
    case SLHIP_FMT_Q4_K:
        return pick({{43, 69, 107}, 17, 60, -8, 58}, {{72, 105, 0}, 37, 83, 8, 42},
                    {{25, 41, 74}, 16, 26, 11, 33}, {{42, 71, 0}, 37, 47, 19, 31});
    case SLHIP_FMT_Q5_K:
        return pick({{50, 81, 134}, 22, 62, -7, 55}, {{84, 131, 0}, 44, 82, 12, 42},
                    {{35, 56, 108}, 20, 28, 11, 36}, {{57, 107, 0}, 43, 48, 22, 33});
    case SLHIP_FMT_Q6_K:
        return pick({{69, 112, 207}, 25, 73, -3, 46}, {{114, 203, 0}, 51, 117, 14, 26},
                    {{48, 77, 164}, 24, 34, 8, 25}, {{77, 157, 0}, 52, 79, 25, 10});
    case SLHIP_FMT_Q2_K:
        return pick({{56, 91, 156}, 9, 99, 4, 28}, {{95, 154, 0}, 21, 217, -37, 29},
                    {{40, 64, 120}, 8, 32, 8, 25}, {{66, 118, 0}, 19, 60, 8, 24});
    case SLHIP_FMT_Q3_K:
        return pick({{66, 107, 186}, 13, 109, 9, 25}, {{109, 187, 0}, 26, 258, -41, 40},
                    {{48, 78, 158}, 9, 36, -1, 30}, {{79, 156, 0}, 22, 73, 7, 25});
    case SLHIP_FMT_Q8_0:
        return pick({{54, 87, 150}, 31, 69, 18, 87}, {{90, 149, 0}, 61, 121, 46, 69},
                    {{33, 54, 112}, 30, 18, 24, 43}, {{56, 111, 0}, 62, 32, 55, 38});
    case SLHIP_FMT_Q4_0:
        return pick({{52, 84, 142}, 16, 74, 4, 58}, {{87, 141, 0}, 33, 128, -4, 52},
                    {{31, 50, 103}, 15, 18, 10, 44}, {{53, 103, 0}, 31, 39, 9, 28});
    case SLHIP_FMT_Q4_1:
        return pick({{43, 69, 107}, 21, 74, 5, 59}, {{71, 102, 0}, 45, 122, 5, 50},
                    {{25, 40, 73}, 20, 25, 6, 37}, {{41, 68, 0}, 46, 42, 23, 31});
    case SLHIP_FMT_Q5_0:
        return pick({{67, 108, 192}, 19, 98, 8, 34}, {{110, 191, 0}, 37, 180, -8, 40},
                    {{46, 74, 153}, 16, 32, 0, 31}, {{76, 153, 0}, 34, 64, 14, 25});
    case SLHIP_FMT_Q5_1:
        return pick({{58, 93, 162}, 21, 85, 13, 44}, {{97, 159, 0}, 39, 156, 4, 43},
                    {{40, 65, 130}, 20, 31, 12, 32}, {{69, 129, 0}, 39, 59, 26, 20});
    default: return {};
    }
}

// Whether a block format's call of few tokens is faster on matvec_mq2 (matvec_mq.hpp), whose smaller blocks (three to five a
// CU) fill the chip evenly where matvec_kw pays for a whole further round, than here: where the estimates of both say so. At
// most one round of matvec_kw's smallest blocks is left to it, unless its waves' stages are uneven (K = 2560: Q6_K f32 x N =
// 4096 12.0 / 9.6) or fewer than the waves (K = 1024: 39 % behind on average over N = 2048 .. 40960); past K = 8192, beyond
// the fit, a clear lead is asked for (K = 14336: 0.6 % from the faster one, 2.1 % without). Past 16 tokens, two launches of
// it win for pairs of many short rows only (K = 1024, N = 16384, T = 17: Q8_0 24.0 / 29.0). Measured at K = 4096, T = 8, us,
// matvec_kw / matvec_mq2: Q6_K bf16 x N = 10240 24.4 / 16.6, N = 8192 14.4 / 13.2; pair N = 20480 72.4 / 52.3; Q4_0 f32 x
// pair N = 14336 38.4 / 31.0, N = 4096 14.2 / 19.6; Q5_K f32 x pair N = 11008 40.3 / 33.8, N = 8192 22.4 / 24.1. Over all
// points measured the choice is on average 0.4 % from the faster one; a line in N alone, for the 32-value formats only, was
// 7 %, at worst 2.0 times.
bool mq2_better(int fmt, const MatvecArgs& a, bool dual)
{
    const int64_t cus = device_cus();
    const KwShape s = kw_shape(fmt, a, dual);
    auto up = [](int64_t n, int64_t d) { return (n + d - 1) / d; };
    const int64_t stages = up(a.K / 256, 8);  // of the wave with the most
    if (a.T > 16) return dual && a.T <= 32 && a.K <= 1024 && a.N > 8192;
    if (s.mt != 1 || (2048 * stages <= a.K + a.K / 4 && a.N <= 16 * cus / (dual ? 2 : 1))) return false;
    const FewCosts c = few_costs(fmt, a.xt == SLHIP_F32, dual);
    const int64_t rounds = up(up(a.N, 16 * s.tn), cus);
    const double k = a.K / 4096.0;
    const double kw = 14.0 + rounds * (28.0 + c.kw[s.tn == 4 ? 2 : s.tn - 1] * (stages / 2.0)) + k * c.kw_rows * (a.N / (32.0 * cus));
    const int64_t blocks = up(a.N, 16 * mq2_row_tiles(fmt, a.xt));
    const double mq = (dual ? 54.0 : 45.0) + k * (c.round * up(blocks, cus) + blocks / (2.0 * cus) * (c.rows + c.token * (a.T / 16.0)));
    return mq < (a.K > 8192 ? 0.87 : 1.0) * kw;
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
