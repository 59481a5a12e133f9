// The tile kernel's launch shapes and their choice (gemv_tile.h). The small-batch entry points come here first when the
// caller leaves the variant to the library (variant < 0).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemv_tile.h"

namespace paia {
namespace {

// Launch shapes, each a sweep's choice over N = 3584..128256, K = 512..18944 (us on MI355X):
//   * W waves split the K of P tiles. BF16 and FP8 run best as 4-wave blocks, several to a CU, so that one block's start and
//     end lie under another's stream (FP8 28672x4096 M = 16 20.6 with 4 waves, 21.5 with 8; 10112x4096 10.0 / 11.1; BF16
//     33000x2048 22.6 / 26.0); but a BF16 row beyond 8 KiB keeps one 4-wave block per CU from having enough in flight
//     (9216x8192 M = 8 34.9 with 4 waves, 26.4 with 8; 4096x14336 M = 4 21.1 / 20.5). INT4 keeps its matrix cores and VALU
//     waiting between a stage's loads and its decode and wants more waves (4096x14336 M = 4 9.9 with 8 waves, 12.4 with
//     4), except for short rows, which leave 8 waves a stage or none each (100000x512 M = 4 9.4 with 4, 12.1 with 8; one
//     tile per CU: 300x1024 2.86 / 2.95, but 2048x2048 3.72 / 3.53).
//   * D stages in flight. One tile per wave: the stages of a K = 4096 row at once (FP8 4096x4096 M = 4 5.06 with four, 5.6
//     with two), two for FP8 at 16 activation rows (registers) and for INT4 up to 8 stages per wave (4096x4096 4.97 /
//     5.16 with four; 4096x14336 10.98 / 9.49). More tiles need fewer, and a second stage soon costs more registers than it
//     brings bytes (FP8 28672x4096 M = 16 P = 4 20.6 with one, 21.5 with two).
//   * FP8 and BF16 weights stream (nt); an INT4 row's 64 bytes share a 128-byte line with the next stage's, which the default
//     policy keeps (4096x14336 M = 4 10.8 against 11.9).
//   * The stages go to the waves in turn for one tile per wave and for INT4 (28672x4096 M = 4 15.8, 17.1 in contiguous
//     ranges), in contiguous ranges otherwise (FP8 14336x4096 M = 16 12.6, 13.3 in turn).
constexpr int kShortK = 2560, kLongBf16K = 4096;
constexpr int kTileMaxRows = (1 << 30) - (1 << 16);

// Rows that are no multiple of 128 bytes (BF16, FP8): every stage's bytes of a row lie in two lines. Read line by line where
// a wave's range pays for its extra line (RING); else plain loads in turn, so that the second stage of a line finds it in
// cache (nt fetched 1.6 times the weights' bytes: BF16 45653x10952 M = 11 250 us, plain in turn 204, RING 155; FP8
// 72800x7024 M = 16 152 / 119 / 100). Several tiles per wave: down to 1280-byte rows (BF16 21595x664 M = 16 9.5 RING, 10.3
// plain; 30000x520 12.2 / 10.7). One tile, which waits on latency more than it streams: K >= 4096 and more than 32 tiles
// (FP8 4000x4944 M = 16 8.6 / 8.8, 1000x3600 6.5 / 4.8; BF16 600x18936 M = 8 22.9 / 28.0, 50x15016 M = 11 20.6 / 14.9), BF16
// from 2400-byte rows on more than 64 tiles (4000x2840 M = 8 6.5 / 7.2, 4090x1208 M = 16 4.9 / 5.3, 1207x2840 7.1 / 7.4, but
// 900x2504 6.4 / 5.2, 700x3592 8.1 / 6.2).
enum { kLines, kRing, kSplit };
template <int F, int P>
int row_form(const BatchParams& b)
{
    if (b.row_bytes % 128 == 0) return kLines;
    if (P > 1) return b.row_bytes >= 1280 ? kRing : kSplit;
    if (F == kBF16 && b.row_bytes >= 2400 && b.N > 64 * kTileRows) return kRing;
    return b.K >= 4096 && b.N > 32 * kTileRows ? kRing : kSplit;
}

template <int F, int MT, int P, int W, int D>
int launch_d(const BatchParams& b, int blocks, hipStream_t st)
{
    if constexpr (TileFmt<F>::kI4F) {
        return launch_tile<F, P, W, W, D, MT, 0, true, false>(b, blocks, st);
    } else {
        switch (row_form<F, P>(b)) {
        case kLines: return launch_tile<F, P, W, W, D, MT, 2, P == 1, false>(b, blocks, st);
        case kRing: return launch_tile<F, P, W, W, D, MT, 2, false, true>(b, blocks, st);
        default: return launch_tile<F, P, W, W, D, MT, 0, true, false>(b, blocks, st);
        }
    }
}
template <int F, int MT, int P>
int launch_p(const BatchParams& b, int blocks, hipStream_t st)
{
    if constexpr (TileFmt<F>::kI4F) {
        if constexpr (P <= 4) {
            if (b.K <= (P == 1 ? 1024 : kShortK)) return launch_d<F, MT, P, 4, P <= 2 ? 2 : 1>(b, blocks, st);
        }
        if constexpr (P == 1) {
            if (b.K > 64 * TileFmt<F>::kCols) return launch_d<F, MT, 1, 8, MT == 16 ? 3 : 4>(b, blocks, st);
        }
        return launch_d<F, MT, P, 8, P <= 2 ? 2 : 1>(b, blocks, st);
    } else {
        if constexpr (F == kBF16 && P <= 3) {
            if (b.K > kLongBf16K && blocks == 0) return launch_d<F, MT, P, 8, P == 1 ? 4 : (P == 2 ? 2 : 1)>(b, blocks, st);
        }
        constexpr int D = P == 1 ? (F == kFP8 && MT == 16 ? 2 : 4) : (P <= 3 || (P == 4 && MT <= 8) ? 2 : 1);
        return launch_d<F, MT, P, 4, D>(b, blocks, st);
    }
}

template <int F, int MT>
int launch_mt(const BatchParams& b, hipStream_t st)
{
    const int cus = device_facts().cus > 0 ? device_facts().cus : 256;
    const int ntiles = (b.N + kTileRows - 1) / kTileRows;
    int P = (ntiles + cus - 1) / cus, blocks = 0;
    if (!TileFmt<F>::kI4F && MT == 4 && ntiles > 4 * cus && b.K > kShortK &&
        (b.row_bytes % 128 == 0 || ntiles <= 16 * cus)) {
        // few activation rows: x is cheap to bring in again for every tile, and a block per tile balances best (FP8
        // 28672x4096 M = 4 18.7 against 19.4 for the best P > 1, BF16 33.9 / 34.7, FP8 128256x4096 73.0 / 74.2); rows with
        // split lines up to 4096 tiles, where their one extra line per range is still cheaper than a longer last wave (FP8
        // 20000x5008 M = 4 18.9 / 19.6, 40000x3008 22.6 / 24.1, but 87988x3680 61.9 / 57.1)
        P = 1;
        blocks = ntiles;
    } else if (P > (b.K <= kShortK ? 4 : 6)) {
        // beyond one block per CU: rounds of two blocks per CU of at most five tiles, for short rows of three of at most
        // four; the fewest blocks where nearly all of them then take P tiles (28672x4096 INT4: 448 of 4 tiles 15.0, 512 of 3
        // or 4 15.4; 33000x2048 needs all 768)
        const int per_round = (b.K <= kShortK ? 3 : 2) * cus, most = b.K <= kShortK ? 4 : 5;
        blocks = per_round * ((ntiles + per_round * most - 1) / (per_round * most));
        P = (ntiles + blocks - 1) / blocks;
        const int fewest = (ntiles + P - 1) / P;
        if (8 * fewest >= 7 * blocks) blocks = fewest;
    }
    switch (P) {
    case 1: return launch_p<F, MT, 1>(b, blocks, st);
    case 2: return launch_p<F, MT, 2>(b, blocks, st);
    case 3: return launch_p<F, MT, 3>(b, blocks, st);
    case 4: return launch_p<F, MT, 4>(b, blocks, st);
    case 5: return launch_p<F, MT, 5>(b, blocks, st);
    default: return launch_p<F, MT, 6>(b, blocks, st);
    }
}

template <int F>
int launch_fmt(const BatchParams& b, hipStream_t st)
{
    if (b.M <= 4) return launch_mt<F, 4>(b, st);
    if (b.M <= 8) return launch_mt<F, 8>(b, st);
    return launch_mt<F, 16>(b, st);
}

}  // namespace

int launch_tile_picked(int kind, const BatchParams& b, hipStream_t st)
{
    // the kernel's index arithmetic: rows in 31 bits, N * 4 bytes of FP8 scales and a launch's threads (at least 64 rows per
    // 256, N this large leaves room for short rows only) in 32, a tile's weights and x behind one 31-bit buffer offset
    if (b.M < 2 || b.M > kMaxBatch || b.N > kTileMaxRows || b.K > (1 << 24)) return kTileRefused;
    switch (kind) {
    case 0: return launch_fmt<kBF16>(b, st);
    case 1: return launch_fmt<kFP8>(b, st);
    case 2: return launch_fmt<kI4>(b, st);
    default: return launch_fmt<kI4ZP>(b, st);
    }
}

}  // namespace paia
