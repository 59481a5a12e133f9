// The tile kernel's launch shapes and their choice (gemv_tile.h). The small-batch entry points come here first when the
// caller leaves the variant to the library (variant < 0).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemv_tile.h"

namespace paia {
namespace {

constexpr int kMaxP = 6;

// Launch shapes: 8 waves split K of P tiles. Stages in flight, D: with one tile per wave all the stages of a K = 4096 row
// (FP8 4096x4096 M = 4: 5.06 us with four, 5.6 with two); INT4's take half the bytes but more decode, and two are enough up
// to 8 stages per wave (4096x4096 4.97 us with two, 5.16 with four; 4096x14336 10.98 with two, 9.49 with four; at 16
// activation rows three, 14.9, for the registers). From P = 3 on one stage of P tiles is enough in flight and a second one
// only costs registers (FP8 9216x8192 M = 16 16.5 us either way, 10112x4096 10.4 against 10.6). FP8 and BF16 weights stream
// (nt); an INT4 row's 64 bytes share a 128-byte line with the next stage's, which the default policy keeps (4096x14336
// M = 4 10.8 us against 11.9). The stages go to the waves in turn for P <= 2 and for INT4 (gate_up 28672x4096 M = 4: 15.8 us
// in turn, 17.1 in contiguous ranges), in contiguous ranges for the wide BF16 and FP8 launches (FP8 14336x4096 M = 16 12.6
// us against 13.3).
template <int F, int MT, int P, int D>
int launch_d(const BatchParams& b, int blocks, hipStream_t st)
{
    constexpr bool I4 = TileFmt<F>::kI4F;
    return launch_tile<F, P, 8, 8, D, MT, I4 ? 0 : 2, I4 || P <= 2>(b, blocks, st);
}
template <int F, int MT, int P>
int launch_p(const BatchParams& b, int blocks, hipStream_t st)
{
    if constexpr (P == 1 && TileFmt<F>::kI4F) {
        if (b.K <= 64 * TileFmt<F>::kCols) return launch_d<F, MT, 1, 2>(b, blocks, st);
        return launch_d<F, MT, 1, MT == 16 ? 3 : 4>(b, blocks, st);
    } else {
        return launch_d<F, MT, P, P == 1 ? 4 : (P == 2 ? 2 : 1)>(b, blocks, st);
    }
}

template <int F, int MT>
int launch_mt(const BatchParams& b, int P, int blocks, hipStream_t st)
{
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
    const int cus = device_facts().cus > 0 ? device_facts().cus : 256;
    const int ntiles = (b.N + kTileRows - 1) / kTileRows;
    // one block per CU while P <= 6 covers the tiles, else rounds of two blocks per CU with P <= 5; fewer blocks where all
    // but the last take P tiles anyway (28672x4096: 448 of 4 tiles 15.0 us, 512 of 3 or 4 15.4; 33000x2048 needs the 512:
    // 413 of 5 tiles leave 99 CUs with one block and 157 with two)
    int P = (ntiles + cus - 1) / cus, blocks = 0;
    if (P > kMaxP) {
        blocks = 2 * cus * ((ntiles + 2 * cus * 5 - 1) / (2 * cus * 5));
        P = (ntiles + blocks - 1) / blocks;
        const int fewest = (ntiles + P - 1) / P;
        if (8 * fewest >= 7 * blocks) blocks = fewest;
    }
    if (b.M <= 4) return launch_mt<F, 4>(b, P, blocks, st);
    if (b.M <= 8) return launch_mt<F, 8>(b, P, blocks, st);
    return launch_mt<F, 16>(b, P, blocks, st);
}

}  // namespace

int launch_tile_picked(int kind, const BatchParams& b, hipStream_t st)
{
    // the kernel's index arithmetic: rows in 31 bits, a tile's weights and x behind one 31-bit buffer offset
    if (b.M < 2 || b.M > kMaxBatch || b.N > (1 << 30) || b.K > (1 << 24)) return kTileRefused;
    switch (kind) {
    case 0: return launch_fmt<kBF16>(b, st);
    case 1: return launch_fmt<kFP8>(b, st);
    case 2: return launch_fmt<kI4>(b, st);
    default: return launch_fmt<kI4ZP>(b, st);
    }
}

}  // namespace paia
