// Which tile a gemm_chain launch (gemm_q8.hip) takes: host arithmetic in plain C++.
#pragma once

namespace sepal::hip {
namespace q8 {

// The tile of a gemm_chain launch: WM x WN waves of 32 MBLK rows x 64 columns.
struct ChainTile {
    int wm, wn, mblk;
    int per_cu;                // blocks a CU holds at once
    double step[2], step2[2];  // us per group with one block on the CU, and with per_cu (per token, per 128)
    double round[2];           // us per tile round besides (prologue, epilogue)
    int rows() const { return 32 * mblk * wm; }
    int cols() const { return 64 * wn; }
    // us of `tiles` tiles: full rounds of per_cu blocks per CU, and a last one that may hold one block per CU
    double cost(int tiles, int groups, int cus, bool per128) const {
        const int slots = per_cu * cus, full = tiles / slots, rest = tiles % slots;
        const int i = per128 ? 1 : 0;
        return full * (groups * step2[i] + round[i]) + (rest == 0 ? 0.0 : groups * (rest <= cus ? step[i] : step2[i]) + round[i]);
    }
};

// Which tile. Large problems take the 128 x 256 tile: the most outputs per operand byte and per instruction. Where its
// grid leaves CUs idle (a narrow N, a last round with few tiles), smaller tiles of the same kernel fill them; every
// output keeps its links' order, so the bits do not depend on the tile. The times below are fitted to forced-tile runs at
// 19456 x 2560, 2560 x 9728, 2560 x 2560 and 7168 x 1024, T 65 .. 4096 (e.g. 2560 x 9728 per token, us: T = 300 128 x 256 80,
// 128 x 128 56, 96 x 128 52, 64 x 128 46, 32 x 128 38; T = 896 82, 56, 54, 85, 94; T = 4096 171, 175, 209, 208, 300). A
// step of a small tile is not a share of the large one's: each wave's converts and multiply-adds, its loads' issue and
// the barrier remain.
constexpr ChainTile kChain128x256{2, 4, 2, 1, {1.05, 1.45}, {1.05, 1.45}, {6.0, 7.0}};
constexpr ChainTile kChain128x128{4, 2, 1, 1, {0.68, 0.80}, {0.68, 0.80}, {4.0, 5.0}};
constexpr ChainTile kChain96x128{3, 2, 1, 1, {0.61, 0.82}, {0.61, 0.82}, {4.0, 4.0}};
constexpr ChainTile kChain64x128{2, 2, 1, 2, {0.49, 0.62}, {1.07, 1.18}, {3.5, 3.5}};
constexpr ChainTile kChain32x128{1, 2, 1, 2, {0.41, 0.68}, {0.73, 0.77}, {3.5, 3.0}};
// the SwiGLU -> int8 epilogue needs 256 columns (one block of 128 outputs)
constexpr ChainTile kChainQ8_128x256{2, 4, 2, 1, {1.70, 1.70}, {1.70, 1.70}, {9.0, 9.0}};
constexpr ChainTile kChainQ8_64x256{2, 4, 1, 1, {0.95, 1.15}, {0.95, 1.15}, {6.0, 7.0}};

// Whole-K sums (gemm_s8, gemm_q8y): no links.
constexpr ChainTile kWhole128x256{2, 4, 2, 1, {0.80, 0.80}, {0.80, 0.80}, {6.0, 6.0}};
constexpr ChainTile kWhole128x128{4, 2, 1, 1, {0.55, 0.55}, {0.55, 0.55}, {4.0, 4.0}};
constexpr ChainTile kWhole96x128{3, 2, 1, 1, {0.50, 0.50}, {0.50, 0.50}, {4.0, 4.0}};
constexpr ChainTile kWhole64x128{2, 2, 1, 2, {0.40, 0.40}, {0.70, 0.70}, {3.5, 3.5}};
constexpr ChainTile kWhole32x128{1, 2, 1, 2, {0.35, 0.35}, {0.55, 0.55}, {3.5, 3.5}};
enum { TILES_CHAIN = 0, TILES_INT8_OUT = 1, TILES_WHOLE = 2 };

struct ChainPlan {
    int full;             // 128 x 256 tiles of the first launch (whole rounds; 0: none)
    const ChainTile* tile;  // of everything, or of what the first launch leaves
};

inline ChainPlan chain_plan(int t, int n, int groups, int kind, bool per128, int cus) {
    static const ChainTile* const sets[3][5] = {
        {&kChain128x256, &kChain128x128, &kChain96x128, &kChain64x128, &kChain32x128},
        {&kChainQ8_128x256, &kChainQ8_64x256},
        {&kWhole128x256, &kWhole128x128, &kWhole96x128, &kWhole64x128, &kWhole32x128},
    };
    const ChainTile& big = *sets[kind][0];
    const ChainTile* const* small = sets[kind] + 1;
    const int count = kind == TILES_INT8_OUT ? 1 : 4;
    const int tiles = (t + 127) / 128 * ((n + 255) / 256), full = tiles / cus * cus;
    ChainPlan best{0, &big};
    double us = big.cost(tiles, groups, cus, per128);
    for (int i = 0; i < count; ++i) {
        const ChainTile& c = *small[i];
        const double whole = c.cost((t + c.rows() - 1) / c.rows() * ((n + c.cols() - 1) / c.cols()), groups, cus, per128);
        if (whole < 0.96 * us) us = whole, best = ChainPlan{0, &c};
        if (full == 0 || full == tiles || 128 % c.rows() != 0) continue;
        // whole rounds of the large tile, then the rest in small ones (a second launch, which starts when the slowest
        // block of the first has ended: 6 us)
        const double mixed = big.cost(full, groups, cus, per128) + 6.0 +
                             c.cost((tiles - full) * (128 / c.rows()) * (256 / c.cols()), groups, cus, per128);
        if (mixed < 0.96 * us) us = mixed, best = ChainPlan{full, &c};
    }
    return best;
}

} // namespace q8
} // namespace sepal::hip
