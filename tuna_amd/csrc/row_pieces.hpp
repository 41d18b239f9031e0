// How the kernels whose lanes hold one packed dword per 16-row tile (gemm_tall.hip, gemm_broad.hip) group those tiles into loads.
#pragma once

namespace tuna {

// Pieces of a lane's weights of a k-step's half: row tiles of 16 in loads of four, two and one dwords.
template <int RT>
struct Pieces {
    static constexpr int fours = RT / 4, twos = (RT & 2) / 2, ones = RT & 1, count = fours + twos + ones;
    static constexpr int width(int p) { return p < fours ? 4 : p < fours + twos ? 2 : 1; }
    static constexpr int first(int p) { return p <= fours ? 4 * p : p <= fours + twos ? 4 * fours + 2 * (p - fours) : RT - 1; }  // row tile
    static constexpr int of(int r) { return r < 4 * fours ? r / 4 : r < 4 * fours + 2 * twos ? fours : count - 1; }
};

}  // namespace tuna
