// The group-scale kernel for 17 rows and more on K-tiled operands (abq_gemm_rows_grouped.hip): what it runs, where its workgroups
// cover the chip, and the plan of a launch.
#pragma once
#include "abq_kernels.h"

namespace abq {

// What it runs: signed 8-bit activations, groups of 128.  (Groups of 64 would need two scale groups per step, activations of at
// most 4 bits other operand reads; neither has been built.)  Its byte offsets are 32 bits wide.
inline bool rows_grouped_runs(int M, int N, int K, int x_bits, int w_bits, int group_size, int act)
{
    return M > 16 && x_bits == 8 && (w_bits == 2 || w_bits == 4 || w_bits == 8) && group_size == 128 && K >= 128 && (!act || N % 32 == 0) &&
           (size_t)N * K * w_bits / 8 < (1ull << 32) && (size_t)M * K < (1ull << 32) && (size_t)N * (K / 128) * 4 < (1ull << 32);
}
// Whether its workgroups, one tile of 16 weight rows and up to 64 rows each at the least, cover most of the 256 compute
// units (W4A8: 2048 x 2048 at 32 rows, 128 workgroups, 4.1 us against 4.0 on the decode kernel's blocks of rows; at 80
// rows, 256, 4.7 against 6.4 on the prefill tiles; 1024 x 1024 at 128 rows, 128, 4.8 against 4.2, at 192 rows, 192, 4.9 against 7.5).
inline bool rows_grouped_covers(int M, int N) { return (long)((N + 15) / 16) * ((M + 63) / 64) >= 192; }
hipError_t launch_rows_grouped_8_2(const GemmArgs &, hipStream_t);
hipError_t launch_rows_grouped_8_4(const GemmArgs &, hipStream_t);
hipError_t launch_rows_grouped_8_8(const GemmArgs &, hipStream_t);
template <int P> inline hipError_t launch_rows_grouped_8(const GemmArgs &a, hipStream_t stream)
{
    return P == 2 ? launch_rows_grouped_8_2(a, stream) : P == 4 ? launch_rows_grouped_8_4(a, stream) : launch_rows_grouped_8_8(a, stream);
}

constexpr int kRowsWaves = 8;

// Steps whose weights are in flight beside the one multiplied: a whole block where the registers hold it beside the
// accumulators, else two.
constexpr int rows_ahead(int p, int t, int mb) { return 4 * t * (p + mb) <= 150 ? 4 : 2; }
// buffers of the activation ring: three steps of 32 rows fit beside the scales, two of 48 or 64
constexpr int rows_ring(int p, int t, int mb) { return mb <= 2 && rows_ahead(p, t, mb) == 4 ? 3 : 2; }
// instances that are built: what registers and LDS hold
constexpr bool rows_built(int p, int t, int mb) { return t * p <= 24 && t * mb <= 18; }
// LDS: the activation rings, then scales, zero points and group sums per wave (the waves' partial tiles take the place of all
// of these at the end) | the rows' scales and zero points, the tiles' zero-point terms
constexpr int rows_scale_loads(int t, int mb, bool zp) { return zp ? 2 * t + mb : t; }
constexpr size_t rows_lds_of_loop(int nw, int p, int t, int mb, bool zp)
{
    return (size_t)nw * (rows_ring(p, t, mb) * mb * 2048 + rows_scale_loads(t, mb, zp) * 256);
}
constexpr size_t rows_lds_of_sum(int nw, int t, int mb) { return (size_t)nw * t * mb * 1024; }
constexpr size_t rows_lds_for_rows(int nw, int p, int t, int mb, bool zp) // where the rows' scales lie
{
    return rows_lds_of_loop(nw, p, t, mb, zp) > rows_lds_of_sum(nw, t, mb) ? rows_lds_of_loop(nw, p, t, mb, zp) : rows_lds_of_sum(nw, t, mb);
}
constexpr size_t rows_lds(int nw, int p, int t, int mb, bool zp) { return rows_lds_for_rows(nw, p, t, mb, zp) + 512 + 512; }

// The plan of a launch.
struct RowsPlan {
    int tiles;      // of 16 weight rows per workgroup; 0: no instance
    int row_blocks; // of 16 rows per workgroup: 2 to 4
    int m_blocks;   // blocks of that many rows
    int waves;
    int rounds; // of the compute units
    size_t lds;
    unsigned grid;
};

// A workgroup fills a compute unit's LDS, so workgroups run in rounds of the 32 compute units of an XCD (the blocks of rows of a set
// of weight rows share one: counted over all 256, 22 sets of eleven blocks passed for one round, but six XCDs had 33 to run); a
// round's time is the weights of its tiles from memory plus the activations from L2, which is about three times as fast.
inline RowsPlan rows_grouped_plan(int w_bits, int M, int N, int K, int act, bool zero_points)
{
    const int m64 = (M + 63) / 64, mb16 = ((M + m64 - 1) / m64 + 15) / 16, mb = mb16 < 2 ? 2 : mb16;
    const int nw = (K / 128 + 3) / 4 < kRowsWaves ? (K / 128 + 3) / 4 : kRowsWaves;
    const long tiles = (N + 15) / 16;
    RowsPlan plan{ 0, mb, (M + mb * 16 - 1) / (mb * 16), nw, 0, 0, 0 };
    double best_cost = 0;
    for (int c : { 1, 2, 3, 4, 6 }) {
        if (!rows_built(w_bits, c, mb) || (act && (c & 1)) || rows_lds(nw, w_bits, c, mb, zero_points) > 160 * 1024)
            continue;
        const long per_xcd = ((tiles + c - 1) / c + 7) / 8 * plan.m_blocks, rounds = (per_xcd + 31) / 32;
        const double cost = (double)rounds * (3.0 * c * (w_bits * 256 + 128) + mb * 2048.0);
        if (plan.tiles == 0 || cost < best_cost) {
            plan.tiles = c;
            plan.rounds = (int)rounds;
            best_cost = cost;
        }
    }
    if (plan.tiles) {
        plan.lds = rows_lds(nw, w_bits, plan.tiles, mb, zero_points);
        plan.grid = (unsigned)(((tiles + plan.tiles - 1) / plan.tiles + 7) / 8 * 8 * plan.m_blocks);
    }
    return plan;
}

} // namespace abq
