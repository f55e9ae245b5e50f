// Pair tiles over the dense nodes of the shared-node path: the work list
// (tiles of the upper triangle, some of them cut into parts over the nodes)
// and the launchers.
#pragma once

#include "ssu_kernels.hpp"

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <functional>
#include <vector>

namespace ssu {

// Tiles are square: 128 x 128 pairs with one sum per pair (weighted), 64 x 64 with
// two (generalized, VAW).
constexpr uint32_t TILE_ROWS_1 = 128, TILE_ROWS_2 = 64;
// workgroups of 256 threads one XCD (32 CUs) holds: two (128) or three (64) waves per SIMD
constexpr uint32_t tile_resident(uint32_t rows) { return rows == TILE_ROWS_1 ? 64 : 96; }
// bytes of one workspace slot: a tile's sums in FP64
constexpr size_t tile_slot_bytes(uint32_t rows) {
    return size_t(rows) * rows * sizeof(double) * (rows == TILE_ROWS_1 ? 1 : 2);
}
constexpr uint32_t TILE_MAX_PARTS = 64;
// The most a plan's workspace slots take together.  Cuts that would take more (up to
// 1.1 GB of sums at 3,000 - 15,000 samples with tens of thousands of dense nodes) give way
// to the best of those that fit: by the rule's own costs 0.1% of the tiles' time over sizes
// to 16,384 samples and 45,000 dense nodes, 14% at the worst of them; half the bytes, 0.8% and 44%.
constexpr size_t TILE_WS_BYTES = size_t(256) << 20;

// One workgroup's work: part p of np of the tile of rows bi * rows .., columns
// bj * rows ..  Parts of one tile hold consecutive workspace slots.
struct TileUnit {
    uint32_t bij;    // bi << 16 | bj; TILE_NONE: nothing
    uint32_t part;   // slot << 12 | p << 6 | (np - 1)
};
constexpr uint32_t TILE_NONE = 0xffffffffu;

// The tiles of an n x n upper triangle in launch order.  Workgroups go to the 8
// XCDs round robin; unit q of XCD x is units[x * per_xcd + q], so that each XCD
// walks a run of neighbouring tiles and shares their operand rows in its L2.
struct TileSet {
    std::vector<TileUnit> units;
    std::vector<TileUnit> split;   // the tiles cut into parts: bij, first slot << 12 | (np - 1)
    uint32_t per_xcd = 0;
    uint32_t slots = 0;            // workspace slots used (parts of cut tiles)
    uint64_t tiles = 0;
};
// rows: the tile's edge; max_nodes: an upper bound on the dense nodes.
TileSet tile_set(uint32_t n, uint32_t rows, uint32_t max_nodes);
// those of `full` that keep(bi, bj) selects, cut as in `full` (so that a tile's
// sums do not depend on the selection)
TileSet tile_subset(const TileSet& full, const std::function<bool(uint32_t, uint32_t)>& keep);

struct TileArgs {
    const void* U;            // operand rows
    const int32_t* rows;      // FP64: operand row of processed node r (nullptr: r itself)
    size_t ldn;               // their stride, a multiple of the tile's edge
    const double* len;        // [K] lengths
    bool scaled;              // FP32 weighted: U's rows hold l u
    const uint32_t* dlist;    // dlist[0] = dense nodes, then their processed-node indices
    uint32_t n;
    const double* S;          // per-sample sums
    bool normalized;
    void* out;                // n x n, the operand's type
    bool add_partial;         // out[i * n + j] (and out2), i < j, hold the rare nodes' shares
    const void* out2;         // two sums: the denominator's share
    double alpha;             // generalized
    const void* C;            // VAW: count rows, as U
    const double* totals;     // VAW: the samples' totals
    uint32_t* flags;          // unnormalised VAW weighted: marks of near-duplicates (below
    float flag_tau;           //   flag_tau of the pair's VAW denominator), as launch_flag_close's,
    GapBand band;             //   among the pairs of the band (the others' shares are not there)
    double* ws;               // workspace slots of tile_slot_bytes
    const TileUnit* units;
    uint32_t n_units, per_xcd;
    const TileUnit* split;
    uint32_t n_split;
};
// Weighted.  FP32: out_ij = (sum over the dense nodes of |x_i - x_j| + the rare
// share) / (S_i + S_j) (or the sum itself), x = l u in FP32 (scaled rows), or of
// l |u_i - u_j| (plain rows).
// FP64: x = S_i + S_j - 2 M in its place, M = sum of l min(u_i, u_j) + the rare
// share, U the embedding (row rows[r] for processed node r).
hipError_t launch_tiles_weighted(bool fp64, const TileArgs& a, hipStream_t st);
// Generalized, 0 <= alpha <= 1: numerator over denominator, each with its share
hipError_t launch_tiles_generalized(bool fp64, const TileArgs& a, hipStream_t st);
// VAW (kind 1: weighted, 2: presence, 3: generalized, 0 <= alpha <= 1): numerator
// over denominator, each with its share (or the numerator, not normalized)
hipError_t launch_tiles_vaw(int kind, bool fp64, const TileArgs& a, hipStream_t st);

// dlist from the dense mask ([ceil(K / 32)] words): dlist[0] = their number,
// then the set bits in increasing order
hipError_t launch_dense_list(uint32_t* dlist, const uint32_t* dmask, uint32_t K, hipStream_t st);

}  // namespace ssu
