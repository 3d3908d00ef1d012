// Arguments and planning of the passes that run several calls of a D2Q9
// lattice at once (tile_kernel.hpp).
#pragma once

#include <algorithm>

#include "node_index.hpp"
#include "step_args.hpp"

namespace lbmc {

struct TilePass {
    const void *src;
    void *dst;
    int calls;           // 1 .. M + 1
    unsigned store;      // bit j: call j of the pass stores rho / u
    int W, H, M;         // tile with margins, margin
    int OW, OH;          // owned nodes
    unsigned mw;         // magic pair of W
    int lw;
    int ntx;             // tiles along x, and their magic pair
    unsigned mt;
    int lt;
    int xoff, yoff;      // multiples of Lx, Ly that are >= M
    int rs[2], ws[2];    // read and write shifts, mod L
    int s0[2];           // t mod L of the pass's first call (stochastic rounding)
};

// Tiles of a lattice: the kernel's capacity (size, tile_capacity), the margin
// M = calls of a pass - 1 and the tile shape.
struct TilePlan {
    bool on = false;
    int size = 0, W = 0, H = 0, M = 0, OW = 0, OH = 0, ntx = 0, nty = 0;
    double us = 0;  // estimated time per call
};

// Kernel capacities: threads per block and nodes per thread.  Sizes 0 and 1
// hold one node per thread, for lattices too small to give every CU a large
// tile; size 2 fills 72 KB of LDS (two blocks per CU) in every format.
struct TileCapacity {
    int threads, per_thread;
};
constexpr TileCapacity tile_capacity(int size, int slot_bytes)
{
    return size == 0 ? TileCapacity{256, 1} : size == 1 ? TileCapacity{512, 1} : TileCapacity{512, 16 / slot_bytes};
}

// Tiles of W x H nodes, margins included, over an Lx x Ly lattice; shrunk to
// the shape that the same number of tiles needs.  At least two calls a pass
// (M >= 1): an even number of passes then covers any run of two calls or more.
inline bool tile_shape(int Lx, int Ly, int size, int W, int H, int M, TilePlan &q)
{
    const int OW = W - 2 * M, OH = H - 2 * M;
    if (M < 1 || OW < 1 || OH < 1) return false;
    q.size = size;
    q.M = M;
    q.ntx = (Lx + OW - 1) / OW;
    q.nty = (Ly + OH - 1) / OH;
    q.OW = (Lx + q.ntx - 1) / q.ntx;
    q.OH = (Ly + q.nty - 1) / q.nty;
    q.W = q.OW + 2 * M;
    q.H = q.OH + 2 * M;
    return true;
}

// Estimated time per call (us) of the passes of a plan.  Measured constants
// (MI355X): 3.5 us for a launch with its first loads and last stores; per
// call of a tile at least the latency of one update (0.5 us, 0.8 us in 64
// bits); per node update 1.2 ns of a CU (2.9 ns in 64 bits, 1.7 ns in 16
// bits, which also round and convert); 20 bytes per ns and CU of memory
// traffic, about half of it hidden under the arithmetic of the other
// resident blocks.
inline double tile_estimate(const TilePlan &q, int slot_bytes, int ncu)
{
    const double ns_node = slot_bytes == 8 ? 2.9 : slot_bytes == 4 ? 1.2 : 1.7;
    const double us_call = slot_bytes == 8 ? 0.8 : 0.5;
    double nodes = 0;
    for (int j = 0; j <= q.M; j++) nodes += (double)(q.W - 2 * j) * (q.H - 2 * j);
    const double tiles = (double)q.ntx * q.nty;
    double per_cu = tiles / ncu;
    if (per_cu < 4) per_cu = std::max(1.0, (double)((long long)(per_cu + 0.999)));
    const double arith = std::max((q.M + 1) * us_call, per_cu * nodes * ns_node * 1e-3);
    const double bytes = per_cu * 9 * (q.H * ((double)q.W * slot_bytes + 96) + q.OH * ((double)q.OW * slot_bytes + 96));
    return (3.5 + arith + 0.5 * bytes / 20e3) / (q.M + 1);
}

// The plan with the smallest estimate (within 10 % of the best of all
// shapes on ten lattices from 64 x 48 to 3392 x 3392, three formats).  In 32
// and 64 bits it beats one call per launch at every size (us per call, one
// call per launch -> passes: 256 x 64 FP64 4.1 -> 1.7, 600 x 300 FP32 6.4 ->
// 3.2, 2048 x 1024 FP32 25.3 -> 15.7, FP64 46.8 -> 39.6, 3392 x 3392 FP32
// 161 -> 78).  The 16-bit one-call kernels move half of FP32's bytes and are
// bound by the same arithmetic plus the conversions, so passes win only
// where launches count: 64 x 48 3.4 -> 1.2, 1500 x 400 11.6 -> 8.0, 2786 x
// 681 equal, 3392 x 3392 80 -> 92; hence the line at 2^20 nodes.
// M up to 7: deeper passes of the small tiles recompute more than they save.
inline TilePlan plan_tiles(int Lx, int Ly, int slot_bytes, int ncu)
{
    TilePlan best;
    if (slot_bytes == 2 && (long long)Lx * Ly > (1LL << 20)) return best;
    for (int size = 0; size <= 2; size++) {
        const TileCapacity cap = tile_capacity(size, slot_bytes);
        const int P = cap.threads * cap.per_thread;
        for (int W = 16; W <= 128; W *= 2)
            for (int M = 1; M <= 7; M++) {
                TilePlan q;
                if (P / W < 8 || !tile_shape(Lx, Ly, size, W, P / W, M, q)) continue;
                q.us = tile_estimate(q, slot_bytes, ncu);
                q.on = true;
                if (!best.on || q.us < best.us) best = q;
            }
    }
    return best;
}

// the geometry half of a pass's arguments
inline void tile_geometry(const TilePlan &q, const int *L, TilePass &p)
{
    p.W = q.W;
    p.H = q.H;
    p.M = q.M;
    p.OW = q.OW;
    p.OH = q.OH;
    p.ntx = q.ntx;
    const FastDiv dw = make_fastdiv(q.W), dt = make_fastdiv(q.ntx);
    p.mw = dw.m;
    p.lw = dw.l;
    p.mt = dt.m;
    p.lt = dt.l;
    p.xoff = (q.M + L[0] - 1) / L[0] * L[0];
    p.yoff = (q.M + L[1] - 1) / L[1] * L[1];
}

}  // namespace lbmc
