// Arguments and planning of the passes that run several calls at once: tiles
// of a D2Q9 lattice (tile_kernel.hpp), marching columns of a D3Q15 one
// (march_kernel.hpp).
#pragma once

#include <algorithm>

#include "node_index.hpp"
#include "step_args.hpp"

namespace lbmc {

constexpr int kMaxPassCalls = 32;  // the bits of TilePass::store

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

// Node classes of a D3Q15 lattice's passes: plain fluid; fluid and solid.
// Lattices with boundary or porous nodes have no passes: the node update with
// every boundary condition needs 133-157 registers (768 threads per block),
// and measured 0.5-1.0 of one call per launch.
enum { MARCH_FLUID = 0, MARCH_SOLID = 1 };

// How a march kernel has its body force (march_kernel.hpp)
enum { MARCH_NO_FORCE = 0, MARCH_NODE_FORCE = 1, MARCH_UNIFORM_FORCE = 2 };

// Two calls of a D3Q15 lattice
struct MarchPass {
    const void *src;
    void *dst;
    long long rstride, wstride;  // elements between the direction arrays of src and dst
    unsigned store;     // bit j: call j of the pass stores rho / u
    int W, H, OW, OH;   // columns of a tile, owned columns
    unsigned mw;        // magic pair of W
    int lw;
    int ntx;            // tiles along x, and their magic pair
    unsigned mn;
    int ln;
    int tiles;          // tiles of a plane, and their magic pair
    unsigned mt;
    int lt;
    int OZ;             // planes of a z range
    int blocks;         // tiles * z ranges
    int per_xcd;        // ceil(blocks / 8); the grid is 8 * per_xcd
    int rs[3], ws[3];   // read and write shifts, mod L
    int cls;            // MARCH_*
};

// Tiles of a lattice: the kernel's capacity (size, tile_capacity), the margin
// M = calls of a pass - 1 and the tile shape.
struct TilePlan {
    bool on = false;
    int size = 0, W = 0, H = 0, M = 0, OW = 0, OH = 0, ntx = 0, nty = 0;
    int OZ = 0, nz = 0;  // D3Q15: planes per z range, z ranges
    double us = 0;       // estimated time per call
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

// Runs of fewer calls go one call per launch (us for 3 calls, one by one and in
// passes of one and two: 2048 x 1024 FP64 143, 185, FP32 76, 86; 1148 x 450
// FP16S 29, 40); with 4 passes are ahead in every format and size that has them
// (1.01 to 1.7 times).
constexpr int kMinPassRun = 4;

// Passes of a run of len calls, K at most in each: an even number, so that the
// state ends in the buffer it started in, of two calls or more each (a pass
// of one call moves what a launch in place moves).  They share out min(len,
// passes * K) calls evenly; the rest, up to three, go one by one.
inline long long tile_passes(long long len, int K)
{
    const long long np = 2 * ((len + 2 * K - 1) / (2 * K));
    return len < 2 * np ? np - 2 : np;
}

// ns of a CU per node update (tile_estimate)
inline double tile_ns(int slot_bytes) { return slot_bytes == 8 ? 2.9 : slot_bytes == 4 ? 1.2 : 1.7; }

// node updates of one tile in a pass, and its bytes
inline double tile_updates(const TilePlan &q, int calls)
{
    double nodes = (double)q.OW * q.OH;
    for (int j = 0; j + 1 < calls; j++) nodes += (double)(q.W - 2 * j) * (q.H - 2 * j);
    return nodes;
}
inline double tile_bytes(const TilePlan &q, int slot_bytes)
{
    return 9 * (q.H * ((double)q.W * slot_bytes + 96) + q.OH * ((double)q.OW * slot_bytes + 96));
}

// Estimated time per call (us) of the passes of a plan.  Measured constants
// (MI355X): 3.5 us for a launch with its first loads and last stores; per
// call of a tile at least the latency of one update (0.5 us, 0.8 us in 64
// bits); per node update 1.2 ns of a CU (2.9 ns in 64 bits, 1.7 ns in 16
// bits, which also round and convert); 20 bytes per ns and CU of memory
// traffic, about half of it hidden under the arithmetic of the other
// resident blocks.
// calls: of a pass of fewer calls than the plan's M + 1.
inline double tile_estimate(const TilePlan &q, int slot_bytes, int ncu, int calls)
{
    const double us_call = slot_bytes == 8 ? 0.8 : 0.5;
    double per_cu = (double)q.ntx * q.nty / ncu;
    if (per_cu < 4) per_cu = std::max(1.0, (double)((long long)(per_cu + 0.999)));
    const double arith = std::max(calls * us_call, per_cu * tile_updates(q, calls) * tile_ns(slot_bytes) * 1e-3);
    return (3.5 + arith + 0.5 * per_cu * tile_bytes(q, slot_bytes) / 20e3) / calls;
}

// The plan with the smallest estimate (within 10 % of the best of all
// shapes on ten lattices from 64 x 48 to 3392 x 3392, three formats).  In 32
// and 64 bits it beats one call per launch at every size (us per call of a
// forced BGK channel, one call per launch -> passes: 256 x 64 FP64 3.8 -> 1.9,
// 600 x 300 FP32 6.2 -> 3.2, 2048 x 1024 FP32 25.2 -> 15.1, FP64 46.4 -> 34.0,
// 3392 x 3392 FP32 160 -> 68).  The 16-bit one-call kernels move half of FP32's bytes and are
// bound by the same arithmetic plus the conversions, so passes win only
// where launches count: 64 x 48 3.3 -> 1.2, 1500 x 400 11.3 -> 7.9, 2786 x
// 681 equal, 3392 x 3392 80 -> 92; hence the line at 2^20 nodes.
// Lattices with nodes of other classes than fluid and solid (boundary,
// prescribed or porous: plain false) take tiles of up to 512 nodes below 1.5e6
// nodes in 16 and 32 bits: a tile that holds such nodes takes longer, and of a
// few rounds of large tiles the last waits for it (MRT between pressure faces,
// tiles of 2048 -> 512 nodes: FP32 512 x 512 7.4 -> 5.4, 1148 x 450 9.3 -> 7.4,
// 1222 x 1000 15.4 -> 13.0, 1400 x 1400 19.6 against 19.0-19.9; FP16S 800 x 640
// 14.6 -> 8.1, one call per launch 11.7; 64 bits hold 1024 and gain 0-5 %).
// M up to 7: deeper passes of the small tiles recompute more than they save.
// calls: the plan for passes of that many (0: the best of all).
inline TilePlan plan_tiles(int Lx, int Ly, int slot_bytes, int ncu, bool plain, int calls = 0)
{
    TilePlan best;
    const long long nodes = (long long)Lx * Ly;
    if (slot_bytes == 2 && nodes > (1LL << 20)) return best;
    const int largest = !plain && slot_bytes <= 4 && nodes < 1500000 ? 1 : 2;
    for (int size = 0; size <= largest; size++) {
        const TileCapacity cap = tile_capacity(size, slot_bytes);
        const int P = cap.threads * cap.per_thread;
        for (int W = 16; W <= 128; W *= 2)
            for (int M = calls ? calls - 1 : 1; M <= (calls ? calls - 1 : 7); M++) {
                TilePlan q;
                if (P / W < 8 || !tile_shape(Lx, Ly, size, W, P / W, M, q)) continue;
                q.us = tile_estimate(q, slot_bytes, ncu, M + 1);
                q.on = true;
                if (!best.on || q.us < best.us) best = q;
            }
    }
    return best;
}

// Tiles of a pass of fewer calls than the lattice's plan q has: q's, or others
// with the margin that these calls need where they are estimated 10 % ahead, 5
// % in 16 bits (below that the planned ones were up to 15 % ahead at 600 x 300,
// 64 x 48).  Runs of 4 calls, us, one call per launch, q's tiles, these: FP32
// 600 x 300 24.7, 26.3, 18.6; 2048 x 1024 102, 99, 76; FP64 2048 x 1024 190,
// 203, 173; FP16S 1148 x 450 40, 48, 30.
inline TilePlan plan_short(const TilePlan &q, int Lx, int Ly, int slot_bytes, int ncu, bool plain, int calls)
{
    const TilePlan s = plan_tiles(Lx, Ly, slot_bytes, ncu, plain, calls);
    return s.on && s.us < (slot_bytes == 2 ? 0.95 : 0.9) * tile_estimate(q, slot_bytes, ncu, calls) ? s : q;
}

// Work of a plan's tiles per call, in ns of one CU (tile_estimate's terms),
// for batches, whose tiles of all members fill the chip together.
inline double tile_work(const TilePlan &q, int slot_bytes)
{
    return (double)q.ntx * q.nty *
           (tile_updates(q, q.M + 1) * tile_ns(slot_bytes) + 0.5 * tile_bytes(q, slot_bytes) / 20) / (q.M + 1);
}

// A batch's run, for batch_passes
struct BatchRun {
    long long nodes;   // of all members
    int slot_bytes;
    int nsteps;
    int store_every;
    bool macro;        // some members prescribe values: the calls that store them run alone
    int every;         // closure members' interval (0: none)
    bool mixed;        // closure members and others, which go in launches of their own
};

// Whether a batch's run pays in passes.  Measured on D2Q9 batches of 4 to 128
// members, 4600 to 6.7 M nodes, us per call in place -> in passes (runs of up
// to 8 calls: per run, which upload less and gain 5-15 us by that).  Not
// - one call, from 8 MB of slots per direction on, which saves no traffic: 6.7
//   M nodes FP32 155 -> 193, FP64 244 -> 317; 2.1 M FP32 95 -> 95;
// - prescribed values stored more often than every 4th call.
// The rest in 32 bits only: tiles of 2048 nodes, four to a thread, make a small
// batch wait for each call (tiles of 1024 in 64 bits are ahead: 16 x 96 x 64
// between pressure faces 7.0 -> 5.5).  Not
// - prescribed values below 2^19 nodes (MRT between pressure faces 16 x 96 x 64
//   6.1 -> 6.9, 8 x 256 x 128 7.8 -> 8.3, 128 x 96 x 64 15.7 -> 15.1), stored now
//   and then below 2^20 (every 12th call 128 x 96 x 64 15.6 -> 17.6, 64 x 256 x 128
//   35 -> 30), every 4th to 6th below 2^22 (64 x 256 x 128 35.3 -> 36.5);
// - the closure every 2nd call, a pass of one call each: 24 x 256 x 128 25.3 ->
//   28.3; beside other members from 2^20 nodes on 28.0 -> 26.2 (4 x 701 x 397);
// - the closure beside other members below 5 * 2^16 nodes, two lists of tiles
//   that each leave part of the chip idle: 8 x 256 x 128, interval 8, 9.0 -> 10.8;
//   64 x 96 x 64 12.0 -> 10.9.
inline bool batch_passes(const BatchRun &r)
{
    if (r.nsteps == 1 && r.nodes * r.slot_bytes > (8LL << 20)) return false;
    const bool stores = r.macro && r.store_every > 0;
    if (stores && r.store_every < 4) return false;
    if (r.slot_bytes != 4) return true;
    if (stores && r.nodes < (r.store_every < 7 ? 1LL << 22 : 1LL << 20)) return false;
    if (r.nsteps <= 8) return true;
    if (r.macro && r.nodes < (1LL << 19)) return false;
    if (r.every == 2) return r.mixed && r.nodes >= (1LL << 20);
    return !(r.every > 2 && r.mixed && r.nodes < (5LL << 16));
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

// Threads per block of the march kernels, by the registers that a column
// needs: 128 are available at 1024 threads (101-128 used), 256 at 512 (161-250
// in 64 bits).
constexpr int march_threads(int slot_bytes) { return slot_bytes == 8 ? 512 : 1024; }

// Collisions that the march kernels take: all but the MRT family with its
// inverse matrix (mfix) and a body force in 32 bits.  That update needs more
// than the 128 registers of a 1024-thread block (measured 131 x 97 x 75 25.0 us
// per call alone against 27.1 in passes, 256^3 363 against 391; without the
// force 24.4 against 17.1 and 359 against 254).
constexpr bool march_takes(int slot_bytes, bool mrt, bool mfix, bool force)
{
    return !(slot_bytes == 4 && mrt && mfix && force);
}

inline void march_shape(const int *L, int W, int H, int nz, TilePlan &q)
{
    q.M = 1;
    q.ntx = (L[0] + W - 3) / (W - 2);
    q.nty = (L[1] + H - 3) / (H - 2);
    q.OW = (L[0] + q.ntx - 1) / q.ntx;
    q.OH = (L[1] + q.nty - 1) / q.nty;
    q.W = q.OW + 2;
    q.H = q.OH + 2;
    q.OZ = (L[2] + nz - 1) / nz;
    q.nz = (L[2] + q.OZ - 1) / q.OZ;
}

// Estimated time per call (us) of the march passes of a plan: 2 us per launch
// and an iteration (one plane of every resident block) of b + c * MB, MB the
// traffic of the resident blocks with e bytes of partial lines at the ends of
// every tile row.  b, c and e fitted to 260 shapes on 11 lattices (within 4-10
// % of the measured times; the chosen shape 0-4 % from the best), apart for
// lattices whose two buffers fit the 256 MB last-level cache.
inline double march_estimate(const TilePlan &q, const int *L, int slot_bytes, int ncu)
{
    const double s = slot_bytes;
    const bool cached = 2.0 * 15 * s * L[0] * L[1] * L[2] <= 260e6;
    const double e = slot_bytes == 8 ? (cached ? 64 : 96) : (cached ? 160 : 64);
    const double b = slot_bytes == 8 ? (cached ? 4.5 : 3.3) : (cached ? 2.7 : 0.6);
    const double c = cached ? 0.015 : slot_bytes == 8 ? 0.075 : 0.135;
    const bool aligned = q.OW * slot_bytes % 128 == 0 && L[0] * slot_bytes % 128 == 0;
    const double bytes = 15 * (q.H * (q.W * s + e) + q.OH * (q.OW * s + (aligned ? 0 : e)));
    const double blocks = (double)q.ntx * q.nty * q.nz;
    const double rounds = (double)((long long)((blocks + ncu - 1) / ncu));
    const double mb = (blocks < ncu ? blocks : ncu) * bytes * 1e-6;
    return (2.0 + rounds * (q.OZ + 2) * (b + c * mb)) / 2;
}

// One call per launch: 2 us, then 6 TB/s where the populations stay in the
// 256 MB last-level cache, 5.6 TB/s from HBM.
inline double march_step_estimate(double nodes, int slot_bytes)
{
    const double bytes = nodes * 15 * slot_bytes;
    return 2.0 + 2 * bytes / (bytes <= 256e6 ? 6e6 : 5.6e6);
}

// The plan with the smallest estimate, or none where one call per launch is
// estimated within 5 % of it (lattices below ~6e5 nodes: too few columns for
// 256 CUs).
// Measured, us per call, one call per launch -> passes: FP32 BGK with
// Smagorinsky, all fluid, 256^3 357 -> 230, 512^3 3005 -> 1774, 128^3 39.1 ->
// 26, 131 x 97 x 75 21.6 -> 13.5; forced duct with solid walls 256^3 366 ->
// 241, 131 x 97 x 75 24.0 -> 15.2; FP64 256^3 771 -> 551, 200 x 150 x 100
// 137 -> 109; MRT, forced duct, FP64 131 x 97 x 75 42 -> 37, 200^3 402 -> 280;
// MRT box FP32 256^3 359 -> 254; 64^3 6.2 against 8.3 in passes (not planned).
// FP64 lattices that fit the last-level cache once but not twice stay with one
// call per launch (128^3: BGK box 73.6 against 74.8, forced ducts 75 against
// 80-97; only boxes of 150-220 MB would gain, 5-15 %).  16-bit lattices have no passes: 256^3
// 192 us against 221, bound by the arithmetic that a pass repeats at the sides.
inline TilePlan plan_march(const int *L, int slot_bytes, int ncu)
{
    TilePlan best;
    if (slot_bytes < 4) return best;
    const double nodes = (double)L[0] * L[1] * L[2], bytes = nodes * 15 * slot_bytes;
    if (slot_bytes == 8 && bytes > 128e6 && bytes <= 256e6) return best;
    best.us = 0.95 * march_step_estimate(nodes, slot_bytes);
    const int T = march_threads(slot_bytes);
    for (int k = 1; k <= 64 && k <= L[0]; k++) {
        const int W = (L[0] + k - 1) / k + 2, H = std::min(T / W, L[1] + 2);
        if (W < 18 && k > 1) break;
        if (H < 3) continue;
        const int tiles = ((L[0] + W - 3) / (W - 2)) * ((L[1] + H - 3) / (H - 2));
        for (int r = 1; r <= 4; r++) {
            // the most z ranges that r rounds of blocks hold
            const int nz = std::max(1, std::min((r * ncu) / tiles, L[2]));
            TilePlan q;
            march_shape(L, W, H, nz, q);
            q.us = march_estimate(q, L, slot_bytes, ncu);
            if (q.us < best.us) {
                best = q;
                best.on = true;
            }
        }
    }
    return best;
}

inline void march_geometry(const TilePlan &q, MarchPass &p)
{
    p.W = q.W;
    p.H = q.H;
    p.OW = q.OW;
    p.OH = q.OH;
    p.ntx = q.ntx;
    p.tiles = q.ntx * q.nty;
    const FastDiv dw = make_fastdiv(q.W), dn = make_fastdiv(q.ntx), dt = make_fastdiv(p.tiles);
    p.mw = dw.m;
    p.lw = dw.l;
    p.mn = dn.m;
    p.ln = dn.l;
    p.mt = dt.m;
    p.lt = dt.l;
    p.OZ = q.OZ;
    p.blocks = p.tiles * q.nz;
    p.per_xcd = (p.blocks + 7) / 8;
}

}  // namespace lbmc
