// Several calls of a D2Q9 lattice in one pass over memory.
//
// A block takes a rectangular tile of W x H nodes: the OW x OH nodes that it
// owns and a margin of M nodes on every side (W = OW + 2 M, H = OH + 2 M).
// The first call reads the tile's arriving populations from device memory
// and leaves the post-collision values in LDS; each further call streams and
// collides inside LDS, valid on a tile that shrinks by one node per side; the
// last one (at most the (M + 1)-th) writes the owned nodes' populations to
// device memory.  Margins are computed by every tile that holds them, from
// the same inputs by the same node update, so every node's values are those
// of the one-call kernels, bit for bit.
//
// Streaming inside LDS is the index shift of the lattice itself: in call j
// of the pass node (x, y) reads and writes direction i at tile slot
// (x - j e_x, y - j e_y), so the update is in place, each slot belongs to one
// node per call and one barrier per call is enough.  A node that is valid in
// call j lies at least j nodes inside the tile, so its slots never wrap.
//
// Tiles of one pass read nodes that other tiles own, so a pass reads one
// population buffer and writes another (src, dst).  The layout of either
// side is an index shift by a number of calls: rs for reading (t mod L to
// continue the stored state of call t; 1 for a buffer holding
// post-collision values at their own nodes) and ws for writing (the same
// numbers; 0 leaves them at their own nodes, aligned rows).
//
// What bounds it: vector-instruction issue.  One call per launch moves 72
// bytes per FP32 node and call; five calls per pass move (36 x 1.7 + 36) / 5
// = 20, and recompute 1.2-1.35 times the nodes, which the arithmetic units
// had to spare.  Measured (MI355X, us per call, one call per launch ->
// passes): FP32 BGK box 4096 x 4096 224 -> 90 (tiles of 64 x 32, M = 4: 187 k
// MLUPS), forced channel 224 -> 105; MRT between pressure faces 2048 x 1024
// FP32 25.1 -> 19.3, FP64 46.9 -> 31.3 (32 x 32, M = 3); small lattices also
// save the launches, FP64 256 x 64 3.8 -> 1.9.  Two blocks of 72 KB LDS per CU hide one block's loads and stores
// under the other's arithmetic: one block of 144 KB (64 x 64 tiles, less
// recomputation) is 2-20 % slower.
#pragma once

#include <hip/hip_runtime.h>

#include "step_kernel.hpp"
#include "tile_pass.hpp"

namespace lbmc {

// LDS element of tile slot id - j (e_y W + e_x) of direction I
template <class L, class S, int I, int P>
__device__ __forceinline__ int tile_slot(int id, int jx, int jy)
{
    return I * P + id - L::ex[I] * jx - L::ey[I] * jy;
}

// One tile of a pass.  T threads, NPT nodes per thread, W * H <= T * NPT.
// update(n, desc, store, v): the update of node n, class descriptor desc, on
// its populations v.
template <class L, class St, int T, int NPT, class Update>
__device__ __forceinline__ void tile_calls(const StepArgs<typename St::C> &a, const TilePass &p, unsigned tile,
                                           typename St::S *lds, Update &&update)
{
    using C = typename St::C;
    using S = typename St::S;
    constexpr int Q = L::Q;
    constexpr int P = T * NPT;
    const int Lx = a.L[0], Ly = a.L[1];
    const int by = fast_div((int)tile, p.mt, p.lt), bx = (int)tile - by * p.ntx;
    const int ox = bx * p.OW, oy = by * p.OH;  // first owned node
    // per node: lattice index, and its depth inside the tile (calls j <= depth
    // are valid; -1 past the tile), bit 8 owned, class descriptor from bit 16
    int node[NPT], info[NPT];
    sfor<0, NPT>([&](auto qq) {
        constexpr int q = decltype(qq)::value;
        const int id = (int)threadIdx.x + q * T;
        const int ty = fast_div(id, p.mw, p.lw), tx = id - ty * p.W;
        int dep = min(min(tx, p.W - 1 - tx), min(ty, p.H - 1 - ty));
        const bool in = id < p.W * p.H;
        const int ux = ox + tx - p.M, uy = oy + ty - p.M;  // before wrapping
        const bool own = in && dep >= p.M && ux < Lx && uy < Ly;
        int gx = ux + p.xoff, gy = uy + p.yoff;
        gx -= fast_div(gx, a.mx, a.lx) * Lx;
        gy -= fast_div(gy, a.my, a.ly) * Ly;
        const int n = gx + gy * Lx;
        node[q] = n;
        dep = in ? min(dep, 127) : -1;
        const unsigned desc = in ? node_class(a, n) : 0u;
        info[q] = (dep & 0xFF) | (own ? 0x100 : 0) | (int)(desc << 16);
    });
    auto depth = [](int w) { return (int)(signed char)(w & 0xFF); };

    const S *const src = (const S *)p.src;
    S *const dst = (S *)p.dst;
    // slot offsets of a node for a shift s: gx and gy relative to the node
    auto offsets = [&](int n, const int *s, int (&dx)[3], int (&dy)[3]) {
        const int gy = fast_div(n, a.mx, a.lx), gx = n - gy * Lx;
        dx[1] = dy[1] = 0;
        dx[2] = gx >= s[0] ? -s[0] : Lx - s[0];
        dx[0] = gx + s[0] < Lx ? s[0] : s[0] - Lx;
        dy[2] = (gy >= s[1] ? -s[1] : Ly - s[1]) * Lx;
        dy[0] = (gy + s[1] < Ly ? s[1] : s[1] - Ly) * Lx;
    };
    auto seed_of = [&](int j) {
        unsigned ts = 0;
        if constexpr (St::stochastic) {
            int sx = p.s0[0] + j, sy = p.s0[1] + j;
            sx -= fast_div(sx, a.mx, a.lx) * Lx;
            sy -= fast_div(sy, a.my, a.ly) * Ly;
            ts = (unsigned)sx + (unsigned)Lx * (unsigned)sy;
        }
        return ts;
    };
    // stored form of a node's post-collision values, direction by direction
    auto stored = [&](int n, unsigned ts, const C (&v)[Q], auto &&put) {
        unsigned r = 0;
        if constexpr (St::stochastic) r = sr_seed(n, ts);
        sfor<0, Q>([&](auto ii) {
            constexpr int i = decltype(ii)::value;
            if constexpr (St::stochastic) {
                put(ii, St::store_sr(v[i], r));
                r = sr_next(r);
            } else {
                put(ii, St::store(v[i]));
            }
        });
    };
    auto to_lds = [&](int id, int n, int jx, int jy, unsigned ts, const C (&v)[Q]) {
        stored(n, ts, v, [&](auto ii, S w) { lds[tile_slot<L, S, decltype(ii)::value, P>(id, jx, jy)] = w; });
    };
    auto to_dst = [&](int n, unsigned ts, const C (&v)[Q]) {
        int dx[3], dy[3];
        offsets(n, p.ws, dx, dy);
        stored(n, ts, v, [&](auto ii, S w) {
            constexpr int i = decltype(ii)::value;
            const unsigned k = (unsigned)(n + dx[L::ex[i] + 1] + dy[L::ey[i] + 1]);
            const unsigned e = sizeof(S) == 2 ? slot_elem(k, a.hs) : k;
            stg((S *)((char *)(dst + (size_t)i * a.npad) + e * (unsigned)sizeof(S)), w);
        });
    };
    // the node's index, opaque: keeps the addresses formed from it beside
    // their use instead of in registers across all the calls of the pass
    auto index = [&](int n) { return (int)lane_offset((unsigned)n); };

    // call 0: from device memory
    {
        constexpr int G = NPT < 2 ? NPT : 2;  // nodes whose loads are in flight together
        const unsigned ts = seed_of(0);
        sfor<0, NPT / G>([&](auto gg) {
            constexpr int g0 = decltype(gg)::value * G;
            C v[G][Q];
            sfor<g0, g0 + G>([&](auto qq) {
                constexpr int q = decltype(qq)::value;
                if (p.calls > 1 ? depth(info[q]) >= 0 : (info[q] & 0x100) != 0) {
                    int dx[3], dy[3];
                    const int n = index(node[q]);
                    offsets(n, p.rs, dx, dy);
                    sfor<0, Q>([&](auto ii) {
                        constexpr int i = decltype(ii)::value;
                        const unsigned k = (unsigned)(n + dx[L::ex[i] + 1] + dy[L::ey[i] + 1]);
                        const unsigned e = sizeof(S) == 2 ? slot_elem(k, a.hs) : k;
                        v[q - g0][i] = St::load(
                            ldg((const S *)((const char *)(src + (size_t)i * a.npad) + e * (unsigned)sizeof(S))));
                    });
                }
            });
            sfor<g0, g0 + G>([&](auto qq) {
                constexpr int q = decltype(qq)::value;
                const bool own = (info[q] & 0x100) != 0;
                if (p.calls > 1 ? depth(info[q]) >= 0 : own) {
                    const int n = index(node[q]);
                    update(n, (uint16_t)((unsigned)info[q] >> 16), (p.store & 1u) != 0 && own, v[q - g0]);
                    if (p.calls > 1) to_lds((int)threadIdx.x + q * T, n, 0, 0, ts, v[q - g0]);
                    else to_dst(n, ts, v[q - g0]);
                }
            });
        });
    }
    auto lds_call = [&](int j, int q, int id, auto &&write) {
        C v[Q];
        sfor<0, Q>([&](auto ii) {
            constexpr int i = decltype(ii)::value;
            v[i] = St::load(lds[tile_slot<L, S, i, P>(id, j, j * p.W)]);
        });
        const int n = index(node[q]);
        const bool st = ((p.store >> j) & 1u) != 0 && (info[q] & 0x100) != 0;
        update(n, (uint16_t)((unsigned)info[q] >> 16), st, v);
        write(n, v);
    };
    // further calls: in LDS
    for (int j = 1; j + 1 < p.calls; j++) {
        __syncthreads();
        const unsigned ts = seed_of(j);
        sfor<0, NPT>([&](auto qq) {
            constexpr int q = decltype(qq)::value;
            const int id = (int)threadIdx.x + q * T;
            if (depth(info[q]) >= j)
                lds_call(j, q, id, [&](int n, const C (&v)[Q]) { to_lds(id, n, j, j * p.W, ts, v); });
        });
    }
    // the last call: the owned nodes, to device memory
    if (p.calls > 1) {
        const int j = p.calls - 1;
        __syncthreads();
        const unsigned ts = seed_of(j);
        sfor<0, NPT>([&](auto qq) {
            constexpr int q = decltype(qq)::value;
            if (info[q] & 0x100)
                lds_call(j, q, (int)threadIdx.x + q * T, [&](int n, const C (&v)[Q]) { to_dst(n, ts, v); });
        });
    }
}

template <class L, class St, int FAM, bool GUO, bool SMAG, int T, int NPT>
__global__ __launch_bounds__(T, 4) void tile_kernel(const StepArgs<typename St::C> a, const TilePass p)
{
    __shared__ typename St::S lds[L::Q * T * NPT];
    tile_calls<L, St, T, NPT>(a, p, blockIdx.x, lds, [&](int n, uint16_t desc, bool st, typename St::C(&v)[L::Q]) {
        node_update_as<L, St, FAM, GUO, SMAG, false>(a, n, desc, st, v);
    });
}

}  // namespace lbmc
