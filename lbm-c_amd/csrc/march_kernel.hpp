// Two calls of a D3Q15 lattice in one pass over memory.
//
// A block takes a tile of W x H columns (x, y) -- the OW x OH columns that it
// owns and one column more on every side -- and marches over the planes of
// its z range, one thread per column.  At plane z it takes the arriving
// populations from device memory, makes the first call there and passes the
// post-collision values of the 12 directions that leave their column
// through LDS to the columns they stream to.  The second call of plane z - 1
// then has all it needs: the e_z = -1 populations from plane z, the e_z = 0
// ones from plane z - 1 and the e_z = +1 ones from plane z - 2, the latter
// two kept in registers since they were passed on.  It writes the owned nodes
// to device memory.  The side columns and the planes before and after the
// range are computed by every block that needs them, from the same inputs by
// the same node update: every node's values are those of the one-call
// kernels, bit for bit.
//
// As in the D2Q9 passes (tile_kernel.hpp) a pass reads one population buffer
// and writes another, with a read and a write shift per axis; a slot's
// address is a uniform plane base per direction plus the column's 32-bit
// offset within a plane.
//
// What bounds it: memory traffic.  A pass reads 60 bytes per FP32 node, the
// side columns again (mostly from L2) and writes 60: 62-65 bytes per node
// and call at 256^3 against 120 with one call per launch.  The march runs at 4.6
// TB/s of that (a bare copy in its order at 4.9-5.2, a linear one at 6.0),
// its arithmetic alone would take 97 of the 218-230 us per call.  Tiles of
// 64 x 13 owned columns: rows of whole lines, 19 % of the columns computed
// twice; 32 x 28 has 12 % but is 11 % slower.  Three calls per pass (own 64
// x 11, two barriers per plane) measured 251 us, two 512-thread blocks per CU
// 257, non-temporal stores 244.
//
// The closure's calls between evaluations take the same passes: at 128^3 FP32
// a call of an interval of 4 takes 41.9 us on average against 47.7 with one
// call per launch, of 8 33.6 against 44.4 (200^3: 144 against 209).  The
// evaluating calls stay alone: their network keeps the vector units busy (85 %
// of their issue slots), and its registers beside the march's do not fit.
#pragma once

#include <hip/hip_runtime.h>

#include "closure_kernel.hpp"
#include "step_kernel.hpp"
#include "tile_pass.hpp"

namespace lbmc {

// x, in its register from here on (a load into it has finished); no instruction
template <class C>
__device__ __forceinline__ void arrived(C &x)
{
    asm volatile("" : "+v"(x));
}

// LDS row of a direction that leaves its column: 1..4 -> 0..3, 7..14 -> 4..11
constexpr int march_row(int i) { return i < 5 ? i - 1 : i - 3; }

// T threads; CLS: the node classes of the lattice (MARCH_*).  One block per
// CU: 4 waves per SIMD at 1024 threads, 2 at 512.  REUSE: calls of the
// learned closure between evaluations (closure_reuse_tau); a column's record
// of a plane is loaded once for both calls.
// FORCE: MARCH_NO_FORCE, or a force per node or the same at every node.  The
// last two are apart because a load of the force in an update waits, in the
// one in-order counter, for the next plane's populations issued before it;
// the compiler places that wait behind the branch that reads a uniform force
// too.  With the load compiled out a forced BGK duct of 256^3 takes 244 us per
// call in FP32 instead of 273, 535 in FP64 instead of 606.
template <class L, class St, int FAM, int FORCE, bool SMAG, bool MFIX, int CLS, int T, bool REUSE>
__global__ __launch_bounds__(T, T / 256) void march_kernel(const StepArgs<typename St::C> args, const MarchPass p)
{
    using C = typename St::C;
    using S = typename St::S;
    constexpr bool GUO = FORCE != MARCH_NO_FORCE;
    StepArgs<C> a = args;
    if constexpr (FORCE == MARCH_UNIFORM_FORCE) a.force[0] = a.force[1] = a.force[2] = nullptr;
    static_assert(L::D == 3 && !St::stochastic, "D3Q15, storage without conversions");
    constexpr int Q = L::Q;
    __shared__ S lds[2][12][T];  // of even and odd planes: one barrier per plane
    const int Lx = a.L[0], Ly = a.L[1], Lz = a.L[2];
    // consecutive tiles of a z range on one XCD (blocks are dealt to the 8
    // XCDs round robin): neighbouring tiles share the lines at their sides in its L2
    const unsigned pos = (blockIdx.x & 7u) * (unsigned)p.per_xcd + (blockIdx.x >> 3);
    if (pos >= (unsigned)p.blocks) return;  // block-uniform
    const int zc = fast_div((int)pos, p.mt, p.lt), tile = (int)pos - zc * p.tiles;
    const int by = fast_div(tile, p.mn, p.ln), bx = tile - by * p.ntx;
    const int z0 = zc * p.OZ, oz = min(p.OZ, Lz - z0);
    const int id = (int)threadIdx.x;
    const bool in = id < p.W * p.H;
    const int cid = in ? id : 0;  // spare threads follow column 0 and write nothing
    const int ty = fast_div(cid, p.mw, p.lw), tx = cid - ty * p.W;
    const int ux = bx * p.OW + tx - 1, uy = by * p.OH + ty - 1;
    const bool own = in && tx >= 1 && tx < p.W - 1 && ty >= 1 && ty < p.H - 1 && ux < Lx && uy < Ly;
    int gx = ux + Lx, gy = uy + Ly;
    gx -= fast_div(gx, a.mx, a.lx) * Lx;
    gy -= fast_div(gy, a.my, a.ly) * Ly;
    const int nxy = gx + gy * Lx;
    const unsigned plane = (unsigned)Lx * (unsigned)Ly;

    // column offsets for the components -1, 0, +1, in elements
    auto columns = [&](const int *s, int (&cx)[3], int (&cy)[3]) {
        cx[1] = gx;
        cx[2] = gx >= s[0] ? gx - s[0] : gx + Lx - s[0];
        cx[0] = gx + s[0] < Lx ? gx + s[0] : gx + s[0] - Lx;
        cy[1] = gy * Lx;
        cy[2] = (gy >= s[1] ? gy - s[1] : gy + Ly - s[1]) * Lx;
        cy[0] = (gy + s[1] < Ly ? gy + s[1] : gy + s[1] - Ly) * Lx;
    };
    int rx[3], ry[3], wx[3], wy[3];
    columns(p.rs, rx, ry);
    columns(p.ws, wx, wy);
    auto wrap_z = [&](int z) { return z < 0 ? z + Lz : (z >= Lz ? z - Lz : z); };
    // slot of direction i of the column at plane z: a uniform plane base and
    // the column's offset
    auto slot = [&](auto ii, const void *f, long long stride, const int *s, int z, const int (&cx)[3], const int (&cy)[3]) -> S * {
        constexpr int i = decltype(ii)::value;
        int q = z - L::ez[i] * s[2];
        q = q < 0 ? q + Lz : (q >= Lz ? q - Lz : q);
        const unsigned off = (unsigned)(cx[L::ex[i] + 1] + cy[L::ey[i] + 1]) * (unsigned)sizeof(S);
        return (S *)((char *)((S *)f + (size_t)i * stride + (size_t)q * plane) + lane_offset(off));
    };
    auto gather = [&](int z, C (&v)[Q]) {
        sfor<0, Q>([&](auto ii) {
            v[decltype(ii)::value] = St::load(ldg((const S *)slot(ii, p.src, p.rstride, p.rs, z, rx, ry)));
        });
    };
    auto record = [&](int z) -> C { return ldg(a.tcache + (nxy + z * (int)plane)); };
    auto solid = [&](int z) -> unsigned {
        if constexpr (CLS == MARCH_FLUID) return 0;
        else return ldg(a.mask + (nxy + z * (int)plane));
    };

    // the update of node n; m, t: its mask byte and recorded relaxation time
    // (the two classes apart, each compiled for its descriptor)
    auto update = [&](int n, unsigned m, bool store, C t, C (&v)[Q]) {
        if (CLS != MARCH_FLUID && m != 0) node_update_as<L, St, FAM, GUO, SMAG, MFIX>(a, n, (uint16_t)CLS_SOLID, store, v);
        else if constexpr (REUSE) closure_reuse_tau<L, St, GUO>(a, n, 0, store, t, v);
        else node_update_as<L, St, FAM, GUO, SMAG, MFIX>(a, n, 0, store, v);
    };

    C flat[5], up1[5], up2[5];  // arrivals held for the second call: e_z = 0 of the last plane, e_z = +1 of the
                                // last plane and of the one before it
    unsigned m1 = 0, m2 = 0;    // mask bytes of this plane's node and of the last plane's, and
    C t1 = 0, t2 = 0;           // their records: loaded a plane ahead like the populations
    // plane k of the range: the first call there, on its populations f, and
    // the second call of plane k - 1; loads plane k + 1 into w meanwhile
    auto plane_calls = [&](int k, C (&f)[Q], C (&w)[Q]) {
        const int z = wrap_z(z0 + k);
        const int n = nxy + z * (int)plane;
        const int zn = wrap_z(z0 + min(k + 1, oz));
        gather(zn, w);
        unsigned mn = solid(zn);
        C tn = 0;
        if constexpr (REUSE) tn = record(zn);
        __builtin_amdgcn_sched_barrier(0);
        S(*row)[T] = lds[k & 1];
        const bool st = (p.store & 1u) != 0 && own && k >= 0 && k < oz;
        update(n, m1, st, t1, f);
        sfor<1, Q>([&](auto ii) {
            constexpr int i = decltype(ii)::value;
            if constexpr (L::ex[i] != 0 || L::ey[i] != 0) row[march_row(i)][id] = St::store(f[i]);
        });
        __syncthreads();
        // post-collision value of the node that direction i arrives from
        auto arrive = [&](auto ii) -> C {
            constexpr int i = decltype(ii)::value;
            if constexpr (L::ex[i] != 0 || L::ey[i] != 0)
                return St::load(row[march_row(i)][id - L::ex[i] - L::ey[i] * p.W]);
            else return f[i];
        };
        const bool second = own && k >= 1;
        const int zs = wrap_z(z0 + k - 1);
        const int ns = nxy + zs * (int)plane;
        C r[Q];
        if (second) {
            int cf = 0, cu = 0;
            sfor<0, Q>([&](auto ii) {
                constexpr int i = decltype(ii)::value;
                if constexpr (L::ez[i] == 0) r[i] = flat[cf++];
                else if constexpr (L::ez[i] == 1) r[i] = up2[cu++];
                else r[i] = arrive(ii);
            });
            update(ns, m2, (p.store & 2u) != 0, t2, r);
        }
        if (own) {
            int cf = 0, cu = 0;
            sfor<0, Q>([&](auto ii) {
                constexpr int i = decltype(ii)::value;
                if constexpr (L::ez[i] == 0) flat[cf++] = arrive(ii);
                else if constexpr (L::ez[i] == 1) {
                    up2[cu] = up1[cu];
                    up1[cu++] = arrive(ii);
                }
            });
        }
        if (second) {
            sfor<0, Q>([&](auto ii) {
                stg(slot(ii, p.dst, p.wstride, p.ws, zs, wx, wy), St::store(r[decltype(ii)::value]));
            });
        }
        // Wait for plane k + 1 here (and, in the same in-order counter, for
        // the stores): a block then runs at most one plane ahead of its
        // memory traffic, and the blocks of an XCD stay close together in z,
        // where the side columns of one are in L2 from the other.  Loads two
        // planes ahead fetch 1.45 GB per pass at 256^3 instead of 1.24 and
        // take 5 % longer.
        sfor<0, Q>([&](auto ii) { arrived(w[decltype(ii)::value]); });
        if constexpr (REUSE) {
            arrived(tn);
            t2 = t1;
            t1 = tn;
        }
        if constexpr (CLS != MARCH_FLUID) arrived(mn);
        m2 = m1;
        m1 = mn;
    };
    // two sets of populations in turn, so that a load in flight stays in its
    // registers
    C va[Q], vb[Q];
    gather(wrap_z(z0 - 1), va);
    m1 = solid(wrap_z(z0 - 1));
    if constexpr (REUSE) t1 = record(wrap_z(z0 - 1));
    sfor<0, Q>([&](auto ii) { arrived(va[decltype(ii)::value]); });
    for (int k = -1;; k += 2) {
        plane_calls(k, va, vb);
        if (k + 1 > oz) break;
        plane_calls(k + 1, vb, va);
        if (k + 2 > oz) break;
    }
}

}  // namespace lbmc
