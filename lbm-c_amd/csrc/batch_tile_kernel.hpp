// Passes of several calls over the D2Q9 members of a batch (tile_kernel.hpp):
// one launch takes a tile of every member through `calls` calls.  Members are
// independent, so plain members and members with the learned closure keep
// their own sequence of launches: plain ones passes over the whole run,
// closure ones an evaluating call (batch_call_kernel, in place) and passes
// with the recorded tau up to the next evaluation.
//
// Bound by vector-instruction issue, like the single-lattice passes.  64
// uneven channels (11.2 M nodes, FP32, MRT and BGK with forcing): 172 -> 102-108
// us per call (five calls a pass, 1.29 nodes computed per node owned);
// with the BGK members' closure evaluated every 8th call 194 -> 134-140 us.
// Tiles are listed by collision variant, so that blocks that run together
// share the instruction cache.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "batch_kernel.hpp"
#include "tile_kernel.hpp"

namespace lbmc {

// A member: arguments of the run's first call, tiles (src = its population
// buffer, dst = its second one) and collision variant (BatchMember)
template <class C>
struct BatchTileMember {
    StepArgs<C> a;
    TilePass p;
    int variant;
};

// One launch: calls offset .. offset + calls - 1 of the run
struct BatchPass {
    int offset, calls;
    unsigned store;    // bit j: call j of the pass stores rho / u
    int first, last;   // reads / leaves the stored layout
    int odd;           // the state is in the second buffer
};

// t mod L of the run's call `offset` along an axis, from that of its first call
template <class C>
__device__ __forceinline__ int call_shift(const StepArgs<C> &a, int d, int offset)
{
    const unsigned v = (unsigned)a.s[d] + (unsigned)offset;  // < 2^32
    const unsigned L = (unsigned)a.L[d];
    return (int)(v % L);
}

template <class St, int T, int NPT>
__global__ __launch_bounds__(T, 4) void batch_tile_kernel(
    const BatchTileMember<typename St::C> *__restrict__ members, const int2 *__restrict__ tiles, const BatchPass bp)
{
    using L = D2Q9;
    using C = typename St::C;
    __shared__ typename St::S lds[L::Q * T * NPT];
    const int2 e = tiles[blockIdx.x];  // (member, tile)
    const BatchTileMember<C> &m = members[e.x];
    const StepArgs<C> &a = m.a;
    TilePass p = m.p;
    if (bp.odd) {
        p.src = m.p.dst;
        p.dst = (void *)m.p.src;
    }
    p.calls = bp.calls;
    p.store = bp.store;
    for (int d = 0; d < 2; d++) {
        p.s0[d] = call_shift(a, d, bp.offset);
        p.rs[d] = bp.first ? p.s0[d] : (a.L[d] > 1 ? 1 : 0);
        p.ws[d] = bp.last ? call_shift(a, d, bp.offset + bp.calls - 1) : 0;
    }
    auto plain = [&](auto fam, auto guo, auto smag) {
        tile_calls<L, St, T, NPT>(a, p, (unsigned)e.y, lds, [&](int n, uint16_t desc, bool st, C(&v)[L::Q]) {
            node_update_as<L, St, decltype(fam)::value, decltype(guo)::value, decltype(smag)::value, false>(a, n, desc,
                                                                                                          st, v);
        });
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using F = std::false_type;
    using Y = std::true_type;
    switch (m.variant) {
    case 0: plain(I0{}, F{}, F{}); break;
    case 1: plain(I0{}, F{}, Y{}); break;
    case 2: plain(I0{}, Y{}, F{}); break;
    case 3: plain(I0{}, Y{}, Y{}); break;
    case 4: plain(I1{}, F{}, F{}); break;
    case 6: plain(I1{}, Y{}, F{}); break;
    default:
        if constexpr (std::is_same<C, float>::value) {
            // between evaluations: the recorded tau
            auto reuse = [&](auto guo) {
                tile_calls<L, St, T, NPT>(a, p, (unsigned)e.y, lds, [&](int n, uint16_t desc, bool st, C(&v)[L::Q]) {
                    closure_reuse_node<L, St, decltype(guo)::value>(a, n, desc, st, v);
                });
            };
            if (m.variant == 9) reuse(Y{});
            else reuse(F{});
        }
        break;
    }
}

// An evaluating call of the closure members, in place in the buffer that
// holds their state: batch_eval_kernel on the call's own shifts.
template <class St, bool RECORD, bool H>
__global__ __launch_bounds__(kBlock, 4) void batch_call_kernel(const BatchTileMember<float> *__restrict__ members,
                                                               const int2 *__restrict__ chunks, int nchunks, int sub,
                                                               const void *__restrict__ mlp, const BatchPass bp)
{
    using L = D2Q9;
    using S = typename St::S;
    constexpr int Q = L::Q;
    __shared__ MlpEval w;
    __shared__ uint4 xb[kBlock];
    {
        const uint4 *src = (const uint4 *)eval_image<H>(mlp);
        uint4 *dst = (uint4 *)&w;
        for (int k = (int)threadIdx.x; k < (int)(sizeof(MlpEval) / 16); k += kBlock) dst[k] = src[k];
    }
    __syncthreads();
    uint4 *xw = xb + (threadIdx.x & ~63u);
    for (int c = (int)blockIdx.x; c < nchunks; c += (int)gridDim.x) {
        const int2 ch = chunks[c];
        if (ch.x < 0) continue;
        const BatchTileMember<float> &m = members[ch.x];
        if (m.variant < 8) continue;  // not a closure member; block-uniform
        const StepArgs<float> &a = m.a;
        S *const f = (S *)(bp.odd ? m.p.dst : (void *)m.p.src);
        const int sx = call_shift(a, 0, bp.offset), sy = call_shift(a, 1, bp.offset);
        const int Lx = a.L[0], Ly = a.L[1];
        for (int j = 0; j < sub; j++) {
            const unsigned t0 = tile_node((unsigned)ch.y, (unsigned)j, kBlock, 0u);
            if (t0 >= (unsigned)a.nnodes) break;
            const unsigned n0 = t0 + threadIdx.x;
            const bool live = n0 < (unsigned)a.nnodes;
            const int n = live ? (int)n0 : a.nnodes - 1;
            const int y = fast_div(n, a.mx, a.lx), x = n - y * Lx;
            const int dx[3] = {x + sx < Lx ? sx : sx - Lx, 0, x >= sx ? -sx : Lx - sx};
            const int dy[3] = {(y + sy < Ly ? sy : sy - Ly) * Lx, 0, (y >= sy ? -sy : Ly - sy) * Lx};
            auto slot = [&](auto ii) -> S * {
                constexpr int i = decltype(ii)::value;
                const unsigned k = (unsigned)(n + dx[L::ex[i] + 1] + dy[L::ey[i] + 1]);
                return (S *)((char *)(f + (size_t)i * a.npad) + lane_offset(k * (unsigned)sizeof(S)));
            };
            float v[Q];
            sfor<0, Q>([&](auto ii) { v[decltype(ii)::value] = St::load(ldg((const S *)slot(ii))); });
            const bool st = (bp.store & 1u) != 0;
            if (m.variant == 9) closure_update<L, St, true, RECORD, H>(a, n, live, st, v, w, xw);
            else closure_update<L, St, false, RECORD, H>(a, n, live, st, v, w, xw);
            if (live) sfor<0, Q>([&](auto ii) { stg(slot(ii), St::store(v[decltype(ii)::value])); });
        }
    }
}

template <class St>
hipError_t launch_batch_tiles(const void *members, const int2 *tiles, int ntiles, const BatchPass &bp, hipStream_t s)
{
    constexpr TileCapacity cap = tile_capacity(2, (int)sizeof(typename St::S));
    hipLaunchKernelGGL((batch_tile_kernel<St, cap.threads, cap.per_thread>), dim3(ntiles), dim3(cap.threads), 0, s,
                       (const BatchTileMember<typename St::C> *)members, tiles, bp);
    return hipGetLastError();
}

}  // namespace lbmc
