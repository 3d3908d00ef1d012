// Batched stepping of several lattices (ensembles of uneven lattices): one
// call for every member is one pass of launches.
//
// The members are ordinary contexts (lbmc_create + lbmc_set_fields + an
// initial condition).  The batch keeps, in device memory, each member's
// kernel arguments (its buffers, its collision variant, the slot offsets of
// the current call t and its closure schedule) and lists of chunks (runs of
// 256-node tiles of one member) over all members and over the closure
// members.  A call is
//   batch_step_kernel     blocks take chunks (striding over the list when
//                         the grid is smaller); a chunk belongs to one
//                         member, so its arguments and collision variant
//                         are uniform over the block; chunks of closure
//                         members that evaluate the network are skipped;
//   batch_eval_kernel     (closure members only) those chunks, with the
//                         network; returns at once when no member evaluates;
// The kernels of call t + j read the members' arguments of that call from
// entry j of a window of kBatchWindow calls in device memory (and the
// evaluation kernel its flag any_eval[j]).  At the end of a window of calls
//   batch_advance_kernel  one block moves every member's state from call t
//                         to t + calls (shift counters, slot offsets, the
//                         macro-store flag, the closure phase), and
//   batch_window_kernel   one block per entry lays out the next window and
//                         its evaluation flags,
// so no kernel takes t as an argument and the state moves on once per
// window.  Because nothing in the launches depends on t, a window of calls
// is captured once into a HIP graph and replayed for any t.  The launch
// shape of the step kernel is chosen by lbmc_batch_autotune (timed
// candidates).
//
// D2Q9 members in 32 and 64 bits that all hold a second population buffer go
// in passes of several calls instead (batch_tile_kernel.hpp, pass_steps).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <mutex>
#include <string>
#include <vector>

#include "batch_kernel.hpp"
#include "batch_tile_kernel.hpp"
#include "ctx.hpp"
#include "dispatch.hpp"
#include "node_index.hpp"


using namespace lbmc;

struct lbmc_batch {
    int count = 0;
    int lattice = 0, storage = 0, device = 0;
    bool cdouble = false;
    std::vector<lbmc_ctx *> members;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    void *dmembers = nullptr;  // BatchMember<C>[count]: the state of call t_next
    void *dwindow = nullptr;   // BatchMember<C>[kBatchWindow][count]: calls t_next + j
    int2 *chunks = nullptr;
    int nchunks = 0;
    int2 *cchunks = nullptr;  // the closure members' chunks
    int ncchunks = 0;
    std::vector<char> chunk_closure;  // which members cchunks holds
    int eval_grid = 0;        // blocks of the evaluation kernel
    int *any_eval = nullptr;  // device flags [kBatchWindow]: some closure member evaluates call t_next + j
    const void *mlp = nullptr;  // closure weights shared by the closure members (a member's image)
    long long nodes = 0;
    int grid = 1;
    int sub = 1;            // 256-node tiles per chunk
    int csub = 1;           //   and per chunk of the closure members' list
    int blocks_per_cu = 0;  // residency cap of the step kernel (0: none)
    int lds = 0;            //   as dynamic LDS bytes per block
    int lds_cu = 0;         // LDS bytes per CU
    int ncu = 256;          // compute units of the device
    long long t_next = -1;  // the call the device arguments describe
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
    int graph_steps = 0;
    // passes of several calls (batch_tile_kernel.hpp): the members' tiles, plain
    // members' first (members of one collision variant together, which share
    // the instruction cache), and the calls of a pass
    std::vector<TilePlan> plans;
    std::vector<char> tile_closure;  // which members the lists below hold as closure members
    int2 *tiles = nullptr;
    int ntiles_plain = 0, ntiles_closure = 0, pass_calls = 0;
    void *dpass = nullptr;  // BatchTileMember<C>[count]: call t0 of the run
    const lbmc_mlp *closure_model = nullptr;
    double closure_lo = 0, closure_hi = 0;
    int closure_fp16 = 0;  // the closure members' network with fp16 operands
    std::string err;
};

namespace {

std::string g_batch_error;

lbmc_status bfail(lbmc_batch *b, lbmc_status st, const char *fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    if (b) b->err = buf;
    else g_batch_error = buf;
    return st;
}

#define B_HIP(b, call)                                                                              \
    do {                                                                                            \
        hipError_t e_ = (call);                                                                     \
        if (e_ != hipSuccess) return bfail((b), LBMC_ERR_DEVICE, "%s: %s", #call, hipGetErrorString(e_)); \
    } while (0)

int member_variant(const lbmc_ctx *c)
{
    const KernelKey &k = c->key;
    if (k.closure) return 8 + (k.guo ? 1 : 0);
    const int bit0 = k.family == 0 ? (k.smag ? 1 : 0) : (k.mfix ? 1 : 0);
    return (k.family << 2) | ((k.guo ? 1 : 0) << 1) | bit0;
}

// Member arguments for call t0, read from the members' current state (so
// that set_fields / set_f on a member between runs is seen).
template <class C>
lbmc_status upload_members(lbmc_batch *b, long long t0, int store_every)
{
    std::vector<BatchMember<C>> hm((size_t)b->count);
    for (int k = 0; k < b->count; k++) {
        const lbmc_ctx *c = b->members[(size_t)k];
        if (c->nsf || c->offsets64 || !c->fields_set)
            return bfail(b, LBMC_ERR_UNSUPPORTED, "batch member %d: sf nodes or state not supported", k);
        if (c->key.closure && (c->closure_model != b->closure_model || c->closure_lo != b->closure_lo ||
                               c->closure_hi != b->closure_hi || c->key.closure_fp16 != b->closure_fp16))
            return bfail(b, LBMC_ERR_UNSUPPORTED, "batch member %d: closure members must share one model, band and operand precision", k);
        BatchMember<C> &m = hm[(size_t)k];
        memset(&m, 0, sizeof(m));
        const int se = store_every > 0 ? store_every : 0;
        fill_args(b->members[(size_t)k], m.a, t0, se > 0 && ((t0 + 1) % se) == 0);
        m.variant = member_variant(b->members[(size_t)k]);
        m.store_every = se;
        m.store_count = se > 0 ? (int)((t0 + 1) % se) : 0;
        // closure interval: the schedule of a single lattice (lbmc_run): the
        // network runs on calls t % K == 0 and on the first call whose
        // state has no valid record
        m.closure_every = c->key.closure ? c->closure_every : 1;
        m.closure_phase = (int)(t0 % m.closure_every);
        if (m.closure_every > 1) m.a.tmode = (!c->tcache_valid || m.closure_phase == 0) ? 1 : 2;
    }
    B_HIP(b, hipMemcpyAsync(b->dmembers, hm.data(), sizeof(BatchMember<C>) * hm.size(), hipMemcpyHostToDevice,
                            b->stream));
    hipLaunchKernelGGL(batch_window_kernel<C>, dim3(kBatchWindow), dim3(256), 0, b->stream,
                       (const BatchMember<C> *)b->dmembers, b->count, (BatchMember<C> *)b->dwindow, b->any_eval);
    B_HIP(b, hipGetLastError());
    B_HIP(b, hipStreamSynchronize(b->stream));
    b->t_next = t0;
    return LBMC_OK;
}

// call t_next + j (j < kBatchWindow) from window entry j
lbmc_status launch_one_step(lbmc_batch *b, int j)
{
    hipError_t e;
    const size_t msz = b->cdouble ? sizeof(BatchMember<double>) : sizeof(BatchMember<float>);
    const void *members = (const char *)b->dwindow + (size_t)j * (size_t)b->count * msz;
    const BatchShape sh{b->grid, b->sub, b->lds};
    const BatchEval ev{b->cchunks, b->mlp ? b->ncchunks : 0, b->eval_grid, b->csub, b->mlp, b->any_eval + j,
                       b->closure_fp16 != 0};
    switch (b->storage) {
    case LBMC_FP64: e = launch_batch_fp64(b->lattice, members, b->chunks, b->nchunks, b->grid, b->sub, b->lds, b->stream); break;
    case LBMC_FP32: e = launch_batch_st<StFP32>(b->lattice, members, b->chunks, b->nchunks, sh, ev, b->stream); break;
    case LBMC_FP16S: e = launch_batch_st<StFP16S>(b->lattice, members, b->chunks, b->nchunks, sh, ev, b->stream); break;
    default: e = launch_batch_st<StBF16S>(b->lattice, members, b->chunks, b->nchunks, sh, ev, b->stream); break;
    }
    if (e != hipSuccess) return bfail(b, LBMC_ERR_DEVICE, "batch step launch: %s", hipGetErrorString(e));
    return LBMC_OK;
}

// the state and the window move on by `calls` (<= kBatchWindow) calls
template <class C>
void launch_advance(lbmc_batch *b, int calls)
{
    hipLaunchKernelGGL(batch_advance_kernel<C>, dim3(1), dim3(256), 0, b->stream, (BatchMember<C> *)b->dmembers,
                       b->count, calls);
    hipLaunchKernelGGL(batch_window_kernel<C>, dim3(kBatchWindow), dim3(256), 0, b->stream,
                       (const BatchMember<C> *)b->dmembers, b->count, (BatchMember<C> *)b->dwindow, b->any_eval);
}

lbmc_status advance(lbmc_batch *b, int calls)
{
    if (b->cdouble) launch_advance<double>(b, calls);
    else launch_advance<float>(b, calls);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return bfail(b, LBMC_ERR_DEVICE, "batch advance launch: %s", hipGetErrorString(e));
    return LBMC_OK;
}

void drop_batch_graph(lbmc_batch *b)
{
    if (b->graph_exec) (void)hipGraphExecDestroy(b->graph_exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    b->graph_exec = nullptr;
    b->graph = nullptr;
    b->graph_steps = 0;
}

constexpr int kBatchGraphSteps = kBatchWindow;

lbmc_status upload(lbmc_batch *b, long long t0, int store_every)
{
    return b->cdouble ? upload_members<double>(b, t0, store_every) : upload_members<float>(b, t0, store_every);
}

// nsteps calls from t0; the device arguments must describe call t0
lbmc_status batch_steps(lbmc_batch *b, long long t0, int nsteps)
{
    int left = nsteps;
    if (left >= kBatchGraphSteps) {
        if (!b->graph_exec) {
            B_HIP(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
            lbmc_status st = LBMC_OK;
            for (int k = 0; k < kBatchGraphSteps && st == LBMC_OK; k++) st = launch_one_step(b, k);
            if (st == LBMC_OK) st = advance(b, kBatchGraphSteps);
            hipGraph_t g = nullptr;
            const hipError_t e = hipStreamEndCapture(b->stream, &g);
            if (st != LBMC_OK) {
                if (g) (void)hipGraphDestroy(g);
                return st;
            }
            if (e != hipSuccess) return bfail(b, LBMC_ERR_DEVICE, "batch graph capture: %s", hipGetErrorString(e));
            b->graph = g;
            B_HIP(b, hipGraphInstantiate(&b->graph_exec, g, nullptr, nullptr, 0));
            b->graph_steps = kBatchGraphSteps;
        }
        while (left >= b->graph_steps) {
            B_HIP(b, hipGraphLaunch(b->graph_exec, b->stream));
            left -= b->graph_steps;
        }
    }
    // the rest of the run: calls of the current window, then one advance
    for (int j = 0; j < left; j++) {
        lbmc_status st = launch_one_step(b, j);
        if (st != LBMC_OK) return st;
    }
    if (left > 0)
        if (lbmc_status st = advance(b, left)) return st;
    b->t_next = t0 + nsteps;
    return LBMC_OK;
}

// List position p of a chunk list runs on XCD p mod 8 (blocks are dealt to
// the XCDs round robin, and the grid is either one block per position or a
// multiple of 8 that strides over the list).  Runs of G = 2^glog consecutive
// chunks (member-major order) go to positions p, p + 8, ..., one XCD: a
// cache line that two neighbouring chunks of a member share -- a chunk
// boundary is rarely line-aligned in the rotated rows of the index shift --
// is then fetched and written back by one L2 instead of two (row_chunk,
// node_index.hpp).  The list is padded to whole groups of 8 runs with
// entries of member -1, which the kernels skip.
static void xcd_order(std::vector<int2> &v, unsigned glog)
{
    if (glog == 0 || v.empty()) return;
    const unsigned n = (unsigned)v.size();
    const unsigned runs = (n + (1u << glog) - 1u) >> glog;
    const unsigned total = ((runs + 7u) / 8u * 8u) << glog;
    std::vector<int2> out(total, make_int2(-1, 0));
    for (unsigned p = 0; p < total; p++) {
        const unsigned c = row_chunk(p, glog);
        if (c < n) out[p] = v[c];
    }
    v.swap(out);
}

// Chunk list for `sub` tiles per chunk: (member, first node) of every chunk,
// member by member (the closure members alone: closure), in XCD order with
// runs of ~1024 nodes (measured best for single D2Q9 lattices: 4 chunks of
// 256 nodes per XCD).  Null without chunks.
lbmc_status upload_chunks(lbmc_batch *b, int sub, bool closure, int2 **list, int *count)
{
    const long long cn = (long long)sub * kBlock;
    std::vector<int2> ch;
    for (int k = 0; k < b->count; k++) {
        const lbmc_ctx *c = b->members[(size_t)k];
        if (closure && !c->key.closure) continue;
        for (long long n = 0; n < c->N; n += cn) ch.push_back(make_int2(k, (int)n));
    }
    xcd_order(ch, sub == 1 ? 2u : sub == 2 ? 1u : 0u);
    *list = nullptr;
    *count = (int)ch.size();
    if (ch.empty()) return LBMC_OK;
    B_HIP(b, dev_malloc((void **)list, sizeof(int2) * ch.size()));
    const hipError_t e = hipMemcpy(*list, ch.data(), sizeof(int2) * ch.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) return LBMC_OK;
    (void)hipFree(*list);
    return bfail(b, LBMC_ERR_DEVICE, "chunk list: %s", hipGetErrorString(e));
}

// the closure members' chunks; the old list stays when there is no memory
lbmc_status build_closure_chunks(lbmc_batch *b, int sub)
{
    int2 *list;
    int count;
    if (lbmc_status st = upload_chunks(b, sub, true, &list, &count)) return st;
    drop_batch_graph(b);  // captured with the old list
    if (b->cchunks) (void)hipFree(b->cchunks);
    b->cchunks = list;
    b->ncchunks = count;
    b->csub = sub;
    b->chunk_closure.clear();
    for (const lbmc_ctx *c : b->members) b->chunk_closure.push_back(c->key.closure ? 1 : 0);
    // evaluation kernel: persistent, 4 blocks per CU (its residency)
    b->eval_grid = std::max(1, std::min(count, 4 * b->ncu));
    return LBMC_OK;
}

lbmc_status build_chunks(lbmc_batch *b, int sub)
{
    int2 *list;
    int count;
    if (lbmc_status st = upload_chunks(b, sub, false, &list, &count)) return st;
    if (lbmc_status st = build_closure_chunks(b, sub)) {
        (void)hipFree(list);
        return st;
    }
    if (b->chunks) (void)hipFree(b->chunks);
    b->chunks = list;
    b->nchunks = count;
    b->sub = sub;
    b->grid = std::min(b->grid, b->nchunks);
    return LBMC_OK;
}

// The closure members as they are now: a member's closure may be switched
// between runs.  Their chunks, and the weights of one of them; the captured
// graph holds both.
lbmc_status follow_closures(lbmc_batch *b)
{
    std::vector<char> closure;
    const void *mlp = b->mlp;
    for (const lbmc_ctx *c : b->members) {
        closure.push_back(c->key.closure ? 1 : 0);
        if (c->key.closure && c->closure_model == b->closure_model) mlp = c->mlp_img;
    }
    if (mlp != b->mlp) drop_batch_graph(b);
    b->mlp = mlp;
    return closure == b->chunk_closure ? LBMC_OK : build_closure_chunks(b, b->csub);
}

// ---- passes of several calls (D2Q9 members in 32 or 64 bits that all hold a
// second population buffer)

bool has_tiles(const lbmc_batch *b)
{
    return b->lattice == LBMC_D2Q9 && (b->storage == LBMC_FP64 || b->storage == LBMC_FP32);
}

// tiles of every member, all of them with the margin of one pass length.
// Allocates, so no member's pass_mu is held (dev_malloc).
lbmc_status build_tiles(lbmc_batch *b)
{
    std::vector<char> closure;
    for (const lbmc_ctx *c : b->members) closure.push_back(c->key.closure ? 1 : 0);
    if (b->tiles && b->dpass && closure == b->tile_closure) return LBMC_OK;
    const int slot = (int)b->members[0]->sbytes;
    const TileCapacity cap = tile_capacity(2, slot);
    const int P = cap.threads * cap.per_thread;
    double best = -1;
    for (int M = 1; M <= 6; M++) {
        std::vector<TilePlan> plans;
        double work = 0;
        for (const lbmc_ctx *c : b->members) {
            TilePlan q;
            double w = -1;
            for (int W = 16; W <= 128; W *= 2) {
                TilePlan t;
                if (!tile_shape(c->L[0], c->L[1], 2, W, P / W, M, t)) continue;
                const double tw = tile_work(t, slot);
                if (w < 0 || tw < w) {
                    w = tw;
                    q = t;
                }
            }
            work += w;
            plans.push_back(q);
        }
        if (best < 0 || work < best) {
            best = work;
            b->plans.swap(plans);
            b->pass_calls = M + 1;
        }
    }
    std::vector<int2> tiles;
    for (int cl = 0; cl < 2; cl++) {
        for (int v = 0; v < 10; v++)
            for (int k = 0; k < b->count; k++)
                if (closure[(size_t)k] == cl && member_variant(b->members[(size_t)k]) == v)
                    for (int t = 0; t < b->plans[(size_t)k].ntx * b->plans[(size_t)k].nty; t++)
                        tiles.push_back(make_int2(k, t));
        (cl ? b->ntiles_closure : b->ntiles_plain) = (int)tiles.size() - (cl ? b->ntiles_plain : 0);
    }
    if (b->tiles) B_HIP(b, hipFree(b->tiles));
    b->tiles = nullptr;
    B_HIP(b, dev_malloc((void **)&b->tiles, sizeof(int2) * tiles.size()));
    B_HIP(b, hipMemcpy(b->tiles, tiles.data(), sizeof(int2) * tiles.size(), hipMemcpyHostToDevice));
    const size_t msz = b->cdouble ? sizeof(BatchTileMember<double>) : sizeof(BatchTileMember<float>);
    if (!b->dpass) B_HIP(b, dev_malloc(&b->dpass, msz * (size_t)b->count));
    b->tile_closure = closure;
    return LBMC_OK;
}

// Whether a run from call t0 goes in passes: it pays, every member with a second
// buffer (their pass_mu held), and closure members on one schedule.  *eval0:
// the closure members evaluate on the first call.
bool can_pass(const lbmc_batch *b, long long t0, int nsteps, int store_every, int *every, bool *eval0)
{
    *every = 0;
    *eval0 = false;
    int seen = 0, ev = 0;
    bool macro = false;
    for (const lbmc_ctx *c : b->members) {
        if (!c->f2 || !c->tile.on || c->nsf || !c->fields_set || c->L[0] >= (1 << 30) || c->L[1] >= (1 << 30)) return false;
        macro = macro || c->has_macro;
        if (!c->key.closure) continue;
        if (*every && c->closure_every != *every) return false;
        *every = c->closure_every;
        seen++;
        ev += (c->closure_every == 1 || !c->tcache_valid || t0 % c->closure_every == 0) ? 1 : 0;
    }
    if (ev != 0 && ev != seen) return false;
    *eval0 = ev != 0;
    return batch_passes(BatchRun{b->nodes, (int)b->members[0]->sbytes, nsteps, store_every, macro, *every,
                                 seen > 0 && seen < b->count});
}

template <class C>
lbmc_status upload_pass_members(lbmc_batch *b, long long t0)
{
    std::vector<BatchTileMember<C>> hm((size_t)b->count);
    for (int k = 0; k < b->count; k++) {
        const lbmc_ctx *c = b->members[(size_t)k];
        if (c->key.closure && (c->closure_model != b->closure_model || c->closure_lo != b->closure_lo ||
                               c->closure_hi != b->closure_hi || c->key.closure_fp16 != b->closure_fp16))
            return bfail(b, LBMC_ERR_UNSUPPORTED, "batch member %d: closure members must share one model, band and operand precision", k);
        BatchTileMember<C> &m = hm[(size_t)k];
        memset(&m, 0, sizeof(m));
        fill_args(c, m.a, t0, 0);
        tile_geometry(b->plans[(size_t)k], c->L, m.p);
        m.p.src = c->f;
        m.p.dst = c->f2;
        m.variant = member_variant(c);
    }
    B_HIP(b, hipMemcpyAsync(b->dpass, hm.data(), sizeof(BatchTileMember<C>) * hm.size(), hipMemcpyHostToDevice,
                            b->stream));
    B_HIP(b, hipStreamSynchronize(b->stream));
    return LBMC_OK;
}

// The run's calls in passes; the device members describe call t0.  Returns
// through *odd_* which buffer the members' states are in.
lbmc_status pass_steps(lbmc_batch *b, long long t0, int nsteps, int store_every, int every, bool eval0, int *odd_plain,
                       int *odd_closure)
{
    auto stores = [&](int k) { return store_every > 0 && (t0 + k + 1) % store_every == 0; };
    bool macro[2] = {false, false};
    for (const lbmc_ctx *c : b->members) macro[c->key.closure ? 1 : 0] |= c->has_macro;
    // calls k .. end - 1 of one kind of members; calls that store the macros
    // of members with prescribed values run alone (lbmc_run)
    auto passes = [&](bool closure, int k, int end, int *odd) -> lbmc_status {
        const int2 *tiles = b->tiles + (closure ? b->ntiles_plain : 0);
        const int ntiles = closure ? b->ntiles_closure : b->ntiles_plain;
        const int begin = k;
        while (k < end) {
            int e = end;
            if (macro[closure ? 1 : 0] && store_every > 0) {
                e = k;
                while (e < end && !stores(e)) e++;
                if (e == k) e = k + 1;
            }
            const int np = (e - k + b->pass_calls - 1) / b->pass_calls, k0 = k;
            for (int q = 0; q < np; q++) {
                BatchPass bp{};
                bp.offset = k0 + (int)((long long)(e - k0) * q / np);
                bp.calls = k0 + (int)((long long)(e - k0) * (q + 1) / np) - bp.offset;
                for (int j = 0; j < bp.calls; j++)
                    if (stores(bp.offset + j)) bp.store |= 1u << j;
                bp.first = bp.offset == begin;
                bp.last = bp.offset + bp.calls == end;
                bp.odd = *odd;
                const hipError_t err = b->cdouble ? launch_batch_tiles_fp64(b->dpass, tiles, ntiles, bp, b->stream)
                                                  : launch_batch_tiles_fp32(b->dpass, tiles, ntiles, bp, b->stream);
                if (err != hipSuccess)
                    return bfail(b, LBMC_ERR_DEVICE, "batch pass launch: %s", hipGetErrorString(err));
                *odd ^= 1;
            }
            k = e;
        }
        return LBMC_OK;
    };
    if (b->ntiles_plain)
        if (lbmc_status st = passes(false, 0, nsteps, odd_plain)) return st;
    if (b->ntiles_closure)
        for (int k = 0; k < nsteps;) {
            if (k == 0 ? eval0 : true) {
                BatchPass bp{};
                bp.offset = k;
                bp.store = stores(k) ? 1u : 0u;
                bp.odd = *odd_closure;
                const hipError_t err = launch_batch_call_fp32(b->dpass, b->cchunks, b->ncchunks, b->eval_grid, b->csub,
                                                              b->mlp, every > 1, b->closure_fp16 != 0, bp, b->stream);
                if (err != hipSuccess)
                    return bfail(b, LBMC_ERR_DEVICE, "batch call launch: %s", hipGetErrorString(err));
                k++;
            }
            // recorded tau up to the next call with t % every == 0
            const int end = (int)std::min<long long>(nsteps, (t0 + k + every - 1) / every * every - t0);
            if (end > k)
                if (lbmc_status st = passes(true, k, end, odd_closure)) return st;
            k = std::max(k, end);
        }
    return LBMC_OK;
}

// Runs (timed: between the batch's events) in passes; *done false: not
// possible, nothing was run
lbmc_status run_in_passes(lbmc_batch *b, long long t0, int nsteps, int store_every, bool timed, bool *done)
{
    *done = false;
    // no memory for the lists: one call per launch needs none
    if (nsteps <= 0 || !has_tiles(b) || build_tiles(b) != LBMC_OK) return LBMC_OK;
    std::vector<std::unique_lock<std::mutex>> locks;
    for (lbmc_ctx *c : b->members) locks.emplace_back(c->pass_mu);
    int every = 0;
    bool eval0 = false;
    if (!can_pass(b, t0, nsteps, store_every, &every, &eval0)) return LBMC_OK;
    if (b->ntiles_closure && (!b->mlp || !b->cchunks)) return LBMC_OK;
    *done = true;
    if (lbmc_status st = b->cdouble ? upload_pass_members<double>(b, t0) : upload_pass_members<float>(b, t0)) return st;
    if (timed) B_HIP(b, hipEventRecord(b->ev0, b->stream));
    int odd[2] = {0, 0};
    const lbmc_status st = pass_steps(b, t0, nsteps, store_every, every, eval0, &odd[0], &odd[1]);
    if (timed && st == LBMC_OK) B_HIP(b, hipEventRecord(b->ev1, b->stream));
    B_HIP(b, hipStreamSynchronize(b->stream));
    for (lbmc_ctx *c : b->members)
        if (odd[c->key.closure ? 1 : 0]) swap_populations(c);
    return st;
}

// after calls were run: every closure member with an interval now holds the
// record of its last evaluation
void mark_records(lbmc_batch *b)
{
    for (lbmc_ctx *c : b->members)
        if (c->key.closure && c->closure_every > 1) c->tcache_valid = true;
}

lbmc_status sync_members(lbmc_batch *b)
{
    for (lbmc_ctx *c : b->members) B_HIP(b, hipStreamSynchronize(c->stream));
    return LBMC_OK;
}

// lbmc_batch_time_steps; passes false: one call per launch
lbmc_status time_calls(lbmc_batch *b, long long t0, int nsteps, int store_every, bool passes, float *ms)
{
    lbmc_status st = sync_members(b);
    if (st == LBMC_OK) st = follow_closures(b);
    bool done = false;
    if (st == LBMC_OK && passes) st = run_in_passes(b, t0, nsteps, store_every, true, &done);
    if (st == LBMC_OK && !done) st = upload(b, t0, store_every);  // outside the timed region
    if (st != LBMC_OK) return st;
    if (!done) {
        B_HIP(b, hipEventRecord(b->ev0, b->stream));
        st = batch_steps(b, t0, nsteps);
        if (st != LBMC_OK) return st;
        B_HIP(b, hipEventRecord(b->ev1, b->stream));
    }
    mark_records(b);
    B_HIP(b, hipEventSynchronize(b->ev1));
    B_HIP(b, hipEventElapsedTime(ms, b->ev0, b->ev1));
    return LBMC_OK;
}

}  // namespace

extern "C" {

const char *lbmc_batch_last_error(const lbmc_batch *b) { return b ? b->err.c_str() : g_batch_error.c_str(); }

lbmc_status lbmc_batch_create(lbmc_ctx *const *members, int count, lbmc_batch **out)
{
    if (!out || !members || count <= 0) return bfail(nullptr, LBMC_ERR_INVALID, "lbmc_batch_create: bad argument");
    *out = nullptr;
    const lbmc_ctx *c0 = members[0];
    if (!c0) return bfail(nullptr, LBMC_ERR_INVALID, "lbmc_batch_create: member 0 is null");
    long long nchunks = 0, nodes = 0;
    const lbmc_mlp *closure_model = nullptr;
    double closure_lo = 0, closure_hi = 0;
    int closure_fp16 = 0;
    const void *closure_img = nullptr;
    for (int k = 0; k < count; k++) {
        const lbmc_ctx *c = members[k];
        if (!c) return bfail(nullptr, LBMC_ERR_INVALID, "lbmc_batch_create: member %d is null", k);
        if (!c->fields_set) return bfail(nullptr, LBMC_ERR_STATE, "lbmc_batch_create: member %d has no fields", k);
        if (c->desc.lattice != c0->desc.lattice || c->storage != c0->storage || c->desc.device != c0->desc.device)
            return bfail(nullptr, LBMC_ERR_INVALID,
                         "lbmc_batch_create: member %d differs in lattice, storage or device from member 0", k);
        if (c->nsf) return bfail(nullptr, LBMC_ERR_UNSUPPORTED, "lbmc_batch_create: member %d has sf boundary nodes", k);
        if (c->key.closure) {
            if (closure_model && (c->closure_model != closure_model || c->closure_lo != closure_lo ||
                                  c->closure_hi != closure_hi || c->key.closure_fp16 != closure_fp16))
                return bfail(nullptr, LBMC_ERR_UNSUPPORTED,
                             "lbmc_batch_create: closure members must share one model, band and operand precision "
                             "(member %d)", k);
            closure_model = c->closure_model;
            closure_fp16 = c->key.closure_fp16;
            closure_lo = c->closure_lo;
            closure_hi = c->closure_hi;
            closure_img = c->mlp_img;
        }
        if (c->offsets64) return bfail(nullptr, LBMC_ERR_UNSUPPORTED, "lbmc_batch_create: member %d is too large", k);
        for (int j = 0; j < k; j++)
            if (members[j] == c) return bfail(nullptr, LBMC_ERR_INVALID, "lbmc_batch_create: member %d repeats %d", k, j);
        nchunks += (c->N + kBlock - 1) / kBlock;
        nodes += c->N;
    }
    if (nchunks >= (1LL << 31)) return bfail(nullptr, LBMC_ERR_UNSUPPORTED, "lbmc_batch_create: too many nodes");
    lbmc_batch *b = new lbmc_batch();
    b->count = count;
    b->lattice = c0->desc.lattice;
    b->storage = c0->storage;
    b->device = c0->desc.device;
    b->cdouble = c0->cbytes == 8;
    b->members.assign(members, members + count);
    b->nchunks = (int)nchunks;
    b->nodes = nodes;
    b->closure_model = closure_model;
    b->closure_fp16 = closure_fp16;
    b->closure_lo = closure_lo;
    b->closure_hi = closure_hi;
    b->mlp = closure_img;
    auto bail = [&](lbmc_status st) {
        g_batch_error = b->err;
        lbmc_batch_destroy(b);
        return st;
    };
    hipError_t e = hipSetDevice(b->device);
    if (e == hipSuccess) e = hipStreamCreate(&b->stream);
    if (e == hipSuccess) e = hipEventCreate(&b->ev0);
    if (e == hipSuccess) e = hipEventCreate(&b->ev1);
    const size_t msz = b->cdouble ? sizeof(BatchMember<double>) : sizeof(BatchMember<float>);
    if (e == hipSuccess) e = dev_malloc(&b->dmembers, msz * (size_t)count);
    if (e == hipSuccess) e = dev_malloc(&b->dwindow, msz * (size_t)count * kBatchWindow);
    if (e == hipSuccess) e = dev_malloc((void **)&b->any_eval, sizeof(int) * kBatchWindow);
    if (e != hipSuccess) return bail(bfail(b, LBMC_ERR_DEVICE, "lbmc_batch_create: %s", hipGetErrorString(e)));
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, b->device) == hipSuccess && prop.multiProcessorCount > 0)
        b->ncu = prop.multiProcessorCount;
    b->grid = b->nchunks;
    if (lbmc_status st = build_chunks(b, 1)) return bail(st);
    // default persistent grid: 8 blocks per CU, at most one block per chunk
    b->grid = (int)std::min<long long>(b->nchunks, 8LL * b->ncu);
    if (hipDeviceGetAttribute(&b->lds_cu, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, b->device) != hipSuccess)
        b->lds_cu = 0;
    if (has_tiles(b)) (void)build_tiles(b);  // tried again by every run
    *out = b;
    return LBMC_OK;
}

lbmc_status lbmc_batch_destroy(lbmc_batch *b)
{
    if (!b) return LBMC_OK;
    (void)hipSetDevice(b->device);
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    drop_batch_graph(b);
    if (b->dmembers) (void)hipFree(b->dmembers);
    if (b->dwindow) (void)hipFree(b->dwindow);
    if (b->chunks) (void)hipFree(b->chunks);
    if (b->cchunks) (void)hipFree(b->cchunks);
    if (b->any_eval) (void)hipFree(b->any_eval);
    if (b->tiles) (void)hipFree(b->tiles);
    if (b->dpass) (void)hipFree(b->dpass);
    if (b->ev0) (void)hipEventDestroy(b->ev0);
    if (b->ev1) (void)hipEventDestroy(b->ev1);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    delete b;
    return LBMC_OK;
}

lbmc_status lbmc_batch_run(lbmc_batch *b, long long t0, int nsteps, int store_every)
{
    if (!b || nsteps < 0 || t0 < 0) return bfail(b, LBMC_ERR_INVALID, "lbmc_batch_run: bad argument");
    B_HIP(b, hipSetDevice(b->device));
    lbmc_status st = sync_members(b);
    if (st == LBMC_OK) st = follow_closures(b);
    bool done = false;
    if (st == LBMC_OK) st = run_in_passes(b, t0, nsteps, store_every, false, &done);
    if (st == LBMC_OK && !done) st = upload(b, t0, store_every);
    if (st == LBMC_OK && !done) st = batch_steps(b, t0, nsteps);
    if (st != LBMC_OK) return st;
    if (nsteps > 0) mark_records(b);
    B_HIP(b, hipStreamSynchronize(b->stream));
    return LBMC_OK;
}

lbmc_status lbmc_batch_time_steps(lbmc_batch *b, long long t0, int nsteps, int store_every, float *ms)
{
    if (!b || nsteps <= 0 || t0 < 0 || !ms) return bfail(b, LBMC_ERR_INVALID, "lbmc_batch_time_steps: bad argument");
    B_HIP(b, hipSetDevice(b->device));
    return time_calls(b, t0, nsteps, store_every, true, ms);
}

// Residency cap of the batch step kernel: at most `per` blocks per CU,
// through dynamic LDS that the kernel does not use (0: no cap).  Not with
// closure members, whose kernel stages the network in static LDS.
void set_blocks_per_cu(lbmc_batch *b, int per)
{
    b->blocks_per_cu = (per >= 3 && per <= 16 && b->lds_cu > 0 && !b->mlp) ? per : 0;
    b->lds = b->blocks_per_cu ? b->lds_cu / b->blocks_per_cu - 1024 : 0;
}

// Times candidate launch shapes over a few steps from the current state and
// keeps the fastest: chunks of 1, 2, 4 or 8 tiles with one block per chunk
// and the resident blocks per CU uncapped or capped at 4 or 6, and
// persistent grids of 2, 4, 8, 16 blocks per CU over one-tile chunks.  These
// are shapes of the one-call launches, so the trials make one call per launch
// also where runs go in passes: the shape then serves the runs that cannot
// (16 members of 64 x 48: 4.6 us per call with 256-node chunks, 12.4 with
// 2048).  Of a pass only the evaluating calls have chunks, the closure members'
// own; they are timed in runs as they go (64 channels, network every call: 245
// us per call with 256-node chunks, 231 with 2048).  The steps advance the
// members' state; callers tune before the timed run.
lbmc_status lbmc_batch_autotune(lbmc_batch *b, long long t0, int steps_per_trial, int *grid, float *ms_per_step)
{
    if (!b || steps_per_trial <= 0 || t0 < 0) return bfail(b, LBMC_ERR_INVALID, "lbmc_batch_autotune: bad argument");
    B_HIP(b, hipSetDevice(b->device));
    const int ncu = b->ncu;
    struct Cand {
        int sub, grid_per_cu, cap;  // grid_per_cu 0: one block per chunk
    };
    std::vector<Cand> cand;
    for (int sub : {1, 2, 4, 8})
        for (int cap : {0, 4, 6}) cand.push_back({sub, 0, cap});
    for (int per : {2, 4, 8, 16}) cand.push_back({1, per, 0});
    float best = -1.f;
    Cand best_c{b->sub, 0, b->blocks_per_cu};
    int best_grid = b->grid;
    long long t = t0;
    // one untimed pass (graph build), then the timed one
    auto trial = [&](bool passes, float *ms) -> lbmc_status {
        for (int k = 0; k < 2; k++, t += steps_per_trial)
            if (lbmc_status st = time_calls(b, t, steps_per_trial, 0, passes, ms)) return st;
        return LBMC_OK;
    };
    for (const Cand &cd : cand) {
        set_blocks_per_cu(b, cd.cap);
        if (cd.cap && !b->blocks_per_cu) continue;  // cap not available
        drop_batch_graph(b);
        if (cd.sub != b->sub || cd.sub != b->csub)
            if (lbmc_status st = build_chunks(b, cd.sub)) return st;
        b->grid = cd.grid_per_cu ? (int)std::min<long long>(b->nchunks, (long long)cd.grid_per_cu * ncu) : b->nchunks;
        float ms = 0.f;
        if (lbmc_status st = trial(false, &ms)) return st;
        if (best < 0.f || ms < best) {
            best = ms;
            best_c = cd;
            best_c.cap = b->blocks_per_cu;
            best_grid = b->grid;
        }
    }
    drop_batch_graph(b);
    if (best_c.sub != b->sub || best_c.sub != b->csub)
        if (lbmc_status st = build_chunks(b, best_c.sub)) return st;
    b->grid = std::min(best_grid, b->nchunks);
    set_blocks_per_cu(b, best_c.cap);
    // runs in passes: their evaluating calls' chunks, and their time per step
    int every = 0;
    bool eval0 = false, passes = has_tiles(b) && b->tiles;
    if (passes) {
        std::vector<std::unique_lock<std::mutex>> locks;
        for (lbmc_ctx *c : b->members) locks.emplace_back(c->pass_mu);
        passes = can_pass(b, t, steps_per_trial, 0, &every, &eval0);
    }
    if (passes) {
        best = -1.f;
        int best_sub = b->csub;
        for (int sub : {1, 2, 4, 8}) {
            if (b->ncchunks && sub != b->csub)
                if (lbmc_status st = build_closure_chunks(b, sub)) return st;
            float ms = 0.f;
            if (lbmc_status st = trial(true, &ms)) return st;
            if (best < 0.f || ms < best) {
                best = ms;
                best_sub = b->csub;
            }
            if (!b->ncchunks) break;  // nothing to choose
        }
        if (best_sub != b->csub)
            if (lbmc_status st = build_closure_chunks(b, best_sub)) return st;
    }
    if (grid) *grid = b->grid;
    if (ms_per_step) *ms_per_step = best / (float)steps_per_trial;
    return LBMC_OK;
}

lbmc_status lbmc_batch_info(const lbmc_batch *b, long long *nodes, int *grid, int *chunks, int *chunk_nodes,
                            int *blocks_per_cu)
{
    if (!b) return LBMC_ERR_INVALID;
    if (nodes) *nodes = b->nodes;
    if (grid) *grid = b->grid;
    if (chunks) *chunks = b->nchunks;
    if (chunk_nodes) *chunk_nodes = b->sub * kBlock;
    if (blocks_per_cu) *blocks_per_cu = b->blocks_per_cu;
    return LBMC_OK;
}

lbmc_status lbmc_batch_set_shape(lbmc_batch *b, int grid, int chunk_nodes, int blocks_per_cu)
{
    if (!b || grid <= 0 || blocks_per_cu < 0 || chunk_nodes < kBlock || chunk_nodes % kBlock ||
        chunk_nodes > 64 * kBlock)
        return bfail(b, LBMC_ERR_INVALID,
                     "lbmc_batch_set_shape: grid > 0, chunk_nodes a multiple of 256 up to 16384, blocks_per_cu >= 0");
    B_HIP(b, hipSetDevice(b->device));
    drop_batch_graph(b);
    if (chunk_nodes / kBlock != b->sub || chunk_nodes / kBlock != b->csub)
        if (lbmc_status st = build_chunks(b, chunk_nodes / kBlock)) return st;
    b->grid = std::min(grid, b->nchunks);
    set_blocks_per_cu(b, blocks_per_cu);
    return LBMC_OK;
}

}  // extern "C"
