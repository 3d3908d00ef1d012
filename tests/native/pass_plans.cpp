// The planner of D2Q9 passes (tile_pass.hpp) on the host: how a run is split,
// and that the tiles of every pass length cover the lattice, have the margin
// of its calls and fit the kernel they are launched with.
#include <cstdio>

#include "../../lbm-c_amd/csrc/tile_pass.hpp"

using namespace lbmc;

namespace {

int failures = 0;

void check(bool ok, const char *what, long long a, long long b, long long c)
{
    if (ok) return;
    std::printf("FAIL %s: %lld %lld %lld\n", what, a, b, c);
    failures++;
}

void splits()
{
    for (int K = 2; K <= kMaxPassCalls; K++)
        for (long long len = 0; len <= 300; len++) {
            const long long np = tile_passes(len, K), in = len < np * K ? len : np * K;
            check(np >= 0 && np % 2 == 0, "even", len, K, np);
            check(len - in < kMinPassRun, "rest", len, K, np);
            check((len >= kMinPassRun) == (np > 0), "shortest", len, K, np);
            for (long long k = 0; k < np; k++) {
                const long long calls = in * (k + 1) / np - in * k / np;
                check(calls >= 2 && calls <= K, "calls of a pass", len, K, calls);
            }
        }
}

void tiles(int Lx, int Ly, int slot, bool plain)
{
    const TilePlan best = plan_tiles(Lx, Ly, slot, 256, plain);
    check(best.on == (slot > 2 || (long long)Lx * Ly <= (1LL << 20)), "planned", Lx, Ly, slot);
    for (int k = 2; best.on && k <= best.M + 1; k++) {
        const TilePlan q = k <= best.M ? plan_short(best, Lx, Ly, slot, 256, plain, k) : best;
        const TileCapacity cap = tile_capacity(q.size, slot);
        check(q.on && q.M + 1 >= k, "margin", Lx, Ly, k);
        check(q.W * q.H <= cap.threads * cap.per_thread, "capacity", Lx, Ly, k);
        check(q.OW == q.W - 2 * q.M && q.OH == q.H - 2 * q.M && q.OW >= 1 && q.OH >= 1, "owned", Lx, Ly, k);
        check((long long)q.OW * q.ntx >= Lx && (long long)q.OH * q.nty >= Ly, "cover", Lx, Ly, k);
        check(tile_estimate(q, slot, 256, k) <= tile_estimate(best, slot, 256, k), "estimate", Lx, Ly, k);
    }
}

// batch_passes at both sides of each of its lines
void batches()
{
    const long long M = 1LL << 20;
    int n = 0;
    auto expect = [&](bool want, const BatchRun &r) { check(batch_passes(r) == want, "batch", n++, r.nodes, r.nsteps); };
    // one call
    expect(true, {2 * M, 4, 1, 0, false, 0, false});
    expect(false, {2 * M + 1, 4, 1, 0, false, 0, false});
    expect(false, {M + 1, 8, 1, 0, false, 0, false});
    expect(true, {1LL << 40, 8, 2, 1, false, 0, false});
    // prescribed values
    for (int nsteps : {2, 100})
        for (int se : {1, 2, 3}) {
            expect(false, {8 * M, 4, nsteps, se, true, 0, false});
            expect(false, {8 * M, 8, nsteps, se, true, 0, false});
        }
    expect(true, {1, 8, 100, 4, true, 0, false});
    expect(true, {1, 4, 8, 0, true, 0, false});
    expect(false, {M / 2 - 1, 4, 9, 0, true, 0, false});
    expect(true, {M / 2, 4, 9, 0, true, 0, false});
    expect(false, {M - 1, 4, 9, 7, true, 0, false});
    expect(true, {M, 4, 9, 7, true, 0, false});
    expect(false, {4 * M - 1, 4, 2, 4, true, 0, false});
    expect(true, {4 * M, 4, 2, 4, true, 0, false});
    expect(true, {1, 4, 100, 1, false, 0, false});
    // closure members
    expect(true, {1, 4, 100, 0, false, 1, true});
    expect(true, {1, 4, 8, 0, false, 2, false});
    expect(false, {8 * M, 4, 9, 0, false, 2, false});
    expect(false, {M - 1, 4, 9, 0, false, 2, true});
    expect(true, {M, 4, 9, 0, false, 2, true});
    expect(true, {1, 4, 9, 0, false, 3, false});
    expect(false, {(5LL << 16) - 1, 4, 9, 0, false, 3, true});
    expect(true, {5LL << 16, 4, 9, 0, false, 3, true});
}

}  // namespace

int main()
{
    splits();
    batches();
    const int L[][2] = {{1, 1},     {3, 5},     {1, 5000},   {64, 48},     {97, 61},     {300, 200},
                        {600, 300}, {900, 500}, {1148, 450}, {1031, 1021}, {2048, 1024}, {3392, 3392}};
    for (const auto &l : L)
        for (int slot : {2, 4, 8})
            for (bool plain : {false, true}) tiles(l[0], l[1], slot, plain);
    if (failures) return 1;
    std::printf("pass plans: ok\n");
    return 0;
}
