// Drives the host side of a context (softmold_amd/csrc/sm_capi.cpp) without a GPU: device memory
// is host memory, allocations can be made to fail, and a kernel's stand-in touches the ends of
// the buffers that it would use, so that the address sanitizer reports one that is gone or
// short.  Usage: context_harness SCENARIO; exit code 0 if it held.
#include "sm_internal.hpp"

#include "../../include/softmold_hip.h"

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <utility>
#include <vector>

namespace {

int g_bad_malloc = -1;      // the device allocation that fails, counted down
bool g_failed = false;      // one did
hipError_t g_last = hipSuccess;
size_t g_bytes = 0;         // device memory allocated so far
int g_clears = 0;           // and clears
size_t g_cells = 0;         // cells of the table that the replicas were given
// The keys that the last key kernel left for a build, as far as a build must agree with it.
struct Keys {
    bool there;
    const void *counts, *desc;
    unsigned cells;
    const void *moved;
    size_t table;
};
Keys g_keys{};
bool g_crowded = false;              // counting builds fall back
int g_builds = 0, g_sorts = 0;       // counting builds, radix sorts

#define EXPECT(cond)                                                       \
    do {                                                                   \
        if (!(cond)) {                                                     \
            std::fprintf(stderr, "line %d: %s\n", __LINE__, #cond);        \
            std::exit(1);                                                  \
        }                                                                  \
    } while (0)

template <class T>
void touch(const T *p, size_t count)
{
    if (count == 0) return;
    const volatile char *c = reinterpret_cast<const volatile char *>(p);
    (void)c[0];
    (void)c[sizeof(T) * count - 1];
}

}  // namespace

extern "C" {
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return std::exchange(g_last, hipSuccess); }
const char *hipGetErrorName(hipError_t e) { return e == hipErrorOutOfMemory ? "hipErrorOutOfMemory" : "hipError"; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = nullptr; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = nullptr; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1.f; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { *g = reinterpret_cast<hipGraph_t>(1); return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) { *e = reinterpret_cast<hipGraphExec_t>(1); return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t *st) { *st = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { *p = std::malloc(bytes); return hipSuccess; }
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipMalloc(void **p, size_t bytes)
{
    if (g_bad_malloc >= 0 && g_bad_malloc-- == 0) {
        g_failed = true;
        return g_last = hipErrorOutOfMemory;
    }
    *p = std::calloc(1, bytes);
    g_bytes += bytes;
    return hipSuccess;
}
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { std::memset(d, v, n); g_clears++; return hipSuccess; }
}

namespace smdev {
int sort_passes(int bits) { return std::min(4, (bits + 7) / 8); }
int move_tiles(int n) { return n / 1024 + 1; }
int move_blocks(int n) { return (n + 255) / 256; }
size_t sort_hist_words() { return 16 * 1024; }
size_t sort_scratch_words(int n, int passes) { return sort_hist_words() + 4 + (size_t)passes * (n / 512 + 2) * 256; }
int build_tiles(int n) { return (n + 511) / 512; }
bool sortw_fits(int n) { return n >= 1 && n <= 524288; }
size_t sortw_words(int n, bool counting) { return kWinKeyWords + (counting ? (size_t)3 * build_tiles(n) * 256 : 0); }
uint32_t *win_scratch(uint32_t *s, int n) { return s + sort_scratch_words(n, 4); }
size_t count_limit(int n)
{
    const long long want = std::min<long long>(std::max<long long>(2ll * n, 1 << 14), kWinCells);
    return (size_t)((want + kCoarseCells - 1) / kCoarseCells * kCoarseCells);
}
WinBook win_book(uint32_t *s, int n, const uint32_t *desc, uint32_t *counts, uint32_t *bucket, uint32_t cells, uint32_t limit)
{
    uint32_t *ws = win_scratch(s, n), *bbox = ws + (size_t)kCoarseCopies * kCoarse;
    return WinBook{desc, ws, bbox, bbox + 16 * 8, counts, bucket, cells, limit};
}
hipError_t noalloc_scratch_init(int) { return hipSuccess; }

static void made_keys(const WinBook &wb, const MoveBook &mb) { g_keys = Keys{true, wb.counts, wb.desc, wb.cells, mb.cnt_b, g_cells}; }
static void take_keys(const WinBook &wb, bool moved)
{
    EXPECT(g_keys.there && g_keys.counts == wb.counts && g_keys.desc == wb.desc && g_keys.cells == wb.cells);
    EXPECT((g_keys.moved != nullptr) == moved && g_keys.table == g_cells);
    g_keys.there = false;
}
static void touch_book(const WinBook &wb)
{
    if (!wb.desc && wb.cells == 0) return;   // no counting build
    EXPECT(wb.counts && wb.bucket && wb.limit > 0 && wb.cells <= wb.limit);
    touch(wb.counts, wb.limit);
    touch(wb.bucket, (size_t)wb.limit * kBucket);
    touch(wb.coarse, kWinKeyWords);
    if (wb.desc) touch(wb.desc, 6);
}
void launch_fill_u32(hipStream_t, uint32_t *p, size_t count, uint32_t v) { std::fill(p, p + count, v); }
void launch_set_step(hipStream_t, DevGlobal *g, long long step) { g->step = g->base = step; }
void launch_first(hipStream_t, const Params &P, const Bead *beads, Bead *out, float4 *, const float4 *, const DevRep *reps,
                  DevGlobal *, uint32_t *key, uint32_t *idx, int, long long, uint32_t *, int, const MoveBook &mb, const WinBook &wb)
{
    touch(beads, P.n);
    touch(out, P.n);
    touch(key, P.n);
    if (idx) touch(idx, P.n);
    touch_book(wb);
    g_cells = 0;
    for (int r = 0; r < P.nrep; r++) g_cells = std::max(g_cells, (size_t)(reps[r].cellbase + reps[r].capacity));
    for (int r = 0; r < P.nrep; r++)
        EXPECT((long long)reps[r].nc[0] * reps[r].nc[1] * reps[r].nc[2] <= reps[r].capacity);
    made_keys(wb, mb);
}
void launch_kick_first(hipStream_t, const Params &P, const Bead *beads, Bead *out, const int2 *, const double4 *, const GenTables &,
                       const float4 *, float4 *, const DevRep *, DevGlobal *, long long, bool, uint32_t *key, uint32_t *,
                       uint32_t *, int, const MoveBook &mb, const WinBook &wb)
{
    touch(beads, P.n);
    touch(out, P.n);
    touch(key, P.n);
    touch_book(wb);
    made_keys(wb, mb);
}
int radix_sort(hipStream_t, SortBuffers &b, int, int)
{
    touch(b.k1, b.n);
    take_keys(WinBook{}, false);
    g_sorts++;
    return 0;
}
void sort_moved(hipStream_t, SortBuffers &, const MoveSort &, int, int) { take_keys(WinBook{}, true); }
void launch_build(hipStream_t, int n, const BuildArgs &a)
{
    touch_book(a.wb);
    take_keys(a.wb, false);
    g_builds++;
    if (g_crowded) ++*a.fallbacks;
    for (const uint32_t *p : {a.k2, a.v0, a.v2, (uint32_t *)a.cells_old, a.cells_now}) touch(p, n);
    touch(a.counts_old, a.wb.limit);
    touch(a.cstart, g_cells);
    touch(a.cend, g_cells);
}
void launch_reorder(hipStream_t, int n, const uint32_t *k, const uint32_t *, const Bead *, Bead *, int *cstart, int *cend, uint32_t *, size_t)
{
    touch(k, n);
    touch(cstart, g_cells);
    touch(cend, g_cells);
}
void launch_pair_force(hipStream_t, const Params &, int, int, const Bead *, const uint32_t *, const uint32_t *, const int *cs,
                       const int *ce, const DevRep *, const float *, float4 *)
{
    touch(cs, g_cells);
    touch(ce, g_cells);
}
void launch_bonded_kick(hipStream_t, const Params &, const Bead *, const int2 *, const double4 *, const GenTables &, const float4 *,
                        float4 *, float4 *, const DevRep *, const DevGlobal *, int, float4 *)
{
}
void launch_pair_gather(hipStream_t, const Params &, int, int, const Bead *, const uint32_t *, const uint32_t *, const int *cs,
                        const int *, const DevRep *, const float *, const double *, double *, int *, int *, unsigned long long *, long long)
{
    touch(cs, g_cells);
}
void launch_sums(hipStream_t, SumKind, const SumArgs &) {}
void launch_pack(hipStream_t, int, int, const PackSrc &, double *, const DevRep *reps, int nrep, const DevGlobal *g, double *head)
{
    std::memcpy(head, (const void *)g, sizeof(long long));
    for (int i = 0; i < 3 * nrep; i++) head[1 + i] = reps[i / 3].L[i % 3];
}
void launch_post(hipStream_t, const double *, size_t, const DevGlobal *g, double *head) { std::memcpy(head, (const void *)g, sizeof(long long)); }
}  // namespace smdev

namespace {

struct System {
    std::vector<double> pos, vel, f, u;
    std::vector<int32_t> type;
    sm_system s{};
    explicit System(int n, double box) : pos(3 * n), vel(3 * n), f{1, 1, 0, 2, 1, 1}, u{1, 1, 1, 2, 1, 1}, type(n, 0)
    {
        for (size_t e = 0; e < pos.size(); e++) pos[e] = box * (double)(e * 7919 % 1000) / 1000;
        s.n_particles = n, s.n_types = 1;
        s.pos = pos.data(), s.vel = vel.data(), s.type = type.data(), s.fconst = f.data(), s.uconst = u.data();
        for (double &l : s.box) l = box;
        s.cutoff = 2, s.dt = 0.02, s.gamma = 1, s.temperature = 3;
    }
};

// A box that needs more cells, uploaded while each of the allocations in turn fails: refused, and
// the context is as it was, or done; either way it goes on with every buffer in place.
int growth_fails()
{
    for (double box : {60.0, 90.0})
        for (int replicas : {1, 2})
            for (int k = 0;; k++) {
                System a(200, 24), b(300, 30);
                const sm_system both[2] = {a.s, b.s};
                sm_ctx *c = nullptr;
                EXPECT(sm_create_batch(both, replicas, &c) == SM_OK);
                EXPECT(sm_run(c, 1, 4) == SM_OK);
                const std::vector<double> L(3 * replicas, box);
                g_bad_malloc = k, g_failed = false;
                const int rc = sm_upload_state(c, nullptr, nullptr, nullptr, L.data());
                g_bad_malloc = -1;
                double e[6], now[6];
                EXPECT(rc == SM_OK || rc == SM_ERR_HIP);
                EXPECT(sm_run(c, 5, 9) == SM_OK && sm_measure(c, e) == SM_OK && sm_init_forces(c) == SM_OK);
                EXPECT(sm_download_state(c, nullptr, nullptr, nullptr, now) == SM_OK);
                EXPECT(now[0] == (rc == SM_OK ? box : 24.0));
                EXPECT(sm_upload_state(c, nullptr, nullptr, nullptr, L.data()) == SM_OK && sm_run(c, 14, 9) == SM_OK);
                EXPECT(sm_destroy(c) == SM_OK);
                if (!g_failed) {
                    EXPECT(k > 1);
                    break;
                }
            }
    return 0;
}

// The launch shapes of a context whose box was uploaded are those of one created with it; a
// chunk that was set stays.
int box_and_shapes()
{
    const auto knob = [](sm_ctx *c, const char *k) {
        int32_t v = -1;
        EXPECT(sm_tune_get(c, k, &v) == SM_OK);
        return v;
    };
    for (const double from : {24.0, 200.0}) {
        const double to = 224.0 - from;
        System a(20000, from), b(20000, to);
        sm_ctx *c = nullptr, *d = nullptr;
        EXPECT(sm_create(&a.s, &c) == SM_OK && sm_create(&b.s, &d) == SM_OK);
        EXPECT(knob(c, "energy_chunk") != knob(d, "energy_chunk"));
        const double L[3] = {to, to, to};
        EXPECT(sm_upload_state(c, nullptr, nullptr, nullptr, L) == SM_OK);
        for (const char *k : {"pair_chunk", "energy_chunk"}) EXPECT(knob(c, k) == knob(d, k));
        EXPECT(sm_tune(c, "pair_chunk", 32) == SM_OK);
        const double back[3] = {from, from, from};
        EXPECT(sm_upload_state(c, nullptr, nullptr, nullptr, back) == SM_OK && knob(c, "pair_chunk") == 32);
        EXPECT(sm_destroy(c) == SM_OK && sm_destroy(d) == SM_OK);
    }
    return 0;
}

// The rest of a step without its first half right before it: another mode, another table or other
// positions in between, or no first half at all.  Every build has the keys that it expects.
int step_phases()
{
    for (const double box : {24.0, 90.0})
        for (int from = 0; from < 3; from++) {
            System a(200, box);
            sm_ctx *c = nullptr;
            EXPECT(sm_create(&a.s, &c) == SM_OK);
            EXPECT(sm_tune(c, "sort_mode", from) == SM_OK && sm_init_forces(c) == SM_OK);
            for (int to = 0; to < 3; to++) {
                EXPECT(sm_step_first(c, 1) == SM_OK && sm_tune(c, "sort_mode", to) == SM_OK);
                EXPECT(sm_step_finish(c, 1, nullptr) == SM_OK);
                EXPECT(sm_step_finish(c, 1, nullptr) == SM_OK);
                EXPECT(sm_step_first(c, 2) == SM_OK && sm_step_first(c, 2) == SM_OK && sm_step_finish(c, 2, nullptr) == SM_OK);
            }
            const double L[3] = {box * 1.5, box * 1.5, box * 1.5};
            EXPECT(sm_tune(c, "sort_mode", from) == SM_OK && sm_step_first(c, 3) == SM_OK);
            EXPECT(sm_upload_state(c, nullptr, nullptr, nullptr, L) == SM_OK && sm_step_finish(c, 3, nullptr) == SM_OK);
            EXPECT(sm_run(c, 4, 9) == SM_OK && sm_step_finish(c, 12, nullptr) == SM_OK);
            EXPECT(sm_destroy(c) == SM_OK);
        }
    return 0;
}

// Builds that keep falling back are left to the sort: in a first long run, and from results; a
// context whose builds count goes on counting, and one that stopped does again when it is told
// to or has another box.
int crowded_cells()
{
    for (const int graph : {0, 1})
        for (const int mode : {0, 2}) {
            System a(200, 24);
            sm_ctx *c = nullptr;
            double e[3];
            const auto runs = [&](int steps, bool counted) {
                g_builds = g_sorts = 0;
                EXPECT(sm_run(c, 1, steps) == SM_OK);
                EXPECT(counted ? g_builds > 0 && g_sorts == 0 : g_builds == 0 && g_sorts > 0);
            };
            g_crowded = false;
            EXPECT(sm_create(&a.s, &c) == SM_OK && sm_tune(c, "sort_mode", mode) == SM_OK);
            EXPECT(sm_init_forces(c) == SM_OK);
            for (int k = 0; k < 3; k++) {
                runs(100, true);
                EXPECT(sm_measure(c, e) == SM_OK);
            }
            // the box gets crowded: seen by the next result
            g_crowded = true;
            runs(100, true);
            EXPECT(sm_sync(c) == SM_OK);
            runs(100, false);
            EXPECT(sm_tune(c, "graph", graph) == SM_OK);
            runs(100, false);
            // told to count again: a first long run finds out after 8 steps
            EXPECT(sm_tune(c, "sort_mode", mode) == SM_OK);
            g_builds = g_sorts = 0;
            EXPECT(sm_run(c, 1, 100) == SM_OK && g_builds == 8 && g_sorts > 0);
            runs(100, false);
            // another box: counted again, and that stays
            const double L[3] = {26, 26, 26};
            g_crowded = false;
            EXPECT(sm_upload_state(c, nullptr, nullptr, nullptr, L) == SM_OK);
            for (int k = 0; k < 3; k++) {
                runs(100, true);
                EXPECT(sm_measure(c, e) == SM_OK);
            }
            EXPECT(sm_destroy(c) == SM_OK);
        }
    return 0;
}

// What making a context takes from the device: the counting builds' buckets follow the cells of
// a small table, and the beads of a small context in a large one; and few clears.
int creation()
{
    struct { int n; double box; size_t mib; } cases[] = {
        {90000, 92, 60},       // 46^3 cells, 107k in the table: 26 MiB of buckets, not 64
        {20000, 200, 36},      // a million cells (8 MiB of table), 40k counted: 10 MiB, not 20
    };
    for (const auto &k : cases) {
        System a(k.n, k.box);
        sm_ctx *c = nullptr;
        g_bytes = 0, g_clears = 0;
        EXPECT(sm_create(&a.s, &c) == SM_OK);
        std::fprintf(stderr, "%d beads: %zu MiB, %d clears\n", k.n, g_bytes >> 20, g_clears);
        EXPECT(g_bytes >> 20 < k.mib && g_clears <= 4);
        EXPECT(sm_destroy(c) == SM_OK);
    }
    return 0;
}

}  // namespace

int main(int argc, char **argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "growth_fails") return growth_fails();
    if (what == "box_and_shapes") return box_and_shapes();
    if (what == "step_phases") return step_phases();
    if (what == "crowded_cells") return crowded_cells();
    if (what == "creation") return creation();
    std::fprintf(stderr, "unknown scenario\n");
    return 2;
}
