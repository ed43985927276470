// Host side of the MI355X MD-step solver: the device context (one or many replica
// systems), step sequencing, hipGraph capture of the step, the launch-shape autotuner,
// and the context part of the C ABI declared in include/softmold_hip.h.
#include "../../include/softmold_hip.h"
#include "sm_adjoint.hpp"
#include "sm_errors.hpp"
#include "sm_internal.hpp"
#include "sm_transfer.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <type_traits>
#include <utility>
#include <vector>

using namespace smdev;
using namespace smapi;

namespace smapi {
thread_local std::string g_err;
}

namespace {

#define HIPCHK(expr)                                                                                   \
    do {                                                                                               \
        hipError_t e_ = (expr);                                                                        \
        if (e_ != hipSuccess)                                                                          \
            throw ApiError(SM_ERR_HIP, std::string(hipGetErrorName(e_)) + " in " #expr " at " __FILE__ \
                                       ":" + std::to_string(__LINE__));                               \
    } while (0)

template <class T>
T *dalloc(size_t count)
{
    void *p = nullptr;
    if (count == 0) count = 1;
    const hipError_t e = hipMalloc(&p, count * sizeof(T));
    if (e != hipSuccess) {
        (void)hipGetLastError();   // reported here, not by the next launch's check
        HIPCHK(e);
    }
    return static_cast<T *>(p);
}

template <class T>
void dfree(T *&p)
{
    if (p) (void)hipFree(p);
    p = nullptr;
}

enum KClass { K_FIRST, K_SORT, K_REORDER, K_PAIR, K_BONDED, K_GATHER, K_SUMS, K_MC, K_KICK_FIRST, K_NCLASS };
const char *kClassName[K_NCLASS] = {"integrate_first+key", "radix_sort", "reorder+cell_table", "pair_force",
                                    "bonded+langevin+kick", "pair_gather_fp64", "energy_sums_fp64",
                                    "mc_move", "bonded+kick+next_first+key"};

// The pair kernels' constant table: each (home type, candidate type) row of the FP32 force
// constants padded to 8 floats {r_m, C1, C2, r_c, C4, C5, 0, 0}, then the culling reach
// r^2 of each candidate type for the force (from those FP32 constants) and for the FP64
// energy gathers (from the FP64 potential constants), kMaxTypes floats each.  A candidate
// type's reach is the largest over the other types, and over both orders of the pair, of
// r_c when the row has an outer branch (C4 or C5 nonzero) and r_m otherwise, capped at the
// cutoff, plus 1e-4.
std::vector<float> pair_table(const std::vector<double> &hf, const std::vector<double> &hu, int nT, double cutoff)
{
    const size_t rows = (size_t)nT * nT;
    std::vector<float> tab(8 * rows + 2 * kMaxTypes, 0.f);
    for (size_t r = 0; r < rows; r++)
        for (int k = 0; k < 6; k++) tab[8 * r + k] = (float)hf[6 * r + k];
    const double rcap = std::sqrt(cutoff * cutoff);
    for (int t = 0; t < nT; t++) {
        double rF = 0.0, rE = 0.0;
        for (int h = 0; h < nT; h++)
            for (const size_t row : {(size_t)h * nT + t, (size_t)t * nT + h}) {
                const float *f = &tab[8 * row];
                const double fm = f[0], fc = f[3], f4 = f[4], f5 = f[5];
                rF = std::fmax(rF, (f4 != 0.0 || f5 != 0.0) ? fc : fm);
                const double *u = &hu[6 * row];
                rE = std::fmax(rE, (u[4] != 0.0 || u[5] != 0.0) ? u[3] : u[0]);
            }
        rF = std::fmin(rF, rcap) + 1e-4;
        rE = std::fmin(rE, rcap) + 1e-4;
        tab[8 * rows + t] = (float)(rF * rF);
        tab[8 * rows + kMaxTypes + t] = (float)(rE * rE);
    }
    return tab;
}

// Whether some (a, b) row of the force or potential table differs from its (b, a) row.  The
// reference evaluates each pair once, with the row of the particle its traversal makes
// first (MD.h:811-819, cellOpt.h:712-926); the pair kernels then pick that row per pair.
bool tables_asymmetric(const std::vector<double> &hf, const std::vector<double> &hu, int nT)
{
    for (int a = 0; a < nT; a++)
        for (int b = a + 1; b < nT; b++)
            for (int k = 0; k < 6; k++)
                if (hf[6 * (a * nT + b) + k] != hf[6 * (b * nT + a) + k] ||
                    hu[6 * (a * nT + b) + k] != hu[6 * (b * nT + a) + k])
                    return true;
    return false;
}

// k_first's step argument: set the device step counter, advance it by one, or leave it
constexpr long long kStepAdvance = -1, kStepKeep = -2;

// host mirror of a replica's layout
struct RepHost {
    int first = 0, count = 0, cfirst = 0, ccount = 0;
    int nbond = 0, nbend = 0;   // generic BOND / BEND records
    long long capacity = 0, cellbase = 0;
};

// Tiles of a segment set: ranges [begin_r, begin_r + len_r) cut into tiles that start at each
// range's start, of kSumTile elements or, in a range of more than kSumTiles of those, a multiple.
struct SegHost {
    std::vector<int4> tile;
    std::vector<int> rep_first;
};

SegHost make_tiles(const std::vector<int> &begin, const std::vector<int> &len)
{
    SegHost h;
    for (size_t r = 0; r < begin.size(); r++) {
        h.rep_first.push_back((int)h.tile.size());
        const int step = kSumTile * (int)(((long long)len[r] + kSumTile * kSumTiles - 1) / (kSumTile * kSumTiles));
        for (int t = 0; t < len[r]; t += step)
            h.tile.push_back(make_int4(begin[r] + t, begin[r] + std::min(len[r], t + step), (int)r, 0));
    }
    h.rep_first.push_back((int)h.tile.size());
    return h;
}

}  // namespace

struct sm_ctx {
    hipStream_t st = nullptr;
    int device = 0;   // the device current at creation, whose stream this is
    Params P{};
    int n = 0;
    int nrep = 0;
    int nchains = 0;
    bool any_mc = false;   // some replica has delta_lxy != 0
    std::vector<RepHost> rh;
    // device state: `slab` holds every buffer whose size stays, `table` cstart and cend, `counting`
    // counts and bucket
    char *slab = nullptr;
    int *table = nullptr;
    uint32_t *counting = nullptr;
    Bead *beads = nullptr, *sbeads = nullptr;
    Bead *beads_alt = nullptr;   // the fused kick + next first half writes positions here, then swaps
    float4 *vel = nullptr, *acc = nullptr, *fpair = nullptr, *fscratch = nullptr;
    uint32_t *k0 = nullptr, *v0 = nullptr, *k1 = nullptr, *v1 = nullptr;
    uint32_t *hist[2] = {nullptr, nullptr};   // sort scratch, double-buffered
    size_t hist_words = 0;
    int sort_parity = 0;                      // scratch the next sort uses
    bool hist_pending = false;                // its histograms hold keys not sorted yet
    // Incremental re-sort (sort_mode 1; 0: every build sorts all keys from index order): the
    // keys by index of this build (kidx[kcur]) and of the previous sort (kidx[1 - kcur]),
    // the sorted order of the previous sort in (sk, sv)[scur] (the new one goes into the
    // other pair), the mover counts and flags, the movers-before words and the mover count.
    // order_valid: those describe the last sort, which was incremental.  Measured on one
    // MI355X: 38.4 against 48.9 us per step at 240k beads (the movers' passes and the
    // merge are latency-bound launches), 126 against 115 us at 3M, 156 against 118 us for
    // the 64-replica sweep of 2.8M; contexts of a million beads or more start in mode 1,
    // single replicas whose builds count beads start in mode 2, and the autotuner tries
    // every mode the context allows.
    int sort_mode = 0;
    uint32_t *kidx[2] = {nullptr, nullptr};
    uint32_t *sk[2] = {nullptr, nullptr}, *sv[2] = {nullptr, nullptr};
    uint32_t *mbefore = nullptr, *cnt_b = nullptr, *cnt_i = nullptr, *cnt_s = nullptr;
    unsigned long long *mflags = nullptr;
    int *mcount = nullptr;
    int kcur = 0, scur = 0;
    bool order_valid = false;
    // Counting builds (sm_internal.hpp).  Window: sort_mode 2, when win_ok (a single replica of
    // at most 256 sort tiles), while the keys have 17 to 24 bits; wdesc + 8p is the window of
    // the build with scratch parity p, which the previous build derived on the device.  Dense:
    // otherwise, sort_mode 0 or 2 with at most 256 tiles, while the cell table holds at most
    // kWinCells cells.  counts[p] and counted[p]: the cells' beads, and the cells counted
    // in, by the build with parity p; k2 then holds the sorted cell indices and v0 the bead
    // indices ((k2, v2) is also the fallback's third buffer pair).  cnt_last: the last build
    // was a counting build, win_last: by a window.
    bool win_ok = false, win_last = false, cnt_last = false;
    uint32_t *k2 = nullptr, *v2 = nullptr, *wdesc = nullptr, *counts[2] = {}, *counted[2] = {}, *bucket = nullptr;
    size_t count_cells = 0;   // cells that counts and bucket hold
    bool counters_ready = false;   // the last build was a counting build with these buffers
    // Builds that keep falling back -- a cell of more beads than a bucket that stays, a vesicle
    // whose window never fits -- count for nothing and then sort in one launch what the radix sort
    // orders faster: per step 165 against 121 us at 192k beads in 16 bilayers, 334 against 224 for
    // a vesicle of 480k.  The device's count of fallbacks comes with every result; where more than
    // half of the builds since the last result fell back, the context stops counting, until its
    // sort mode is set or a box uploaded.  counts_known: a result has told about this context's
    // builds; a first long run asks for one after 8 steps (run()).
    bool count_off = false, counts_known = false;
    uint32_t fallbacks_seen = 0;
    long long counted_builds = 0;   // launched since
    void learn()
    {
        constexpr int kEnough = 4;   // the first build of a window always falls back
        if (counted_builds < kEnough) return;
        const uint32_t now = link.fallbacks();
        counts_known = true;
        if (2ll * (uint32_t)(now - fallbacks_seen) > counted_builds && !count_off) {
            drop_graph();
            forget_keys();
            count_off = true;
        }
        fallbacks_seen = now;
        counted_builds = 0;
    }
    void count_again()
    {
        if (count_off) {
            drop_graph();
            forget_keys();
        }
        count_off = counts_known = false;
    }
    bool win_now() const
    {
        return sort_mode == 2 && win_ok && bucket && !count_off && sort_bits >= 17 && sort_bits <= 24;
    }
    bool dense_now() const
    {
        return !win_now() && sort_mode != 1 && bucket && !count_off && capacity <= kWinCells && sortw_fits(n);
    }
    bool count_now() const { return dense_now() || win_now(); }
    // room to count in windows, or in the whole table while that is small; without the memory for
    // it the builds sort
    void alloc_counts()
    {
        if (!sortw_fits(n)) return;
        // a window is a part of the table, so a small table's cells are enough for either
        size_t cells = win_ok ? count_limit(n) : 0;
        if (capacity <= kWinCells) cells = ((size_t)capacity + kCoarseCells - 1) / kCoarseCells * kCoarseCells;
        if (cells <= count_cells) return;
        counters_ready = false;
        count_cells = 0;
        bucket = nullptr;
        counts[0] = counts[1] = nullptr;
        dfree(counting);
        try {
            counting = dalloc<uint32_t>(cells * (kBucket + 2));
        } catch (const ApiError &) {
            return;
        }
        bucket = counting;
        for (int p = 0; p < 2; p++) counts[p] = counting + cells * (kBucket + p);
        count_cells = cells;
    }
    int *cstart = nullptr, *cend = nullptr;
    long long capacity = 0;   // cells in the dense table, all replicas
    int sort_bits = 0;
    DevRep *reps = nullptr;
    DevGlobal *glob = nullptr;
    HostLink link;             // results on their way to the host
    // The boxes as last read or set, 3 per replica, and the box moves launched since: a box
    // lies within moves * |delta_lxy| of them, so most runs need no read-back to know that the
    // cell table is large enough.
    std::vector<double> boxL, deltaL;
    long long moves_since = 0;
    float *fconstF = nullptr;   // pair table: padded FP32 force rows, then the reach tables
    double *uconstD = nullptr;
    double *fconstD = nullptr;   // FP64 force rows (the force kernel's pair-count hook)
    int2 *chainPerBead = nullptr, *chainList = nullptr;
    double4 *cconstD = nullptr;
    // generic BOND / BEND records, per bead (CSR); gptr == nullptr when there are none
    int *gptr = nullptr;
    GenEnt *gent = nullptr;
    double2 *gconstD = nullptr;
    GenTables gen() const { return GenTables{gptr, gent, gconstD}; }
    // host copies of the constants (the adjoint changes them)
    std::vector<double> hfconst, huconst;
    std::vector<double4> hcconst;
    double *adjF = nullptr, *adjDF = nullptr, *adjDU = nullptr;   // FP64 F table, d/dtheta tables
    // the adjoint's workspace (AdjointRun)
    char *adj_ws = nullptr;
    size_t adj_ws_bytes = 0;
    char *adj_workspace(size_t bytes)
    {
        if (bytes > adj_ws_bytes) {
            free_adj_workspace();
            adj_ws = dalloc<char>(bytes);
            adj_ws_bytes = bytes;
        }
        return adj_ws;
    }
    void free_adj_workspace()
    {
        dfree(adj_ws);
        adj_ws = nullptr;
        adj_ws_bytes = 0;
    }
    // sm_param_derivative: the U table's d/dUmin and d/dUmax forms of one type pair, their
    // culling tables, and the CHAIN constant sets with (k_bond, k_bend) = (1, 0) and (0, 1)
    double *pdU = nullptr;
    float *pdTab = nullptr;
    double4 *pdC = nullptr;
    int pd_a = -1, pd_b = -1;
    size_t pd_tab = 0;
    double *ebead = nullptr, *edelta = nullptr;   // a term per bead; a box-move step keeps its dU in edelta
    double *dres = nullptr;                      // meas [R][3], then dU [R][2]; or one call's 8 R results
    SegTiles segB{}, segC{};
    int *dcounts = nullptr, *dpairs = nullptr;
    long long pairs_cap = 0;
    unsigned long long *dnp = nullptr;
    int chunk = 8, echunk = 8;   // sorted slots per wave: the force and the counts; the FP64 energy traversals
    bool chunk_set = false;      // by sm_tune or the autotuner
    int pair_variant = 0;
    // box-move steps: the pair dU in the same traversal as the step's pair force (1) or in
    // a gather of its own after the kick (0, as the adjoint uses)
    bool mc_fused = true;
    int sorted_sel = 0;   // which sort buffer pair holds the sorted result
    // captured 8-step graph
    bool use_graph = false;
    // one graph per sort-scratch parity and bead buffer at the start of the block (8 sorts and 8
    // changes of buffer return to them): [2 * parity + (beads is not beads_home)]
    hipGraph_t graph[4] = {};
    hipGraphExec_t gexec[4] = {};
    const Bead *beads_home = nullptr;
    // profiling
    bool prof = false;
    struct Rec { int cls; hipEvent_t a, b; };
    std::vector<Rec> recs;
    std::vector<hipEvent_t> pool;
    double prof_ms[K_NCLASS] = {};
    long long prof_cnt[K_NCLASS] = {};

    const uint32_t *skey() const { return sort_mode == 1 ? sk[scur] : (cnt_last ? k2 : (sorted_sel ? k1 : k0)); }
    const uint32_t *sidx() const { return sort_mode == 1 ? sv[scur] : (cnt_last ? v0 : (sorted_sel ? v1 : v0)); }
    // the key kernel's outputs and bookkeeping for the next sort
    uint32_t *key_out() const { return sort_mode == 1 ? kidx[kcur] : k0; }
    // bead indices for the every-key sort (a counting build's are in its buckets)
    uint32_t *idx_out() const { return sort_mode == 1 || count_now() ? nullptr : v0; }
    WinBook win_keys(int p) const
    {
        if (!count_now()) return WinBook{};
        const bool win = win_now();
        return win_book(hist[p], n, win ? wdesc + 8 * p : nullptr, counts[p], bucket, win ? 0u : (uint32_t)capacity,
                        (uint32_t)count_cells);
    }
    // whether the last build counted its beads, and did not fall back to sorting them (waits for
    // the stream); its window and flag: its scratch is cleared only by the next build
    bool counted_last()
    {
        if (!cnt_last) return false;
        const int lp = 1 - sort_parity;
        uint32_t wx = 1, flag = 0;
        if (win_last) HIPCHK(hipMemcpyAsync(&wx, wdesc + 8 * lp + 3, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
        const uint32_t *f = win_book(hist[lp], n, nullptr, nullptr, nullptr, 0u, 0u).flag;
        HIPCHK(hipMemcpyAsync(&flag, f, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        return wx != 0 && flag == 0;
    }
    // a key kernel ran without its sort: zero what it added to the sort's scratch
    void restart_hist(uint32_t *gh)
    {
        launch_fill_u32(st, gh, sort_hist_words(), 0u);
        launch_fill_u32(st, win_scratch(gh, n), kWinKeyWords, 0u);
        if (counts[0]) launch_fill_u32(st, counts[sort_parity], count_cells, 0u);
    }
    // keys that no build has taken, made for another sort mode, table or state: gone
    void forget_keys()
    {
        if (hist_pending) restart_hist(hist[sort_parity]);
        hist_pending = false;
    }
    // before a key kernel: its scratch holds nothing yet
    void begin_keys()
    {
        forget_keys();   // keys computed twice before a sort: start over
        hist_pending = true;
        // a counting build clears the counters of the one right before it only
        if (count_now() && !counters_ready)
            for (uint32_t *c : counts) launch_fill_u32(st, c, count_cells, 0u);
    }
    MoveBook move_book() const
    {
        if (sort_mode != 1) return MoveBook{nullptr, nullptr};
        return MoveBook{order_valid ? kidx[1 - kcur] : nullptr, cnt_b};
    }
    double *meas_dev() const { return dres; }
    double *du_dev() const { return dres + 3 * (size_t)nrep; }

    ~sm_ctx()
    {
        if (st) (void)hipStreamSynchronize(st);
        drop_graph();
        link.destroy();
        for (auto &r : recs) { (void)hipEventDestroy(r.a); (void)hipEventDestroy(r.b); }
        for (auto e : pool) (void)hipEventDestroy(e);
        dfree(slab); dfree(table); dfree(counting); dfree(dpairs);
        free_adj_workspace();
        dfree(adjF); dfree(adjDF); dfree(adjDU); dfree(pdU); dfree(pdTab); dfree(pdC);
        if (st) (void)hipStreamDestroy(st);
    }

    void drop_graph()
    {
        for (int p = 0; p < 4; p++) {
            if (gexec[p]) (void)hipGraphExecDestroy(gexec[p]);
            if (graph[p]) (void)hipGraphDestroy(graph[p]);
            gexec[p] = nullptr;
            graph[p] = nullptr;
        }
    }

    // ---- profiling helpers ----
    hipEvent_t ev()
    {
        if (!pool.empty()) {
            hipEvent_t e = pool.back();
            pool.pop_back();
            return e;
        }
        hipEvent_t e;
        HIPCHK(hipEventCreate(&e));
        return e;
    }
    template <class F>
    void timed(int cls, F &&f)
    {
        if (!prof) {
            f();
            return;
        }
        Rec r{cls, ev(), ev()};
        HIPCHK(hipEventRecord(r.a, st));
        f();
        HIPCHK(hipEventRecord(r.b, st));
        recs.push_back(r);
        if (recs.size() >= 8192) harvest();
    }
    void harvest()
    {
        HIPCHK(hipStreamSynchronize(st));
        for (auto &r : recs) {
            float ms = 0.f;
            HIPCHK(hipEventElapsedTime(&ms, r.a, r.b));
            prof_ms[r.cls] += ms;
            prof_cnt[r.cls]++;
            pool.push_back(r.a);
            pool.push_back(r.b);
        }
        recs.clear();
    }

    void check_launch() { HIPCHK(hipGetLastError()); }

    std::vector<DevRep> read_reps()
    {
        std::vector<DevRep> h(nrep);
        HIPCHK(hipMemcpyAsync(h.data(), reps, sizeof(DevRep) * nrep, hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        return h;
    }
    void write_reps(const std::vector<DevRep> &h)
    {
        HIPCHK(hipMemcpyAsync(reps, h.data(), sizeof(DevRep) * nrep, hipMemcpyHostToDevice, st));
        HIPCHK(hipStreamSynchronize(st));
    }
    DevGlobal read_glob()
    {
        DevGlobal g;
        HIPCHK(hipMemcpyAsync(&g, glob, sizeof g, hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        return g;
    }

    void check_flags() { check_bits(link.fetch(st, glob, nullptr, 0, nullptr)); }
    // the flags of a result, and what its count of fallbacks says
    void check_bits(int flags)
    {
        learn();
        if (flags & FLAG_BAD_POSITION)
            throw ApiError(SM_ERR_STATE, "a particle position left the box or became non-finite");
        if (flags & FLAG_SORT_TIMEOUT)
            throw ApiError(SM_ERR_STATE, "cell-key sort look-back timed out");
        if (flags & FLAG_SORT_COUNT)
            throw ApiError(SM_ERR_STATE, "incremental cell sort: inconsistent mover count");
        if (flags & FLAG_CELL_OVERFLOW)
            throw ApiError(SM_ERR_STATE, "an accepted box move would exceed the cell table or make fewer than 3 cells per axis");
    }
    // `count` doubles of results to the host, and the state checked
    void fetch(const double *src, size_t count, double *dst) { check_bits(link.fetch(st, glob, src, count, dst)); }

    // the device's boxes were set back to an earlier state's: read them when next needed
    void forget_boxes() { moves_since = 1ll << 40; }

    // the current box lengths (boxL), read back if box moves were launched since
    void know_boxes()
    {
        if (moves_since == 0) return;
        link.fetch_boxes(st, glob, reps, nrep, boxL.data());
        moves_since = 0;
    }

    // cells that replica r needs for every box that `moves` MC moves from boxL can reach;
    // kUnbounded when the moves could take the box anywhere (the device then refuses the
    // accepted move that outgrows the table)
    static constexpr long long kUnbounded = (long long)9e18;
    long long cells_needed(int r, long long moves) const
    {
        const double dL = deltaL[r], *L = &boxL[3 * (size_t)r];
        const double grow = (double)moves * std::fabs(dL);
        double Lmax[3], Lmin[2];
        for (int d = 0; d < 2; d++) {
            Lmax[d] = L[d] + grow;
            Lmin[d] = std::max(L[d] - grow, 1e-300);
        }
        Lmax[2] = (moves > 0 && dL != 0) ? L[2] * (L[0] * L[1]) / (Lmin[0] * Lmin[1]) : L[2];
        double need = 1.0;   // a product that may pass 2^63 while the bound is loose
        for (int d = 0; d < 3; d++) need *= std::floor(Lmax[d] / P.cutoff) + 1.0;
        return need < 9e18 ? (long long)need : kUnbounded;
    }

    // Dense cell table sized for every box the next `moves` MC moves can reach, in every
    // replica; a replica that outgrows its reservation moves every cell base (keys are
    // recomputed each step, so only the table is reallocated).  A table that cannot be had
    // leaves the context as it was.
    void ensure_capacity(long long moves)
    {
        auto grows = [&](int r) {
            const long long need = cells_needed(r, moves);
            return need > rh[r].capacity && need != kUnbounded;
        };
        bool relayout = false;
        for (int r = 0; r < nrep && !relayout; r++) relayout = cells_needed(r, moves_since + moves) > rh[r].capacity;
        if (!relayout) return;
        know_boxes();
        relayout = false;
        for (int r = 0; r < nrep && !relayout; r++) relayout = grows(r);
        if (!relayout) return;
        std::vector<DevRep> hr = read_reps();
        std::vector<RepHost> laid = rh;
        long long base = 0;
        for (int r = 0; r < nrep; r++) {
            if (grows(r)) {
                const long long need = cells_needed(r, moves);
                laid[r].capacity = need + need / 8;
            }
            laid[r].cellbase = base;
            if (laid[r].capacity > 0xFFFFFFFFll || (base += laid[r].capacity) > 0xFFFFFFFFll)
                unsupported("cell tables of all replicas exceed 2^32 cells");
            hr[r].cellbase = laid[r].cellbase;
            hr[r].capacity = laid[r].capacity;
        }
        int *grown = dalloc<int>(2 * (size_t)base);
        try {
            HIPCHK(hipMemsetAsync(grown, 0xFF, 2 * sizeof(int) * (size_t)base, st));
        } catch (...) {
            dfree(grown);
            throw;
        }
        drop_graph();
        forget_keys();
        dfree(table);
        table = grown;
        cstart = table;
        cend = table + base;
        rh = std::move(laid);
        capacity = base;
        write_reps(hr);
        int bits = 1;
        while ((1ll << bits) < base) bits++;
        sort_bits = bits;
        alloc_counts();
    }

    // The launch shapes that follow from the box: at creation and when one is uploaded (box moves
    // change it by percents).  Chunks that were set or tuned stay.
    void launch_rules()
    {
        const int flat = nrep == 1 && boxL[2] / P.cutoff < 64.0 ? 1 : 0;
        if (flat != P.flat) drop_graph();   // captured launches hold it, and the chunks that it sets
        P.flat = flat;
        if (chunk_set) return;
        // sorted slots per wave in the pair kernels: short chunks keep small systems filling the
        // chip and even out flat ones, longer ones cut the overhead per wave (every chunk gives
        // the same forces).  Whole steps in us at 2, 4, 8, 16 slots: 1.5k vesicle 27.1, 28 at 4;
        // 18k bilayer 48.0, 46.7; 90k vesicle 63.7, 62.3, 61.7; 120k 74.5, 72.5, 71.7; 300k
        // bilayer 148 at 4, 158, 178; 990k bilayer 450 at 4, 451, 468; 3M bilayer 1216 at 4,
        // 1188, 1191; 1.35M vesicle 530 at 8, 522; 3M vesicle 1123 at 8, 1098; 1.5M beads in 64
        // bilayers 648 at 8, 658.
        const int many = P.flat ? 1000000 : 100000;
        chunk = n < 10000 ? 2 : (n < many ? 4 : (n < 2000000 || P.flat ? 8 : 16));
        // The energy traversals do more per candidate.  Force with dU and U in us: 1.5k vesicle
        // 24 and 15.0 at 2, 31 and 19.4 at 8; 12k bilayer 57 and 29.4 at 2, 46 and 25.4 at 8; 37k
        // vesicle 54 and 29.2 at 2, 51 and 27.1 at 4, 49 and 29.6 at 8; 90k bilayer 84 and 44.2
        // at 4, 82 and 43.0 at 8; 1.2M vesicle 687 and 325 at 8, 677 and 317 at 16; 1.2M bilayer
        // 653 and 311 at 8, 667 and 317 at 16.
        echunk = n < 10000 ? 2 : (P.flat ? 8 : (n < 50000 ? 4 : (n < 1000000 ? 8 : 16)));
    }

    // keys (optionally after Verlet::first) with the next sort's digit histograms, sort,
    // reorder + dense cell table (clearing the other sort scratch)
    // away: the beads go to the other buffer
    void first_and_keys(int integrate, long long step_set, bool for_sort = true, bool away = false)
    {
        uint32_t *gh = for_sort ? hist[sort_parity] : nullptr;
        if (for_sort) begin_keys();
        const int passes = sort_passes(sort_bits);
        timed(K_FIRST, [&] {
            if (for_sort)
                launch_first(st, P, beads, away ? beads_alt : beads, vel, acc, reps, glob, key_out(), idx_out(),
                             integrate, step_set, gh, passes, move_book(), win_keys(sort_parity));
            else   // keys only (no sort follows): into the mover buffer, which no sort state holds
                launch_first(st, P, beads, beads, vel, acc, reps, glob, k0, nullptr, integrate, step_set, nullptr, passes,
                             MoveBook{nullptr, nullptr});
        });
        if (away) std::swap(beads, beads_alt);
    }
    void sort_and_reorder()
    {
        // a step's rest without its first half, or with something in between that the keys do not
        // fit: the keys of the positions there are
        if (!hist_pending) first_and_keys(0, kStepKeep);
        const int p = sort_parity;
        const bool count = count_now();
        win_last = count && win_now();
        cnt_last = counters_ready = count;
        if (count) {
            counted_builds++;
            timed(K_REORDER, [&] {
                launch_build(st, n, BuildArgs{k0, v0, k1, v1, k2, v2, win_keys(p), counts[1 - p], counted[1 - p],
                                              counted[p], wdesc ? wdesc + 8 * (1 - p) : nullptr, beads, sbeads, cstart,
                                              cend, hist[1 - p], hist_words, reps, hist[p],
                                              win_scratch(hist[p], n) + kWinKeyWords, &glob->flags, &glob->fallbacks, build_tiles(n)});
            });
            order_valid = false;
            sort_parity = 1 - p;
            hist_pending = false;
            return;
        }
        if (sort_mode == 1) {
            timed(K_SORT, [&] {
                SortBuffers sb{k0, v0, k1, v1, {hist[0], hist[1]}, &glob->flags, n, 0};
                const MoveSort m{kidx[kcur], order_valid ? kidx[1 - kcur] : nullptr, sk[scur], sv[scur], cstart, cend,
                                 cnt_b, cnt_i, cnt_s, mflags, mbefore, mcount, sk[1 - scur], sv[1 - scur]};
                sort_moved(st, sb, m, sort_bits, p);
            });
            scur = 1 - scur;
            kcur = 1 - kcur;
            order_valid = true;
        } else {
            timed(K_SORT, [&] {
                SortBuffers sb{k0, v0, k1, v1, {hist[0], hist[1]}, &glob->flags, n, 0};
                sorted_sel = radix_sort(st, sb, sort_bits, p);
            });
            order_valid = false;
        }
        timed(K_REORDER, [&] {
            launch_reorder(st, n, skey(), sidx(), beads, sbeads, cstart, cend, hist[1 - p], hist_words);
        });
        sort_parity = 1 - p;
        hist_pending = false;
    }
    void build(int integrate, long long step_set)
    {
        first_and_keys(integrate, step_set);
        sort_and_reorder();
    }
    void pair_force()
    {
        timed(K_PAIR, [&] {
            launch_pair_force(st, P, chunk, pair_variant, sbeads, skey(), sidx(), cstart, cend, reps, fconstF, fpair);
        });
    }
    void bonded(int mode, float4 *fchain_out)
    {
        timed(K_BONDED, [&] {
            launch_bonded_kick(st, P, beads, chainPerBead, cconstD, gen(), fpair, vel, acc, reps, glob, mode,
                               fchain_out);
        });
    }
    // {U_pair, U_chain, K} of every replica into dres[3r + 0..2] (device)
    void measure_device()
    {
        timed(K_GATHER, [&] {
            launch_pair_gather(st, P, echunk, GATHER_U, sbeads, skey(), sidx(), cstart, cend, reps, fconstF, uconstD, ebead,
                               nullptr, nullptr, nullptr, 0);
        });
        timed(K_SUMS, [&] {
            SumArgs a = sums(ebead, meas_dev());
            launch_sums(st, SUM_MEASURE, a);
            if (gptr) {
                launch_gen_energy(st, n, gen(), beads, reps, 0, ebead);
                add_column(ebead, meas_dev() + 1, 3);
            }
        });
    }
    SumArgs sums(const double *x, double *out) const
    {
        SumArgs a{};
        a.B = segB;
        a.C = segC;
        a.x = x;
        a.vel = vel;
        a.chains = chainList;
        a.cconst = cconstD;
        a.beads = beads;
        a.reps = reps;
        a.out = out;
        a.n = n;
        return a;
    }
    // the pair force with each bead's share of U_pair in ebead: one traversal of 32 us where the
    // force and U took 23 and 24 at 12k beads
    void pair_force_u()
    {
        timed(K_PAIR, [&] {
            launch_pair_force_u(st, P, echunk, sbeads, skey(), sidx(), cstart, cend, reps, fconstF, uconstD, fpair,
                                ebead);
        });
    }
    // out[2r + 0..1] += {U_pair (from ebead), U_chain}
    void add_energies(double *out)
    {
        timed(K_SUMS, [&] {
            launch_sums(st, SUM_ENERGY, sums(ebead, out));
            if (gptr) {
                launch_gen_energy(st, n, gen(), beads, reps, 0, ebead);
                add_column(ebead, out + 1, 2);
            }
        });
    }
    void add_column(const double *x, double *out, int stride) const
    {
        SumArgs a = sums(x, out);
        a.stride = stride;
        a.add = 1;
        launch_sums(st, SUM_COLUMN, a);
    }
    // U(old) - U(scaled) of every replica with its trial scale into dres[3R + 2r + 0..1]
    void delta_device()
    {
        timed(K_GATHER, [&] {
            launch_pair_gather(st, P, echunk, GATHER_DU, sbeads, skey(), sidx(), cstart, cend, reps, fconstF, uconstD, edelta,
                               nullptr, nullptr, nullptr, 0);
        });
        delta_sums();
    }
    // the replicas' pair dU from the beads' (edelta), with the CHAIN and generic-record part
    void delta_sums()
    {
        timed(K_SUMS, [&] {
            launch_sums(st, SUM_DELTA, sums(edelta, du_dev()));
            if (gptr) {
                launch_gen_energy(st, n, gen(), beads, reps, 1, ebead);
                add_column(ebead, du_dev() + 1, 2);
            }
        });
    }
    void mc_move()
    {
        timed(K_MC, [&] { launch_mc_propose(st, nrep, reps, glob); });
        delta_device();
        mc_decide();
    }
    void mc_decide()
    {
        moves_since++;
        timed(K_MC, [&] {
            launch_mc_decide(st, P, reps, glob, du_dev());
            launch_rescale(st, n, beads, reps);
        });
    }
    // A box-move step's pair force with its pair dU: the trial scale is drawn first (it
    // depends on the step's key only), then one traversal gives the forces and each owned
    // pair's U(old) - U(scaled) at the positions the force sees, which the kick leaves as
    // they are.  The bonded dU and the decision follow the kick (mc_finish).
    void pair_force_mc()
    {
        timed(K_MC, [&] { launch_mc_propose(st, nrep, reps, glob); });
        pair_force_du();
    }
    // the pair force with the pair dU under each replica's current trial scale
    void pair_force_du()
    {
        timed(K_PAIR, [&] {
            launch_pair_force_du(st, P, echunk, sbeads, skey(), sidx(), cstart, cend, reps, fconstF, uconstD, fpair,
                                 edelta);
        });
    }
    void pair_step(bool mc)
    {
        if (mc && mc_fused)
            pair_force_mc();
        else
            pair_force();
    }
    void mc_finish()
    {
        if (mc_fused) {
            delta_sums();
            mc_decide();
        } else {
            mc_move();
        }
    }
    bool mc_step(long long step) const { return step % 8 == 0 && step != 0 && any_mc; }

    // Step s's bonded + Langevin forces and second half kick, with step s + 1's first half,
    // keys and digit histograms, as one kernel (same arithmetic as bonded() then
    // step_first(s + 1)); the new positions land in the other bead buffer.  from_base: s counts
    // from the captured block's start.
    void kick_first(long long s, bool from_base = false)
    {
        uint32_t *gh = hist[sort_parity];
        begin_keys();
        const int passes = sort_passes(sort_bits);
        timed(K_KICK_FIRST, [&] {
            launch_kick_first(st, P, beads, beads_alt, chainPerBead, cconstD, gen(), fpair, vel, reps, glob, s,
                              from_base, key_out(), idx_out(), gh, passes, move_book(), win_keys(sort_parity));
        });
        std::swap(beads, beads_alt);
    }

    void step_first(long long step_set) { first_and_keys(1, step_set); }
    void step_finish(bool measure, bool mc)
    {
        sort_and_reorder();
        pair_step(mc);
        bonded(KICK_STEP, nullptr);
        if (measure) measure_device();
        if (mc) mc_finish();
    }
    // Steps s .. s+7 with s % 8 == 1 as one graph: the step counter advances on the
    // device, so the same graph serves every such block; the MC move (if any replica
    // has one) falls on the block's last step.  The kernels are run()'s: seven fused kicks, and
    // the block's first half step moves the beads to the other buffer too, so that the block
    // ends in the buffer it began in and the next replays the same graph.  16 steps of the
    // 12k-bead bilayer with their download took 831 us with the halves apart, 793 now.
    void graph_block(long long s)
    {
        if ((sort_mode == 1 && !order_valid) || (count_now() && !counters_ready)) {
            // the graph would replay a first sort without a previous order, or a first counting
            // build: step this block eagerly, after which there is one to capture against
            eager(s, s + 8);
            return;
        }
        forget_keys();   // the graph's are the first
        const int p = sort_parity, q = 2 * p + (beads != beads_home ? 1 : 0);
        if (!gexec[q]) {
            HIPCHK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
            first_and_keys(1, kStepAdvance, true, true);
            for (int k = 0; k < 8; k++) {
                const bool mc = k == 7 && any_mc;
                sort_and_reorder();
                pair_step(mc);
                if (k < 7) {
                    kick_first(k + 1, true);
                    continue;
                }
                bonded(KICK_STEP, nullptr);
                if (mc) mc_finish();
            }
            hipError_t e = hipStreamEndCapture(st, &graph[q]);
            if (e != hipSuccess) {
                graph[q] = nullptr;
                HIPCHK(e);
            }
            HIPCHK(hipGraphInstantiate(&gexec[q], graph[q], nullptr, nullptr, 0));
            if (any_mc) moves_since--;   // capture only recorded the move, and the builds
            if (cnt_last) counted_builds -= 8;
        }
        sort_parity = p;   // and the toggles
        if (any_mc) moves_since++;
        if (cnt_last) counted_builds += 8;
        // the block advances from step s - 1
        launch_set_step(st, glob, s - 1);
        HIPCHK(hipGraphLaunch(gexec[q], st));
    }

    // Steps [s, end): one without a box move ends in the fused kernel that also does the next
    // step's first half; a box-move step and the last step end unfused.
    void eager(long long s, long long end)
    {
        bool first_done = false;
        for (; s < end; s++) {
            if (!first_done) step_first(s);
            const bool mc = mc_step(s);
            sort_and_reorder();
            pair_step(mc);
            first_done = !mc && s + 1 < end;
            if (first_done) {
                kick_first(s);
                continue;
            }
            bonded(KICK_STEP, nullptr);
            if (mc) mc_finish();
        }
    }

    void run(long long first, long long nsteps)
    {
        long long moves = 0;
        for (long long s = first; s < first + nsteps; s++)
            if (mc_step(s)) moves++;
        if (moves) ensure_capacity(moves);
        long long s = first;
        const long long end = first + nsteps;
        if (nsteps >= 64 && count_now() && !counts_known) {
            eager(s, s + 8);
            s += 8;
            try {
                (void)link.fetch(st, glob, nullptr, 0, nullptr);
                learn();
            } catch (const ApiError &) {   // a wait that is refused where it is called: the next result tells
                counts_known = true;
            }
        }
        if (use_graph && !prof) {
            const long long lead = std::min(end, s + (9 - s % 8) % 8);   // up to the next s % 8 == 1
            eager(s, lead);
            for (s = lead; end - s >= 8; s += 8) graph_block(s);
        }
        eager(s, end);
    }
};

// ---------------------------------------------------------------------------------------
// validation and upload
// ---------------------------------------------------------------------------------------
namespace {

void validate(const sm_system *s)
{
    if (!s) invalid("null system");
    const int n = s->n_particles;
    if (n <= 0) invalid("n_particles must be positive");
    if (!s->pos || !s->type || !s->vel) invalid("pos, type and vel are required");
    if (s->n_types < 1 || s->n_types > kMaxTypes)
        unsupported("n_types must be in [1, " + std::to_string(kMaxTypes) + "]");
    if (!s->fconst || !s->uconst) invalid("fconst and uconst are required");
    if (!(s->cutoff > 0)) invalid("cutoff must be positive");
    if (!(s->dt > 0)) invalid("dt must be positive");
    if (!(s->gamma > 0)) invalid("gamma must be > 0");
    if (!(s->sigma_temperature >= 0)) invalid("sigma_temperature must be >= 0");
    for (int d = 0; d < 3; d++) {
        if (!(s->box[d] > 0)) invalid("box lengths must be positive");
        if ((int)(s->box[d] / s->cutoff) < 3) unsupported("fewer than 3 cells along an axis");
    }
    const int nT = s->n_types;
    for (int i = 0; i < n; i++) {
        if (s->type[i] < 0 || s->type[i] >= nT) invalid("particle " + std::to_string(i) + " has a type outside [0, nTypes)");
        for (int d = 0; d < 3; d++) {
            double p = s->pos[3 * (size_t)i + d];
            if (!(p >= 0 && p <= s->box[d]))
                invalid("particle " + std::to_string(i) + " position is out of bounds");
        }
    }
    // the reference's force takes the branch at row offset int(r / r_m) * 3 (MD.h:819),
    // which stays inside the row for every r below the cutoff only while 2 r_m >= cutoff
    for (int r = 0; r < nT * nT; r++)
        if (!(2.0 * s->fconst[6 * r] >= s->cutoff))
            unsupported("two-body row " + std::to_string(r / nT) + "," + std::to_string(r % nT) +
                        ": r_m below half the cutoff (the reference's branch offset int(r/r_m)*3 leaves the row)");
    if (s->n_chain_blocks < 0) invalid("negative chain block count");
    if (s->n_chain_blocks > 0 && (!s->chain || !s->chain_const)) invalid("chain blocks without data");
    // CHAIN blocks (start, nChains, length): inside the particles, each bead in one chain
    // at most (the reference checks its chains' bonds against nParticles, system.h:515-535)
    std::vector<char> chained(s->n_chain_blocks > 0 ? n : 0, 0);
    for (int b = 0; b < s->n_chain_blocks; b++) {
        const int start = s->chain[3 * b], cnt = s->chain[3 * b + 1], len = s->chain[3 * b + 2];
        if (len < 3 || len > 0xFFFF) unsupported("CHAIN length must be in [3, 65535]");
        if (cnt < 0 || start < 0 || (long long)start + (long long)cnt * len > n) invalid("CHAIN block out of range");
        for (int i = start; i < start + cnt * len; i++) {
            if (chained[i]) unsupported("a bead belongs to two CHAIN records");
            chained[i] = 1;
        }
    }
    if (s->n_bonds < 0 || s->n_bends < 0 || s->n_balls < 0) invalid("negative BOND / BEND / BALL record count");
    if ((s->n_bonds > 0 && (!s->bond || !s->bond_const)) || (s->n_bends > 0 && (!s->bend || !s->bend_const)) ||
        (s->n_balls > 0 && (!s->ball || !s->ball_const)))
        invalid("BOND / BEND / BALL records without data");
    auto in_range = [&](const int32_t *t, int m) {
        for (int k = 0; k < m; k++)
            if (t[k] < 0 || t[k] >= n) invalid("a BOND / BEND / BALL record names a particle out of range");
        for (int k = 0; k < m; k++)
            for (int l = k + 1; l < m; l++)
                if (t[k] == t[l]) invalid("a BOND / BEND / BALL record repeats a particle");
    };
    for (int j = 0; j < s->n_bonds; j++) in_range(s->bond + 2 * j, 2);
    for (int j = 0; j < s->n_bends; j++) in_range(s->bend + 3 * j, 3);
    for (int j = 0; j < s->n_balls; j++) in_range(s->ball + 2 * j, 2);
}

// replicas of one context share the interaction constants, cutoff and time step
void validate_batch(const sm_system *s, int nrep)
{
    long long total = 0, blocks = 0;
    for (int r = 0; r < nrep; r++) {
        validate(&s[r]);
        total += s[r].n_particles;
        blocks += s[r].n_chain_blocks;
        if (r == 0) continue;
        const sm_system &a = s[0], &b = s[r];
        if (b.n_types != a.n_types || b.cutoff != a.cutoff || b.dt != a.dt)
            unsupported("replicas must share n_types, cutoff and dt");
        const size_t nt = 6 * (size_t)a.n_types * a.n_types;
        if (std::memcmp(a.fconst, b.fconst, nt * sizeof(double)) != 0 ||
            std::memcmp(a.uconst, b.uconst, nt * sizeof(double)) != 0)
            unsupported("replicas must share the two-body constant tables");
    }
    if (total > 0x7FFFFFFF) unsupported("more than 2^31-1 beads in one context");
    if (blocks > 0x8000) unsupported("too many CHAIN constant sets");
}

sm_ctx *create(const sm_system *s, int nrep)
{
    validate_batch(s, nrep);
    sm_ctx *c = new sm_ctx();
    try {
        c->nrep = nrep;
        c->rh.resize(nrep);
        int n = 0, nch = 0;
        for (int r = 0; r < nrep; r++) {
            c->rh[r].first = n;
            c->rh[r].count = s[r].n_particles;
            n += s[r].n_particles;
        }
        c->n = n;
        c->P.n = n;
        c->P.nrep = nrep;
        c->P.nT = s[0].n_types;
        c->P.cutoff = s[0].cutoff;
        c->P.dt = s[0].dt;
        HIPCHK(hipStreamCreate(&c->st));
        // the device's fixed scratch for the entry points that allocate nothing, looked up
        // once per device while it is current
        HIPCHK(hipGetDevice(&c->device));
        HIPCHK(noalloc_scratch_init(c->device));
        c->link.create(nrep);

        // chains: per-bead role table and per-chain list, replica after replica
        std::vector<int2> perBead(n, make_int2(-1, 0));
        std::vector<int2> list;
        std::vector<double4> ccD;
        for (int r = 0; r < nrep; r++) {
            const int off = c->rh[r].first;
            c->rh[r].cfirst = (int)list.size();
            for (int b = 0; b < s[r].n_chain_blocks; b++) {
                // ranges, lengths, overlaps and the constant-set count checked by validate_batch()
                const int start = s[r].chain[3 * b], cnt = s[r].chain[3 * b + 1], len = s[r].chain[3 * b + 2];
                const double *cc = s[r].chain_const + 4 * b;
                const int cid = (int)ccD.size();
                ccD.push_back(make_double4(cc[0], cc[1], cc[2], cc[3]));
                for (int k = 0; k < cnt; k++) {
                    const int st0 = off + start + k * len;
                    list.push_back(make_int2(st0, len | (cid << 16)));
                    for (int j = 0; j < len; j++) perBead[st0 + j] = make_int2(st0, len | (cid << 16));
                }
            }
            c->rh[r].ccount = (int)list.size() - c->rh[r].cfirst;
        }
        nch = (int)list.size();
        c->nchains = nch;

        // generic BOND / BEND records: each record listed under each of its beads
        std::vector<int> gcount(n + 1, 0);
        std::vector<GenEnt> grec;
        std::vector<double2> gcst;
        for (int r = 0; r < nrep; r++) {
            // indices checked by validate()
            const int off = c->rh[r].first;
            auto bead = [&](int32_t b) { return off + b; };
            c->rh[r].nbond = s[r].n_bonds;
            c->rh[r].nbend = s[r].n_bends;
            for (int j = 0; j < s[r].n_bonds; j++) {
                grec.push_back(GenEnt{0, bead(s[r].bond[2 * j]), bead(s[r].bond[2 * j + 1]), -1});
                gcst.push_back(make_double2(s[r].bond_const[2 * j], s[r].bond_const[2 * j + 1]));
            }
            for (int j = 0; j < s[r].n_balls; j++) {
                grec.push_back(GenEnt{2, bead(s[r].ball[2 * j]), bead(s[r].ball[2 * j + 1]), -1});
                gcst.push_back(make_double2(s[r].ball_const[2 * j], s[r].ball_const[2 * j + 1]));
            }
            for (int j = 0; j < s[r].n_bends; j++) {
                grec.push_back(GenEnt{1, bead(s[r].bend[3 * j]), bead(s[r].bend[3 * j + 1]), bead(s[r].bend[3 * j + 2])});
                gcst.push_back(make_double2(s[r].bend_const[2 * j], s[r].bend_const[2 * j + 1]));
            }
        }
        std::vector<int> gptrH;
        std::vector<GenEnt> gentH;
        std::vector<double2> gcstH;
        if (!grec.empty()) {
            auto members = [](const GenEnt &g, int out[3]) {
                out[0] = g.p1;
                out[1] = g.p2;
                out[2] = g.p3;
                return g.kind == 1 ? 3 : 2;
            };
            for (const GenEnt &g : grec) {
                int mb[3];
                const int m = members(g, mb);
                for (int k = 0; k < m; k++) gcount[mb[k] + 1]++;
            }
            gptrH.assign(n + 1, 0);
            for (int i = 0; i < n; i++) gptrH[i + 1] = gptrH[i] + gcount[i + 1];
            gentH.resize(gptrH[n]);
            gcstH.resize(gptrH[n]);
            std::vector<int> fill(gptrH.begin(), gptrH.end() - 1);
            for (size_t e = 0; e < grec.size(); e++) {
                int mb[3];
                const int m = members(grec[e], mb);
                for (int k = 0; k < m; k++) {
                    gentH[fill[mb[k]]] = grec[e];
                    gcstH[fill[mb[k]]++] = gcst[e];
                }
            }
        }

        // host staging
        std::vector<Bead> hb(n);
        std::vector<float4> hv(n), ha(n);
        std::vector<DevRep> hr(nrep);
        for (int r = 0; r < nrep; r++) {
            const sm_system &q = s[r];
            const int off = c->rh[r].first;
            for (int i = 0; i < q.n_particles; i++) {
                const size_t k = 3 * (size_t)i;
                Bead &b = hb[off + i];
                b.x = q.pos[k];
                b.y = q.pos[k + 1];
                b.z = q.pos[k + 2];
                b.type = q.type[i];
                b.rep = r;
                hv[off + i] = make_float4((float)q.vel[k], (float)q.vel[k + 1], (float)q.vel[k + 2], 0.f);
                ha[off + i] = q.acc ? make_float4((float)q.acc[k], (float)q.acc[k + 1], (float)q.acc[k + 2], 0.f)
                                    : make_float4(0.f, 0.f, 0.f, 0.f);
            }
            DevRep &R = hr[r];
            std::memset(&R, 0, sizeof R);
            for (int d = 0; d < 3; d++) {
                R.L[d] = q.box[d];
                R.nc[d] = (int)(q.box[d] / q.cutoff);
                R.cs[d] = q.box[d] / R.nc[d];
                R.scale[d] = 1.0;
            }
            R.first = c->rh[r].first;
            R.count = c->rh[r].count;
            R.cfirst = c->rh[r].cfirst;
            R.ccount = c->rh[r].ccount;
            R.seed = q.seed;
            R.temperature = q.temperature;
            R.gamma = q.gamma;
            const double Ts = q.sigma_temperature > 0 ? q.sigma_temperature : q.temperature;
            R.sigma = std::sqrt((6.0 * Ts * q.gamma) / q.dt);
            R.sigma_fixed = q.sigma_temperature > 0 ? 1 : 0;
            R.delta_lxy = q.delta_lxy;
            R.tension = q.tension;
            c->boxL.insert(c->boxL.end(), q.box, q.box + 3);
            c->deltaL.push_back(q.delta_lxy);
            if (q.delta_lxy != 0) c->any_mc = true;
        }
        const int nT = s[0].n_types;
        const size_t nconst = 6 * (size_t)nT * nT;
        c->hfconst.assign(s[0].fconst, s[0].fconst + nconst);
        c->huconst.assign(s[0].uconst, s[0].uconst + nconst);
        c->P.asym = tables_asymmetric(c->hfconst, c->huconst, nT) ? 1 : 0;
        const std::vector<float> fF = pair_table(c->hfconst, c->huconst, nT, s[0].cutoff);
        c->hcconst = ccD;

        // segment tiles: beads (molecule order == sorted order per replica) and chains
        std::vector<int> bb(nrep), bl(nrep), cb(nrep), cl(nrep);
        for (int r = 0; r < nrep; r++) {
            bb[r] = c->rh[r].first; bl[r] = c->rh[r].count;
            cb[r] = c->rh[r].cfirst; cl[r] = c->rh[r].ccount;
        }
        const SegHost tb = make_tiles(bb, bl), tc = make_tiles(cb, cl);

        c->win_ok = nrep == 1 && sortw_fits(n);
        c->sort_mode = n >= 1000000 ? 1 : (c->win_ok ? 2 : 0);
        c->hist_words = sort_scratch_words(n, 4) + sortw_words(n, sortw_fits(n));
        // Every buffer whose size stays, in one allocation: each of some 50 cost 10 us and, past the
        // runtime's cache of freed memory, 250 us more to free.  Twice over one list: its size, then
        // the addresses; what starts as zeros comes last and has one clear.
        size_t zeros_at = 0, bytes = 0;
        for (int pass = 0; pass < 2; pass++) {
            if (pass) c->slab = dalloc<char>(bytes);
            size_t at = 0;
            const auto take = [&](auto *&p, size_t count) {
                using T = std::remove_reference_t<decltype(*p)>;
                if (pass) p = reinterpret_cast<T *>(c->slab + at);
                at += (sizeof(T) * std::max<size_t>(count, 1) + 255) / 256 * 256;
            };
            for (Bead **p : {&c->beads, &c->sbeads, &c->beads_alt}) take(*p, n);
            for (float4 **p : {&c->vel, &c->acc, &c->fscratch}) take(*p, n);
            for (uint32_t **p : {&c->k0, &c->v0, &c->k1, &c->v1, &c->kidx[0], &c->kidx[1], &c->sk[0], &c->sk[1], &c->sv[0],
                                 &c->sv[1], &c->mbefore})
                take(*p, n);
            if (sortw_fits(n))
                for (uint32_t **p : {&c->k2, &c->v2}) take(*p, n);
            take(c->cnt_b, move_blocks(n));
            take(c->cnt_i, move_tiles(n));
            take(c->cnt_s, move_tiles(n));
            take(c->mflags, ((size_t)n + 63) / 64);
            take(c->mcount, 1);
            take(c->reps, nrep);
            take(c->glob, 1);
            take(c->fconstF, fF.size());
            take(c->uconstD, nconst);
            take(c->fconstD, nconst);
            take(c->chainPerBead, n);
            take(c->chainList, list.size());
            take(c->cconstD, ccD.size());
            take(c->ebead, n);
            take(c->edelta, n);
            take(c->dres, 8 * (size_t)nrep);
            take(c->dcounts, n);
            take(c->dnp, 1);
            if (!gentH.empty()) {
                take(c->gptr, gptrH.size());
                take(c->gent, gentH.size());
                take(c->gconstD, gcstH.size());
            }
            for (auto [S, h] : {std::make_pair(&c->segB, &tb), std::make_pair(&c->segC, &tc)}) {
                take(S->tile, h->tile.size());
                take(S->rep_first, h->rep_first.size());
                take(S->tilesum, kSumCols * h->tile.size());
            }
            zeros_at = at;
            take(c->fpair, n);
            for (uint32_t **p : {&c->hist[0], &c->hist[1]}) take(*p, c->hist_words);
            if (c->win_ok) take(c->wdesc, 16);
            if (sortw_fits(n))
                for (uint32_t **p : {&c->counted[0], &c->counted[1]}) take(*p, n);
            for (SegTiles *S : {&c->segB, &c->segC}) take(S->ticket, (size_t)kTicketWords * nrep);
            bytes = at;
        }
        c->beads_home = c->beads;
        HIPCHK(hipMemsetAsync(c->slab + zeros_at, 0, bytes - zeros_at, c->st));
        auto upseg = [&](SegTiles &S, const SegHost &h) {
            S.ntiles = (int)h.tile.size();
            if (!h.tile.empty())
                HIPCHK(hipMemcpyAsync(S.tile, h.tile.data(), sizeof(int4) * h.tile.size(), hipMemcpyHostToDevice, c->st));
            HIPCHK(hipMemcpyAsync(S.rep_first, h.rep_first.data(), sizeof(int) * h.rep_first.size(),
                                  hipMemcpyHostToDevice, c->st));
        };
        upseg(c->segB, tb);
        upseg(c->segC, tc);

        DevGlobal g{};
        hipStream_t st = c->st;
        HIPCHK(hipMemcpyAsync(c->beads, hb.data(), sizeof(Bead) * n, hipMemcpyHostToDevice, st));
        HIPCHK(hipMemcpyAsync(c->vel, hv.data(), sizeof(float4) * n, hipMemcpyHostToDevice, st));
        HIPCHK(hipMemcpyAsync(c->acc, ha.data(), sizeof(float4) * n, hipMemcpyHostToDevice, st));
        HIPCHK(hipMemcpyAsync(c->reps, hr.data(), sizeof(DevRep) * nrep, hipMemcpyHostToDevice, st));
        HIPCHK(hipMemcpyAsync(c->glob, &g, sizeof g, hipMemcpyHostToDevice, st));
        HIPCHK(hipMemcpyAsync(c->fconstF, fF.data(), sizeof(float) * fF.size(), hipMemcpyHostToDevice, st));
        HIPCHK(hipMemcpyAsync(c->uconstD, s[0].uconst, sizeof(double) * nconst, hipMemcpyHostToDevice, st));
        HIPCHK(hipMemcpyAsync(c->fconstD, s[0].fconst, sizeof(double) * nconst, hipMemcpyHostToDevice, st));
        HIPCHK(hipMemcpyAsync(c->chainPerBead, perBead.data(), sizeof(int2) * n, hipMemcpyHostToDevice, st));
        if (!gentH.empty()) {
            HIPCHK(hipMemcpyAsync(c->gptr, gptrH.data(), sizeof(int) * gptrH.size(), hipMemcpyHostToDevice, st));
            HIPCHK(hipMemcpyAsync(c->gent, gentH.data(), sizeof(GenEnt) * gentH.size(), hipMemcpyHostToDevice, st));
            HIPCHK(hipMemcpyAsync(c->gconstD, gcstH.data(), sizeof(double2) * gcstH.size(), hipMemcpyHostToDevice,
                                  st));
        }
        if (!list.empty()) {
            HIPCHK(hipMemcpyAsync(c->chainList, list.data(), sizeof(int2) * list.size(), hipMemcpyHostToDevice, st));
            HIPCHK(hipMemcpyAsync(c->cconstD, ccD.data(), sizeof(double4) * ccD.size(), hipMemcpyHostToDevice, st));
        }
        c->launch_rules();
        c->ensure_capacity(0);
        HIPCHK(hipStreamSynchronize(st));
    } catch (...) {
        delete c;
        throw;
    }
    return c;
}

}  // namespace

// ---------------------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------------------
extern "C" {

const char *sm_last_error(void) { return g_err.c_str(); }
const char *sm_version(void) { return "softmold-mi355x 0.2 (gfx950)"; }

int sm_create(const sm_system *s, sm_ctx **out)
{
    if (!out) {
        g_err = "null output pointer";
        return SM_ERR_INVALID;
    }
    *out = nullptr;
    return guarded([&] { *out = create(s, 1); });
}

int sm_create_batch(const sm_system *systems, int32_t n_replicas, sm_ctx **out)
{
    if (!out) {
        g_err = "null output pointer";
        return SM_ERR_INVALID;
    }
    *out = nullptr;
    return guarded([&] {
        if (!systems || n_replicas < 1) invalid("need at least one replica");
        *out = create(systems, n_replicas);
    });
}

int sm_destroy(sm_ctx *c)
{
    return guarded([&] { delete c; });
}

int sm_replicas(sm_ctx *c, int32_t *n_replicas, int32_t *first, int32_t *count)
{
    return guarded([&] {
        if (!c) invalid("null context");
        if (n_replicas) *n_replicas = c->nrep;
        for (int r = 0; r < c->nrep; r++) {
            if (first) first[r] = c->rh[r].first;
            if (count) count[r] = c->rh[r].count;
        }
    });
}

int sm_sync(sm_ctx *c)
{
    return guarded([&] {
        if (!c) invalid("null context");
        c->check_flags();   // waits for the stream
    });
}

int sm_download_state(sm_ctx *c, double *pos, double *vel, double *acc, double *box)
{
    return guarded([&] {
        if (!c) invalid("null context");
        // positions, velocities and accelerations in one pass; the boxes and flags with them
        const PackSrc src{c->beads, c->vel, c->acc};
        int flags;
        if (pos || vel || acc)
            flags = c->link.fetch_beads(c->st, c->n, src, pos, vel, acc, c->glob, c->reps, c->nrep, c->boxL.data());
        else
            flags = c->link.fetch_boxes(c->st, c->glob, c->reps, c->nrep, c->boxL.data());
        c->moves_since = 0;
        if (box) std::copy(c->boxL.begin(), c->boxL.end(), box);
        c->check_bits(flags);
    });
}

int sm_upload_state(sm_ctx *c, const double *pos, const double *vel, const double *acc, const double *box)
{
    return guarded([&] {
        if (!c) invalid("null context");
        const int n = c->n;
        std::vector<double> L(c->boxL.size());
        if (box) {
            std::copy(box, box + L.size(), L.begin());
            for (const double l : L) {
                if (!(l > 0)) invalid("box lengths must be positive");
                if ((int)(l / c->P.cutoff) < 3) unsupported("fewer than 3 cells along an axis");
            }
        } else if (pos) {
            c->know_boxes();
            L = c->boxL;
        }
        if (pos) {
            for (int r = 0; r < c->nrep; r++)
                for (int i = c->rh[r].first; i < c->rh[r].first + c->rh[r].count; i++)
                    for (int d = 0; d < 3; d++) {
                        const double p = pos[3 * (size_t)i + d];
                        if (!(p >= 0 && p <= L[3 * (size_t)r + d]))
                            invalid("particle " + std::to_string(i) + " position is out of bounds");
                    }
        }
        if (box) {   // the cells that it needs, before anything changes
            struct Tried {
                sm_ctx *c;
                std::vector<double> was;
                long long since;
                ~Tried()
                {
                    c->boxL.swap(was);
                    c->moves_since = since;
                }
            } tried{c, c->boxL, c->moves_since};
            c->boxL = L;
            c->moves_since = 0;
            c->ensure_capacity(0);
        }
        if (pos || box) c->forget_keys();
        if (pos) c->link.send_positions(c->st, n, pos, c->beads);
        auto up3 = [&](float4 *dst, const double *src) {
            std::vector<float4> h(n);
            for (int i = 0; i < n; i++)
                h[i] = make_float4((float)src[3 * (size_t)i], (float)src[3 * (size_t)i + 1], (float)src[3 * (size_t)i + 2], 0.f);
            HIPCHK(hipMemcpyAsync(dst, h.data(), sizeof(float4) * n, hipMemcpyHostToDevice, c->st));
            HIPCHK(hipStreamSynchronize(c->st));
        };
        if (vel) up3(c->vel, vel);
        if (acc) up3(c->acc, acc);
        if (box) {
            std::vector<DevRep> hr = c->read_reps();
            for (int r = 0; r < c->nrep; r++)
                for (int d = 0; d < 3; d++) {
                    hr[r].L[d] = L[3 * (size_t)r + d];
                    hr[r].nc[d] = (int)(hr[r].L[d] / c->P.cutoff);
                    hr[r].cs[d] = hr[r].L[d] / hr[r].nc[d];
                }
            c->write_reps(hr);
            c->boxL = L;
            c->moves_since = 0;
            c->launch_rules();
            c->count_again();
        }
    });
}

int sm_set_temperature(sm_ctx *c, double T)
{
    return guarded([&] {
        if (!c) invalid("null context");
        if (!(T >= 0)) invalid("temperature must be >= 0");
        std::vector<DevRep> hr = c->read_reps();
        for (auto &R : hr) {
            R.temperature = T;
            if (!R.sigma_fixed) R.sigma = std::sqrt((6.0 * T * R.gamma) / c->P.dt);
        }
        c->write_reps(hr);
    });
}

int sm_init_forces(sm_ctx *c)
{
    return guarded([&] {
        if (!c) invalid("null context");
        c->build(0, 0);
        c->pair_force();
        c->bonded(KICK_INIT, nullptr);
        c->check_launch();
    });
}

int sm_second_half(sm_ctx *c)
{
    return guarded([&] {
        if (!c) invalid("null context");
        launch_second(c->st, c->n, c->beads, c->acc, c->vel, (float)(c->P.dt * 0.5));
        c->check_launch();
    });
}

int sm_step_first(sm_ctx *c, int64_t step)
{
    return guarded([&] {
        if (!c) invalid("null context");
        if (step < 0) invalid("negative step index");
        // the cell table must hold this step's box move before the keys are computed
        if (c->mc_step(step)) c->ensure_capacity(1);
        c->step_first(step);
        c->check_launch();
    });
}

int sm_step_finish(sm_ctx *c, int64_t step, double *measure)
{
    return guarded([&] {
        if (!c) invalid("null context");
        const bool mc = c->mc_step(step);
        c->step_finish(measure != nullptr, mc);
        c->check_launch();
        if (measure) c->fetch(c->meas_dev(), 3 * (size_t)c->nrep, measure);
    });
}

int sm_run(sm_ctx *c, int64_t first, int32_t nsteps)
{
    return guarded([&] {
        if (!c) invalid("null context");
        if (nsteps < 0 || first < 0) invalid("negative step index or count");
        c->run(first, nsteps);
        c->check_launch();
    });
}

int sm_mc_stats(sm_ctx *c, int64_t *trials, int64_t *accepted)
{
    return guarded([&] {
        if (!c) invalid("null context");
        std::vector<DevRep> hr = c->read_reps();
        for (int r = 0; r < c->nrep; r++) {
            if (trials) trials[r] = hr[r].trials;
            if (accepted) accepted[r] = hr[r].accepted;
        }
    });
}

int sm_mc_hist(sm_ctx *c, int32_t replica, int32_t cap, double *accepted, double *rejected, int32_t *n_out)
{
    return guarded([&] {
        if (!c || !n_out || cap < 0) invalid("bad argument");
        if (replica < 0 || replica >= c->nrep) invalid("replica index out of range");
        std::vector<DevRep> hr = c->read_reps();
        const DevRep &R = hr[replica];
        const double dL = R.delta_lxy;
        int nb = 0;
        if (dL != 0) nb = (int)(2.0 * dL / (dL / 101.0)) + 1;
        if (nb > kHistBins) nb = kHistBins;
        *n_out = nb;
        const int m = nb < cap ? nb : cap;
        for (int i = 0; i < m; i++) {
            if (accepted) accepted[i] = R.hist_accept[i];
            if (rejected) rejected[i] = R.hist_reject[i];
        }
    });
}

int sm_measure(sm_ctx *c, double *out)
{
    return guarded([&] {
        if (!c || !out) invalid("null argument");
        c->build(0, kStepKeep);
        c->measure_device();
        c->check_launch();
        c->fetch(c->meas_dev(), 3 * (size_t)c->nrep, out);
    });
}

int sm_bond_stats(sm_ctx *c, double *out)
{
    return guarded([&] {
        if (!c || !out) invalid("null argument");
        const int R = c->nrep;
        std::vector<double> h((size_t)4 * R, 0.0);
        if (c->gptr) {
            for (int what = 0; what < 4; what++) {
                launch_gen_stats(c->st, c->n, c->gen(), c->beads, c->reps, what, c->ebead);
                SumArgs a = c->sums(c->ebead, c->dres + what);
                a.stride = 4;
                launch_sums(c->st, SUM_COLUMN, a);
            }
            c->check_launch();
            (void)c->link.fetch(c->st, c->glob, c->dres, h.size(), h.data());
        }
        for (int r = 0; r < R; r++) {
            // the divisions on the host, as the reference writes them: lBond / nBond even
            // when nBond is 0; the bend sums divided only when nBend > 1
            const int nb = c->rh[r].nbond, ne = c->rh[r].nbend;
            double *o = out + 4 * (size_t)r;
            const double zero = 0.0;
            o[0] = h[4 * r] / (nb ? (double)nb : zero);
            o[1] = h[4 * r + 1];
            o[2] = h[4 * r + 2];
            o[3] = h[4 * r + 3];
            if (ne > 1)
                for (int k = 1; k < 4; k++) o[k] /= (double)ne;
        }
    });
}

// the replicas' radii from their heads: `work` holds 8 doubles a replica, the radii last
static void vesicle_radius(sm_ctx *c, int32_t head_type, double *work, double *radius)
{
    SumArgs a = c->sums(nullptr, work);
    a.radius = work + 7 * (size_t)c->nrep;
    a.head = head_type;
    launch_sums(c->st, SUM_HEADS, a);
    launch_sums(c->st, SUM_HEAD_DIST, a);
    c->check_launch();
    (void)c->link.fetch(c->st, c->glob, a.radius, (size_t)c->nrep, radius);
}

int sm_vesicle_radius(sm_ctx *c, int32_t head_type, double *radius)
{
    return guarded([&] {
        if (!c || !radius) invalid("null argument");
        vesicle_radius(c, head_type, c->dres, radius);
    });
}

int sm_vesicle_radius_noalloc(sm_ctx *c, int32_t head_type, double *radius)
{
    return guarded([&] {
        if (!c || !radius) invalid("null argument");
        const int R = c->nrep;
        if (R > kNoAllocMaxReplicas)
            unsupported("sm_vesicle_radius_noalloc: " + std::to_string(R) + " replicas exceed its fixed scratch of " +
                        std::to_string(kNoAllocMaxReplicas) + "; use sm_vesicle_radius");
        double *w = noalloc_scratch(c->device);
        if (!w) throw ApiError(SM_ERR_STATE, "fixed scratch of this device was not set up");
        // every word read is written first by this call, so nothing is cleared
        vesicle_radius(c, head_type, w, radius);
    });
}

int sm_compute_forces(sm_ctx *c, double *pair_out, double *chain_out)
{
    return guarded([&] {
        if (!c) invalid("null context");
        c->build(0, kStepKeep);
        c->pair_force();
        c->bonded(KICK_NONE, c->fscratch);
        c->check_launch();
        if (pair_out || chain_out) {
            c->check_bits(c->link.fetch_beads(c->st, c->n, PackSrc{nullptr, c->fpair, c->fscratch}, nullptr, pair_out,
                                              chain_out, c->glob, c->reps, c->nrep, nullptr));
        } else {
            c->check_flags();
        }
    });
}

int sm_cell_keys(sm_ctx *c, int32_t *keys)
{
    return guarded([&] {
        if (!c || !keys) invalid("null argument");
        c->first_and_keys(0, kStepKeep, false);   // no sort follows: leave its histograms alone
        c->check_launch();
        std::vector<uint32_t> h(c->n);
        HIPCHK(hipMemcpyAsync(h.data(), c->k0, sizeof(uint32_t) * c->n, hipMemcpyDeviceToHost, c->st));
        HIPCHK(hipStreamSynchronize(c->st));
        for (int r = 0; r < c->nrep; r++)
            for (int i = c->rh[r].first; i < c->rh[r].first + c->rh[r].count; i++)
                keys[i] = (int32_t)((long long)h[i] - c->rh[r].cellbase);
        c->check_flags();
    });
}

int sm_pair_count(sm_ctx *c, int32_t *counts, int64_t *total)
{
    return guarded([&] {
        if (!c) invalid("null context");
        c->build(0, kStepKeep);
        launch_pair_gather(c->st, c->P, c->chunk, GATHER_COUNT, c->sbeads, c->skey(), c->sidx(), c->cstart, c->cend,
                           c->reps, c->fconstF, c->uconstD, nullptr, c->dcounts, nullptr, nullptr, 0);
        c->check_launch();
        std::vector<int32_t> h(c->n);
        HIPCHK(hipMemcpyAsync(h.data(), c->dcounts, sizeof(int32_t) * c->n, hipMemcpyDeviceToHost, c->st));
        HIPCHK(hipStreamSynchronize(c->st));
        long long t = 0;
        for (int i = 0; i < c->n; i++) t += h[i];
        if (counts) std::memcpy(counts, h.data(), sizeof(int32_t) * c->n);
        if (total) *total = t / 2;
        c->check_flags();
    });
}

int sm_force_pair_count(sm_ctx *c, int32_t *counts, int64_t *total)
{
    return guarded([&] {
        if (!c) invalid("null context");
        if (c->pair_variant != 0) unsupported("the force pair count follows the one-phase force kernel (pair_variant 0)");
        c->build(0, kStepKeep);
        launch_pair_gather(c->st, c->P, c->chunk, GATHER_FCOUNT, c->sbeads, c->skey(), c->sidx(), c->cstart, c->cend,
                           c->reps, c->fconstF, c->fconstD, nullptr, c->dcounts, nullptr, nullptr, 0);
        c->check_launch();
        std::vector<int32_t> h(c->n);
        HIPCHK(hipMemcpyAsync(h.data(), c->dcounts, sizeof(int32_t) * c->n, hipMemcpyDeviceToHost, c->st));
        HIPCHK(hipStreamSynchronize(c->st));
        long long t = 0;
        for (int i = 0; i < c->n; i++) t += h[i];
        if (counts) std::memcpy(counts, h.data(), sizeof(int32_t) * c->n);
        if (total) *total = t / 2;
        c->check_flags();
    });
}

int sm_pair_list(sm_ctx *c, int32_t *pairs, int64_t cap, int64_t *n_out)
{
    return guarded([&] {
        if (!c || cap < 0) invalid("bad argument");
        if (cap > c->pairs_cap) {
            dfree(c->dpairs);
            c->dpairs = dalloc<int>(2 * (size_t)cap);
            c->pairs_cap = cap;
        }
        c->build(0, kStepKeep);
        HIPCHK(hipMemsetAsync(c->dnp, 0, sizeof(unsigned long long), c->st));
        launch_pair_gather(c->st, c->P, c->chunk, GATHER_LIST, c->sbeads, c->skey(), c->sidx(), c->cstart, c->cend,
                           c->reps, c->fconstF, c->uconstD, nullptr, c->dcounts, c->dpairs, c->dnp, cap);
        c->check_launch();
        unsigned long long np = 0;
        HIPCHK(hipMemcpyAsync(&np, c->dnp, sizeof np, hipMemcpyDeviceToHost, c->st));
        HIPCHK(hipStreamSynchronize(c->st));
        const long long keep = std::min<long long>((long long)np, cap);
        if (pairs && keep > 0) {
            HIPCHK(hipMemcpyAsync(pairs, c->dpairs, sizeof(int32_t) * 2 * (size_t)keep, hipMemcpyDeviceToHost, c->st));
            HIPCHK(hipStreamSynchronize(c->st));
        }
        if (n_out) *n_out = (int64_t)np;
        c->check_flags();
    });
}

int sm_potential_delta(sm_ctx *c, const double *scale, double *du_pair, double *du_chain)
{
    return guarded([&] {
        if (!c || !scale) invalid("null argument");
        c->link.send_scale(c->st, c->reps, c->nrep, scale);
        c->build(0, kStepKeep);
        if (c->mc_fused) {   // the traversal a box-move step runs (it also leaves the pair forces)
            c->pair_force_du();
            c->delta_sums();
        } else {
            c->delta_device();
        }
        c->check_launch();
        std::vector<double> h(2 * (size_t)c->nrep);
        const int flags = c->link.fetch(c->st, c->glob, c->du_dev(), h.size(), h.data());
        for (int r = 0; r < c->nrep; r++) {
            if (du_pair) du_pair[r] = h[2 * r];
            if (du_chain) du_chain[r] = h[2 * r + 1];
        }
        c->check_bits(flags);
    });
}

int sm_tune(sm_ctx *c, const char *knob, int32_t value)
{
    return guarded([&] {
        if (!c || !knob) invalid("null argument");
        if (std::strcmp(knob, "pair_chunk") == 0) {
            if (value < 1 || value > 4096) invalid("pair_chunk must be in [1, 4096]");
            c->chunk = c->echunk = value;
            c->chunk_set = true;
        } else if (std::strcmp(knob, "pair_variant") == 0) {
            if (value < 0 || value > 1) invalid("pair_variant must be 0 or 1");
            c->pair_variant = value;
        } else if (std::strcmp(knob, "graph") == 0) {
            if (value < 0 || value > 1) invalid("graph must be 0 or 1");
            c->use_graph = value != 0;
        } else if (std::strcmp(knob, "sort_mode") == 0) {
            if (value < 0 || value > 2) invalid("sort_mode must be 0, 1 or 2");
            if (value == 2 && !c->win_ok) invalid("sort_mode 2 needs a single replica of at most 524288 beads");
            c->forget_keys();
            c->count_again();
            c->sort_mode = value;
            c->order_valid = false;
        } else if (std::strcmp(knob, "mc_fused") == 0) {
            if (value < 0 || value > 1) invalid("mc_fused must be 0 or 1");
            c->mc_fused = value != 0;
        } else {
            invalid(std::string("unknown knob ") + knob);
        }
        c->drop_graph();
    });
}

int sm_tune_get(sm_ctx *c, const char *knob, int32_t *value)
{
    return guarded([&] {
        if (!c || !knob || !value) invalid("null argument");
        if (std::strcmp(knob, "pair_chunk") == 0) *value = c->chunk;
        else if (std::strcmp(knob, "energy_chunk") == 0) *value = c->echunk;
        else if (std::strcmp(knob, "pair_variant") == 0) *value = c->pair_variant;
        else if (std::strcmp(knob, "graph") == 0) *value = c->use_graph ? 1 : 0;
        else if (std::strcmp(knob, "sort_mode") == 0) *value = c->sort_mode;
        else if (std::strcmp(knob, "mc_fused") == 0) *value = c->mc_fused ? 1 : 0;
        else if (std::strcmp(knob, "sort_window_path") == 0) *value = c->win_last && c->counted_last() ? 1 : 0;
        else if (std::strcmp(knob, "sort_count_path") == 0) *value = c->counted_last() ? 1 : 0;
        else invalid(std::string("unknown knob ") + knob);
    });
}

int sm_autotune(sm_ctx *c, int32_t steps, double *best_ms_per_step)
{
    return guarded([&] {
        if (!c) invalid("null context");
        if (steps < 8 || steps > 100000) invalid("steps per trial must be in [8, 100000]");
        if (c->prof) invalid("profiling is on");
        const DevGlobal entry = c->read_glob();
        const long long s0 = entry.step + 1;
        // every trial starts from the same state; reserve cells for the trials' moves
        // first so that no trial moves the cell bases
        long long moves = 0;
        for (long long s = s0; s < s0 + steps; s++)
            if (c->mc_step(s)) moves++;
        c->ensure_capacity(moves);
        const int n = c->n;
        Bead *b0 = dalloc<Bead>(n);
        float4 *v0 = dalloc<float4>(n), *a0 = dalloc<float4>(n);
        DevRep *r0 = dalloc<DevRep>(c->nrep);
        DevGlobal *g0 = dalloc<DevGlobal>(1);
        hipEvent_t e0 = nullptr, e1 = nullptr;
        auto cleanup = [&] {
            dfree(b0); dfree(v0); dfree(a0); dfree(r0); dfree(g0);
            if (e0) (void)hipEventDestroy(e0);
            if (e1) (void)hipEventDestroy(e1);
        };
        try {
            hipStream_t st = c->st;
            auto copy = [&](void *d, const void *s, size_t bytes) {
                HIPCHK(hipMemcpyAsync(d, s, bytes, hipMemcpyDeviceToDevice, st));
            };
            auto save = [&] {
                copy(b0, c->beads, sizeof(Bead) * n); copy(v0, c->vel, sizeof(float4) * n);
                copy(a0, c->acc, sizeof(float4) * n); copy(r0, c->reps, sizeof(DevRep) * c->nrep);
                copy(g0, c->glob, sizeof(DevGlobal));
            };
            auto restore = [&] {
                c->forget_boxes();
                copy(c->beads, b0, sizeof(Bead) * n); copy(c->vel, v0, sizeof(float4) * n);
                copy(c->acc, a0, sizeof(float4) * n); copy(c->reps, r0, sizeof(DevRep) * c->nrep);
                copy(c->glob, g0, sizeof(DevGlobal));
                c->fallbacks_seen = entry.fallbacks;
                c->counted_builds = 0;
            };
            HIPCHK(hipEventCreate(&e0));
            HIPCHK(hipEventCreate(&e1));
            save();
            // launch shapes that leave every result bit-identical: the chunk of the one-phase
            // pair kernel (a cell is processed the same way whatever chunk holds it), the
            // graph replay (the same kernels on the same stream) and the sort mode (both
            // give the same order)
            struct Cand { int chunk, variant, graph, sort; };
            std::vector<Cand> cands;
            for (int ch : {2, 4, 8, 16, 32, 64}) cands.push_back({ch, 0, 1, c->sort_mode});
            double best = 1e300;
            Cand bestc{c->chunk, c->pair_variant, c->use_graph ? 1 : 0, c->sort_mode};
            auto trial = [&](const Cand &k) {
                c->chunk = c->echunk = k.chunk;   // as sm_tune sets them
                c->pair_variant = k.variant;
                c->use_graph = k.graph != 0;
                if (c->sort_mode != k.sort) {
                    c->sort_mode = k.sort;
                    c->order_valid = false;
                    c->count_again();
                }
                c->drop_graph();
                restore();
                c->run(s0, 8);          // warm: first launches, graph capture
                const bool counted = c->count_now();
                c->check_flags();
                restore();
                if (counted != c->count_now()) {   // it stopped counting: warm again
                    c->run(s0, 8);
                    restore();
                }
                HIPCHK(hipEventRecord(e0, st));
                c->run(s0, steps);
                HIPCHK(hipEventRecord(e1, st));
                HIPCHK(hipEventSynchronize(e1));
                c->check_launch();
                float ms = 0.f;
                HIPCHK(hipEventElapsedTime(&ms, e0, e1));
                const double per = ms / steps;
                if (per < best) {
                    best = per;
                    bestc = k;
                }
            };
            for (const auto &k : cands) trial(k);
            const Cand b0 = bestc;
            for (int m = 0; m <= 2; m++)   // the other sort modes
                if (m != b0.sort && (m != 2 || c->win_ok)) trial({b0.chunk, b0.variant, 1, m});
            trial({bestc.chunk, bestc.variant, 0, bestc.sort});       // is the graph worth it here
            c->chunk = c->echunk = bestc.chunk;
            c->chunk_set = true;
            c->pair_variant = bestc.variant;
            c->use_graph = bestc.graph != 0;
            if (c->sort_mode != bestc.sort) {
                c->sort_mode = bestc.sort;
                c->order_valid = false;
                c->count_again();
            }
            c->drop_graph();
            restore();
            HIPCHK(hipStreamSynchronize(st));
            c->check_flags();
            if (best_ms_per_step) *best_ms_per_step = best;
        } catch (...) {
            (void)hipStreamSynchronize(c->st);
            cleanup();
            throw;
        }
        cleanup();
    });
}

}  // extern "C"

// ---------------------------------------------------------------------------------------
// interaction constants as adjoint parameters
// ---------------------------------------------------------------------------------------
namespace {

void check_pair(const sm_ctx *c, int a, int b)
{
    if (a < 0 || b < 0 || a >= c->P.nT || b >= c->P.nT) invalid("type index out of range");
}

// laradjiRevaleeFC / laradjiRevaleePC rows (potentials/laradjiRevalee.h:84-152) of the
// type pair (a, b) and (b, a) from Umin, Umax, keeping each row's r_m and r_c
void set_pair_rows(sm_ctx *c, int a, int b, double umin, double umax)
{
    const int nT = c->P.nT;
    for (int pass = 0; pass < 2; pass++) {
        const size_t row = 6 * (size_t)(pass ? b * nT + a : a * nT + b);
        double *F = &c->hfconst[row], *U = &c->huconst[row];
        const double rm = F[0], rc = F[3];
        F[1] = (2.0 * (umax - umin)) / (rm * rm);
        F[2] = 0;
        F[4] = (6.0 * umin) / ((rc - rm) * (rc - rm));
        F[5] = (6.0 * umin) / ((rc - rm) * (rc - rm) * (rc - rm));
        U[0] = rm;
        U[1] = (umax - umin) / (rm * rm);
        U[2] = umin;
        U[3] = rc;
        U[4] = (3.0 * umin) / ((rc - rm) * (rc - rm));
        U[5] = (2.0 * umin) / ((rc - rm) * (rc - rm) * (rc - rm));
    }
}

void upload_constants(sm_ctx *c)
{
    const size_t nt = c->hfconst.size();
    // a captured graph holds the pair kernels of the tables' symmetry
    const int asym = tables_asymmetric(c->hfconst, c->huconst, c->P.nT) ? 1 : 0;
    if (asym != c->P.asym) {
        c->P.asym = asym;
        c->drop_graph();
    }
    const std::vector<float> fF = pair_table(c->hfconst, c->huconst, c->P.nT, c->P.cutoff);
    HIPCHK(hipMemcpyAsync(c->fconstF, fF.data(), sizeof(float) * fF.size(), hipMemcpyHostToDevice, c->st));
    HIPCHK(hipMemcpyAsync(c->uconstD, c->huconst.data(), sizeof(double) * nt, hipMemcpyHostToDevice, c->st));
    HIPCHK(hipMemcpyAsync(c->fconstD, c->hfconst.data(), sizeof(double) * nt, hipMemcpyHostToDevice, c->st));
    if (!c->hcconst.empty())
        HIPCHK(hipMemcpyAsync(c->cconstD, c->hcconst.data(), sizeof(double4) * c->hcconst.size(),
                              hipMemcpyHostToDevice, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
}

// FP64 F table and the d/d(Umin), d/d(Umax) tables of the (a, b) rows
void upload_adjoint_tables(sm_ctx *c, int a, int b)
{
    const int nT = c->P.nT;
    const size_t nt = 6 * (size_t)nT * nT;
    std::vector<double> dF(2 * nt, 0.0), dU(2 * nt, 0.0);
    for (int pass = 0; pass < 2; pass++) {
        const size_t row = 6 * (size_t)(pass ? b * nT + a : a * nT + b);
        const double rm = c->hfconst[row], rc = c->hfconst[row + 3];
        const double w = rc - rm;
        double *Fmin = &dF[row], *Fmax = &dF[nt + row], *Umin = &dU[row], *Umax = &dU[nt + row];
        Fmin[1] = -2.0 / (rm * rm);
        Fmin[4] = 6.0 / (w * w);
        Fmin[5] = 6.0 / (w * w * w);
        Fmax[1] = 2.0 / (rm * rm);
        Umin[1] = -1.0 / (rm * rm);
        Umin[2] = 1.0;
        Umin[4] = 3.0 / (w * w);
        Umin[5] = 2.0 / (w * w * w);
        Umax[1] = 1.0 / (rm * rm);
    }
    if (!c->adjF) {
        c->adjF = dalloc<double>(nt);
        c->adjDF = dalloc<double>(2 * nt);
        c->adjDU = dalloc<double>(2 * nt);
    }
    HIPCHK(hipMemcpyAsync(c->adjF, c->hfconst.data(), sizeof(double) * nt, hipMemcpyHostToDevice, c->st));
    HIPCHK(hipMemcpyAsync(c->adjDF, dF.data(), sizeof(double) * 2 * nt, hipMemcpyHostToDevice, c->st));
    HIPCHK(hipMemcpyAsync(c->adjDU, dU.data(), sizeof(double) * 2 * nt, hipMemcpyHostToDevice, c->st));
}

// The tables sm_param_derivative runs the energy kernels with.  U is linear in each
// laradjiRevaleePC row's entries {r_m, C1, C2, r_c, C4, C5} with r_m and r_c fixed
// (laradjiRevalee.h:124-152), and those entries are linear in Umin and Umax, so the FP64
// potential gather run on a table whose (a, b) and (b, a) rows hold the entries'
// derivatives (every row keeping its r_m and r_c, every other coefficient 0) sums
// dU_pair/dUmin or dU_pair/dUmax.  harmonicP and bendP are linear in k_bond and k_bend
// (MD.h:422-431,769-789), so the CHAIN energy with (k_bond, k_bend) = (1, 0) or (0, 1) is
// dU_chain/dk_bond or dU_chain/dk_bend.  Depends only on r_m, r_c, l0 and the cos-theta
// term, which the fitting parameters leave alone; rebuilt when the pair changes.
void upload_param_derivative_tables(sm_ctx *c, int a, int b)
{
    if (c->pdU && c->pd_a == a && c->pd_b == b) return;
    const int nT = c->P.nT;
    const size_t nt = 6 * (size_t)nT * nT;
    std::vector<double> dU(2 * nt, 0.0);
    for (size_t row = 0; row < nt; row += 6)
        for (int p = 0; p < 2; p++) {
            dU[p * nt + row] = c->huconst[row];
            dU[p * nt + row + 3] = c->huconst[row + 3];
        }
    for (int pass = 0; pass < 2; pass++) {
        const size_t row = 6 * (size_t)(pass ? b * nT + a : a * nT + b);
        const double rm = c->huconst[row], rc = c->huconst[row + 3];
        const double w = rc - rm;
        double *Umin = &dU[row], *Umax = &dU[nt + row];
        Umin[1] = -1.0 / (rm * rm);
        Umin[2] = 1.0;
        Umin[4] = 3.0 / (w * w);
        Umin[5] = 2.0 / (w * w * w);
        Umax[1] = 1.0 / (rm * rm);
    }
    std::vector<double> dUmin(dU.begin(), dU.begin() + nt), dUmax(dU.begin() + nt, dU.end());
    const std::vector<float> t0 = pair_table(c->hfconst, dUmin, nT, c->P.cutoff);
    const std::vector<float> t1 = pair_table(c->hfconst, dUmax, nT, c->P.cutoff);
    std::vector<double4> cc;
    for (const double4 &k : c->hcconst) cc.push_back(make_double4(k.x, 1.0, k.z, 0.0));
    for (const double4 &k : c->hcconst) cc.push_back(make_double4(k.x, 0.0, k.z, 1.0));
    if (!c->pdU) {
        c->pdU = dalloc<double>(2 * nt);
        c->pd_tab = t0.size();
        c->pdTab = dalloc<float>(2 * c->pd_tab);
        c->pdC = dalloc<double4>(cc.size());
    }
    HIPCHK(hipMemcpyAsync(c->pdU, dU.data(), sizeof(double) * 2 * nt, hipMemcpyHostToDevice, c->st));
    HIPCHK(hipMemcpyAsync(c->pdTab, t0.data(), sizeof(float) * c->pd_tab, hipMemcpyHostToDevice, c->st));
    HIPCHK(hipMemcpyAsync(c->pdTab + c->pd_tab, t1.data(), sizeof(float) * c->pd_tab, hipMemcpyHostToDevice, c->st));
    if (!cc.empty())
        HIPCHK(hipMemcpyAsync(c->pdC, cc.data(), sizeof(double4) * cc.size(), hipMemcpyHostToDevice, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    c->pd_a = a;
    c->pd_b = b;
}

// The adjoint's trajectory in a context: the solver's beads, velocities, replicas and step
// counter stand aside (put back on every way out) while the steps run on copies in the
// context's workspace, a buffer of beads per step, so a step's positions stay for the reverse
// pass without a copy.
//
// What bounds a gradient is launches and recomputation: at 12k beads a step's kernels take 5
// to 40 us each.  The reverse pass needs each step's positions only, 32 bytes a bead; the steps
// since the last checkpoint are kept as the forward pass makes them, and checkpoints are set no
// closer than kKeepBytes allows, so a trajectory that fits is run once and not twice.  With
// the copies of each step's beads and replicas, the objective read back after each step and
// the workspace allocated anew, 24 steps took 5.5 ms instead of 3.5.
struct AdjointRun {
    static constexpr size_t kKeepBytes = 256ull << 20;    // positions kept whatever checkpoint asks for
    static constexpr size_t kIdleBytes = 512ull << 20;    // workspace a context holds between calls

    sm_ctx *c;
    const int n, nrep, S;   // beads, replicas, steps
    int k, nseg;            // steps between checkpoints, segments
    struct State {
        Bead *beads;
        float4 *vel, *acc;
        DevRep *reps;
        DevGlobal *glob;
    };
    State own;                        // the context's
    Bead *own_alt;
    bool own_fused;
    uint32_t own_fallbacks;           // with the counts of builds in the context's step counter
    long long own_builds;
    // x[t]: a segment's positions after its t-th step, before that step's box move.  An
    // objective alone needs the step before only: two buffers in turns (at), and no segments.
    std::vector<Bead *> x;
    const bool keep;
    Bead *at(int t) const { return x[keep ? t : t & 1]; }
    std::vector<State> checkpoint;    // states at steps k, 2k, ...; [0] at step 0
    DevRep *pre = nullptr, *post = nullptr;   // a segment's box moves: the replicas before and after each
    double *sums = nullptr;           // sums over the steps of U_pair, U_chain per replica
    double4 *X = nullptr, *V = nullptr, *A = nullptr, *A_next = nullptr, *F = nullptr, *HV = nullptr;
    double *g = nullptr, *gs = nullptr;

    AdjointRun(sm_ctx *ctx, int steps, int want_k, bool grad) : c(ctx), n(ctx->n), nrep(ctx->nrep), S(steps), keep(grad)
    {
        const long long fit = (long long)(kKeepBytes / (sizeof(Bead) * (size_t)n));
        k = keep ? (int)std::min<long long>(S, std::max<long long>(want_k, fit)) : S;
        nseg = (S + k - 1) / k;
        own = State{c->beads, c->vel, c->acc, c->reps, c->glob};
        own_alt = c->beads_alt;
        own_fused = c->mc_fused;
        own_fallbacks = c->fallbacks_seen;
        own_builds = c->counted_builds;
        // two passes over one list: the workspace's size, then its addresses
        State cur{};
        for (int pass = 0; pass < 2; pass++) {
            size_t at = 0;
            char *base = pass ? c->adj_workspace(words) : nullptr;
            auto take = [&](auto *&p, size_t count) {
                using T = std::remove_reference_t<decltype(*p)>;
                p = reinterpret_cast<T *>(base + at);
                at += (sizeof(T) * count + 255) / 256 * 256;
            };
            x.resize(keep ? k + 2 : 2);
            for (Bead *&b : x) take(b, n);
            auto state = [&](State &s, bool beads) {
                if (beads) take(s.beads, n);
                take(s.vel, n);
                take(s.acc, n);
                take(s.reps, nrep);
                take(s.glob, 1);
            };
            state(cur, false);
            checkpoint.resize(nseg - 1);
            for (State &s : checkpoint) state(s, true);
            take(sums, 2 * (size_t)nrep);
            if (keep) {
                take(pre, (size_t)(k / 8 + 1) * nrep);
                take(post, (size_t)(k / 8 + 1) * nrep);
                for (double4 **p : {&X, &V, &A, &A_next, &F, &HV}) take(*p, n);
                take(g, kNTheta * (size_t)n);
                take(gs, kNTheta * (size_t)nrep);
            }
            words = at;
        }
        copy(x[0], own.beads, n);
        copy(cur.vel, own.vel, n);
        copy(cur.acc, own.acc, n);
        copy(cur.reps, own.reps, nrep);
        copy(cur.glob, own.glob, 1);
        c->beads = x[0];
        c->vel = cur.vel;
        c->acc = cur.acc;
        c->reps = cur.reps;
        c->glob = cur.glob;
        // the forward run and the recomputed segments take their box-move dU the same way
        // (the gather after the kick), so they make the same decisions
        c->mc_fused = false;
        c->drop_graph();
    }
    ~AdjointRun()
    {
        (void)hipStreamSynchronize(c->st);
        c->beads = own.beads;
        c->beads_alt = own_alt;
        c->vel = own.vel;
        c->acc = own.acc;
        c->reps = own.reps;
        c->glob = own.glob;
        c->mc_fused = own_fused;
        c->fallbacks_seen = own_fallbacks;
        c->counted_builds = own_builds;
        c->forget_boxes();
        if (c->adj_ws_bytes > kIdleBytes) c->free_adj_workspace();
    }
    AdjointRun(const AdjointRun &) = delete;
    AdjointRun &operator=(const AdjointRun &) = delete;

    // index among the segment's box moves of the one at step s
    int move(int s, int s0) const { return s / 8 - s0 / 8 - 1; }

    // Steps s0 + 1 .. s1 (a segment's, from its state with the positions in x[0]): the context
    // is left in the state at s1.  objective: add each step's energies to the sums.
    void steps(int s0, int s1, bool objective)
    {
        const size_t rn = nrep;
        copy(at(1), at(0), n);
        c->beads = at(1);
        c->step_first(s0 + 1);
        for (int s = s0 + 1; s <= s1; s++) {
            const int t = s - s0;
            const bool mc = c->mc_step(s);
            c->sort_and_reorder();
            c->pair_force_u();   // in the recomputed segments too, whose steps must be the same
            if (objective) c->add_energies(sums);
            if (!mc && s < s1) {
                c->beads_alt = at(t + 1);
                c->kick_first(s);   // at(t) stays as it is
                continue;
            }
            c->bonded(KICK_STEP, nullptr);
            if (mc) {
                if (keep) copy(pre + move(s, s0) * rn, c->reps, rn);
                copy(at(t + 1), at(t), n);
                c->beads = at(t + 1);
                c->mc_move();
                if (keep) copy(post + move(s, s0) * rn, c->reps, rn);
                if (s < s1) c->step_first(s + 1);
            }
        }
    }
    void save(const State &to)
    {
        copy(to.beads, c->beads, n);
        copy(to.vel, c->vel, n);
        copy(to.acc, c->acc, n);
        copy(to.reps, c->reps, nrep);
        copy(to.glob, c->glob, 1);
    }
    void load(const State &from)
    {
        copy(x[0], from.beads, n);
        copy(c->vel, from.vel, n);
        copy(c->acc, from.acc, n);
        copy(c->reps, from.reps, nrep);
        copy(c->glob, from.glob, 1);
    }

private:
    size_t words = 0;   // the workspace's bytes
    template <class T>
    void copy(T *to, const T *from, size_t count)
    {
        if (to != from) HIPCHK(hipMemcpyAsync(to, from, sizeof(T) * count, hipMemcpyDeviceToDevice, c->st));
    }
};

}  // namespace

extern "C" {

int sm_set_params(sm_ctx *c, int32_t type_a, int32_t type_b, const double *theta)
{
    return guarded([&] {
        if (!c || !theta) invalid("null argument");
        check_pair(c, type_a, type_b);
        set_pair_rows(c, type_a, type_b, theta[0], theta[1]);
        for (auto &k : c->hcconst) {
            k.y = theta[2];
            k.w = theta[3];
        }
        upload_constants(c);
    });
}

int sm_get_params(sm_ctx *c, int32_t type_a, int32_t type_b, double *theta)
{
    return guarded([&] {
        if (!c || !theta) invalid("null argument");
        check_pair(c, type_a, type_b);
        const double *F = &c->hfconst[6 * (size_t)(type_a * c->P.nT + type_b)];
        const double rm = F[0], rc = F[3];
        const double umin = F[4] * (rc - rm) * (rc - rm) / 6.0;
        theta[0] = umin;
        theta[1] = F[1] * rm * rm / 2.0 + umin;
        theta[2] = c->hcconst.empty() ? 0.0 : c->hcconst[0].y;
        theta[3] = c->hcconst.empty() ? 0.0 : c->hcconst[0].w;
    });
}

int sm_param_derivative(sm_ctx *c, int32_t type_a, int32_t type_b, double *out)
{
    return guarded([&] {
        if (!c || !out) invalid("null argument");
        check_pair(c, type_a, type_b);
        upload_param_derivative_tables(c, type_a, type_b);
        c->build(0, kStepKeep);
        launch_pair_gather_u2(c->st, c->P, c->echunk, c->sbeads, c->skey(), c->sidx(), c->cstart, c->cend, c->reps,
                              c->pdTab, c->pdU, c->ebead, c->edelta);
        // the measurement words are free between calls (each measurement copies its own out)
        SumArgs a = c->sums(c->ebead, c->dres);
        a.y = c->edelta;
        a.cconst = c->pdC;
        a.cconst2 = c->pdC + c->hcconst.size();
        launch_sums(c->st, SUM_PARAM, a);
        c->check_launch();
        const int flags = c->link.fetch(c->st, c->glob, c->dres, 4 * (size_t)c->nrep, out);
        c->check_bits(flags);
    });
}

int sm_adjoint(sm_ctx *c, int32_t type_a, int32_t type_b, int32_t nsteps, int32_t checkpoint, double *J,
               double *grad)
{
    return guarded([&] {
        if (!c || !J) invalid("null argument");
        if (nsteps < 1 || checkpoint < 1 || checkpoint > nsteps) invalid("need 1 <= checkpoint <= nsteps");
        const int R = c->nrep;
        check_pair(c, type_a, type_b);
        const int n = c->n, S = nsteps;
        const double obj = 1.0 / S;
        long long moves = 0;
        for (long long s = 1; s <= S; s++)
            if (c->mc_step(s)) moves++;
        c->ensure_capacity(moves);
        upload_adjoint_tables(c, type_a, type_b);
        AdjointRun run(c, S, checkpoint, grad != nullptr);
        const int k = run.k, nseg = run.nseg;
        hipStream_t st = c->st;

        // forward: init forces, then steps 1..S, J = mean of U after each kick
        HIPCHK(hipMemsetAsync(run.sums, 0, sizeof(double) * 2 * (size_t)R, st));
        c->build(0, 0);
        c->pair_force();
        c->bonded(KICK_INIT, nullptr);
        for (int seg = 0; seg < nseg; seg++) {
            if (seg + 1 < nseg) run.save(run.checkpoint[seg]);
            run.steps(seg * k, std::min(S, seg * k + k), true);
            if (seg + 1 < nseg) HIPCHK(hipMemcpyAsync(run.x[0], c->beads, sizeof(Bead) * n, hipMemcpyDeviceToDevice, st));
            if (seg + 1 < nseg) c->beads = run.x[0];
        }
        c->check_launch();
        std::vector<double> h(2 * (size_t)R);
        c->check_bits(c->link.fetch(st, c->glob, run.sums, h.size(), h.data()));
        for (int r = 0; r < R; r++) J[r] = (h[2 * r] + h[2 * r + 1]) * obj;
        if (!grad) return;

        const auto zero = [&](void *p, size_t bytes) { HIPCHK(hipMemsetAsync(p, 0, bytes, st)); };
        for (double4 *p : {run.X, run.V, run.A}) zero(p, sizeof(double4) * n);
        zero(run.g, sizeof(double) * kNTheta * n);
        const int nT = c->P.nT;
        const AdjTables T{c->adjF, c->adjDF, c->adjDU, 6 * (type_a * nT + type_b), 6 * (type_b * nT + type_a)};
        auto pair_terms = [&](double o, int hv) {
            launch_adj_pair(st, c->P, c->sbeads, c->skey(), c->sidx(), c->cstart, c->cend, c->reps, T, run.A, run.F,
                            run.HV, run.g, o, hv);
        };
        auto chain_terms = [&](double o, int hv) {
            launch_adj_chain(st, c->P, c->beads, c->chainPerBead, c->cconstD, c->reps, run.A, run.F, run.HV, run.g, o,
                             hv);
            if (c->gptr) launch_adj_gen(st, c->P, c->gen(), c->beads, c->reps, run.A, run.F, run.HV, hv);
        };
        for (int seg = nseg - 1; seg >= 0; seg--) {
            const int s0 = seg * k, s1 = std::min(S, s0 + k);
            if (seg + 1 < nseg) {   // the last segment's positions are there from the forward pass
                run.load(run.checkpoint[seg]);
                run.steps(s0, s1, false);
            }
            for (int s = s1; s > s0; s--) {
                const bool mc = c->mc_step(s);
                const DevRep *post = c->reps;
                c->beads = run.x[s - s0];
                if (mc) {
                    const size_t m = (size_t)run.move(s, s0) * R;
                    HIPCHK(hipMemcpyAsync(c->reps, run.pre + m, sizeof(DevRep) * R, hipMemcpyDeviceToDevice, st));
                    post = run.post + m;
                }
                c->build(0, kStepKeep);
                pair_terms(obj, 1);
                const int prep = s - 1 >= 1 ? 1 : 0;
                if (c->gptr) {
                    chain_terms(obj, 1);
                    launch_adj_step(st, c->P, c->beads, post, mc ? 1 : 0, run.X, run.V, run.A, run.A_next, run.F,
                                    run.HV, obj, prep);
                } else {
                    launch_adj_chain_step(st, c->P, c->beads, c->chainPerBead, c->cconstD, c->reps, post, mc ? 1 : 0,
                                          run.X, run.V, run.A, run.A_next, run.F, run.HV, run.g, obj, prep);
                }
                std::swap(run.A, run.A_next);
            }
        }
        // a_0 = F(x_0) + ...: its adjoint meets dF/dtheta at the initial positions
        c->beads = run.x[0];
        c->build(0, kStepKeep);
        pair_terms(0.0, 0);
        chain_terms(0.0, 0);
        // per replica: grad[r * kNTheta + p]
        static_assert(kNTheta == 4, "SUM_COLUMNS sums four");
        launch_sums(st, SUM_COLUMNS, c->sums(run.g, run.gs));
        c->check_launch();
        (void)c->link.fetch(st, c->glob, run.gs, kNTheta * (size_t)R, grad);
    });
}

int sm_profile_enable(sm_ctx *c, int32_t on)
{
    return guarded([&] {
        if (!c) invalid("null context");
        c->harvest();
        c->prof = on != 0;
        for (int k = 0; k < K_NCLASS; k++) { c->prof_ms[k] = 0; c->prof_cnt[k] = 0; }
    });
}

int sm_profile_read(sm_ctx *c, int32_t cap, const char **names, double *avg_ms, int64_t *count, int32_t *n_out)
{
    return guarded([&] {
        if (!c) invalid("null context");
        c->harvest();
        int m = 0;
        for (int k = 0; k < K_NCLASS && m < cap; k++, m++) {
            if (names) names[m] = kClassName[k];
            if (avg_ms) avg_ms[m] = c->prof_cnt[k] ? c->prof_ms[k] / (double)c->prof_cnt[k] : 0.0;
            if (count) count[m] = c->prof_cnt[k];
        }
        if (n_out) *n_out = m;
    });
}

}  // extern "C"
