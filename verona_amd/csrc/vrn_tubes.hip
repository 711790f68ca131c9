// vrn_tubes.hip -- thousands of independent 1D relativistic shock tubes of
// uneven length advanced by one persistent, hipGraph-launched kernel.
//
// Each tube follows Verona1D.HARM_HLL (src/1dim/algos.jl:58-315): SoA
// primitives (rho, u, u^x) without ghost cells, reconstruction into PR[i-1],
// PL[i] over the reference's index range, a face flux for every face,
// midpoint RK2 (Uhalf = U - dt/2 dx dF, then U -= dt/dx dF) on cells
// 1 .. N-3 (0-based; cells 0, N-2, N-1 are never updated), and the 3x3
// Newton con2prim of src/1dim/structs.jl:78-105 on every cell, warm-started
// from P^n in both stages.  Face states the reconstruction never writes keep
// the tube's initial primitives, as the reference's deepcopy'd PR/PL do.
//
// Execution: a persistent grid of workgroups pulls tube indices from an
// atomic queue (tubes pre-sorted longest first, LPT) and runs every step of
// a tube inside one workgroup; tubes are independent, so no grid-wide
// synchronisation is needed.  Within a tube the workgroup streams over the
// cells in chunks of blockDim cells, one cell per lane, exchanging face
// states and fluxes through LDS with a carry across chunks.  Where that leaves
// most of the GPU idle (few tubes, or a few long ones), ranges of the tubes
// run in workgroups of their own, several steps a launch, with halos wide
// enough for these steps (k_tubes_split; split_plan and ranges_faster choose).
//
// This file holds the C ABI and the exact-form kernels; the kernels
// themselves are in vrn_tubes_kern.hpp, compiled again as the fast FP64 form
// in vrn_tubes_fast.hip (vrn_tubes_set_precision selects one).
#include "../../include/verona_hip.h"
#include "vrn_tubes_kern.hpp"
#include "vrn_xfer.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <numeric>
#include <string>
#include <tuple>
#include <vector>

// fast FP64 form of the tube kernels (vrn_tubes_fast.hip)
void vrn_fast_launch_tubes_split(hipStream_t s, const vrn::TubeArgs &a, int rec, int riem, int block, int nseg);
void vrn_fast_launch_tubes(hipStream_t s, const vrn::TubeArgs &a, int rec, int riem, int block, int grid);

using namespace vrn;

namespace {
thread_local std::string t_err;
int tfail(int code, const char *fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    t_err = buf;
    return code;
}
#define TCHK(expr)                                                                        \
    do {                                                                                  \
        hipError_t e_ = (expr);                                                           \
        if (e_ != hipSuccess) return tfail(VRN_E_HIP, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)
}  // namespace

struct vrn_tubes {
    vrn_xfer::Hold hold;
    int ntubes = 0;
    long ncell = 0;
    double gamma = 5.0 / 3.0;
    double *buf = nullptr;
    long *off = nullptr;
    int *order = nullptr;
    double *dt = nullptr, *dx = nullptr;
    unsigned int *queue = nullptr;
    hipStream_t s = nullptr;
    TubeArgs args{};
    int rec = VRN_REC_PPM, riemann = VRN_RIEMANN_HLLC;
    int precision = VRN_PREC_FP64;
    bool params = false;
    // captured graph
    hipGraphExec_t gexec = nullptr;
    hipGraph_t graph = nullptr;
    // what it was captured with: launch shape, steps, method (con2prim limits
    // among it), precision and state buffer
    std::tuple<int, int, int, int, int, int, double, int, const double *> g_key{};
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    float last_ms = 0.f;
    // k_tubes_split: 0 never, 1 where it is the faster, 2 wherever split_plan
    // has a plan; steps a launch (0: no plan) and ranges
    int split = 1;
    int split_k = 0, nseg = 0;
    // for ranges_faster: lengths (longest first), their sum, and the time of a
    // stage in ranges and in whole tubes in the best launch shape
    std::vector<long> len;
    double cells = 0.0, t_ranges = 0.0, t_whole = 0.0;
    TubeSeg *seg = nullptr;
    double *Psave[3] = {nullptr, nullptr, nullptr}, *Usave[3] = {nullptr, nullptr, nullptr};
};

namespace {

constexpr int SPLIT_BLOCK = 256;
constexpr int SPLIT_CELLS = 62 * (SPLIT_BLOCK / 64);
constexpr int SPLIT_STEPS = 4096;

// Ranges for k_tubes_split at k steps a launch (tubes that fit a workgroup
// whole need no halo); the cells they hold in all, halos included.
long split_ranges(const int64_t *lengths, const std::vector<int> &order, int k, std::vector<TubeSeg> *out)
{
    const int halo = 2 * TUBE_REACH * k, useful = SPLIT_CELLS - 2 * halo;
    long cells = 0;
    for (int t : order) {
        const long N = lengths[t];
        const long n = N <= SPLIT_CELLS ? 1 : (N + useful - 1) / useful;
        cells += N + (n - 1) * 2 * halo;
        if (out)
            for (long j = 0; j < n; j++) out->push_back({t, (int)(N * j / n), (int)(N * (j + 1) / n)});
    }
    return cells;
}

// The plan for ranges: 0 if a batch is better run as whole tubes by persistent
// workgroups (k_tubes) in any launch shape, else the steps a launch of
// k_tubes_split and its ranges.  For exact PPM + HLLC: persistent workgroups of
// 256 threads take about 8 us a stage for each 256 cells of the longest tube,
// and 3.9e-5 us a cell when the chip is full; ranges take at least 6 us a stage,
// 4.4e-5 us a cell (halos included) and 3 us a launch.  So ranges win while
// tubes are too few or too uneven to fill the chip, and persistent workgroups
// when it is full.  32 steps, persistent / ranges: 8 tubes of 1000 to 3000 cells
// 3.29 / 0.41 ms; 256 of 4000 8.8 / 3.4; 1024 of 256 to 8192 17.2 / 13.3; 2000 of
// 100 to 700 (HLL) 3.15 / 3.40; 1280 of 500 2.22 / 2.87; 4096 of 256 to 8192 43.9 /
// 50.4.  In other launch shapes whole tubes may be the faster where there is a
// plan too: ranges_faster.
int split_plan(int ntubes, const int64_t *lengths, const std::vector<int> &order, std::vector<TubeSeg> &seg)
{
    long total = 0;
    for (int t = 0; t < ntubes; t++) total += lengths[t];
    const double whole = std::max(8.0 * (double)((lengths[order[0]] + 255) / 256), 3.9e-5 * (double)total);
    int best = 0;
    double least = whole;
    for (int k = 1; k <= 16; k *= 2) {
        const double stage = std::max(6.0, 4.4e-5 * (double)split_ranges(lengths, order, k, nullptr)) + 1.5 / k;
        if (stage < least) {
            least = stage;
            best = k;
        }
    }
    if (best) split_ranges(lengths, order, best, &seg);
    return best;
}

// us a stage in ranges and as whole tubes in the best launch shape, for
// ranges_faster, of a batch that has a plan
void stage_times(vrn_tubes *c, const std::vector<TubeSeg> &seg)
{
    double waves = 0.0, lanes = 0.0;
    for (const TubeSeg &g : seg) waves += c->len[0] <= SPLIT_CELLS ? (g.hi - g.lo + 61) / 62 : SPLIT_BLOCK / 64;
    const double n = (double)seg.size();
    if (c->len[0] <= SPLIT_CELLS)  // no halo, all steps in a launch
        c->t_ranges = n <= 1280 ? 0.0065 * c->cells / SPLIT_CELLS : 0.0035 * n + 0.00075 * waves;
    else
        c->t_ranges = 0.0035 * n + 0.00075 * waves + 2.1 / c->split_k;
    c->t_ranges = std::max(4.4, 3.6 + c->t_ranges);
    auto face_lanes = [&](size_t t) { return (double)((c->len[t] + 64) / 64 * 64); };
    double most = 0.0;
    for (size_t t = 0; t < c->len.size(); t++) lanes += face_lanes(t);
    for (size_t j = 0; 256 * j < c->len.size(); j++) most = std::max(most, (j + 1) * face_lanes(256 * j));
    const bool full = lanes / 256 > most || lanes > 1e6;
    c->t_whole = std::max(5.9, 2.9 + (full ? 0.0085 : 0.0072) * std::max(most, lanes / 256));
}

// Whether a batch that has a plan is faster in ranges than as whole tubes by
// `grid` workgroups of `block` threads.  Times of a stage in us, the geometric
// mean of both forms and four methods (minmod + HLL, PPM + HLL, PPM + HLLC,
// WENO-Z + HLLC), measured on 60 batches of 1 to 3000 tubes of 16 to 12000
// cells:
//  * ranges take 3.6 + 0.0065 a full workgroup (4.4 at least) and 2.1 for a
//    launch, which has 2 k stages (standard deviation 8 %);
//  * whole tubes in the best of 12 shapes take 2.9 + 0.0072 a cell of the
//    busiest CU, 0.0085 where all CUs are busy or a million cells no longer
//    fit the L2s, 5.9 at least (8 %);
//  * in a given shape a workgroup goes through its tubes in chunks of `block`
//    cells, each 2.8 plus 0.24 for each wave that the CU runs at a time (20 at
//    most; a batch of few tubes fills some CUs before others) (17 %);
//  * ranges / whole tubes of a form and reconstruction lies off the mean by
//    the factors below.
// Whole tubes in the best shape / ranges: 122 of 390 6.6 / 6.2, 256 of 500 7.4 /
// 9.0, 512 of 500 10.5 / 13.3, 256 of 1000 10.1 / 12.5, 64 of 1000 9.0 / 6.0, 256
// of 2000 19 / 21, 400 of 2000 34 / 29; by 512 workgroups of 128 threads ranges
// win in all of them (512 of 500 19).  Run in ranges whatever the shape, 306 of
// 5952 runs (496 of a plan, 12 shapes) took 5 to 47 % longer than whole tubes in
// their shape; by this rule 100 do, 54 of them by more than 10 %, and 58 are whole that
// ranges would run 5 % faster or more.
bool ranges_faster(const vrn_tubes *c, int block, int grid)
{
    const long n = (long)c->len.size(), w = block / 64, G = std::min<long>(grid, 256 * (20 / w));
    auto chunks = [&](long t) { return (double)((c->len[t] + block) / block); };
    double mean = 0.0, most = 0.0;
    for (long t = 0; t < n; t++) mean += chunks(t) / (double)G;
    for (long j = 0; G * j < n; j++) most = std::max(most, (j + 1) * chunks(G * j));
    const double per_cu = std::max(1.0, std::min((double)G / 256, std::max(1.0, (double)n / 128)));
    const double chunk = 2.8 + 0.24 * per_cu * (double)w * (c->cells > 1e6 ? 1.3 : 1.0);
    static const double off[3][2] = {{0.98, 0.86}, {1.11, 1.00}, {1.03, 0.94}};  // minmod, PPM, WENO-Z
    static_assert(VRN_REC_MINMOD == 0 && VRN_REC_PPM == 1 && VRN_REC_WENOZ == 2, "rows of off");
    const double ranges = c->t_ranges * off[c->rec][c->precision == VRN_PREC_FP64_FAST];
    return ranges < std::max(c->t_whole, 1.6 + std::max(mean, most) * chunk);
}

}  // namespace

extern "C" {

const char *vrn_tubes_last_error(void) { return t_err.c_str(); }

int vrn_tubes_create(int ntubes, const int64_t *lengths, double gamma, vrn_tubes **out)
{
    if (!out || !lengths || ntubes <= 0) return tfail(VRN_E_ARG, "bad arguments");
    *out = nullptr;
    long total = 0;
    for (int t = 0; t < ntubes; t++) {
        if (lengths[t] < 8) return tfail(VRN_E_ARG, "tube %d shorter than 8 cells", t);
        total += lengths[t];
    }
    vrn_tubes *c = new vrn_tubes();
    c->ntubes = ntubes;
    c->ncell = total;
    c->gamma = gamma;
    std::vector<long> off(ntubes + 1, 0);
    for (int t = 0; t < ntubes; t++) off[t + 1] = off[t] + lengths[t];
    std::vector<int> order(ntubes);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return lengths[a] > lengths[b]; });
    std::vector<TubeSeg> seg;
    c->split_k = split_plan(ntubes, lengths, order, seg);
    c->nseg = (int)seg.size();
    if (c->split_k) {
        for (int t : order) c->len.push_back(lengths[t]);
        c->cells = (double)total;
        stage_times(c, seg);
    }
    // one allocation for the state (P, Ph, U, Uh, P0, Psave, Usave x 3
    // variables) and the tables, the constant ones of which (off, order, seg)
    // are copied together
    const size_t nd = (size_t)total * 21, nt = (size_t)ntubes;
    const size_t b_off = sizeof(long) * (nt + 1), b_seg = sizeof(TubeSeg) * seg.size(), b_ord = sizeof(int) * nt;
    std::vector<char> tab(b_off + b_seg + b_ord);
    std::memcpy(tab.data(), off.data(), b_off);
    if (b_seg) std::memcpy(tab.data() + b_off, seg.data(), b_seg);
    std::memcpy(tab.data() + b_off + b_seg, order.data(), b_ord);
    hipError_t e = hipStreamCreate(&c->s);
    if (e == hipSuccess)
        e = hipMalloc(&c->buf, sizeof(double) * (nd + 2 * nt) + tab.size() + sizeof(unsigned int));
    if (e == hipSuccess) {
        c->dt = c->buf + nd;
        c->dx = c->dt + nt;
        char *t = reinterpret_cast<char *>(c->dx + nt);
        c->off = reinterpret_cast<long *>(t);
        c->seg = reinterpret_cast<TubeSeg *>(t + b_off);
        c->order = reinterpret_cast<int *>(t + b_off + b_seg);
        c->queue = reinterpret_cast<unsigned int *>(t + b_off + b_seg + b_ord);
        e = hipMemcpy(t, tab.data(), tab.size(), hipMemcpyHostToDevice);
    }
    if (e == hipSuccess) e = hipEventCreate(&c->ev0);
    if (e == hipSuccess) e = hipEventCreate(&c->ev1);
    if (e != hipSuccess) {
        vrn_tubes_destroy(c);
        return tfail(VRN_E_NOMEM, "allocation failed: %s", hipGetErrorString(e));
    }
    double *p = c->buf;
    TubeArgs &a = c->args;
    for (int v = 0; v < 3; v++) a.P[v] = p + (0 * 3 + v) * total;
    for (int v = 0; v < 3; v++) a.Ph[v] = p + (1 * 3 + v) * total;
    for (int v = 0; v < 3; v++) a.U[v] = p + (2 * 3 + v) * total;
    for (int v = 0; v < 3; v++) a.Uh[v] = p + (3 * 3 + v) * total;
    for (int v = 0; v < 3; v++) a.P0[v] = p + (4 * 3 + v) * total;
    for (int v = 0; v < 3; v++) c->Psave[v] = p + (5 * 3 + v) * total;
    for (int v = 0; v < 3; v++) c->Usave[v] = p + (6 * 3 + v) * total;
    a.off = c->off;
    a.order = c->order;
    a.dt = c->dt;
    a.dx = c->dx;
    a.queue = c->queue;
    a.ntubes = ntubes;
    a.g = gamma;
    *out = c;
    return 0;
}

int vrn_tubes_destroy(vrn_tubes *c)
{
    if (!c) return 0;
    if (c->s) (void)hipStreamSynchronize(c->s);
    if (c->gexec) (void)hipGraphExecDestroy(c->gexec);
    if (c->graph) (void)hipGraphDestroy(c->graph);
    if (c->ev0) (void)hipEventDestroy(c->ev0);
    if (c->ev1) (void)hipEventDestroy(c->ev1);
    (void)hipFree(c->buf);
    if (c->s) (void)hipStreamDestroy(c->s);
    delete c;
    return 0;
}

// Upload concatenated SoA primitives (rho, u, u^x; each ncell doubles, tubes
// back to back) with per-tube dt and dx; computes U = PtoU(P) and keeps the
// initial primitives for the face states the reconstruction never writes.
int vrn_tubes_upload(vrn_tubes *c, const double *rho, const double *u, const double *ux,
                     const double *dt, const double *dx)
{
    if (!c || !rho || !u || !ux || !dt || !dx) return tfail(VRN_E_ARG, "null argument");
    const size_t b = sizeof(double) * c->ncell;
    const double *src[3] = {rho, u, ux};
    for (int v = 0; v < 3; v++) {
        TCHK(vrn_xfer::h2d(c->args.P[v], src[v], b, c->s));
        TCHK(hipMemcpyAsync((void *)c->args.P0[v], c->args.P[v], b, hipMemcpyDeviceToDevice, c->s));
    }
    TCHK(hipMemcpyAsync(c->dt, dt, sizeof(double) * c->ntubes, hipMemcpyHostToDevice, c->s));
    TCHK(hipMemcpyAsync(c->dx, dx, sizeof(double) * c->ntubes, hipMemcpyHostToDevice, c->s));
    hipLaunchKernelGGL(k_tubes_p2u, dim3(1024), dim3(256), 0, c->s, c->args, c->ncell);
    TCHK(hipGetLastError());
    TCHK(hipStreamSynchronize(c->s));
    return 0;
}

int vrn_tubes_download(vrn_tubes *c, double *rho, double *u, double *ux)
{
    if (!c || !rho || !u || !ux) return tfail(VRN_E_ARG, "null argument");
    const size_t b = sizeof(double) * c->ncell;
    double *dst[3] = {rho, u, ux};
    for (int v = 0; v < 3; v++) TCHK(vrn_xfer::d2h(dst[v], c->args.P[v], b, c->s));
    return 0;
}

int vrn_tubes_set_method(vrn_tubes *c, int rec, int riemann, int n_iter, double tol)
{
    if (!c || rec < 0 || rec > 2 || riemann < 0 || riemann > 1 || n_iter < 0)
        return tfail(VRN_E_ARG, "bad method");
    c->rec = rec;
    c->riemann = riemann;
    c->args.n_iter = n_iter;
    c->args.tol = tol;
    c->params = true;
    return 0;
}

// Arithmetic of the tube kernels: VRN_PREC_FP64 (default) reproduces the
// oracle bit for bit; VRN_PREC_FP64_FAST is the same algorithm with FMA
// contraction and reciprocal-based division (vrn_tubes_fast.hip).
int vrn_tubes_set_precision(vrn_tubes *c, int precision)
{
    if (!c) return tfail(VRN_E_ARG, "null");
    if (precision != VRN_PREC_FP64 && precision != VRN_PREC_FP64_FAST)
        return tfail(VRN_E_ARG, "tubes support VRN_PREC_FP64 and VRN_PREC_FP64_FAST (got %d)", precision);
    c->precision = precision;
    return 0;
}

static void launch_tubes(vrn_tubes *c, int block, int grid)
{
    // VRN_REC_* / VRN_RIEMANN_* equal the kernels' REC_* / RIEM_* values
    if (c->precision == VRN_PREC_FP64_FAST)
        vrn_fast_launch_tubes(c->s, c->args, c->rec, c->riemann, block, grid);
    else
        vrn::launch_tubes_kernels(c->s, c->args, c->rec, c->riemann, block, grid);
}

// Whether c's tubes are run in ranges when the launch shape is this.
static bool in_ranges(const vrn_tubes *c, int block, int grid)
{
    return c->split_k && c->split && (c->split == 2 || ranges_faster(c, block, grid));
}

// Steps of the launches of nsteps steps in ranges: as many as the halos are
// wide for, or, where every tube lies in one workgroup and needs none, up to
// SPLIT_STEPS (the kernel's halo, 6 cells a step, stays far inside an int, and
// a launch of 30 ms or more makes its 3 us nothing).
static int launch_steps(const vrn_tubes *c, int nsteps)
{
    return std::min(c->nseg == c->ntubes ? SPLIT_STEPS : c->split_k, nsteps);
}

// nsteps steps by k_tubes_split.  The two state buffers change places at each
// launch.
static int run_split(vrn_tubes *c, int nsteps)
{
    const int most = launch_steps(c, nsteps);
    for (int done = 0; done < nsteps;) {
        TubeArgs &a = c->args;
        a.seg = c->seg;
        a.ksteps = std::min(most, nsteps - done);
        for (int v = 0; v < 3; v++) {
            a.Pn[v] = a.Ph[v];
            a.Un[v] = a.Uh[v];
        }
        if (c->precision == VRN_PREC_FP64_FAST)
            vrn_fast_launch_tubes_split(c->s, a, c->rec, c->riemann, SPLIT_BLOCK, c->nseg);
        else
            vrn::launch_tubes_split(c->s, a, c->rec, c->riemann, SPLIT_BLOCK, c->nseg);
        TCHK(hipGetLastError());
        for (int v = 0; v < 3; v++) {
            std::swap(a.P[v], a.Ph[v]);
            std::swap(a.U[v], a.Uh[v]);
        }
        done += a.ksteps;
    }
    return 0;
}

static int check_shape(int nsteps, int block, int grid)
{
    if (nsteps < 0 || block < 64 || block > 1024 || (block & 63) || grid < 1)
        return tfail(VRN_E_ARG, "bad launch shape (block %d, grid %d)", block, grid);
    return 0;
}

// Advance every tube by nsteps steps: split over workgroups where in_ranges
// says so, else with `grid` persistent workgroups of `block` threads.
// use_graph != 0 captures (queue reset + persistent kernel) into a hipGraph once
// per g_key and replays it.  *ms (may be NULL) receives the device time of the
// launches.  Blocks.
int vrn_tubes_run(vrn_tubes *c, int nsteps, int block, int grid, int use_graph, double *ms)
{
    if (!c || !c->params) return tfail(VRN_E_STATE, "vrn_tubes_set_method first");
    if (int r = check_shape(nsteps, block, grid)) return r;
    c->args.nsteps = nsteps;
    if (in_ranges(c, block, grid)) {
        TCHK(hipEventRecord(c->ev0, c->s));
        if (int r = run_split(c, nsteps)) return r;
        TCHK(hipEventRecord(c->ev1, c->s));
    } else if (use_graph) {
        const decltype(c->g_key) key{block, grid, nsteps, c->rec, c->riemann, c->args.n_iter, c->args.tol, c->precision,
                                     c->args.P[0]};
        const bool stale = !c->gexec || c->g_key != key;
        if (stale) {
            if (c->gexec) (void)hipGraphExecDestroy(c->gexec);
            if (c->graph) (void)hipGraphDestroy(c->graph);
            c->gexec = nullptr;
            c->graph = nullptr;
            TCHK(hipStreamBeginCapture(c->s, hipStreamCaptureModeThreadLocal));
            launch_tubes(c, block, grid);
            TCHK(hipStreamEndCapture(c->s, &c->graph));
            TCHK(hipGraphInstantiate(&c->gexec, c->graph, nullptr, nullptr, 0));
            c->g_key = key;
        }
        TCHK(hipEventRecord(c->ev0, c->s));
        TCHK(hipGraphLaunch(c->gexec, c->s));
        TCHK(hipEventRecord(c->ev1, c->s));
    } else {
        TCHK(hipEventRecord(c->ev0, c->s));
        launch_tubes(c, block, grid);
        TCHK(hipGetLastError());
        TCHK(hipEventRecord(c->ev1, c->s));
    }
    TCHK(hipStreamSynchronize(c->s));
    float t = 0.f;
    TCHK(hipEventElapsedTime(&t, c->ev0, c->ev1));
    c->last_ms = t;
    if (ms) *ms = t;
    return 0;
}

// Whether batches are run in ranges: never (0), where that is the faster (1,
// the default) or wherever there is a plan for it (2).
int vrn_tubes_set_split(vrn_tubes *c, int mode)
{
    if (!c || mode < 0 || mode > 2) return tfail(VRN_E_ARG, "null, or mode outside 0..2");
    c->split = mode;
    return 0;
}

// How a run of nsteps steps in a launch shape is launched: the steps of its
// launches in ranges and the ranges, both 0 for whole tubes.
int vrn_tubes_plan(vrn_tubes *c, int nsteps, int block, int grid, int *steps, int *ranges)
{
    if (!c) return tfail(VRN_E_ARG, "null");
    if (int r = check_shape(nsteps, block, grid)) return r;
    const bool r = in_ranges(c, block, grid);
    if (steps) *steps = r ? launch_steps(c, nsteps) : 0;
    if (ranges) *ranges = r ? c->nseg : 0;
    return 0;
}

// Save / restore the state (P, U) so the autotuner can try launch shapes on
// the real data without advancing it.
int vrn_tubes_checkpoint(vrn_tubes *c, int restore)
{
    if (!c) return tfail(VRN_E_ARG, "null");
    const size_t b = sizeof(double) * c->ncell;
    for (int v = 0; v < 3; v++) {
        if (restore) {
            TCHK(hipMemcpyAsync(c->args.P[v], c->Psave[v], b, hipMemcpyDeviceToDevice, c->s));
            TCHK(hipMemcpyAsync(c->args.U[v], c->Usave[v], b, hipMemcpyDeviceToDevice, c->s));
        } else {
            TCHK(hipMemcpyAsync(c->Psave[v], c->args.P[v], b, hipMemcpyDeviceToDevice, c->s));
            TCHK(hipMemcpyAsync(c->Usave[v], c->args.U[v], b, hipMemcpyDeviceToDevice, c->s));
        }
    }
    TCHK(hipStreamSynchronize(c->s));
    return 0;
}

int vrn_tubes_info(vrn_tubes *c, int64_t *ncell, int *cu_count)
{
    if (!c) return tfail(VRN_E_ARG, "null");
    if (ncell) *ncell = c->ncell;
    if (cu_count) {
        int dev = 0;
        TCHK(hipGetDevice(&dev));
        TCHK(hipDeviceGetAttribute(cu_count, hipDeviceAttributeMultiprocessorCount, dev));
    }
    return 0;
}

}  // extern "C"
