// search.hip -- host driver and C ABI (include/episdet.h) of the gfx950
// epistasis search.
//
// The reference's EpistasisDetectionSearch (search-pairs.cu:9-246,
// search-triplets.cu:8-305) runs a host loop of rounds, each a binary GEMM
// plus an objective kernel.  Here the default path is one persistent launch
// that walks the whole set space from a device work queue and fuses counting,
// FP32 scoring and candidate selection; candidates are then re-scored in FP64
// and reduced on the host with a deterministic tie rule.  The reference-shaped
// round loop is kept as the PLAIN path (and as the exact fallback).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstddef>
#include <cstring>
#include <atomic>
#include <thread>
#include <vector>
#include <tuple>
#include <mutex>
#include <map>

#include "episdet.h"
#include "kernels_mfma.hpp"
#include "kernels_mfma_pairs.hpp"
#include "kernels_mfma3.hpp"
#include "kernels_mfma4.hpp"
#include "kernels_mfma_pairs2.hpp"
#include "kernels_mfma5.hpp"
#include "kernels_seed.hpp"

using namespace episdet;

namespace {

constexpr int BLOCK = 256;            // the reference's BLOCK_SIZE (Makefile:2)
constexpr int PLAIN_GROUP = 16;       // 3-way rounds per FP4 count launch of the plain path
constexpr size_t SEED_WORDS = 2 * SEED_BLOCKS + SEED_MAX_PAIRS;   // block bests, picked pairs
constexpr int PLAIN_GROUP2 = 32;      // 2-way rounds per FP4 count launch of the plain path
// Words per plane row on the device: the samples rounded up to 1024 (the
// reference's own padding), a whole chunk of every kernel that stages
// through LDS DMA (16 or 32 words) and half a chunk of MFMA version 1, which
// reads the missing half of its last chunk as zeros.
constexpr int W_ALIGN = 32;
static_assert(M2_KW % 16 == 0 && 32 % M2_KW == 0 && MF_KW == 2 * W_ALIGN, "chunk widths divide the row alignment");
constexpr int NUM_STREAMS = 8;        // the reference's NUM_STREAMS (Makefile:2)
constexpr unsigned DEFAULT_CAP = 1u << 20;
// Candidates copied back with the control block right after a search (a
// search that appends more fetches the rest in a second copy).
constexpr unsigned STAGE_CAND = 1024;
constexpr size_t STAGE_BYTES = 256 + (size_t)STAGE_CAND * (sizeof(unsigned long long) + sizeof(float) + sizeof(double));

#define HIPCHK(expr)                                                                                    \
    do {                                                                                                \
        hipError_t e_ = (expr);                                                                         \
        if (e_ != hipSuccess) {                                                                         \
            std::fprintf(stderr, "episdet: %s failed: %s (%s:%d)\n", #expr, hipGetErrorString(e_),      \
                         __FILE__, __LINE__);                                                           \
            return EPISDET_ERR_HIP;                                                                     \
        }                                                                                               \
    } while (0)

#define CHK(expr)                                                                                       \
    do {                                                                                                \
        int r_ = (expr);                                                                                \
        if (r_ != EPISDET_OK) return r_;                                                                \
    } while (0)

double now_s()
{
    return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

struct ScoreTables {
    bool ready = false;
    double *t64 = nullptr;    // K2: ln m!; MI: log2(m/N) (FP64 re-scoring)
    double t_max = 0;         // K2: max |ln m! - c m| over the table
    double shift_c = 0;       // K2 shift per cell, c = ln N - 1
    float invN = 0, k0 = 0;   // FP32 constants of the fused scoring
    double term_err = 0;      // measured error of the FP32 terms (k_term_error)
};

struct Ctl {                  // device control block; hot words on lines of their own (QLINE)
    unsigned long long queue[QLINE];
    unsigned long long xq[8][QLINE];    // per-XCD queues (fetch_xcd), right after the queue
    alignas(8 * QLINE) unsigned best32; // score bound
    alignas(8 * QLINE) unsigned cand_count;   // candidates appended; with cand_over, CandOut::cand_count[0..1]
    unsigned cand_over;       // sticky overflow flag (the count can wrap past 2^32)
    unsigned bad_snp;         // lowest SNP with a sample in both planes (k_singles), or ~0
    alignas(8 * QLINE) unsigned long long best64;
    unsigned long long checksum;
};
static_assert(offsetof(Ctl, cand_over) == offsetof(Ctl, cand_count) + sizeof(unsigned),
              "the overflow flag follows the candidate count");

}  // namespace

// Device memory of the no-allocation search (episdet_run_noalloc): control
// block, argument block, candidate slots, work-unit groups and, when the
// dataset has not built them yet, the FP64 score table and the 3-way pair
// table.  The runtime reserves it on every device when the module loads and
// keeps it until the process ends.  In host code the name stands for a
// host-side shadow, not a device address: host code uses only the address
// hipGetSymbolAddress returns for the current device (scratch_device).
constexpr size_t SCRATCH_BYTES = 64ull << 20;
static __device__ __align__(256) unsigned char scratch[SCRATCH_BYTES];

namespace {

constexpr unsigned SCRATCH_CAND = 1u << 18;     // candidate slots of a no-allocation search

// The regions of `scratch` one no-allocation call uses (device addresses),
// and the two timing events it uses (the dataset's).  Set for the duration of the call on its host
// thread (t_scr); every device allocation site of the search checks it.
struct ScratchPlan {
    Ctl *ctl = nullptr;
    void *jobargs = nullptr;
    unsigned long long *jobstart = nullptr;
    unsigned long long *err = nullptr;
    unsigned long long *cand = nullptr;
    float *cand_s32 = nullptr;
    double *cand_s64 = nullptr;
    unsigned long long *gstart = nullptr;
    int2 *groups = nullptr;
    size_t max_groups = 0;
    double *t64 = nullptr;          // when the dataset has no FP64 table for the score
    uint4 *pairs = nullptr;         // when a 3-way dataset has no pair table
    hipEvent_t ev[2] = {nullptr, nullptr};
};
thread_local const ScratchPlan *t_scr = nullptr;

// Every device allocation of the search goes through here.  Inside a
// no-allocation call it fails instead of allocating (the call then returns
// an error), so such a call can never reach hipMalloc.
hipError_t dev_malloc(void **p, size_t bytes)
{
    if (t_scr) {
        *p = nullptr;
        return hipErrorNotSupported;
    }
    return hipMalloc(p, bytes);
}

// Two timing events: inside a no-allocation call the dataset's own (made
// with the dataset), else two new ones destroyed with the Timer.
struct Timer {
    hipEvent_t e0 = nullptr, e1 = nullptr;
    bool own = false;
    int make()
    {
        if (t_scr) {
            e0 = t_scr->ev[0];
            e1 = t_scr->ev[1];
            return EPISDET_OK;
        }
        own = true;
        HIPCHK(hipEventCreate(&e0));
        HIPCHK(hipEventCreate(&e1));
        return EPISDET_OK;
    }
    ~Timer()
    {
        if (own) {
            if (e0) (void)hipEventDestroy(e0);
            if (e1) (void)hipEventDestroy(e1);
        }
    }
};

}  // namespace

struct episdet_dataset {
    int dev = 0;
    int n = 0, nrows = 0, N[2] = {0, 0}, W[2] = {0, 0};
    uint32_t *planes[2] = {nullptr, nullptr};
    uint4 *singles = nullptr;
    uint4 *pairs = nullptr;
    ScoreTables tab[2];
    hipStream_t stream = nullptr;
    Ctl *ctl = nullptr;
    unsigned long long *cand = nullptr;
    float *cand_s32 = nullptr;
    double *cand_s64 = nullptr;
    unsigned cand_cap = 0;
    int cu = 0;
    void *jobargs = nullptr;                  // device copy of one kernel argument block
    unsigned long long *jobstart = nullptr;   // {0, units} for a batch of one
    unsigned long long *gstart = nullptr;     // 3-way work-unit groups (k_groups), and the tile they are for
    int2 *groups = nullptr;
    int group_tile[3] = {0, 0, 0};            // TY, TZ, X per unit; 0: none yet
    unsigned long long *seed = nullptr;       // best pairs of the seeding kernels (SEED_WORDS)
    hipEvent_t ev[3] = {nullptr, nullptr, nullptr};   // search start / end, re-score end
    unsigned char *stage = nullptr;           // pinned, device-mapped: candidate count + the first candidates
    unsigned char *stage_dev = nullptr;       // the device's address of `stage`
    std::vector<unsigned long long> topk_packed;   // last top-k result, best first
    std::vector<double> topk_scores;
};

namespace {

int check_device(int *cu)
{
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count < 1) return EPISDET_ERR_NO_DEVICE;
    hipDeviceProp_t prop;
    HIPCHK(hipGetDeviceProperties(&prop, 0));
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
        std::fprintf(stderr, "episdet: device 0 is %s, gfx950 required\n", prop.gcnArchName);
        return EPISDET_ERR_NO_DEVICE;
    }
    if (cu) *cu = prop.multiProcessorCount;
    return EPISDET_OK;
}

// Runs f(part, parts) on up to `most` threads, in the calling one if no
// other can be started.
template <typename F>
void on_threads(int most, F &&f)
{
    const int parts = std::max(1, std::min(most, (int)std::thread::hardware_concurrency()));
    std::vector<std::thread> th;
    int started = 1;
    try {
        th.reserve((size_t)parts);
        for (; started < parts; started++) th.emplace_back(f, started, parts);
    } catch (...) {
        // the parts that got no thread run below
    }
    f(0, parts);
    for (int p = started; p < parts; p++) f(p, parts);
    for (std::thread &t : th) t.join();
}

// Pinned, device-mapped staging for dataset uploads, shared by the process: one
// upload uses it at a time (another that finds it taken copies from pageable
// memory), 24 MB at most, given back when the process exits.  The runtime
// moves pageable memory at about 20 GB/s; six threads fill this and the repacking
// kernel reads it over the link, 64 MB in about 1.6 ms.
constexpr int UP_THREADS = 6;
constexpr size_t UP_SLOT = 4u << 20;
std::mutex g_up_mu;
unsigned char *g_up = nullptr, *g_up_dev = nullptr;

// Called with g_up_mu held.
bool upload_pool()
{
    if (g_up) return true;
    if (hipHostMalloc((void **)&g_up, UP_SLOT * UP_THREADS, hipHostMallocMapped | hipHostMallocPortable) != hipSuccess) {
        g_up = nullptr;
        (void)hipGetLastError();
        return false;
    }
    if (hipHostGetDevicePointer((void **)&g_up_dev, g_up, 0) != hipSuccess) {
        (void)hipHostFree(g_up);
        g_up = nullptr;
        return false;
    }
    std::atexit([] { (void)hipHostFree(g_up); });
    return true;
}

// One class's planes through the pool: each thread fills its slot with the
// next SNPs' rows and launches their repacking, and waits for that before it fills the
// slot again.  Called with g_up_mu held and the pool there.
int upload_pooled(episdet_dataset *ds, int c, const unsigned *src, int in_w)
{
    const size_t snp_bytes = sizeof(uint32_t) * 2 * (size_t)in_w;
    const int per = (int)std::max<size_t>(1, UP_SLOT / snp_bytes);
    const int chunks = (ds->n + per - 1) / per;
    std::atomic<int> next{0}, rc{EPISDET_OK};
    const auto work = [&](int part, int) {
        hipEvent_t ev = nullptr;
        bool used = false;
        if (hipSetDevice(ds->dev) != hipSuccess || hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) {
            rc = EPISDET_ERR_HIP;
            return;
        }
        for (int k = next++; k < chunks && rc == EPISDET_OK; k = next++) {
            const int s0 = k * per, s1 = std::min(ds->n, s0 + per);
            if (used && hipEventSynchronize(ev) != hipSuccess) rc = EPISDET_ERR_HIP;
            std::memcpy(g_up + UP_SLOT * part, src + (size_t)s0 * 2 * in_w, snp_bytes * (size_t)(s1 - s0));
            // the last chunk also clears the rows past the last SNP
            const int snps = (k + 1 == chunks ? ds->nrows : s1) - s0;
            const size_t words = (size_t)snps * 2 * ds->W[c];
            hipLaunchKernelGGL(k_repack, dim3((unsigned)std::min<size_t>((words + 255) / 256, 4096)), dim3(256), 0,
                               ds->stream, (const uint32_t *)(g_up_dev + UP_SLOT * part), in_w, ds->planes[c],
                               ds->W[c], ds->n, s0, snps, ds->N[c]);
            if (hipGetLastError() != hipSuccess || hipEventRecord(ev, ds->stream) != hipSuccess) rc = EPISDET_ERR_HIP;
            used = true;
        }
        // the slot is not to be filled by the next upload while it is read
        if (used && hipEventSynchronize(ev) != hipSuccess) rc = EPISDET_ERR_HIP;
        (void)hipEventDestroy(ev);
    };
    on_threads(std::min(UP_THREADS, chunks), work);
    return rc;
}

int ensure_cand(episdet_dataset *ds, unsigned cap)
{
    if (ds->cand_cap >= cap) return EPISDET_OK;
    if (t_scr) return EPISDET_ERR_SCRATCH;           // the slots of `scratch` are all there is
    if (ds->cand) (void)hipFree(ds->cand);
    ds->cand = nullptr;
    ds->cand_s32 = nullptr;
    ds->cand_s64 = nullptr;
    ds->cand_cap = 0;
    // packed indices, FP64 scores and FP32 scores in one block
    if (dev_malloc((void **)&ds->cand, (2 * sizeof(unsigned long long) + sizeof(float)) * (size_t)cap) != hipSuccess) {
        ds->cand = nullptr;
        return EPISDET_ERR_ALLOC;
    }
    ds->cand_s64 = (double *)(ds->cand + cap);
    ds->cand_s32 = (float *)(ds->cand_s64 + cap);
    ds->cand_cap = cap;
    return EPISDET_OK;
}

// Host tables.  FP64: exactly the oracle's (lgamma / log2 of glibc), so FP64
// scores agree bit for bit.  FP32: the shifted K2 table or the MI table.
// ln m! for the small K2 terms (g_lnfact), once per process; glibc lgamma in
// FP64, rounded to FP32.
int ensure_lnfact()
{
    static std::mutex mu;
    static bool done = false;
    std::lock_guard<std::mutex> lk(mu);
    if (done) return EPISDET_OK;
    std::vector<float> h(LNF_SMALL);
    for (int m = 0; m < LNF_SMALL; m++) h[m] = (float)std::lgamma((double)m + 1.0);
    HIPCHK(hipMemcpyToSymbol(HIP_SYMBOL(g_lnfact), h.data(), sizeof(float) * LNF_SMALL));
    done = true;
    return EPISDET_OK;
}

// FP32 shares of the classes for the MI terms (mi_dterm): Nc/N rounded, and
// 1 minus that rounded.
void mi_shares(const episdet_dataset *ds, float q[2])
{
    q[0] = (float)((double)ds->N[0] / (double)(ds->N[0] + ds->N[1]));
    q[1] = 1.f - q[0];
}

int ensure_tables(episdet_dataset *ds, int score)
{
    ScoreTables &t = ds->tab[score];
    if (t.ready) return EPISDET_OK;
    CHK(ensure_lnfact());
    const int N = ds->N[0] + ds->N[1];
    const int len = N + 2;
    std::vector<double> h64(len, 0.0);
    t.shift_c = std::log((double)N) - 1.0;
    t.invN = (float)(1.0 / (double)N);
    t.k0 = (float)(0.5 * std::log((double)N) - 1.0 + 0.5 * std::log(2.0 * M_PI));
    if (score == EPISDET_SCORE_K2) {
        // (lgamma_r: lgamma's own sign variable is shared by the threads)
        on_threads(len >= (1 << 14) ? 8 : 1, [&](int part, int parts) {
            const int m1 = (int)((long long)len * (part + 1) / parts);
            int sign;
            for (int m = (int)((long long)len * part / parts); m < m1; m++) h64[m] = lgamma_r((double)m + 1.0, &sign);
        });
        double mx = 0;
        for (int m = 0; m < len; m++) mx = std::max(mx, std::fabs(h64[m] - t.shift_c * (double)m));
        t.t_max = mx;
    } else {
        h64[0] = 0.0;
        on_threads(len >= (1 << 14) ? 8 : 1, [&](int part, int parts) {
            const int m1 = (int)((long long)N * (part + 1) / parts);
            for (int m = 1 + (int)((long long)N * part / parts); m <= m1; m++) h64[m] = std::log2((double)m / (double)N);
        });
    }
    // inside a no-allocation call the table and the error word live in
    // `scratch` (the caller restores the dataset's tables afterwards)
    if (t_scr) t.t64 = t_scr->t64;
    else if (dev_malloc((void **)&t.t64, sizeof(double) * len) != hipSuccess) return EPISDET_ERR_ALLOC;
    if (!t.t64) return EPISDET_ERR_INTERNAL;
    HIPCHK(hipMemcpy(t.t64, h64.data(), sizeof(double) * len, hipMemcpyHostToDevice));
    // error of the FP32 terms over every argument this dataset can produce
    unsigned long long *d_err = t_scr ? t_scr->err : nullptr;
    if (!d_err && dev_malloc((void **)&d_err, sizeof(unsigned long long)) != hipSuccess) return EPISDET_ERR_ALLOC;
    const unsigned long long zero = 0ull;
    HIPCHK(hipMemcpy(d_err, &zero, sizeof zero, hipMemcpyHostToDevice));
    const int blocks = std::min(1024, (len + 255) / 256);
    float q[2];
    mi_shares(ds, q);
    hipLaunchKernelGGL(k_term_error, dim3(blocks), dim3(256), 0, ds->stream, score, N, t.invN, t.k0,
                       (float)t.shift_c, t.shift_c, t.t64, q[0], q[1], d_err);
    HIPCHK(hipGetLastError());
    unsigned long long bits = 0;
    HIPCHK(hipMemcpyAsync(&bits, d_err, sizeof bits, hipMemcpyDeviceToHost, ds->stream));
    HIPCHK(hipStreamSynchronize(ds->stream));
    if (!t_scr) (void)hipFree(d_err);
    std::memcpy(&t.term_err, &bits, sizeof bits);
    if (!(t.term_err >= 0.0 && t.term_err < 1e3)) return EPISDET_ERR_INTERNAL;
    t.ready = true;
    return EPISDET_OK;
}

double ulp32(double x)
{
    if (x <= 0) return std::ldexp(1.0, -149);
    return std::ldexp(1.0, std::ilogb(x) - 23);
}

// FP32 scoring context and its error bound.  The bound covers the table
// rounding (half an ulp of the largest entry per lookup), the two rounded
// operations per cell, the compensated cell sum and the final subtraction;
// the candidate margin is twice that.
ScoreCtx make_ctx(const episdet_dataset *ds, int score, int order)
{
    const ScoreTables &t = ds->tab[score];
    const int ncells = order == 3 ? 27 : 9;
    const int N = ds->N[0] + ds->N[1];
    const double u = std::ldexp(1.0, -24);
    ScoreCtx sc;
    sc.score = score;
    sc.ncells = ncells;
    sc.k2_total = 0.f;
    sc.k0 = t.k0;
    sc.c = (float)t.shift_c;
    sc.invN = t.invN;
    const double qc = (double)ds->N[0] / N, qt = (double)ds->N[1] / N;
    mi_shares(ds, sc.mi_q);
    sc.mi_scale = (float)(1.0 / ((double)N * std::log(2.0)));
    double eps;
    if (score == EPISDET_SCORE_K2) {
        sc.k2_total = (float)(ncells * t.shift_c);
        // per cell: three terms, each off by at most term_err, and two
        // roundings of sums below 3T; then the compensated sum and the
        // final subtraction
        const double T = t.t_max + t.term_err;
        const double sum_bound = ncells * 3.0 * T;
        eps = ncells * (3.0 * t.term_err + 2.0 * ulp32(3.0 * T)) + 2.0 * u * sum_bound + ulp32(sum_bound) +
              ulp32(ncells * t.shift_c);
    } else {
        // The 2 ncells terms D >= 0 each err by at most term_err relative
        // (measured), their sum by 2 ncells roundings, and the scale by two
        // more, so the FP32 MI errs by at most (term_err + (2 ncells + 3) u)
        // times the MI, which never exceeds H(Y).  Rounding the classes'
        // shares to FP32 moves the MI by N KL(pi || fl(pi)) / (N ln 2), of
        // order u^2: the absolute 4u covers it.  Counts of 2^24 and more
        // round to FP32 (x and n by u relative each), which moves D by
        // |ln(x/y)| x u + |d| u <= (2 D + x + |d|) u; the x and |d| of a
        // table add up to at most 3N, so the MI moves by at most
        // 2u MI + 3u / ln 2 in bits: 16u covers both.
        const double hY = -qc * std::log2(qc) - qt * std::log2(qt);
        eps = hY * (t.term_err + (2.0 * ncells + 3.0) * u) * (1.0 + 1e-6) + 4.0 * u +
              (N >= (1 << 24) ? 16.0 * u : 0.0);
    }
    sc.margin = (float)(2.0 * eps);
    // Badness lower bound (bound_exceeds): lb_max - lb_scale * S, and
    // for K2 + lb_lnw * sum_c log2 max(n_c, 1) + lb_off.
    // Its FP32 error: each (cas - pi n)^2 / n errs by about 2 |d| ulp(N) / n
    // <= 2 ulp(N) since |d| <= n (taken 4 times over), lb_scale times that
    // over the cells; K2's N H(pi) rounds by under 1e-7 N, and a further
    // absolute term covers the sums' roundings and the log2 of the cell
    // products (each product within 4 roundings, each log2 below 125 within
    // a few ulps: under 1e-5 relative of the log sum, 25 ncells at most).
    const double K = std::max(-std::log1p(-qc) / (qc * qc), -std::log(qc) / (qt * qt)) * (1.0 + 1e-6);
    sc.lb_pi = (float)qc;
    double scale, lbmax, extra, lnw = 0.0, off = 0.0, top;
    if (score == EPISDET_SCORE_K2) {
        scale = K;
        lbmax = -(double)N * (qc * std::log(qc) + qt * std::log(qt));
        top = lbmax;
        extra = 1e-7 * N + 1.0;
        // The Stirling term multiplies 5 cells in FP32: only while every
        // cell, at most N, is below 2^25 (the VALU path takes larger N).
        if (N < (1 << 25)) {
            lnw = 0.5 * std::log(2.0);
            off = -ncells * 0.5 * std::log(M_PI / 2.0) * (1.0 + 1e-6);
            // sum_c ln max(n_c, 1) over cells adding up to N is at most
            // ncells ln(N / ncells) when N >= e ncells, else N / e
            const double lnsum =
                N >= std::exp(1.0) * ncells ? ncells * std::log((double)N / ncells) : N / std::exp(1.0);
            top = lbmax + 0.5 * lnsum + 1.0;
            extra += lnw * 25.0 * ncells * 1e-5;
        }
    } else {
        scale = K / ((double)N * std::log(2.0));
        lbmax = 0.0;
        top = 0.0;
        extra = 1e-6;
    }
    sc.lb_scale = (float)scale;
    sc.lb_max = (float)lbmax;
    sc.lb_lnw = (float)lnw;
    sc.lb_off = (float)off;
    sc.lb_top = (float)top;
    // quick_bound (FP32 cells): with M = sqrt(S N), every marginal's |D| is at
    // most M (Cauchy-Schwarz), so a base cell or marginal errs by at most u M
    // and a cell derived from errors e1 + e2 + e3 by at most that plus 3 u M:
    // over the 27 cells 1 (8 of them), 6 (12), 16 (6) and 36 (1) times u M,
    // 57.3 u M in the 2-norm (9 cells: below that).  With T >= 1 below D^2 / T,
    // sqrt(S') >= sqrt(S) (1 - 57.3 u sqrt(N)); the sum's own roundings are
    // under 1e-5.  Cell totals and the sum of their bits are exact below 2^23
    // samples; with more, the quick bound is off.
    const double eta = 57.3 * u * std::sqrt((double)N);
    const bool quick = N < (1 << 23) && (score != EPISDET_SCORE_K2 || lnw > 0.0);
    sc.fb_scale = quick ? (float)(scale / ((1.0 - eta) * (1.0 - eta)) * (1.0 + 1e-5)) : 0.f;
    sc.fb_lnw = (float)(lnw * std::ldexp(1.0, -23));
    // Second bound, sum of f(D) = D^2 r (k + a r |D|) over the cells: f is
    // convex in |D| with |D| f' <= 3 f, so with cells off by delta the sum
    // loses at most 3 sum |delta| r |D| w <= 3 sqrt(1.125 wmax) |delta| sqrt(sum f)
    // (Cauchy-Schwarz; r <= 1.125, w = k + a r |D| <= wmax = k + 1.125 a), and
    // |delta| <= eta sqrt(S) <= eta sqrt(sum f / k).
    const double kpi = 1.0 / (2.0 * qc * qt);
    const double slope = std::max({0.0, (-std::log1p(-qc) / (qc * qc) - kpi) / qc, (-std::log(qc) / (qt * qt) - kpi) / qt});
    const double loss = 3.0 * eta * std::sqrt(1.125 * (1.0 + 1.125 * slope / kpi));
    const double widen = scale / K * (1.0 + 1e-6) / (1.0 - loss) * (1.0 + 1e-5);
    // (a class of a few samples among many: the second bound rules out nothing)
    sc.tb_k = loss < 0.5 ? (float)(kpi * widen) : 1e30f;
    sc.tb_a = loss < 0.5 ? (float)(slope * widen) : 0.f;
    sc.lb_slack = (float)(2.0 * sc.margin + scale * ncells * 8.0 * ulp32((double)N) + extra);
    return sc;
}

struct DevList {   // device allocations released together
    std::vector<void *> ptrs;
    ~DevList()
    {
        for (void *p : ptrs) (void)hipFree(p);
    }
    template <typename T>
    int alloc(T **dst, size_t n)
    {
        *dst = nullptr;
        if (dev_malloc((void **)dst, sizeof(T) * std::max<size_t>(n, 1)) != hipSuccess) return EPISDET_ERR_ALLOC;
        ptrs.push_back((void *)*dst);
        return EPISDET_OK;
    }
    template <typename T>
    int put(T **dst, const T *src, size_t n)
    {
        CHK(alloc(dst, n));
        if (n && hipMemcpy((void *)*dst, (const void *)src, sizeof(T) * n, hipMemcpyHostToDevice) != hipSuccess)
            return EPISDET_ERR_HIP;
        return EPISDET_OK;
    }
};

// Streams (default priority) with one event each, destroyed together.
struct StreamSet {
    std::vector<hipStream_t> st;
    std::vector<hipEvent_t> ev;
    int create(int k)
    {
        for (int i = 0; i < k; i++) {
            hipStream_t q;
            HIPCHK(hipStreamCreateWithFlags(&q, hipStreamNonBlocking));
            st.push_back(q);
            hipEvent_t e;
            HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
            ev.push_back(e);
        }
        return EPISDET_OK;
    }
    ~StreamSet()
    {
        for (hipEvent_t e : ev) (void)hipEventDestroy(e);
        for (hipStream_t q : st) (void)hipStreamDestroy(q);
    }
};

// Inverse of the kernels' order-preserving double key (d2key).
double key2d_host(unsigned long long k)
{
    const unsigned long long u = (k >> 63) ? (k & 0x7FFFFFFFFFFFFFFFull) : ~k;
    double d;
    std::memcpy(&d, &u, sizeof d);
    return d;
}

int ensure_pairs(episdet_dataset *ds, bool rebuild = false);

int launch_blocks(const void *kernel, int cu)
{
    int per = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, 256, 0) != hipSuccess || per < 1) per = 1;
    return per * cu;
}

// ---------------------------------------------------------------- tiles --

struct Tri3Tile {
    int A, B;
};
constexpr Tri3Tile TRI_TILES[] = {{2, 4}, {2, 2}, {2, 4}, {4, 2}};   // id 0 = default
constexpr int PAIR_TILES[] = {4, 2, 4};                               // R; id 0 = default

template <int A, int B, int MODE>
int launch_tri(episdet_dataset *ds, TriArgs &a, int grid, hipStream_t s)
{
    hipLaunchKernelGGL((k_triplets_valu<A, B, MODE>), dim3(grid), dim3(256), 0, s, a);
    HIPCHK(hipGetLastError());
    return EPISDET_OK;
}

template <int MODE>
int dispatch_tri(episdet_dataset *ds, int tile, TriArgs &a, int grid_override, hipStream_t s)
{
    const Tri3Tile t = TRI_TILES[tile];
    auto pick = [&](const void *k) { return grid_override > 0 ? grid_override : launch_blocks(k, ds->cu); };
    if (t.A == 2 && t.B == 4) return launch_tri<2, 4, MODE>(ds, a, pick((const void *)k_triplets_valu<2, 4, MODE>), s);
    if (t.A == 2 && t.B == 2) return launch_tri<2, 2, MODE>(ds, a, pick((const void *)k_triplets_valu<2, 2, MODE>), s);
    if (t.A == 4 && t.B == 2) return launch_tri<4, 2, MODE>(ds, a, pick((const void *)k_triplets_valu<4, 2, MODE>), s);
    return EPISDET_ERR_INVALID;
}

// MFMA tiles: 0 = version 2 (64 x 64 units, one 512-thread workgroup per
// CU), 1 = version 1 (32 x 64 units, register-staged chunks), 2 = version 3
// (64 x 32 units, two 256-thread workgroups per CU), 3 and 4 = version 4
// (pairs of X against 32 x 32, two workgroups per CU; 512-sample chunks
// triple-buffered, or 1024-sample chunks double-buffered), 5 = version 5
// (version 4's unit with the classes contracted in sequence by all waves).
constexpr int MFMA_TILES = 6;
inline int mfma_ty(int tile) { return tile == 1 ? MF_TY : (tile == 2 ? M3_TY : (tile >= 3 ? M4_TY : M2_TY)); }
inline int mfma_tz(int tile) { return tile == 1 ? MF_TZ : (tile == 2 ? M3_TZ : (tile >= 3 ? M4_TZ : M2_TZ)); }
inline int mfma_xstep(int tile) { return tile >= 3 ? 2 : 1; }   // X values per work unit
inline int mfma_threads(int tile) { return tile >= 2 ? 256 : 512; }
template <int MODE>
const void *mfma_kernel(int tile)
{
    if (tile == 1) return (const void *)k_triplets_mfma<MODE>;
    if (tile == 2) return (const void *)k_triplets_mfma3<MODE>;
    if (tile == 3) return (const void *)k_triplets_mfma4<MODE, 16>;
    if (tile == 4) return (const void *)k_triplets_mfma4<MODE, 32>;
    if (tile == 5) return (const void *)k_triplets_mfma5<MODE>;
    return (const void *)k_triplets_mfma2<MODE>;
}
template <int MODE>
void launch_tri_mfma(int tile, int blocks, const BatchTri &bt, hipStream_t s)
{
    if (tile == 1) hipLaunchKernelGGL((k_triplets_mfma<MODE>), dim3(blocks), dim3(512), 0, s, bt);
    else if (tile == 2) hipLaunchKernelGGL((k_triplets_mfma3<MODE>), dim3(blocks), dim3(256), 0, s, bt);
    else if (tile == 3) hipLaunchKernelGGL((k_triplets_mfma4<MODE, 16>), dim3(blocks), dim3(256), 0, s, bt);
    else if (tile == 4) hipLaunchKernelGGL((k_triplets_mfma4<MODE, 32>), dim3(blocks), dim3(256), 0, s, bt);
    else if (tile == 5) hipLaunchKernelGGL((k_triplets_mfma5<MODE>), dim3(blocks), dim3(256), 0, s, bt);
    else hipLaunchKernelGGL((k_triplets_mfma2<MODE>), dim3(blocks), dim3(512), 0, s, bt);
}

static_assert(sizeof(TriArgs) <= 1024 && sizeof(PairArgs) <= 1024, "argument slot too small");

InitArgs init_args(const episdet_dataset *ds, unsigned long long u0 = 0, unsigned seed_key = 0)
{
    return InitArgs{ds->ctl->queue,      &ds->ctl->best32, &ds->ctl->cand_count, &ds->ctl->best64,
                    &ds->ctl->checksum, u0,               seed_key};
}

// Resets the dataset's control block on its stream (queue at u0, global
// bound at seed_key, 0: +inf; no candidates) and writes a kernel's argument
// block to the dataset's slot, for a batch of one.
template <typename A>
int init_single(episdet_dataset *ds, const A &a, unsigned long long units, unsigned long long u0 = 0,
                unsigned seed_key = 0)
{
    hipLaunchKernelGGL((k_init_args<A>), dim3(1), dim3(64), 0, ds->stream, init_args(ds, u0, seed_key), a,
                       (A *)ds->jobargs, ds->jobstart, units);
    HIPCHK(hipGetLastError());
    return EPISDET_OK;
}

// The caller has written `a` to the dataset's argument slot (init_single).
template <int MODE>
int dispatch_tri_mfma(episdet_dataset *ds, int tile, TriArgs &a, hipStream_t s)
{
    const void *k = mfma_kernel<MODE>(tile);
    int per = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k, mfma_threads(tile), 0) != hipSuccess || per < 1)
        per = 1;
    BatchTri bt;
    bt.jobs = (const TriArgs *)ds->jobargs;
    bt.job_start = ds->jobstart;
    bt.njobs = 1;
    bt.total = a.nunits;
    bt.queue = a.queue;
    launch_tri_mfma<MODE>(tile, per * ds->cu, bt, s);
    HIPCHK(hipGetLastError());
    return EPISDET_OK;
}

// The MFMA path accumulates counts in FP32: exact while every class has
// fewer than 2^24 samples.
size_t plane_bytes(const episdet_dataset *ds, int c) { return (size_t)ds->nrows * 2 * ds->W[c] * sizeof(uint32_t); }

// The MFMA kernels accumulate counts in FP32, exact while every class has
// fewer than 2^24 samples, and address each class's planes with 32-bit byte
// offsets.
bool mfma_ok(const episdet_dataset *ds)
{
    return ds->N[0] < (1 << 24) && ds->N[1] < (1 << 24) && plane_bytes(ds, 0) < (1ull << 32) &&
           plane_bytes(ds, 1) < (1ull << 32);
}

template <int MODE>
int launch_pairs_batch(int R, int cu, const BatchPair &bp, hipStream_t s)
{
    if (R == 4) {
        int grid = launch_blocks((const void *)k_pairs_valu<4, MODE>, cu);
        hipLaunchKernelGGL((k_pairs_valu<4, MODE>), dim3(grid), dim3(256), 0, s, bp);
    } else if (R == 2) {
        int grid = launch_blocks((const void *)k_pairs_valu<2, MODE>, cu);
        hipLaunchKernelGGL((k_pairs_valu<2, MODE>), dim3(grid), dim3(256), 0, s, bp);
    } else if constexpr (MODE == MODE_SEARCH) {
        int grid = launch_blocks((const void *)k_pairs_valu<1, MODE>, cu);
        hipLaunchKernelGGL((k_pairs_valu<1, MODE>), dim3(grid), dim3(256), 0, s, bp);
    } else {
        return EPISDET_ERR_INTERNAL;
    }
    HIPCHK(hipGetLastError());
    return EPISDET_OK;
}

// MFMA pair tiles: 0 = 128 x 64 units, one 512-thread workgroup per CU (also
// the pair-table builder); 1 = 64 x 64 units, two 256-thread workgroups per
// CU.
constexpr int MFMA_PAIR_TILES = 2;
template <int MODE>
const void *pairs_mfma_kernel(int tile)
{
    if constexpr (MODE != MODE_PAIRTABLE)
        if (tile == 1) return (const void *)k_pairs_mfma2<MODE>;
    return (const void *)k_pairs_mfma<MODE>;
}
inline int pairs_mfma_threads(int tile) { return tile == 1 ? 256 : 512; }

template <int MODE>
int launch_pairs_mfma(int tile, int blocks, const BatchPair &bp, hipStream_t s)
{
    if constexpr (MODE != MODE_PAIRTABLE) {
        if (tile == 1) {
            hipLaunchKernelGGL((k_pairs_mfma2<MODE>), dim3(blocks), dim3(256), 0, s, bp);
            HIPCHK(hipGetLastError());
            return EPISDET_OK;
        }
    }
    hipLaunchKernelGGL((k_pairs_mfma<MODE>), dim3(blocks), dim3(512), 0, s, bp);
    HIPCHK(hipGetLastError());
    return EPISDET_OK;
}

// PairArgs for the FP4-MFMA pair kernel (128 x 64 units, B-tile-major) or
// the VALU pair kernel (square 16R tiles, triangular).
void fill_pairs(episdet_dataset *ds, PairArgs &a, bool mfma, int tile);

template <int MODE>
int dispatch_pairs(episdet_dataset *ds, bool mfma, int tile, PairArgs &a, hipStream_t s, int R = 0)
{
    BatchPair bp;
    bp.jobs = (const PairArgs *)ds->jobargs;
    bp.job_start = ds->jobstart;
    bp.njobs = 1;
    bp.total = a.nunits;
    bp.queue = a.queue;
    bp.xcd = mfma && (tile == 0 || tile == 1);
    if (mfma) {
        int per = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, pairs_mfma_kernel<MODE>(tile), pairs_mfma_threads(tile),
                                                         0) != hipSuccess ||
            per < 1)
            per = 1;
        return launch_pairs_mfma<MODE>(tile, per * ds->cu, bp, s);
    }
    return launch_pairs_batch<MODE>(R ? R : PAIR_TILES[tile], ds->cu, bp, s);
}

// Groups of 3-way units: (Y tile, Z tile) pairs that hold at least one
// X < Y < Z, each with the number of X values it needs.
void build_groups(int n, int TY, int TZ, std::vector<int2> &groups, std::vector<unsigned long long> &gstart,
                  int xstep = 1)
{
    groups.clear();
    gstart.clear();
    unsigned long long acc = 0;
    const int nty = (n + TY - 1) / TY, ntz = (n + TZ - 1) / TZ;
    for (int ty = 0; ty < nty; ty++)
        for (int tz = 0; tz < ntz; tz++) {
            const int units = group_units(n, TY, TZ, xstep, ty, tz);
            if (units <= 0) continue;
            groups.push_back(make_int2(ty, tz));
            gstart.push_back(acc);
            acc += (unsigned long long)units;
        }
    gstart.push_back(acc);
}

void fill_tri_common(episdet_dataset *ds, TriArgs &a)
{
    std::memset(&a, 0, sizeof a);
    a.p0 = ds->planes[0];
    a.p1 = ds->planes[1];
    a.bytes0 = (unsigned)std::min<size_t>(plane_bytes(ds, 0), 0xFFFFFFFFu);
    a.bytes1 = (unsigned)std::min<size_t>(plane_bytes(ds, 1), 0xFFFFFFFFu);
    a.W0 = ds->W[0];
    a.W1 = ds->W[1];
    a.n = ds->n;
    a.N0 = ds->N[0];
    a.N1 = ds->N[1];
    a.singles = ds->singles;
    a.pairs = ds->pairs;
    a.queue = ds->ctl->queue;
    a.checksum = &ds->ctl->checksum;
    a.co.best_key = &ds->ctl->best32;
    a.co.cand_count = &ds->ctl->cand_count;
    a.co.cand = ds->cand;
    a.co.cand_s32 = ds->cand_s32;
    a.co.cand_cap = ds->cand_cap;
}

void fill_pair_common(episdet_dataset *ds, PairArgs &a, int T)
{
    std::memset(&a, 0, sizeof a);
    a.p0 = ds->planes[0];
    a.p1 = ds->planes[1];
    a.bytes0 = (unsigned)std::min<size_t>(plane_bytes(ds, 0), 0xFFFFFFFFu);
    a.bytes1 = (unsigned)std::min<size_t>(plane_bytes(ds, 1), 0xFFFFFFFFu);
    a.W0 = ds->W[0];
    a.W1 = ds->W[1];
    a.n = ds->n;
    a.N0 = ds->N[0];
    a.N1 = ds->N[1];
    a.singles = ds->singles;
    a.ntiles = (ds->n + T - 1) / T;
    a.nunits = (unsigned long long)a.ntiles * (a.ntiles + 1) / 2;
    a.queue = ds->ctl->queue;
    a.checksum = &ds->ctl->checksum;
    a.co.best_key = &ds->ctl->best32;
    a.co.cand_count = &ds->ctl->cand_count;
    a.co.cand = ds->cand;
    a.co.cand_s32 = ds->cand_s32;
    a.co.cand_cap = ds->cand_cap;
}

void fill_pairs(episdet_dataset *ds, PairArgs &a, bool mfma, int tile)
{
    if (mfma && tile == 1) {
        fill_pair_common(ds, a, P3_TB);     // 64 x 64 tiles, triangular order or XCD blocks
        a.blocked = a.ntiles >= 16;
        if (a.blocked) a.nunits = blocked_units(a.ntiles);
    } else if (mfma) {
        fill_pair_common(ds, a, P2_TB);     // 128 x 64 tiles, B-tile-major or XCD blocks
        a.blocked = a.ntiles >= 16;
        a.nunits = a.blocked ? p2_blocked_units(ds->n) : p2_units(a.ntiles);
    } else {
        fill_pair_common(ds, a, 16 * PAIR_TILES[tile]);
    }
}

// The 3-way pair table, built once per dataset; rebuild = true builds it
// again in place (the planes never change, so this only makes the build
// part of a call's cost).  Not waited for: what follows on the dataset's
// stream reads it.
int ensure_pairs(episdet_dataset *ds, bool rebuild)
{
    if (ds->pairs && !rebuild) return EPISDET_OK;
    const size_t bytes = (size_t)ds->n * ds->n * 2 * sizeof(uint4);
    if (ds->pairs) {
        // built before: the same buffer
    } else if (t_scr) {
        ds->pairs = t_scr->pairs;        // restored by the no-allocation call
        if (!ds->pairs) return EPISDET_ERR_INTERNAL;
    } else if (dev_malloc((void **)&ds->pairs, bytes) != hipSuccess) {
        ds->pairs = nullptr;
        return EPISDET_ERR_ALLOC;
    }
    PairArgs a;
    const bool mfma = mfma_ok(ds);
    fill_pairs(ds, a, mfma, 0);
    a.pairs = ds->pairs;
    CHK(init_single(ds, a, a.nunits));
    return dispatch_pairs<MODE_PAIRTABLE>(ds, mfma, 0, a, ds->stream);
}

inline bool better(int score, double s, unsigned long long p, double bs, unsigned long long bp)
{
    if (score == EPISDET_SCORE_K2) {
        if (s < bs) return true;
        if (s > bs) return false;
    } else {
        if (s > bs) return true;
        if (s < bs) return false;
    }
    return p < bp;
}

void unpack(int order, unsigned long long p, int idx[3])
{
    if (order == 3) {
        idx[0] = (int)(p & 0x1FFFFF);
        idx[1] = (int)((p >> 21) & 0x1FFFFF);
        idx[2] = (int)((p >> 42) & 0x1FFFFF);
    } else {
        idx[0] = (int)(p & 0xFFFFFFFFu);
        idx[1] = (int)(p >> 32);
        idx[2] = -1;
    }
}

// Arguments of the FP64 re-scoring of the sets in ds->cand (count unset).
RescoreArgs rescore_args(const episdet_dataset *ds, int order, int score)
{
    RescoreArgs r;
    std::memset(&r, 0, sizeof r);
    r.p0 = ds->planes[0];
    r.p1 = ds->planes[1];
    r.W0 = ds->W[0];
    r.W1 = ds->W[1];
    r.n = ds->n;
    r.N0 = ds->N[0];
    r.N1 = ds->N[1];
    r.order = order;
    r.score = score;
    r.singles = ds->singles;
    r.pairs = ds->pairs;
    r.t64 = ds->tab[score].t64;
    r.cand = ds->cand;
    r.out_s64 = ds->cand_s64;
    return r;
}

// FP64 re-scoring of `count` packed sets already on the device in ds->cand.
int rescore(episdet_dataset *ds, int order, int score, int count, double *ms)
{
    if (count <= 0) {
        *ms = 0;
        return EPISDET_OK;
    }
    RescoreArgs r = rescore_args(ds, order, score);
    r.count = count;
    Timer tm;
    CHK(tm.make());
    HIPCHK(hipEventRecord(tm.e0, ds->stream));
    hipLaunchKernelGGL(k_rescore, dim3(count), dim3(64), 0, ds->stream, r);
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(tm.e1, ds->stream));
    HIPCHK(hipEventSynchronize(tm.e1));
    float f = 0;
    HIPCHK(hipEventElapsedTime(&f, tm.e0, tm.e1));
    *ms = f;
    return EPISDET_OK;
}

// Re-scored candidates gathered over one or more launches: the winner (FP64
// score, then the lowest packed index), the FP32-vs-FP64 error over every
// candidate, and for top-k the best topk so far.
struct Collected {
    int score = 0, topk = 0;
    bool have = false;
    double bs = 0;                  // FP64 score of the winner
    unsigned long long bp = ~0ull;  // its packed index
    float b32 = 0.f;                // its FP32 score
    double maxabs = 0, maxrel = 0;
    long long count = 0;
    std::vector<std::pair<double, unsigned long long>> top;   // better() order, at most topk
};

// Adds `count` re-scored candidates (host copies) to acc.
int collect_host(const unsigned long long *hp, const float *h32, const double *h64, int count, Collected &acc)
{
    if (count <= 0) return EPISDET_OK;
    const int score = acc.score;
    for (int i = 0; i < count; i++) {
        if (std::isnan(h64[i])) return EPISDET_ERR_INTERNAL;   // inconsistent count tables
        const double s32 = score == EPISDET_SCORE_K2 ? (double)h32[i] : -(double)h32[i];
        const double err = std::fabs(s32 - h64[i]);
        acc.maxabs = std::max(acc.maxabs, err);
        if (h64[i] != 0) acc.maxrel = std::max(acc.maxrel, err / std::fabs(h64[i]));
        if (!acc.have || better(score, h64[i], hp[i], acc.bs, acc.bp)) {
            acc.have = true;
            acc.bs = h64[i];
            acc.bp = hp[i];
            acc.b32 = (float)s32;
        }
    }
    if (acc.topk > 1) {
        for (int i = 0; i < count; i++) acc.top.emplace_back(h64[i], hp[i]);
        const size_t m = std::min<size_t>((size_t)acc.topk, acc.top.size());
        std::partial_sort(acc.top.begin(), acc.top.begin() + m, acc.top.end(),
                          [&](const std::pair<double, unsigned long long> &a,
                              const std::pair<double, unsigned long long> &b) {
                              return better(score, a.first, a.second, b.first, b.second);
                          });
        acc.top.resize(m);
    }
    acc.count += count;
    return EPISDET_OK;
}

// Adds the `count` candidates re-scored on the device (ds->cand,
// ds->cand_s32, ds->cand_s64) to acc.
int collect(episdet_dataset *ds, int count, Collected &acc)
{
    if (count <= 0) return EPISDET_OK;
    std::vector<unsigned long long> hp(count);
    std::vector<float> h32(count);
    std::vector<double> h64(count);
    HIPCHK(hipMemcpy(hp.data(), ds->cand, sizeof(unsigned long long) * count, hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(h32.data(), ds->cand_s32, sizeof(float) * count, hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(h64.data(), ds->cand_s64, sizeof(double) * count, hipMemcpyDeviceToHost));
    return collect_host(hp.data(), h32.data(), h64.data(), count, acc);
}

// The parts of a dataset's pinned staging area (k_rescore_after's HostStage),
// by their host (base = stage) or device (base = stage_dev) addresses.
unsigned *stage_ctl(unsigned char *base) { return (unsigned *)base; }
unsigned long long *stage_packed(unsigned char *base) { return (unsigned long long *)(base + 256); }
float *stage_s32(unsigned char *base) { return (float *)(base + 256 + 8 * (size_t)STAGE_CAND); }
double *stage_s64(unsigned char *base) { return (double *)(base + 256 + 12 * (size_t)STAGE_CAND); }

HostStage host_stage(episdet_dataset *ds, unsigned cap)
{
    HostStage hs;
    hs.ctl = stage_ctl(ds->stage_dev);
    hs.packed = stage_packed(ds->stage_dev);
    hs.s32 = stage_s32(ds->stage_dev);
    hs.s64 = stage_s64(ds->stage_dev);
    hs.slots = std::min<unsigned>(cap, STAGE_CAND);
    return hs;
}

// Adds the `count` candidates a search left: from the staging area if they
// all fit it.
int collect_staged(episdet_dataset *ds, int count, Collected &acc)
{
    if (count > (int)STAGE_CAND) return collect(ds, count, acc);
    return collect_host(stage_packed(ds->stage), stage_s32(ds->stage), stage_s64(ds->stage), count, acc);
}

// Writes the gathered winner (and, for top-k, the ranking) into res and ds.
int finish(episdet_dataset *ds, int order, const Collected &acc, episdet_result *res)
{
    if (!acc.have) return EPISDET_ERR_INTERNAL;   // the winner is always a candidate
    res->best_score = acc.bs;
    res->best_score_f32 = acc.b32;
    res->packed = acc.bp;
    unpack(order, acc.bp, res->idx);
    res->fp32_max_abs_err = acc.maxabs;
    res->fp32_max_rel_err = acc.maxrel;
    res->candidates = acc.count;
    if (acc.topk > 1) {
        ds->topk_packed.resize(acc.top.size());
        ds->topk_scores.resize(acc.top.size());
        for (size_t i = 0; i < acc.top.size(); i++) {
            ds->topk_packed[i] = acc.top[i].second;
            ds->topk_scores[i] = acc.top[i].first;
        }
    }
    return EPISDET_OK;
}

// Winner of `count` candidates already re-scored and staged by the device.
int collect_best(episdet_dataset *ds, int order, int score, int count, episdet_result *res)
{
    Collected acc;
    acc.score = score;
    CHK(collect_staged(ds, count, acc));
    return finish(ds, order, acc, res);
}

// One fused kernel configuration for one dataset and search: the argument
// block; the 3-way work-unit groups are the dataset's (ensure_groups).
struct FusedPlan {
    int order = 0, score = 0, path = 0, tile = 0;
    bool mfma = false;
    TriArgs ta{};
    PairArgs pa{};
    ScoreCtx sc{};
    unsigned long long nunits = 0;
    unsigned seed_key = 0;       // starting global bound (best32), 0: none
    int pr = 0;                  // VALU 2-way: units of 16 pr x 16 pr
    int seed_pairs = 0;          // 3-way: > 0: the launch starts from the triplets of this many best pairs
    void group_tile(int (&t)[3]) const
    {
        t[0] = mfma ? mfma_ty(tile) : 16 * TRI_TILES[tile].A;
        t[1] = mfma ? mfma_tz(tile) : 16 * TRI_TILES[tile].B;
        t[2] = mfma ? mfma_xstep(tile) : 1;
    }
};

// The 3-way work-unit groups of a tile in the dataset's buffers, listed on
// its stream; kept while searches use the same tile.  *ngroups and *nunits: their
// numbers.  Every tile is at least 32 x 32, which sizes the buffers.
int ensure_groups(episdet_dataset *ds, const int (&t)[3], int *ngroups, unsigned long long *nunits)
{
    const size_t side = ((size_t)ds->n + 31) / 32, most = side * (side + 1) / 2;
    if (!t_scr && !ds->gstart) {
        if (dev_malloc((void **)&ds->gstart, sizeof(unsigned long long) * (most + 1)) != hipSuccess ||
            dev_malloc((void **)&ds->groups, sizeof(int2) * most) != hipSuccess) {
            if (ds->gstart) (void)hipFree(ds->gstart);
            ds->gstart = nullptr;
            ds->groups = nullptr;
            return EPISDET_ERR_ALLOC;
        }
    }
    const int nty = (ds->n + t[0] - 1) / t[0], ntz = (ds->n + t[1] - 1) / t[1];
    size_t g = 0;
    unsigned long long u = 0;
    for (int ty = 0; ty < nty; ty++)
        for (int tz = (int)((long long)ty * t[0] / t[1]); tz < ntz; tz++) {
            const int k = group_units(ds->n, t[0], t[1], t[2], ty, tz);
            u += (unsigned long long)k;
            g += k > 0;
        }
    if (g == 0) return EPISDET_ERR_INVALID;
    if (g > most || (t_scr && g > t_scr->max_groups)) return EPISDET_ERR_INTERNAL;
    *ngroups = (int)g;
    *nunits = u;
    if (!t_scr && std::memcmp(ds->group_tile, t, sizeof t) == 0) return EPISDET_OK;
    hipLaunchKernelGGL(k_groups, dim3(1), dim3(1024), 0, ds->stream, ds->n, t[0], t[1], t[2], ds->groups, ds->gstart);
    HIPCHK(hipGetLastError());
    if (!t_scr) std::memcpy(ds->group_tile, t, sizeof t);
    return EPISDET_OK;
}

bool tile_valid(int order, int path, int tile)
{
    if (tile < 0) return false;
    if (path == EPISDET_PATH_FUSED_MFMA) return tile < (order == 3 ? MFMA_TILES : MFMA_PAIR_TILES);
    if (order == 3) return tile < (int)(sizeof TRI_TILES / sizeof TRI_TILES[0]);
    return tile < (int)(sizeof PAIR_TILES / sizeof PAIR_TILES[0]);
}

// Tables, pair table and candidate buffer must exist (ensure_*) before.
int plan_fused(episdet_dataset *ds, int order, int score, int path, int tile, FusedPlan &pl, int topk = 0)
{
    pl.order = order;
    pl.score = score;
    pl.path = path;
    pl.tile = tile;
    pl.mfma = path == EPISDET_PATH_FUSED_MFMA;
    if (pl.mfma && !mfma_ok(ds)) return EPISDET_ERR_INVALID;
    if (!tile_valid(order, path, tile)) return EPISDET_ERR_INVALID;
    pl.sc = make_ctx(ds, score, order);
    if (order == 3) {
        int t[3], ngroups = 0;
        pl.group_tile(t);
        CHK(ensure_groups(ds, t, &ngroups, &pl.nunits));
        fill_tri_common(ds, pl.ta);
        pl.ta.sc = pl.sc;
        pl.ta.gstart = ds->gstart;
        pl.ta.groups = ds->groups;
        pl.ta.ngroups = ngroups;
        pl.ta.nunits = pl.nunits;
    } else {
        fill_pairs(ds, pl.pa, pl.mfma, tile);
        if (!pl.mfma) {
            pl.pr = PAIR_TILES[tile];
            // VALU tile 1 with at most 3/2 units of 16 x 16 a CU (432 SNPs):
            // units of that size, one pair a thread, so a quarter of the serial
            // work each.  A search, 32 x 32 and 16 x 16 units: 53 and 49 us at
            // 64 x 500, 63 and 57 at 400 x 4000, 61 and 53 at 256 x 4096 (MI).
            // From two units a CU their turns cost more: 57 and 60 us at 512 x
            // 2048, 59 and 65 at 640 x 2000.  Not for top-k, which may ask for
            // 1024 sets of a unit.
            const unsigned long long t = (unsigned long long)(ds->n + 15) / 16, u = t * (t + 1) / 2;
            if (pl.pr == 2 && !topk && 2 * u <= 3ull * (unsigned long long)ds->cu) {
                pl.pr = 1;
                fill_pair_common(ds, pl.pa, 16);
            }
        }
        pl.pa.sc = pl.sc;
        pl.nunits = pl.pa.nunits;
    }
    return EPISDET_OK;
}

// Most sets one work unit of a plan can append: a candidate buffer at least
// this large always holds a launch over any one unit.
unsigned long long unit_sets_max(const FusedPlan &pl)
{
    if (pl.order == 3) {
        if (pl.mfma) return (unsigned long long)mfma_xstep(pl.tile) * mfma_ty(pl.tile) * mfma_tz(pl.tile);
        const Tri3Tile t = TRI_TILES[pl.tile];
        return 256ull * t.A * t.B;
    }
    if (pl.mfma) return pl.tile == 0 ? (unsigned long long)P2_TA * P2_TB : (unsigned long long)P3_TA * P3_TB;
    return 256ull * PAIR_TILES[pl.tile] * PAIR_TILES[pl.tile];
}

// A starting global bound for a 3-way search, on its stream between the reset
// of the control block and the search (kernels_seed.hpp): the best FP32
// badness among the triplets that contain one of the best pairs, or for top-k
// the k-th best.  Some sets reach it, as they reach the minimum a workgroup
// publishes, so the winner, the k best and every set tied with them still
// become candidates; the score bounds then skip FP32 scores from the first unit on when
// strongly associated triplets have associated pairs.
constexpr int SEED_PAIRS = 4;
SeedArgs seed_args_of(episdet_dataset *ds, int score, const ScoreCtx &sc, int npairs, bool topk)
{
    SeedArgs a;
    std::memset(&a, 0, sizeof a);
    a.r = rescore_args(ds, 3, score);
    a.r.cand = nullptr;
    a.r.out_s64 = nullptr;
    a.sc = sc;
    a.blk = ds->seed;
    a.pick = ds->seed + 2 * SEED_BLOCKS;
    a.blocks = std::min(SEED_BLOCKS, ds->n - 1);
    a.npairs = npairs;
    a.best_key = &ds->ctl->best32;
    a.s32 = topk ? ds->cand_s32 : nullptr;     // free until the search appends
    return a;
}

int seed_from_pairs(episdet_dataset *ds, const FusedPlan &pl, int topk)
{
    const SeedArgs a = seed_args_of(ds, pl.score, pl.sc, pl.seed_pairs, topk != 0);
    const int m = a.npairs * ds->n;
    hipLaunchKernelGGL(k_seed_pairs<SeedArgs>, dim3(a.blocks), dim3(256), 0, ds->stream, a);
    hipLaunchKernelGGL(k_seed_pick<SeedArgs>, dim3(1), dim3(SEED_BLOCKS), 0, ds->stream, a);
    hipLaunchKernelGGL(k_seed_triplets<SeedArgs>, dim3((m + 3) / 4), dim3(256), 0, ds->stream, a);
    if (topk)
        hipLaunchKernelGGL(k_seed_kth, dim3(1), dim3(1024), 0, ds->stream, ds->cand_s32, m, (unsigned)topk,
                           &ds->ctl->best32);
    HIPCHK(hipGetLastError());
    return EPISDET_OK;
}

// Pairs whose triplets seed a 3-way search (0: none): 4 for the best set; for
// the k best enough to hold about 2 k triplets, if those fit the candidate
// slots they are kept in.  A no-allocation call goes without, and so does a
// top-k search whose caller sets the candidate slots: those are chosen to
// force the windowed rerun, whose windows start from exact scores.
int seed_pairs(const episdet_dataset *ds, int topk, bool own_cap)
{
    if (t_scr || ds->n < 4) return 0;
    if (!topk) return SEED_PAIRS;
    if (own_cap) return 0;
    const int p = std::min({std::max(SEED_PAIRS, (2 * topk + ds->n - 3) / (ds->n - 2)), SEED_MAX_PAIRS, ds->n - 1});
    return (long long)p * ds->n <= (long long)ds->cand_cap ? p : 0;
}

// Issues the plan over work units [u0, u1) (the whole search is
// [0, nunits)) with `cap` candidate slots and the global bound starting at
// seed_key (0: +inf), between events e0 and e1 on the dataset's stream; does
// not wait for it.  The argument block is uploaded before e0, so the events
// time the search kernel alone.
int issue_fused(episdet_dataset *ds, FusedPlan &pl, int topk, unsigned long long u0, unsigned long long u1,
                unsigned cap, unsigned seed_key, hipEvent_t e0, hipEvent_t e1)
{
    if (cap > ds->cand_cap) return EPISDET_ERR_INTERNAL;
    TriArgs &ta = pl.ta;
    PairArgs &pa = pl.pa;
    ta.co.cand = pa.co.cand = ds->cand;
    ta.co.cand_s32 = pa.co.cand_s32 = ds->cand_s32;
    ta.co.cand_cap = pa.co.cand_cap = cap;
    ta.co.topk = pa.co.topk = (unsigned)topk;
    // the launch covers units [u0, u1): the queue starts at u0 and the
    // kernels stop at nunits (restored below)
    ta.nunits = pa.nunits = u1;
    struct Restore {
        FusedPlan &pl;
        ~Restore() { pl.ta.nunits = pl.pa.nunits = pl.nunits; }
    } restore{pl};
    const int order = pl.order, tile = pl.tile;
    const bool mfma = pl.mfma;
    int rc = EPISDET_OK;
    // the batched kernels read their argument block from device memory (the
    // VALU 3-way kernel takes it by value, and only finds a copy there)
    if (order == 3) CHK(init_single(ds, ta, ta.nunits, u0, seed_key));
    else CHK(init_single(ds, pa, pa.nunits, u0, seed_key));
    if (pl.seed_pairs > 0) CHK(seed_from_pairs(ds, pl, topk));
    // the kernels that tighten the top-k bound from the candidates' own scores
    // (tighten_topk) must find +inf in slots not written yet
    if (topk && mfma && (order == 3 ? tile >= 3 : tile == 1)) {
        hipLaunchKernelGGL(k_fill_f32, dim3(4 * ds->cu), dim3(256), 0, ds->stream, ds->cand_s32, cap, INFINITY);
        HIPCHK(hipGetLastError());
    }
    HIPCHK(hipEventRecord(e0, ds->stream));
    if (topk)
        rc = order == 3 ? (mfma ? dispatch_tri_mfma<MODE_TOPK>(ds, tile, ta, ds->stream)
                                : dispatch_tri<MODE_TOPK>(ds, tile, ta, 0, ds->stream))
                        : dispatch_pairs<MODE_TOPK>(ds, mfma, tile, pa, ds->stream);
    else
        rc = order == 3 ? (mfma ? dispatch_tri_mfma<MODE_SEARCH>(ds, tile, ta, ds->stream)
                                : dispatch_tri<MODE_SEARCH>(ds, tile, ta, 0, ds->stream))
                        : dispatch_pairs<MODE_SEARCH>(ds, mfma, tile, pa, ds->stream, pl.pr);
    HIPCHK(hipEventRecord(e1, ds->stream));
    return rc;
}

// issue_fused, waiting for the search: its kernel time in *ms.
int launch_fused(episdet_dataset *ds, FusedPlan &pl, int topk, unsigned long long u0, unsigned long long u1,
                 unsigned cap, unsigned seed_key, float *ms)
{
    Timer tm;
    CHK(tm.make());
    int rc = issue_fused(ds, pl, topk, u0, u1, cap, seed_key, tm.e0, tm.e1);
    const bool synced = hipEventSynchronize(tm.e1) == hipSuccess;
    float k = 0;
    if (synced) (void)hipEventElapsedTime(&k, tm.e0, tm.e1);
    if (rc == EPISDET_OK && !synced) rc = EPISDET_ERR_HIP;
    *ms = k;
    return rc;
}

// The whole search in one synchronisation: the launch, then on the same
// stream the FP64 re-scoring of the candidates it appended (count read on the
// device), which also writes the candidate count, the overflow flag and the
// first STAGE_CAND candidates into the dataset's pinned staging area.
// hc->cand_count and hc->cand_over receive the count and the flag; the
// search's and the re-scoring's device times go to *kms, *rms.
int launch_fused_rescored(episdet_dataset *ds, FusedPlan &pl, int topk, unsigned cap, unsigned seed_key, float *kms,
                          float *rms, Ctl *hc)
{
    int rc = issue_fused(ds, pl, topk, 0, pl.nunits, cap, seed_key, ds->ev[0], ds->ev[1]);
    if (rc == EPISDET_OK) {
        const RescoreArgs r = rescore_args(ds, pl.order, pl.score);
        const HostStage hs = host_stage(ds, cap);
        const unsigned grid = std::min<unsigned>(cap, 16u * (unsigned)ds->cu);
        hipLaunchKernelGGL(k_rescore_after, dim3(grid), dim3(64), 0, ds->stream, r, &ds->ctl->cand_count, cap,
                           (const float *)ds->cand_s32, hs);
        if (hipGetLastError() != hipSuccess) rc = EPISDET_ERR_HIP;
    }
    if (rc == EPISDET_OK && hipEventRecord(ds->ev[2], ds->stream) != hipSuccess) rc = EPISDET_ERR_HIP;
    // wait even after an error, so no kernel is left writing the staging area
    const bool synced = hipStreamSynchronize(ds->stream) == hipSuccess;
    if (rc != EPISDET_OK) return rc;
    if (!synced) return EPISDET_ERR_HIP;
    HIPCHK(hipEventElapsedTime(kms, ds->ev[0], ds->ev[1]));
    HIPCHK(hipEventElapsedTime(rms, ds->ev[1], ds->ev[2]));
    std::memset(hc, 0, sizeof *hc);
    hc->cand_count = stage_ctl(ds->stage)[0];
    hc->cand_over = stage_ctl(ds->stage)[1];
    return EPISDET_OK;
}

int choose_kernel(episdet_dataset *ds, int order, int score, int *path, int *tile, bool tune, bool single = false);

// Order-preserving key of a float, as f2key in the kernels.
unsigned f2key_host(float f)
{
    unsigned u;
    std::memcpy(&u, &f, sizeof u);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// ------------------------------------------------------------ autotuner --
//
// For each shape (order, score, n, W0, W1) the tuner times every kernel
// configuration that can run it on a window of work units from the middle
// of its queue (three waves of resident workgroups, or the whole search if
// it is smaller), counts the sets in that window exactly, and predicts the
// whole search as time x all sets / window sets.  The fastest prediction is
// cached for the process and used by AUTO.

struct TuneKey {
    int order, score, n, W0, W1;
    bool operator<(const TuneKey &o) const
    {
        return std::tie(order, score, n, W0, W1) < std::tie(o.order, o.score, o.n, o.W0, o.W1);
    }
};
struct TuneChoice {
    int path, tile;
};
std::mutex g_tune_mu;
std::map<TuneKey, TuneChoice> g_tune;

void host_unrank_tri(unsigned long long u, long long &ta, long long &tb)
{
    long long b = (long long)((std::sqrt(8.0 * (double)u + 1.0) - 1.0) * 0.5);
    while ((unsigned long long)(b + 1) * (unsigned long long)(b + 2) / 2 <= u) b++;
    while ((unsigned long long)b * (unsigned long long)(b + 1) / 2 > u) b--;
    tb = b;
    ta = (long long)(u - (unsigned long long)b * (unsigned long long)(b + 1) / 2);
}

void host_unrank_p2(unsigned long long u, long long &ta, long long &tb)
{
    long long m = (long long)((std::sqrt(4.0 * (double)u + 1.0) - 1.0) * 0.5);
    while ((unsigned long long)(m + 1) * (unsigned long long)(m + 2) <= u) m++;
    while ((unsigned long long)m * (unsigned long long)(m + 1) > u) m--;
    const unsigned long long e = (unsigned long long)m * (unsigned long long)(m + 1);
    if (u < e + (unsigned long long)(m + 1)) {
        tb = 2 * m;
        ta = (long long)(u - e);
    } else {
        tb = 2 * m + 1;
        ta = (long long)(u - (unsigned long long)(m + 1) * (unsigned long long)(m + 1));
    }
}

// Valid sets (X < Y < Z < n, or A < B < n) in work units [u0, u1) of a plan.
unsigned long long count_sets(const episdet_dataset *ds, const FusedPlan &pl, unsigned long long u0,
                              unsigned long long u1)
{
    const long long n = ds->n;
    unsigned long long total = 0;
    if (pl.order == 3) {
        const long long TY = pl.mfma ? mfma_ty(pl.tile) : 16 * TRI_TILES[pl.tile].A;
        const long long TZ = pl.mfma ? mfma_tz(pl.tile) : 16 * TRI_TILES[pl.tile].B;
        const long long XS = pl.mfma ? mfma_xstep(pl.tile) : 1;
        std::vector<int2> groups;
        std::vector<unsigned long long> gstart;
        build_groups(ds->n, (int)TY, (int)TZ, groups, gstart, (int)XS);
        size_t g = (size_t)(std::upper_bound(gstart.begin(), gstart.end(), u0) - gstart.begin()) - 1;
        for (unsigned long long u = u0; u < u1; u++) {
            while (g + 1 < groups.size() && gstart[g + 1] <= u) g++;
            const long long ylo = (long long)groups[g].x * TY, zlo = (long long)groups[g].y * TZ;
            const long long zhi = std::min(zlo + TZ, n);
            for (long long X = XS * (long long)(u - gstart[g]); X < XS * (long long)(u - gstart[g] + 1); X++)
                for (long long Y = std::max(ylo, X + 1); Y < std::min(ylo + TY, n); Y++) {
                    const long long z0 = std::max(zlo, Y + 1);
                    if (zhi > z0) total += (unsigned long long)(zhi - z0);
                }
        }
    } else {
        const bool p2 = pl.mfma && pl.tile == 0;   // 128 x 64 order; the others are triangular
        const long long TA = p2 ? P2_TA : (pl.mfma ? P3_TA : 16 * pl.pr);
        const long long TB = p2 ? P2_TB : (pl.mfma ? P3_TB : 16 * pl.pr);
        for (unsigned long long u = u0; u < u1; u++) {
            long long ta, tb;
            if (p2 && pl.pa.blocked) {
                int a, b;
                if (!p2_blocked_unrank(u, (int)n, a, b)) continue;
                ta = a;
                tb = b;
            } else if (p2) {
                host_unrank_p2(u, ta, tb);
            } else if (pl.mfma && pl.pa.blocked) {
                int a, b;
                if (!blocked_unrank(u, pl.pa.ntiles, a, b)) continue;
                ta = a;
                tb = b;
            } else {
                host_unrank_tri(u, ta, tb);
            }
            const long long b0 = tb * TB, bhi = std::min(b0 + TB, n);
            for (long long A = ta * TA; A < std::min(ta * TA + TA, n); A++) {
                const long long blo = std::max(b0, A + 1);
                if (bhi > blo) total += (unsigned long long)(bhi - blo);
            }
        }
    }
    return total;
}

int occupancy_blocks(const void *k, int threads, int cu)
{
    int per = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k, threads, 0) != hipSuccess || per < 1) per = 1;
    return per * cu;
}

// Workgroups a plan's search launch keeps resident.
unsigned long long resident_blocks(const episdet_dataset *ds, const FusedPlan &pl)
{
    const int cu = ds->cu;
    if (pl.order == 3) {
        if (pl.mfma)
            return (unsigned long long)occupancy_blocks(mfma_kernel<MODE_SEARCH>(pl.tile), mfma_threads(pl.tile), cu);
        const Tri3Tile t = TRI_TILES[pl.tile];
        if (t.A == 2 && t.B == 2) return (unsigned long long)launch_blocks((const void *)k_triplets_valu<2, 2, MODE_SEARCH>, cu);
        if (t.A == 4 && t.B == 2) return (unsigned long long)launch_blocks((const void *)k_triplets_valu<4, 2, MODE_SEARCH>, cu);
        return (unsigned long long)launch_blocks((const void *)k_triplets_valu<2, 4, MODE_SEARCH>, cu);
    }
    if (pl.mfma)
        return (unsigned long long)occupancy_blocks(pairs_mfma_kernel<MODE_SEARCH>(pl.tile), pairs_mfma_threads(pl.tile),
                                                    cu);
    if (pl.pr == 1) return (unsigned long long)launch_blocks((const void *)k_pairs_valu<1, MODE_SEARCH>, cu);
    if (pl.pr == 2) return (unsigned long long)launch_blocks((const void *)k_pairs_valu<2, MODE_SEARCH>, cu);
    return (unsigned long long)launch_blocks((const void *)k_pairs_valu<4, MODE_SEARCH>, cu);
}

// Times every configuration for this dataset's shape; fills `table` (may be
// null) and returns the fastest in path / tile.
int tune_kernel(episdet_dataset *ds, int order, int score, std::vector<episdet_tune_entry> *table, int *path,
                int *tile)
{
    std::vector<std::pair<int, int>> cands;
    if (mfma_ok(ds)) {
        cands.push_back({EPISDET_PATH_FUSED_MFMA, 0});
        for (int t = 1; t < (order == 3 ? MFMA_TILES : MFMA_PAIR_TILES); t++)
            cands.push_back({EPISDET_PATH_FUSED_MFMA, t});
    }
    if (order == 3) {
        cands.push_back({EPISDET_PATH_FUSED_VALU, 0});
        cands.push_back({EPISDET_PATH_FUSED_VALU, 1});
        cands.push_back({EPISDET_PATH_FUSED_VALU, 3});
    } else {
        cands.push_back({EPISDET_PATH_FUSED_VALU, 0});
        cands.push_back({EPISDET_PATH_FUSED_VALU, 1});
    }
    CHK(ensure_tables(ds, score));
    if (order == 3) CHK(ensure_pairs(ds));
    CHK(ensure_cand(ds, DEFAULT_CAP));
    const double all_sets = (double)episdet_n_choose_k((unsigned)ds->n, (unsigned)order);
    double best = INFINITY;
    for (const auto &c : cands) {
        FusedPlan pl;
        CHK(plan_fused(ds, order, score, c.first, c.second, pl));
        const unsigned long long k = std::min<unsigned long long>(pl.nunits, 3 * resident_blocks(ds, pl));
        const unsigned long long u0 = (pl.nunits - k) / 2;
        const unsigned long long sets = count_sets(ds, pl, u0, u0 + k);
        float ms = 0;
        CHK(launch_fused(ds, pl, 0, u0, u0 + k, ds->cand_cap, 0, &ms));   // first launch loads the code object
        CHK(launch_fused(ds, pl, 0, u0, u0 + k, ds->cand_cap, 0, &ms));
        const double est = sets ? (double)ms * all_sets / (double)sets : INFINITY;
        if (table) {
            episdet_tune_entry e;
            std::memset(&e, 0, sizeof e);
            e.path = c.first;
            e.tile = c.second;
            e.est_ms = est;
            e.sample_ms = ms;
            e.sample_sets = (long long)sets;
            table->push_back(e);
        }
        if (est < best) {
            best = est;
            *path = c.first;
            *tile = c.second;
        }
    }
    return best < INFINITY ? EPISDET_OK : EPISDET_ERR_INTERNAL;
}

// The kernel AUTO runs: the tuned choice for this shape if there is one (or
// tune now when asked), else the FP4-MFMA kernels wherever they are exact
// (fewer than 2^24 samples per class, planes below 4 GiB per class) and the
// VALU kernels otherwise.
int choose_kernel(episdet_dataset *ds, int order, int score, int *path, int *tile, bool tune, bool single)
{
    const TuneKey key{order, score, ds->n, ds->W[0], ds->W[1]};
    {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        auto it = g_tune.find(key);
        if (it != g_tune.end()) {
            *path = it->second.path;
            *tile = it->second.tile;
            return EPISDET_OK;
        }
    }
    if (tune) {
        CHK(tune_kernel(ds, order, score, nullptr, path, tile));
        std::lock_guard<std::mutex> lk(g_tune_mu);
        g_tune[key] = TuneChoice{*path, *tile};
        return EPISDET_OK;
    }
    // A small 2-way search of few samples on its own (not in a batch, whose
    // graph runs MFMA kernels): the VALU kernel of 32 x 32 units spreads it
    // over more workgroups than the MFMA kernel's 64 x 64 units, which leave
    // most CUs idle.  Whole K2 searches at 2048 samples took 53 / 59 / 61 us
    // against 73 / 76 / 69 us at 64 / 256 / 512 SNPs, but 77 against 73 us at 1024
    // SNPs, and with more samples a unit's count is the longer part and the
    // matrix cores win: 87 against 81 us at 256 x 8192, 155 against 98 us at 300 x
    // 20000, 416 against 226 us at 100 x 100000.  So the VALU kernel is chosen
    // below 1e9 set-samples and up to 4096 samples.
    if (single && order == 2 &&
        ds->N[0] + ds->N[1] <= 4096 &&
        (double)episdet_n_choose_k((unsigned)ds->n, 2) * (double)(ds->N[0] + ds->N[1]) < 1e9) {
        *path = EPISDET_PATH_FUSED_VALU;
        *tile = 1;
        return EPISDET_OK;
    }
    *path = mfma_ok(ds) ? EPISDET_PATH_FUSED_MFMA : EPISDET_PATH_FUSED_VALU;
    // 3-way: version 4 (pairs of X, two workgroups per CU) with 1024-sample
    // chunks measured fastest at both 4096 x 262144 (6.79 s against 7.08 s
    // with 512-sample chunks and 7.27 s for version 2) and 8192 x 65536
    // (16.2 s against 16.8 s, 17.0 s for version 3, 18.4 s for version 2).
    // 2-way: the 64 x 64 kernel with the classes in sequence (tile 1)
    // measured 11.9 ms against 12.8 ms at 16384 x 65536 (40/60 classes).
    // 3-way with uneven classes: version 5 (tile 5) takes the same time for
    // any split, version 4 is 12% faster at 50/50 but slower once the
    // smaller class has under ~2/3 of the larger's samples (2048 SNPs x
    // 131072 samples: 452 / 517 / 581 / 659 ms for version 4 at 50/50,
    // 40/60, 30/70, 20/80 against 505 / 512 / 512 / 513 ms for version 5).
    if (*path != EPISDET_PATH_FUSED_MFMA) *tile = 0;
    else if (order == 2) *tile = 1;
    else *tile = 100LL * std::min(ds->W[0], ds->W[1]) < 65LL * std::max(ds->W[0], ds->W[1]) ? 5 : 4;
    return EPISDET_OK;
}

// Key of the smallest float at or above badness + margin / 2, or 0 when
// that is not finite.  A launch seeded with it keeps as candidates every set
// whose exact badness is at or below `badness` (each FP32 badness is within
// half the margin of the exact one).
unsigned seed_key_above(double badness, float margin)
{
    const double bound = badness + 0.5 * (double)margin;
    float f = (float)bound;
    if ((double)f < bound) f = std::nextafter(f, INFINITY);
    if (!std::isfinite(f)) return 0u;
    return f2key_host(f);
}

// Exact answer after a candidate overflow (heavy ties, degenerate data): the
// work queue is searched again in consecutive unit windows, each re-scored
// in FP64 and gathered before the next, so no window holds more candidates
// than the buffer.  A window of cap / unit_sets_max(pl) units can never
// overflow; windows start larger when the first launch's count allows and
// double while they stay well below the cap.  Each window's global bound
// starts at the best exact badness gathered so far (the k-th best for
// top-k) plus half the margin, which keeps every set that can still win.
int run_sliced(episdet_dataset *ds, FusedPlan &pl, int topk, unsigned cap, const Ctl &first, Collected &acc,
               double *kms_total, double *rms_total)
{
    const unsigned long long floor_step = std::max<unsigned long long>(1ull, cap / unit_sets_max(pl));
    unsigned long long step = floor_step;
    // the first launch appended at least cand_count sets when that exceeds
    // the cap (more if the count wrapped, which the shrinking below absorbs)
    if (first.cand_count > cap)
        step = std::max(step, (unsigned long long)((double)pl.nunits * (double)cap / (2.0 * first.cand_count)));
    const float margin = pl.sc.margin;
    for (unsigned long long u = 0; u < pl.nunits;) {
        const unsigned long long u1 = std::min(pl.nunits, u + step);
        unsigned seed = pl.seed_key;
        const bool bounded = topk ? (int)acc.top.size() >= topk : acc.have;
        if (bounded) {
            const double s = topk ? acc.top.back().first : acc.bs;
            const unsigned k = seed_key_above(pl.score == EPISDET_SCORE_K2 ? s : -s, margin);
            if (k && (!seed || k < seed)) seed = k;
        }
        float kms = 0;
        CHK(launch_fused(ds, pl, topk, u, u1, cap, seed, &kms));
        *kms_total += kms;
        Ctl hc;
        HIPCHK(hipMemcpy(&hc, ds->ctl, sizeof hc, hipMemcpyDeviceToHost));
        if (hc.cand_over || hc.cand_count > cap) {
            if (step <= floor_step) return EPISDET_ERR_INTERNAL;   // cannot happen: see above
            step = std::max(floor_step, step / 4);
            continue;
        }
        double rms = 0;
        CHK(rescore(ds, pl.order, pl.score, (int)hc.cand_count, &rms));
        *rms_total += rms;
        CHK(collect(ds, (int)hc.cand_count, acc));
        u = u1;
        if (hc.cand_count < cap / 8) step *= 2;
    }
    return EPISDET_OK;
}

// Fused search: one persistent launch, then FP64 re-scoring of the
// candidates.  With o->topk > 1 the candidates cover the topk best sets.
int run_fused(episdet_dataset *ds, const episdet_options *o, episdet_result *res)
{
    const int order = o->order, score = o->score;
    int path = o->path, tile = o->tile;
    const int topk = o->topk > 1 ? o->topk : 0;
    if (topk > EPISDET_TOPK_MAX) return EPISDET_ERR_INVALID;
    CHK(ensure_tables(ds, score));
    if (order == 3) CHK(ensure_pairs(ds));
    if (path == EPISDET_PATH_AUTO) CHK(choose_kernel(ds, order, score, &path, &tile, o->autotune != 0, true));
    FusedPlan pl;
    CHK(plan_fused(ds, order, score, path, tile, pl, topk));
    // Candidate slots of this search: the requested capacity, by default 1M
    // and for top-k at least what the resident blocks append before the
    // bound settles (about 2k sets each); never fewer than one work unit's
    // sets, which is all a window of the sliced rerun needs.
    unsigned long long cap = DEFAULT_CAP;
    if (o->candidate_cap > 0) cap = (unsigned long long)o->candidate_cap;
    else if (topk) cap = std::max<unsigned long long>(cap, std::min<unsigned long long>(1ull << 26, 32ull * topk * ds->cu));
    cap = std::max(cap, unit_sets_max(pl));
    // a no-allocation call has the slots of `scratch` (at least one unit's)
    if (t_scr) cap = std::min<unsigned long long>(cap, ds->cand_cap);
    CHK(ensure_cand(ds, (unsigned)cap));
    const ScoreCtx &sc = pl.sc;
    if (order == 3) pl.seed_pairs = seed_pairs(ds, topk, o->candidate_cap > 0);
    res->seeded = pl.seed_pairs > 0;

    Collected acc;
    acc.score = score;
    acc.topk = topk;
    float kms = 0, rms = 0;
    Ctl hc;
    CHK(launch_fused_rescored(ds, pl, topk, (unsigned)cap, pl.seed_key, &kms, &rms, &hc));
    double kms_total = kms, rms_total = 0;
    if (!hc.cand_over && hc.cand_count <= cap) {
        // re-scored on the device behind the search; the first STAGE_CAND
        // candidates are already on the host
        rms_total = rms;
        CHK(collect_staged(ds, (int)hc.cand_count, acc));
    } else {
        // more sets within the FP32 margin than slots: search again in
        // windows, from the bound that the launch arrived at
        Ctl end;
        HIPCHK(hipMemcpy(&end, ds->ctl, sizeof end, hipMemcpyDeviceToHost));
        pl.seed_pairs = 0;
        if (end.best32 < 0xFF800000u) pl.seed_key = end.best32;
        CHK(run_sliced(ds, pl, topk, (unsigned)cap, hc, acc, &kms_total, &rms_total));
        res->fallback = 1;
    }
    res->kernel_ms = kms_total;
    res->rescore_ms = rms_total;
    res->margin = sc.margin;
    res->tile = tile;
    CHK(finish(ds, order, acc, res));
    res->path = path;
    return EPISDET_OK;
}

// Reference-shaped path (search-pairs.cu:137-211, search-triplets.cu:162-273):
// a host loop of rounds of 256 on NUM_STREAMS streams, each a count kernel
// writing the round's int32 AND-count tables to HBM and an FP64 objective
// kernel that derives, scores and keeps the round's best set.  3-way rounds
// are (Y block, X, Z block >= Y block); 2-way rounds are block pairs
// (A block <= B block).  Each stream keeps its best (exact score, lowest
// packed index); the host takes the best of the streams, so ties of any
// size give the same exact answer.
int run_plain(episdet_dataset *ds, const episdet_options *o, episdet_result *res)
{
    const int order = o->order, score = o->score;
    CHK(ensure_tables(ds, score));
    if (order == 3) CHK(ensure_pairs(ds));
    const int n = ds->n, nb = (n + BLOCK - 1) / BLOCK;
    // tile 1: the 3-way count kernel on the matrix cores (the 64 x 64 FP4
    // kernel writing its AND-counts), PLAIN_GROUP rounds of one (Y block,
    // Z block) and consecutive X per launch so that a launch fills the GPU
    // (16 workgroups per round); tile 0: the VALU count kernel, one round
    // per launch, as the reference's loop
    const bool mfma = o->tile == 1;
    if (o->tile != 0 && !(mfma && mfma_ok(ds))) return EPISDET_ERR_INVALID;
    const int group = mfma ? (order == 3 ? PLAIN_GROUP : PLAIN_GROUP2) : 1;
    const size_t slot = (size_t)2 * 256 * 256 * (order == 3 ? 8 : 4);
    DevList dl;
    uint32_t *counts = nullptr;
    unsigned long long *blk = nullptr, *sbest = nullptr, *flag = nullptr;
    CHK(dl.alloc(&counts, slot * NUM_STREAMS * group));
    CHK(dl.alloc(&blk, (size_t)NUM_STREAMS * 2 * 512));      // [stream][parity][256][2]
    CHK(dl.alloc(&sbest, (size_t)NUM_STREAMS * 2));          // [stream][2]
    CHK(dl.alloc(&flag, 1));
    hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(64), 0, ds->stream, sbest, NUM_STREAMS * 2, ~0ull);
    hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(64), 0, ds->stream, flag, 1, 0ull);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(ds->stream));
    StreamSet ss;
    CHK(ss.create(NUM_STREAMS));
    hipEvent_t e0, e1;
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    HIPCHK(hipEventRecord(e0, ds->stream));
    for (int i = 0; i < NUM_STREAMS; i++) HIPCHK(hipStreamWaitEvent(ss.st[i], e0, 0));

    const int plain_tile = 1;   // 32 x 32 (Y, Z) per workgroup: 64 workgroups per round
    TriArgs ta;
    if (order == 3) fill_tri_common(ds, ta);
    PairArgs pa{};
    if (mfma && order == 3) {
        CHK(init_single(ds, ta, 0));    // the planes and sizes the count kernel reads
        HIPCHK(hipStreamSynchronize(ds->stream));   // it runs on other streams
    }
    if (mfma && order == 2) {
        fill_pairs(ds, pa, true, 0);
        CHK(init_single(ds, pa, 0));
        HIPCHK(hipStreamSynchronize(ds->stream));
    }
    PlainObjArgs po;
    std::memset(&po, 0, sizeof po);
    po.singles = ds->singles;
    po.pairs = ds->pairs;
    po.order = order;
    po.n = n;
    po.N0 = ds->N[0];
    po.N1 = ds->N[1];
    po.score = score;
    po.t64 = ds->tab[score].t64;
    po.nan_flag = (unsigned *)flag;
    const Tri3Tile t = TRI_TILES[plain_tile];
    const int grid_count = (256 / (16 * t.A)) * (256 / (16 * t.B));
    long long rounds = 0, per_stream[NUM_STREAMS] = {};
    const long long limit = o->plain_rounds > 0 ? o->plain_rounds : -1;
    // the objective kernel of one round whose counts are at c, on stream s
    auto objective = [&](int X, int yb, int zb, const uint32_t *c, int s) -> int {
        const long long k = per_stream[s];
        po.counts = c;
        po.X = X;
        po.yb = yb;
        po.zb = zb;
        po.blk_out = blk + ((size_t)s * 2 + (k & 1)) * 512;
        po.blk_in = k ? blk + ((size_t)s * 2 + ((k - 1) & 1)) * 512 : nullptr;
        po.best = sbest + 2 * s;
        hipLaunchKernelGGL(k_objective_plain, dim3(256), dim3(256), 0, ss.st[s], po);
        HIPCHK(hipGetLastError());
        per_stream[s]++;
        rounds++;
        return EPISDET_OK;
    };
    // one round: count kernel, then the objective kernel, on stream s
    auto round = [&](int X, int yb, int zb) -> int {
        const int s = (int)(rounds % NUM_STREAMS);
        uint32_t *c = counts + slot * s;
        if (order == 3) {
            ta.X = X;
            ta.yb = yb;
            ta.zb = zb;
            ta.counts = c;
            CHK(dispatch_tri<MODE_COUNTS>(ds, plain_tile, ta, grid_count, ss.st[s]));
        } else {
            hipLaunchKernelGGL(k_pairs_counts, dim3(16), dim3(256), 0, ss.st[s], ds->planes[0], ds->W[0],
                               ds->planes[1], ds->W[1], yb, zb, c);
        }
        return objective(X, yb, zb, c, s);
    };
    // cnt rounds (X0 .. X0 + cnt - 1, yb, zb): one FP4 count launch, then
    // their objective kernels, on one stream
    long long launches = 0;
    auto mfma_rounds = [&](int X0, int cnt, int yb, int zb) -> int {
        const int s = (int)(launches++ % NUM_STREAMS);
        uint32_t *c = counts + slot * group * s;
        BatchTri bt;
        bt.jobs = (const TriArgs *)ds->jobargs;
        bt.job_start = ds->jobstart;
        bt.njobs = 1;
        bt.total = 0;
        bt.queue = nullptr;
        bt.X0 = X0;
        bt.yb = yb;
        bt.zb = zb;
        bt.rounds = cnt;
        bt.counts = c;
        bt.slot = slot;
        hipLaunchKernelGGL((k_triplets_mfma2<MODE_COUNTS>), dim3(16 * cnt), dim3(512), 0, ss.st[s], bt);
        HIPCHK(hipGetLastError());
        for (int r = 0; r < cnt; r++) CHK(objective(X0 + r, yb, zb, c + slot * r, s));
        return EPISDET_OK;
    };
    // cnt 2-way rounds (A block ab, B blocks bb0 .. bb0 + cnt - 1): one FP4
    // count launch of the 128 x 64 pair kernel, then their objectives
    auto mfma_pair_rounds = [&](int ab, int bb0, int cnt) -> int {
        const int s = (int)(launches++ % NUM_STREAMS);
        uint32_t *c = counts + slot * group * s;
        BatchPair bp;
        bp.jobs = (const PairArgs *)ds->jobargs;
        bp.job_start = ds->jobstart;
        bp.njobs = 1;
        bp.total = 0;
        bp.queue = nullptr;
        bp.ab = ab;
        bp.bb0 = bb0;
        bp.rounds = cnt;
        bp.counts = c;
        bp.slot = slot;
        hipLaunchKernelGGL((k_pairs_mfma<MODE_COUNTS>), dim3(8 * cnt), dim3(512), 0, ss.st[s], bp);
        HIPCHK(hipGetLastError());
        for (int r = 0; r < cnt; r++) CHK(objective(0, ab, bb0 + r, c + slot * r, s));
        return EPISDET_OK;
    };
    bool stop = false;
    if (mfma && order == 2) {
        for (int ab = 0; ab < nb && !stop; ab++)
            for (int bb0 = ab; bb0 < nb; bb0 += group) {
                long long cnt = std::min(group, nb - bb0);
                if (limit >= 0) cnt = std::min(cnt, limit - rounds);
                if (cnt <= 0) {
                    stop = true;
                    break;
                }
                CHK(mfma_pair_rounds(ab, bb0, (int)cnt));
            }
    } else if (mfma) {
        for (int yb = 0; yb < nb && !stop; yb++)
            for (int zb = yb; zb < nb && !stop; zb++) {
                const int xend = std::min((yb + 1) * BLOCK, n);
                for (int X0 = 0; X0 < xend; X0 += group) {
                    long long cnt = std::min(group, xend - X0);
                    if (limit >= 0) cnt = std::min(cnt, limit - rounds);
                    if (cnt <= 0) {
                        stop = true;
                        break;
                    }
                    CHK(mfma_rounds(X0, (int)cnt, yb, zb));
                }
            }
    } else if (order == 3) {
        for (int yb = 0; yb < nb && !stop; yb++)
            for (int X = 0; X < std::min((yb + 1) * BLOCK, n) && !stop; X++)
                for (int zb = yb; zb < nb; zb++) {
                    if (limit >= 0 && rounds >= limit) {
                        stop = true;
                        break;
                    }
                    CHK(round(X, yb, zb));
                }
    } else {
        for (int ab = 0; ab < nb && !stop; ab++)
            for (int bb = ab; bb < nb; bb++) {
                if (limit >= 0 && rounds >= limit) {
                    stop = true;
                    break;
                }
                CHK(round(0, ab, bb));
            }
    }
    for (int i = 0; i < NUM_STREAMS; i++) {
        if (per_stream[i]) {
            hipLaunchKernelGGL(k_plain_fold, dim3(1), dim3(64), 0, ss.st[i],
                               blk + ((size_t)i * 2 + ((per_stream[i] - 1) & 1)) * 512, sbest + 2 * i);
            HIPCHK(hipGetLastError());
        }
        HIPCHK(hipEventRecord(ss.ev[i], ss.st[i]));
        HIPCHK(hipStreamWaitEvent(ds->stream, ss.ev[i], 0));
    }
    HIPCHK(hipEventRecord(e1, ds->stream));
    HIPCHK(hipEventSynchronize(e1));
    float kms = 0;
    HIPCHK(hipEventElapsedTime(&kms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    res->kernel_ms = kms;
    res->rounds_run = rounds;

    unsigned long long hb[NUM_STREAMS * 2], hflag = 0;
    HIPCHK(hipMemcpy(hb, sbest, sizeof hb, hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(&hflag, flag, sizeof hflag, hipMemcpyDeviceToHost));
    if (hflag) return EPISDET_ERR_INTERNAL;   // inconsistent count tables
    unsigned long long bk = ~0ull, bp = ~0ull;
    for (int i = 0; i < NUM_STREAMS; i++)
        if (hb[2 * i] < bk || (hb[2 * i] == bk && hb[2 * i + 1] < bp)) {
            bk = hb[2 * i];
            bp = hb[2 * i + 1];
        }
    if (bp == ~0ull) return rounds ? EPISDET_ERR_INTERNAL : EPISDET_ERR_INVALID;
    const double bad = key2d_host(bk);
    res->best_score = score == EPISDET_SCORE_K2 ? bad : -bad;
    res->best_score_f32 = (float)res->best_score;
    res->packed = bp;
    unpack(order, bp, res->idx);
    res->candidates = 0;
    res->path = EPISDET_PATH_PLAIN;
    res->tile = mfma ? 1 : 0;
    return EPISDET_OK;
}

long long sets_total(int order, int n) { return (long long)episdet_n_choose_k((unsigned)n, (unsigned)order); }

}  // namespace

// ================================================================ C ABI ==

extern "C" {

unsigned long long episdet_n_choose_k(unsigned n, unsigned k)
{
    unsigned long long r = 1;
    for (unsigned i = 1; i <= k; i++) {
        r = r * n / i;
        n = n - 1;
    }
    return r;
}

long long episdet_reference_rounds(int order, int numSNPs)
{
    const long long nb = (numSNPs + BLOCK - 1) / BLOCK;
    if (order == 2) return nb * (nb + 1) / 2;
    long long r = 0;
    for (long long yb = 0; yb < nb; yb++) r += std::min((yb + 1) * BLOCK, (long long)numSNPs) * (nb - yb);
    return r;
}

const char *episdet_status_string(int status)
{
    switch (status) {
    case EPISDET_OK: return "ok";
    case EPISDET_ERR_INVALID: return "invalid argument";
    case EPISDET_ERR_NO_DEVICE: return "no gfx950 device";
    case EPISDET_ERR_HIP: return "HIP runtime error";
    case EPISDET_ERR_ALLOC: return "allocation failed";
    case EPISDET_ERR_CANDIDATES: return "candidate buffer overflow";
    case EPISDET_ERR_GENOTYPES: return "a sample is marked in both genotype planes of a SNP";
    case EPISDET_ERR_SCRATCH: return "the search needs more than the no-allocation entry point's scratch memory";
    default: return "internal error";
    }
}

int episdet_device_info(char *name, int name_len, int *compute_units, int *clock_khz)
{
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count < 1) return EPISDET_ERR_NO_DEVICE;
    hipDeviceProp_t prop;
    HIPCHK(hipGetDeviceProperties(&prop, 0));
    if (name && name_len > 0) {
        std::snprintf(name, (size_t)name_len, "%s (%s)", prop.name, prop.gcnArchName);
    }
    if (compute_units) *compute_units = prop.multiProcessorCount;
    if (clock_khz) *clock_khz = prop.clockRate;
    return EPISDET_OK;
}

int episdet_device_synchronize(void)
{
    return hipDeviceSynchronize() == hipSuccess ? EPISDET_OK : EPISDET_ERR_HIP;
}

// Single counts, and the check that no sample is marked in both genotype
// planes of a SNP (such input has no genotype for that sample, and the
// derived counts of the SNP would be inconsistent).  Never captured: it
// synchronises.
// With wait = false (a rebuild before a fused search: the planes never
// change after the dataset passed the check) the counts are recomputed on
// the dataset's stream with no wait of their own; the search that follows
// on that stream reads them.  Work on other streams (the plain path's, a
// batch graph's) needs wait = true.
static int compute_singles(episdet_dataset *ds, bool wait = true)
{
    unsigned *bad = &ds->ctl->bad_snp;
    if (wait) HIPCHK(hipMemsetAsync(bad, 0xFF, sizeof(unsigned), ds->stream));
    hipLaunchKernelGGL(k_singles, dim3(ds->n), dim3(64), 0, ds->stream, ds->planes[0], ds->W[0], ds->planes[1],
                       ds->W[1], ds->n, ds->singles, bad);
    HIPCHK(hipGetLastError());
    if (!wait) return EPISDET_OK;
    unsigned hb = 0;
    HIPCHK(hipMemcpyAsync(&hb, bad, sizeof hb, hipMemcpyDeviceToHost, ds->stream));
    HIPCHK(hipStreamSynchronize(ds->stream));
    if (hb != ~0u) return EPISDET_ERR_GENOTYPES;
    return EPISDET_OK;
}

int episdet_dataset_create(const unsigned *cases, const unsigned *controls, int numSNPs, int numCases,
                           int numControls, int casesWords, int controlsWords, episdet_dataset **out)
{
    if (!out) return EPISDET_ERR_INVALID;
    *out = nullptr;
    if (!cases || !controls || numSNPs < 2 || numSNPs > 0x1FFFFF || numCases < 1 || numControls < 1)
        return EPISDET_ERR_INVALID;
    // N = numCases + numControls, and N + 2 table entries, stay in int
    if ((long long)numCases + numControls >= (1LL << 30)) return EPISDET_ERR_INVALID;
    if (casesWords * 32LL < numCases || controlsWords * 32LL < numControls) return EPISDET_ERR_INVALID;
    int cu = 0;
    CHK(check_device(&cu));
    HIPCHK(hipSetDevice(0));
    episdet_dataset *ds = new (std::nothrow) episdet_dataset();
    if (!ds) return EPISDET_ERR_ALLOC;
    ds->cu = cu;
    ds->n = numSNPs;
    ds->nrows = ((numSNPs + BLOCK - 1) / BLOCK) * BLOCK;
    ds->N[0] = numCases;
    ds->N[1] = numControls;
    const int in_w[2] = {casesWords, controlsWords};
    const unsigned *src[2] = {cases, controls};
    int rc = EPISDET_OK;
    if (hipStreamCreateWithFlags(&ds->stream, hipStreamNonBlocking) != hipSuccess) rc = EPISDET_ERR_HIP;
    // control block, argument slot and the seeding kernels' pairs in one block
    if (rc == EPISDET_OK && hipMalloc(&ds->ctl, sizeof(Ctl) + 1024 + 256 + sizeof(unsigned long long) * SEED_WORDS) != hipSuccess) {
        ds->ctl = nullptr;
        rc = EPISDET_ERR_ALLOC;
    }
    if (rc == EPISDET_OK) {
        unsigned char *at = (unsigned char *)(ds->ctl + 1);
        ds->jobargs = at;
        ds->jobstart = (unsigned long long *)(at + 1024);
        ds->seed = (unsigned long long *)(at + 1024 + 256);
    }
    for (int e = 0; e < 3 && rc == EPISDET_OK; e++)
        if (hipEventCreate(&ds->ev[e]) != hipSuccess) rc = EPISDET_ERR_HIP;
    if (rc == EPISDET_OK && hipHostMalloc((void **)&ds->stage, STAGE_BYTES, hipHostMallocMapped) != hipSuccess) {
        ds->stage = nullptr;
        rc = EPISDET_ERR_ALLOC;
    }
    if (rc == EPISDET_OK && hipHostGetDevicePointer((void **)&ds->stage_dev, ds->stage, 0) != hipSuccess)
        rc = EPISDET_ERR_HIP;
    for (int c = 0; c < 2 && rc == EPISDET_OK; c++) {
        const int Wv = (ds->N[c] + 31) / 32;
        ds->W[c] = ((Wv + W_ALIGN - 1) / W_ALIGN) * W_ALIGN;
        const size_t in_bytes = sizeof(uint32_t) * (size_t)numSNPs * 2 * in_w[c];
        const size_t dev_words = (size_t)ds->nrows * 2 * ds->W[c];
        if (hipMalloc(&ds->planes[c], sizeof(uint32_t) * dev_words) != hipSuccess) {
            rc = EPISDET_ERR_ALLOC;
            break;
        }
        // Large planes go through the pinned pool (a pair search of 4096 x
        // 65536 from host buffers: 5.4 ms without, 3.9 with); below 4 MB a class
        // starting threads is the longer part, and a slot has to hold a SNP's rows.
        if (in_bytes >= UP_SLOT && sizeof(uint32_t) * 2 * (size_t)in_w[c] <= UP_SLOT) {
            std::unique_lock<std::mutex> lk(g_up_mu, std::try_to_lock);
            if (lk.owns_lock() && upload_pool()) {
                rc = upload_pooled(ds, c, src[c], in_w[c]);
                continue;
            }
        }
        uint32_t *stage = nullptr;
        if (hipMalloc(&stage, in_bytes) != hipSuccess) {
            rc = EPISDET_ERR_ALLOC;
            break;
        }
        if (hipMemcpyAsync(stage, src[c], in_bytes, hipMemcpyHostToDevice, ds->stream) != hipSuccess) rc = EPISDET_ERR_HIP;
        if (rc == EPISDET_OK) {
            const int grid = (int)std::min<size_t>((dev_words + 255) / 256, 65536);
            hipLaunchKernelGGL(k_repack, dim3(grid), dim3(256), 0, ds->stream, stage, in_w[c], ds->planes[c], ds->W[c],
                               numSNPs, 0, ds->nrows, ds->N[c]);
            if (hipGetLastError() != hipSuccess) rc = EPISDET_ERR_HIP;
        }
        if (hipStreamSynchronize(ds->stream) != hipSuccess) rc = EPISDET_ERR_HIP;
        (void)hipFree(stage);
    }
    if (rc == EPISDET_OK && hipMalloc(&ds->singles, sizeof(uint4) * numSNPs) != hipSuccess) rc = EPISDET_ERR_ALLOC;
    if (rc == EPISDET_OK) rc = compute_singles(ds);
    if (rc != EPISDET_OK) {
        episdet_dataset_destroy(ds);
        return rc;
    }
    *out = ds;
    return EPISDET_OK;
}

void episdet_dataset_destroy(episdet_dataset *ds)
{
    if (!ds) return;
    (void)hipDeviceSynchronize();
    for (int c = 0; c < 2; c++) {
        if (ds->planes[c]) (void)hipFree(ds->planes[c]);
        if (ds->tab[c].t64) (void)hipFree(ds->tab[c].t64);
    }
    if (ds->singles) (void)hipFree(ds->singles);
    if (ds->pairs) (void)hipFree(ds->pairs);
    if (ds->ctl) (void)hipFree(ds->ctl);
    if (ds->gstart) (void)hipFree(ds->gstart);
    if (ds->groups) (void)hipFree(ds->groups);
    if (ds->cand) (void)hipFree(ds->cand);
    for (hipEvent_t e : ds->ev)
        if (e) (void)hipEventDestroy(e);
    if (ds->stage) (void)hipHostFree(ds->stage);
    if (ds->stream) (void)hipStreamDestroy(ds->stream);
    delete ds;
}

int episdet_run(episdet_dataset *ds, const episdet_options *opt, episdet_result *res)
{
    if (!ds || !opt || !res) return EPISDET_ERR_INVALID;
    if (opt->order != 2 && opt->order != 3) return EPISDET_ERR_INVALID;
    if (opt->score != EPISDET_SCORE_K2 && opt->score != EPISDET_SCORE_MI) return EPISDET_ERR_INVALID;
    if (ds->n < opt->order) return EPISDET_ERR_INVALID;
    if (opt->topk > 1 && (opt->path == EPISDET_PATH_PLAIN || opt->topk > EPISDET_TOPK_MAX)) return EPISDET_ERR_INVALID;
    std::memset(res, 0, sizeof *res);
    const double t0 = now_s();
    if (opt->rebuild) {
        CHK(compute_singles(ds, opt->path == EPISDET_PATH_PLAIN));
        if (opt->order == 3) CHK(ensure_pairs(ds, true));
        res->prep_ms = (now_s() - t0) * 1e3;
    }
    int rc;
    switch (opt->path) {
    case EPISDET_PATH_AUTO:
    case EPISDET_PATH_FUSED_VALU:
    case EPISDET_PATH_FUSED_MFMA: rc = run_fused(ds, opt, res); break;
    case EPISDET_PATH_PLAIN: rc = run_plain(ds, opt, res); break;
    default: rc = EPISDET_ERR_INVALID;
    }
    res->wall_s = now_s() - t0;
    res->rounds = episdet_reference_rounds(opt->order, ds->n);
    res->sets = sets_total(opt->order, ds->n);
    if (opt->path == EPISDET_PATH_PLAIN && opt->order == 3 && res->rounds_run < res->rounds && res->rounds > 0)
        res->sets = (long long)((double)res->sets * (double)res->rounds_run / (double)res->rounds);
    return rc;
}

}  // extern "C"

namespace {

// Per-device set-up of the no-allocation search: the device address of
// `scratch` (each device holds its own copy at its own address), taken once
// with that device current.
constexpr int SCRATCH_MAX_DEVICES = 64;
struct ScratchDevice {
    unsigned char *base = nullptr;
};
std::mutex g_scratch_mu;      // no-allocation calls of this process run one at a time
ScratchDevice g_scratch_dev[SCRATCH_MAX_DEVICES];

// Called with g_scratch_mu held and `dev` current.
int scratch_device(int dev, ScratchDevice **out)
{
    if (dev < 0 || dev >= SCRATCH_MAX_DEVICES) return EPISDET_ERR_INVALID;
    ScratchDevice &sd = g_scratch_dev[dev];
    if (!sd.base) {
        void *ptr = nullptr;
        HIPCHK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        if (!ptr) return EPISDET_ERR_INTERNAL;
        sd.base = (unsigned char *)ptr;
    }
    *out = &sd;
    return EPISDET_OK;
}

// Bytes of `scratch` a no-allocation search of this dataset needs, and the
// regions it takes (device addresses from base).
size_t scratch_layout(const episdet_dataset *ds, int order, int score, unsigned char *base, ScratchPlan &sp)
{
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t at = off;
        off = (off + bytes + 255) & ~(size_t)255;
        return base + at;
    };
    sp.ctl = (Ctl *)take(sizeof(Ctl));
    sp.jobargs = take(1024);
    sp.jobstart = (unsigned long long *)take(2 * sizeof(unsigned long long));
    sp.err = (unsigned long long *)take(sizeof(unsigned long long));
    sp.cand = (unsigned long long *)take(sizeof(unsigned long long) * SCRATCH_CAND);
    sp.cand_s32 = (float *)take(sizeof(float) * SCRATCH_CAND);
    sp.cand_s64 = (double *)take(sizeof(double) * SCRATCH_CAND);
    if (order == 3) {
        // every 3-way unit enumeration uses Y and Z tiles of at least 32 SNPs
        const size_t t = ((size_t)ds->n + 31) / 32;
        sp.max_groups = t * (t + 1) / 2;
        sp.gstart = (unsigned long long *)take(sizeof(unsigned long long) * (sp.max_groups + 1));
        sp.groups = (int2 *)take(sizeof(int2) * sp.max_groups);
    }
    if (!ds->tab[score].ready) sp.t64 = (double *)take(sizeof(double) * ((size_t)ds->N[0] + ds->N[1] + 2));
    if (order == 3 && !ds->pairs) sp.pairs = (uint4 *)take((size_t)ds->n * ds->n * 2 * sizeof(uint4));
    return off;
}

}  // namespace

extern "C" {

int episdet_run_noalloc(episdet_dataset *ds, const episdet_options *opt, episdet_result *res)
{
    if (!ds || !opt || !res) return EPISDET_ERR_INVALID;
    if (opt->order != 2 && opt->order != 3) return EPISDET_ERR_INVALID;
    if (opt->score != EPISDET_SCORE_K2 && opt->score != EPISDET_SCORE_MI) return EPISDET_ERR_INVALID;
    // the plain path, the rebuild and the tuner allocate buffers of their own
    if (opt->path == EPISDET_PATH_PLAIN || opt->rebuild || opt->autotune) return EPISDET_ERR_INVALID;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    HIPCHK(hipSetDevice(ds->dev));
    ScratchDevice *sd = nullptr;
    CHK(scratch_device(ds->dev, &sd));
    ScratchPlan sp;
    if (scratch_layout(ds, opt->order, opt->score, sd->base, sp) > SCRATCH_BYTES) {
        std::fprintf(stderr,
                     "episdet: episdet_run_noalloc: a %d-way search of %d SNPs x %d samples needs more than the "
                     "%zu MiB of its static scratch memory\n",
                     opt->order, ds->n, ds->N[0] + ds->N[1], SCRATCH_BYTES >> 20);
        return EPISDET_ERR_SCRATCH;
    }
    // timing events: the dataset's own, made when it was created
    sp.ev[0] = ds->ev[0];
    sp.ev[1] = ds->ev[1];
    // Point the dataset's per-search buffers at `scratch` for this call and
    // restore them afterwards; the FP64 table and the pair table built in
    // `scratch` are forgotten, since the next call overwrites them.
    struct Bind {
        episdet_dataset *ds;
        int score;
        Ctl *ctl;
        void *jobargs;
        unsigned long long *jobstart, *cand;
        float *cand_s32;
        double *cand_s64;
        unsigned cand_cap;
        uint4 *pairs;
        ScoreTables tab;
        unsigned long long *gstart;
        int2 *groups;
        ~Bind()
        {
            t_scr = nullptr;
            ds->ctl = ctl;
            ds->jobargs = jobargs;
            ds->jobstart = jobstart;
            ds->cand = cand;
            ds->cand_s32 = cand_s32;
            ds->cand_s64 = cand_s64;
            ds->cand_cap = cand_cap;
            ds->pairs = pairs;
            ds->tab[score] = tab;
            ds->gstart = gstart;
            ds->groups = groups;
        }
    } bind{ds,           opt->score,    ds->ctl,      ds->jobargs, ds->jobstart, ds->cand,
           ds->cand_s32, ds->cand_s64, ds->cand_cap, ds->pairs,   ds->tab[opt->score],
           ds->gstart,   ds->groups};
    ds->ctl = sp.ctl;
    ds->jobargs = sp.jobargs;
    ds->jobstart = sp.jobstart;
    ds->cand = sp.cand;
    ds->cand_s32 = sp.cand_s32;
    ds->cand_s64 = sp.cand_s64;
    ds->cand_cap = SCRATCH_CAND;
    ds->gstart = sp.gstart;
    ds->groups = sp.groups;
    t_scr = &sp;
    return episdet_run(ds, opt, res);
}

int episdet_autotune(episdet_dataset *ds, int order, int score, episdet_tune_entry *entries, int capacity,
                     int *count, int *chosen)
{
    if (!ds || (order != 2 && order != 3) || (score != EPISDET_SCORE_K2 && score != EPISDET_SCORE_MI) ||
        ds->n < order || !count || !chosen || capacity < 0 || (capacity > 0 && !entries))
        return EPISDET_ERR_INVALID;
    std::vector<episdet_tune_entry> table;
    int path = 0, tile = 0;
    CHK(tune_kernel(ds, order, score, &table, &path, &tile));
    {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        g_tune[TuneKey{order, score, ds->n, ds->W[0], ds->W[1]}] = TuneChoice{path, tile};
    }
    *count = (int)table.size();
    *chosen = -1;
    for (int i = 0; i < (int)table.size(); i++) {
        if (i < capacity) entries[i] = table[i];
        if (table[i].path == path && table[i].tile == tile) *chosen = i;
    }
    return EPISDET_OK;
}

int episdet_run_topk(episdet_dataset *ds, const episdet_options *opt, int k, unsigned long long *packed,
                     double *scores, int *count, episdet_result *res)
{
    if (!ds || !opt || !packed || !scores || !count || !res || k < 1 || k > EPISDET_TOPK_MAX)
        return EPISDET_ERR_INVALID;
    episdet_options o = *opt;
    o.topk = k;
    ds->topk_packed.clear();
    ds->topk_scores.clear();
    CHK(episdet_run(ds, &o, res));
    if (k == 1) {
        packed[0] = res->packed;
        scores[0] = res->best_score;
        *count = 1;
        return EPISDET_OK;
    }
    const int m = (int)ds->topk_packed.size();
    for (int i = 0; i < m; i++) {
        packed[i] = ds->topk_packed[i];
        scores[i] = ds->topk_scores[i];
    }
    *count = m;
    return EPISDET_OK;
}

int episdet_search(int order, int score, const unsigned *cases, const unsigned *controls, int numSNPs, int numCases,
                   int numControls, unsigned numSNPsWithPadding, int numCasesWithPadding, int numControlsWithPadding,
                   int *roundsCounter, double *searchTime, float *outputFromGpu, unsigned long long *packedIndices)
{
    if (!roundsCounter || !searchTime || !outputFromGpu || !packedIndices) return EPISDET_ERR_INVALID;
    if (numCasesWithPadding % 32 != 0 || numControlsWithPadding % 32 != 0) return EPISDET_ERR_INVALID;
    if ((long long)numSNPsWithPadding < numSNPs) return EPISDET_ERR_INVALID;
    const double t0 = now_s();
    episdet_dataset *ds = nullptr;
    CHK(episdet_dataset_create(cases, controls, numSNPs, numCases, numControls, numCasesWithPadding / 32,
                               numControlsWithPadding / 32, &ds));
    // The reference prints one line per outer block of its host loop from
    // inside the search (search-pairs.cu:137-139, search-triplets.cu:162-164).
    // The search here is one persistent launch, so the lines come first.
    for (long long start = 0; start < (long long)numSNPsWithPadding; start += BLOCK)
        std::printf("Outer loop iteration %d out of %d\n", (int)(start / BLOCK), (int)(numSNPsWithPadding / BLOCK));
    std::fflush(stdout);
    episdet_options o;
    std::memset(&o, 0, sizeof o);
    o.order = order;
    o.score = score;
    o.path = EPISDET_PATH_AUTO;
    episdet_result r;
    const int rc = episdet_run(ds, &o, &r);
    episdet_dataset_destroy(ds);
    *searchTime = now_s() - t0;
    if (rc != EPISDET_OK) return rc;
    *roundsCounter = (int)episdet_reference_rounds(order, numSNPs);
    *outputFromGpu = (float)r.best_score;
    *packedIndices = r.packed;
    return EPISDET_OK;
}

// ------------------------------------------------------ batched search --

// Candidate slots of a batched job: the requested capacity (default 1M),
// never fewer than one work unit's sets of its MFMA tile.
static unsigned batch_cap(const episdet_options &o, int order, int tile)
{
    const unsigned long long unit = order == 3 ? (unsigned long long)mfma_xstep(tile) * mfma_ty(tile) * mfma_tz(tile)
                                               : (tile == 0 ? (unsigned long long)P2_TA * P2_TB
                                                            : (unsigned long long)P3_TA * P3_TB);
    const unsigned long long want = o.candidate_cap > 0 ? (unsigned long long)o.candidate_cap : DEFAULT_CAP;
    return (unsigned)std::max(want, unit);
}

int episdet_run_batch(episdet_dataset *const *dss, const episdet_options *opts, int njobs, episdet_result *results,
                      double *batch_ms)
{
    if (!dss || !opts || !results || njobs <= 0) return EPISDET_ERR_INVALID;
    const double t0 = now_s();
    // 3-way jobs by MFMA tile, 2-way jobs by MFMA pair tile, the rest
    std::vector<int> tri[MFMA_TILES], pairs[MFMA_PAIR_TILES], solo;
    std::vector<int> kpath(njobs), ktile(njobs);
    for (int j = 0; j < njobs; j++) {
        episdet_dataset *ds = dss[j];
        const episdet_options &o = opts[j];
        std::memset(&results[j], 0, sizeof(episdet_result));
        if (!ds || (o.order != 2 && o.order != 3) || (o.score != EPISDET_SCORE_K2 && o.score != EPISDET_SCORE_MI) ||
            ds->n < o.order || o.topk > 1)
            return EPISDET_ERR_INVALID;
        const double tp = now_s();
        if (o.rebuild) CHK(compute_singles(ds, false));
        CHK(ensure_tables(ds, o.score));
        if (o.order == 3) CHK(ensure_pairs(ds, o.rebuild != 0));
        CHK(ensure_cand(ds, o.candidate_cap > 0 ? (unsigned)o.candidate_cap : DEFAULT_CAP));
        results[j].prep_ms = (now_s() - tp) * 1e3;
        kpath[j] = o.path;
        ktile[j] = o.tile;
        if (o.path == EPISDET_PATH_AUTO) CHK(choose_kernel(ds, o.order, o.score, &kpath[j], &ktile[j], o.autotune != 0));
    }
    // AUTO jobs of one order share one kernel: the MFMA tile their per-shape
    // choices give the most work (sets x samples).  One graph branch per order
    // packs the CUs better than one branch per tile: on the 64-job workload
    // the per-job choices, spread over seven kernels, took 1.75 s against
    // 1.51 s for one 3-way and one 2-way kernel.
    for (int order = 2; order <= 3; order++) {
        const int ntiles = order == 3 ? MFMA_TILES : MFMA_PAIR_TILES;
        std::vector<double> work(ntiles, 0.0);
        for (int j = 0; j < njobs; j++)
            if (opts[j].order == order && opts[j].path == EPISDET_PATH_AUTO && kpath[j] == EPISDET_PATH_FUSED_MFMA &&
                ktile[j] >= 0 && ktile[j] < ntiles)
                work[ktile[j]] += (double)episdet_n_choose_k((unsigned)dss[j]->n, (unsigned)order) *
                                  (double)(dss[j]->N[0] + dss[j]->N[1]);
        const int win = (int)(std::max_element(work.begin(), work.end()) - work.begin());
        if (work[win] <= 0.0) continue;
        for (int j = 0; j < njobs; j++)
            if (opts[j].order == order && opts[j].path == EPISDET_PATH_AUTO && mfma_ok(dss[j])) {
                kpath[j] = EPISDET_PATH_FUSED_MFMA;
                ktile[j] = win;
            }
    }
    std::vector<const episdet_dataset *> seen;     // datasets already in the graph
    for (int j = 0; j < njobs; j++) {
        episdet_dataset *ds = dss[j];
        const episdet_options &o = opts[j];
        // 3-way and 2-way jobs go to the batched FP4-MFMA kernel of their
        // tile; anything else runs on its own afterwards.
        // A dataset's control block and candidate buffer hold one search at a
        // time, so a second job on the same dataset runs after the graph.
        const bool dup = std::find(seen.begin(), seen.end(), ds) != seen.end();
        const bool batchable = kpath[j] == EPISDET_PATH_FUSED_MFMA && mfma_ok(ds) && ktile[j] >= 0 &&
                               ktile[j] < (o.order == 3 ? MFMA_TILES : MFMA_PAIR_TILES);
        if (dup || !batchable) {
            solo.push_back(j);
            continue;
        }
        seen.push_back(ds);
        CHK(ensure_cand(ds, batch_cap(o, o.order, ktile[j])));
        if (o.order == 3) tri[ktile[j]].push_back(j);
        else pairs[ktile[j]].push_back(j);
    }
    DevList dl;
    int cu = dss[0]->cu;
    // per-job kernel arguments
    std::vector<TriArgs> ta[MFMA_TILES];
    std::vector<unsigned long long> tstart[MFMA_TILES];
    std::vector<SeedArgs> seeds;
    int seed_blocks = 0, seed_sets = 0;
    for (int tl = 0; tl < MFMA_TILES; tl++) {
        ta[tl].resize(tri[tl].size());
        tstart[tl].assign(1, 0ull);
        for (size_t k = 0; k < tri[tl].size(); k++) {
            episdet_dataset *ds = dss[tri[tl][k]];
            const int t[3] = {mfma_ty(tl), mfma_tz(tl), mfma_xstep(tl)};
            int ngroups;
            unsigned long long nunits;
            CHK(ensure_groups(ds, t, &ngroups, &nunits));
            TriArgs &a = ta[tl][k];
            fill_tri_common(ds, a);
            a.co.cand_cap = batch_cap(opts[tri[tl][k]], 3, tl);
            a.sc = make_ctx(ds, opts[tri[tl][k]].score, 3);
            a.gstart = ds->gstart;
            a.groups = ds->groups;
            a.ngroups = ngroups;
            a.nunits = nunits;
            tstart[tl].push_back(tstart[tl].back() + nunits);
            const int np = seed_pairs(ds, 0, false);
            if (np > 0) {
                seeds.push_back(seed_args_of(ds, opts[tri[tl][k]].score, a.sc, np, false));
                seed_blocks = std::max(seed_blocks, seeds.back().blocks);
                seed_sets = std::max(seed_sets, np * ds->n);
            }
            results[tri[tl][k]].seeded = np > 0;
        }
    }
    std::vector<PairArgs> pa[MFMA_PAIR_TILES];
    std::vector<unsigned long long> pstart[MFMA_PAIR_TILES];
    for (int tl = 0; tl < MFMA_PAIR_TILES; tl++) {
        pa[tl].resize(pairs[tl].size());
        pstart[tl].assign(1, 0ull);
        for (size_t k = 0; k < pairs[tl].size(); k++) {
            episdet_dataset *ds = dss[pairs[tl][k]];
            fill_pairs(ds, pa[tl][k], true, tl);
            pa[tl][k].co.cand_cap = batch_cap(opts[pairs[tl][k]], 2, tl);
            pa[tl][k].sc = make_ctx(ds, opts[pairs[tl][k]].score, 2);
            pstart[tl].push_back(pstart[tl].back() + pa[tl][k].nunits);
        }
    }
    std::vector<int> batched;
    for (int tl = 0; tl < MFMA_TILES; tl++) batched.insert(batched.end(), tri[tl].begin(), tri[tl].end());
    for (int tl = 0; tl < MFMA_PAIR_TILES; tl++) batched.insert(batched.end(), pairs[tl].begin(), pairs[tl].end());
    std::vector<RescoreJob> rj(batched.size());
    std::vector<unsigned long long *> qp(batched.size());
    std::vector<unsigned *> bp(batched.size()), cp(batched.size());
    for (size_t k = 0; k < batched.size(); k++) {
        episdet_dataset *ds = dss[batched[k]];
        rj[k].r = rescore_args(ds, opts[batched[k]].order, opts[batched[k]].score);
        rj[k].count = &ds->ctl->cand_count;
        rj[k].cap = batch_cap(opts[batched[k]], opts[batched[k]].order, ktile[batched[k]]);
        rj[k].cand_s32 = ds->cand_s32;
        rj[k].hs = host_stage(ds, rj[k].cap);
        qp[k] = ds->ctl->queue;
        bp[k] = &ds->ctl->best32;
        cp[k] = &ds->ctl->cand_count;
    }
    TriArgs *d_ta[MFMA_TILES] = {};
    PairArgs *d_pa[MFMA_PAIR_TILES] = {};
    unsigned long long *d_tstart[MFMA_TILES] = {}, *d_pstart[MFMA_PAIR_TILES] = {}, *d_bq = nullptr;
    RescoreJob *d_rj = nullptr;
    SeedArgs *d_seeds = nullptr;
    unsigned long long **d_qp = nullptr;
    unsigned **d_bp = nullptr, **d_cp = nullptr;
    constexpr int NQ = MFMA_TILES + MFMA_PAIR_TILES;   // one work queue per batched kernel
    constexpr int QW = 9 * QLINE;                      // each: the queue, then 8 per-XCD queues
    const std::vector<unsigned long long> zeros(NQ * QW, 0ull);
    for (int tl = 0; tl < MFMA_TILES; tl++) {
        if (tri[tl].empty()) continue;
        CHK(dl.put(&d_ta[tl], ta[tl].data(), ta[tl].size()));
        CHK(dl.put(&d_tstart[tl], tstart[tl].data(), tstart[tl].size()));
    }
    for (int tl = 0; tl < MFMA_PAIR_TILES; tl++) {
        if (pairs[tl].empty()) continue;
        CHK(dl.put(&d_pa[tl], pa[tl].data(), pa[tl].size()));
        CHK(dl.put(&d_pstart[tl], pstart[tl].data(), pstart[tl].size()));
    }
    CHK(dl.put(&d_bq, zeros.data(), zeros.size()));
    CHK(dl.put(&d_seeds, seeds.data(), seeds.size()));
    CHK(dl.put(&d_rj, rj.data(), rj.size()));
    CHK(dl.put(&d_qp, qp.data(), qp.size()));
    CHK(dl.put(&d_bp, bp.data(), bp.size()));
    CHK(dl.put(&d_cp, cp.data(), cp.size()));

    // the count tables and group lists are built on the datasets' streams,
    // side by side; the graph runs on its own
    for (int j = 0; j < njobs; j++) HIPCHK(hipStreamSynchronize(dss[j]->stream));
    double gms = 0;
    if (!batched.empty()) {
        hipStream_t st, br[NQ];
        HIPCHK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
        const auto used = [&](int q) { return !(q < MFMA_TILES ? tri[q] : pairs[q - MFMA_TILES]).empty(); };
        hipEvent_t fork, seeded, join[NQ];
        HIPCHK(hipEventCreateWithFlags(&fork, hipEventDisableTiming));
        HIPCHK(hipEventCreateWithFlags(&seeded, hipEventDisableTiming));
        for (int q = 0; q < NQ; q++)
            if (used(q)) {
                HIPCHK(hipStreamCreateWithFlags(&br[q], hipStreamNonBlocking));
                HIPCHK(hipEventCreateWithFlags(&join[q], hipEventDisableTiming));
            }
        hipGraph_t graph;
        hipGraphExec_t exec;
        // one graph: reset, then one branch per batched kernel (each 3-way
        // and 2-way MFMA tile) running side by side, so each fills the CUs
        // the others' tails leave idle, then FP64 re-scoring
        HIPCHK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
        const int nb = (int)batched.size();
        hipLaunchKernelGGL(k_init_many, dim3((std::max(nb, NQ * QW) + 63) / 64), dim3(64), 0, st, d_qp, d_bp, d_cp, nb,
                           d_bq, NQ * QW);
        HIPCHK(hipEventRecord(fork, st));
        for (int q = 0; q < NQ; q++)
            if (used(q)) HIPCHK(hipStreamWaitEvent(br[q], fork, 0));
        // the 3-way jobs' starting bounds, beside the 2-way kernels, whose
        // workgroups so get their CUs first: started together with the
        // 3-way ones they held LDS for 9.2 ms to do 0.1 ms of work
        if (!seeds.empty()) {
            for (size_t k = 0; k < seeds.size(); k += 65535) {       // a grid's y extent
                const SeedMany sm{d_seeds + k};
                const unsigned nj = (unsigned)std::min<size_t>(seeds.size() - k, 65535);
                hipLaunchKernelGGL(k_seed_pairs<SeedMany>, dim3(seed_blocks, nj), dim3(256), 0, st, sm);
                hipLaunchKernelGGL(k_seed_pick<SeedMany>, dim3(1, nj), dim3(SEED_BLOCKS), 0, st, sm);
                hipLaunchKernelGGL(k_seed_triplets<SeedMany>, dim3((seed_sets + 3) / 4, nj), dim3(256), 0, st, sm);
            }
            HIPCHK(hipEventRecord(seeded, st));
        }
        for (int tl = 0; tl < MFMA_TILES; tl++) {
            if (tri[tl].empty()) continue;
            if (!seeds.empty()) HIPCHK(hipStreamWaitEvent(br[tl], seeded, 0));
            BatchTri bt;
            bt.jobs = d_ta[tl];
            bt.job_start = d_tstart[tl];
            bt.njobs = (int)tri[tl].size();
            bt.total = tstart[tl].back();
            bt.queue = d_bq + QW * tl;
            launch_tri_mfma<MODE_SEARCH>(tl, occupancy_blocks(mfma_kernel<MODE_SEARCH>(tl), mfma_threads(tl), cu), bt,
                                         br[tl]);
        }
        for (int tl = 0; tl < MFMA_PAIR_TILES; tl++) {
            if (pairs[tl].empty()) continue;
            BatchPair bpr;
            bpr.jobs = d_pa[tl];
            bpr.job_start = d_pstart[tl];
            bpr.njobs = (int)pairs[tl].size();
            bpr.total = pstart[tl].back();
            bpr.queue = d_bq + QW * (MFMA_TILES + tl);
            bpr.xcd = tl == 0 || tl == 1;
            // a failed launch shows at the end of the capture
            (void)launch_pairs_mfma<MODE_SEARCH>(
                tl, occupancy_blocks(pairs_mfma_kernel<MODE_SEARCH>(tl), pairs_mfma_threads(tl), cu), bpr,
                br[MFMA_TILES + tl]);
        }
        for (int q = 0; q < NQ; q++) {
            if (!used(q)) continue;
            HIPCHK(hipEventRecord(join[q], br[q]));
            HIPCHK(hipStreamWaitEvent(st, join[q], 0));
        }
        hipLaunchKernelGGL(k_rescore_batch, dim3(8 * cu), dim3(64), 0, st, d_rj, nb);
        HIPCHK(hipStreamEndCapture(st, &graph));
        HIPCHK(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
        hipEvent_t e0, e1;
        HIPCHK(hipEventCreate(&e0));
        HIPCHK(hipEventCreate(&e1));
        HIPCHK(hipEventRecord(e0, st));
        HIPCHK(hipGraphLaunch(exec, st));
        HIPCHK(hipEventRecord(e1, st));
        HIPCHK(hipStreamSynchronize(st));
        float f = 0;
        HIPCHK(hipEventElapsedTime(&f, e0, e1));
        gms = f;
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        (void)hipGraphExecDestroy(exec);
        (void)hipGraphDestroy(graph);
        (void)hipEventDestroy(fork);
        (void)hipEventDestroy(seeded);
        for (int q = 0; q < NQ; q++) {
            if (!used(q)) continue;
            (void)hipEventDestroy(join[q]);
            (void)hipStreamDestroy(br[q]);
        }
        (void)hipStreamDestroy(st);
    }
    for (size_t k = 0; k < batched.size(); k++) {
        const int j = batched[k];
        episdet_dataset *ds = dss[j];
        const unsigned count = stage_ctl(ds->stage)[0], over = stage_ctl(ds->stage)[1];
        if (count == 0 || over || count > batch_cap(opts[j], opts[j].order, ktile[j])) {
            solo.push_back(j);     // overflow: exact rerun on its own
            continue;
        }
        episdet_result &r = results[j];
        CHK(collect_best(ds, opts[j].order, opts[j].score, (int)count, &r));
        // the graph's device time; its re-scoring kernel is part of it
        // (rescore_ms stays 0 for batched jobs)
        r.kernel_ms = gms;
        r.tile = ktile[j];
        r.margin = make_ctx(ds, opts[j].score, opts[j].order).margin;
        r.path = EPISDET_PATH_FUSED_MFMA;
        r.rounds = episdet_reference_rounds(opts[j].order, ds->n);
        r.sets = sets_total(opts[j].order, ds->n);
    }
    for (int j : solo) {
        const double pm = results[j].prep_ms;
        episdet_options o = opts[j];
        o.rebuild = 0;
        CHK(episdet_run(dss[j], &o, &results[j]));
        results[j].prep_ms = pm;
    }
    const double wall = now_s() - t0;
    for (int j = 0; j < njobs; j++) results[j].wall_s = wall;
    if (batch_ms) *batch_ms = gms;
    return EPISDET_OK;
}

int episdet_search_batch(const episdet_job *jobs, int njobs, const episdet_options *opt, episdet_result *results,
                         double *batch_ms)
{
    if (!jobs || njobs <= 0 || !results) return EPISDET_ERR_INVALID;
    std::vector<episdet_dataset *> dss(njobs, nullptr);
    std::vector<episdet_options> opts(njobs);
    int rc = EPISDET_OK;
    for (int j = 0; j < njobs && rc == EPISDET_OK; j++) {
        const episdet_job &jb = jobs[j];
        rc = episdet_dataset_create(jb.cases, jb.controls, jb.numSNPs, jb.numCases, jb.numControls, jb.casesWords,
                                    jb.controlsWords, &dss[j]);
        std::memset(&opts[j], 0, sizeof(episdet_options));
        if (opt) opts[j] = *opt;
        opts[j].order = jb.order;
        opts[j].score = jb.score;
    }
    if (rc == EPISDET_OK) rc = episdet_run_batch(dss.data(), opts.data(), njobs, results, batch_ms);
    for (episdet_dataset *ds : dss) episdet_dataset_destroy(ds);
    return rc;
}

int episdet_tables(episdet_dataset *ds, int order, const int *sets, int m, unsigned *out)
{
    if (!ds || !sets || !out || m < 0 || (order != 2 && order != 3)) return EPISDET_ERR_INVALID;
    if (m == 0) return EPISDET_OK;
    for (int i = 0; i < m; i++) {
        for (int o = 0; o < order; o++) {
            const int v = sets[i * order + o];
            if (v < 0 || v >= ds->n || (o > 0 && v <= sets[i * order + o - 1])) return EPISDET_ERR_INVALID;
        }
    }
    if (order == 3) CHK(ensure_pairs(ds));
    std::vector<unsigned long long> hp(m);
    for (int i = 0; i < m; i++) {
        const int *s = sets + (size_t)i * order;
        hp[i] = order == 3 ? ((unsigned long long)s[0] | ((unsigned long long)s[1] << 21) |
                              ((unsigned long long)s[2] << 42))
                           : ((unsigned long long)s[0] | ((unsigned long long)s[1] << 32));
    }
    const int nc = order == 3 ? 27 : 9;
    unsigned long long *d_sets = nullptr;
    uint32_t *d_cells = nullptr;
    if (hipMalloc(&d_sets, sizeof(unsigned long long) * m) != hipSuccess) return EPISDET_ERR_ALLOC;
    if (hipMalloc(&d_cells, sizeof(uint32_t) * (size_t)m * 2 * nc) != hipSuccess) {
        (void)hipFree(d_sets);
        return EPISDET_ERR_ALLOC;
    }
    HIPCHK(hipMemcpy(d_sets, hp.data(), sizeof(unsigned long long) * m, hipMemcpyHostToDevice));
    RescoreArgs r;
    std::memset(&r, 0, sizeof r);
    r.p0 = ds->planes[0];
    r.p1 = ds->planes[1];
    r.W0 = ds->W[0];
    r.W1 = ds->W[1];
    r.n = ds->n;
    r.N0 = ds->N[0];
    r.N1 = ds->N[1];
    r.order = order;
    r.singles = ds->singles;
    r.pairs = ds->pairs;
    r.cand = d_sets;
    r.count = m;
    r.out_cells = d_cells;
    hipLaunchKernelGGL(k_rescore, dim3(m), dim3(64), 0, ds->stream, r);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(ds->stream));
    HIPCHK(hipMemcpy(out, d_cells, sizeof(uint32_t) * (size_t)m * 2 * nc, hipMemcpyDeviceToHost));
    (void)hipFree(d_sets);
    (void)hipFree(d_cells);
    return EPISDET_OK;
}

static int dump_or_checksum(episdet_dataset *ds, int order, int path, int tile, unsigned *out, size_t capacity,
                            unsigned long long *checksum)
{
    if (!ds || (order != 2 && order != 3)) return EPISDET_ERR_INVALID;
    if (path != EPISDET_PATH_FUSED_VALU && path != EPISDET_PATH_AUTO && path != EPISDET_PATH_FUSED_MFMA)
        return EPISDET_ERR_INVALID;
    const bool mfma = path == EPISDET_PATH_FUSED_MFMA;
    if (mfma && !mfma_ok(ds)) return EPISDET_ERR_INVALID;
    if (!tile_valid(order, mfma ? EPISDET_PATH_FUSED_MFMA : EPISDET_PATH_FUSED_VALU, tile)) return EPISDET_ERR_INVALID;
    const int nc = order == 3 ? 27 : 9;
    const unsigned long long total = episdet_n_choose_k((unsigned)ds->n, (unsigned)order);
    if (total == 0) {                  // fewer SNPs than a set holds
        if (checksum) *checksum = 0ull;
        return EPISDET_OK;
    }
    uint32_t *d_dump = nullptr;
    if (out) {
        if (capacity < total * 2 * nc) return EPISDET_ERR_INVALID;
        if (hipMalloc(&d_dump, sizeof(uint32_t) * total * 2 * nc) != hipSuccess) return EPISDET_ERR_ALLOC;
    }
    if (order == 3) CHK(ensure_pairs(ds));
    int rc;
    if (order == 3) {
        const Tri3Tile vt = TRI_TILES[mfma ? 0 : tile];
        const int t[3] = {mfma ? mfma_ty(tile) : 16 * vt.A, mfma ? mfma_tz(tile) : 16 * vt.B, mfma ? mfma_xstep(tile) : 1};
        TriArgs ta;
        fill_tri_common(ds, ta);
        rc = ensure_groups(ds, t, &ta.ngroups, &ta.nunits);
        if (rc != EPISDET_OK) {
            if (d_dump) (void)hipFree(d_dump);
            return rc;
        }
        ta.gstart = ds->gstart;
        ta.groups = ds->groups;
        ta.dump = d_dump;
        CHK(init_single(ds, ta, ta.nunits));
        if (mfma)
            rc = out ? dispatch_tri_mfma<MODE_DUMP>(ds, tile, ta, ds->stream)
                     : dispatch_tri_mfma<MODE_CHECKSUM>(ds, tile, ta, ds->stream);
        else
            rc = out ? dispatch_tri<MODE_DUMP>(ds, tile, ta, 0, ds->stream)
                     : dispatch_tri<MODE_CHECKSUM>(ds, tile, ta, 0, ds->stream);
    } else {
        PairArgs pa;
        fill_pairs(ds, pa, mfma, tile);
        pa.dump = d_dump;
        CHK(init_single(ds, pa, pa.nunits));
        rc = out ? dispatch_pairs<MODE_DUMP>(ds, mfma, tile, pa, ds->stream)
                 : dispatch_pairs<MODE_CHECKSUM>(ds, mfma, tile, pa, ds->stream);
    }
    HIPCHK(hipStreamSynchronize(ds->stream));
    if (rc == EPISDET_OK && out)
        HIPCHK(hipMemcpy(out, d_dump, sizeof(uint32_t) * total * 2 * nc, hipMemcpyDeviceToHost));
    if (rc == EPISDET_OK && checksum) {
        Ctl hc;
        HIPCHK(hipMemcpy(&hc, ds->ctl, sizeof hc, hipMemcpyDeviceToHost));
        *checksum = hc.checksum;
    }
    if (d_dump) (void)hipFree(d_dump);
    return rc;
}

int episdet_dump_tables(episdet_dataset *ds, int order, int path, int tile, unsigned *out, size_t capacity)
{
    if (!out) return EPISDET_ERR_INVALID;
    return dump_or_checksum(ds, order, path, tile, out, capacity, nullptr);
}

int episdet_checksum(episdet_dataset *ds, int order, int path, int tile, unsigned long long *checksum)
{
    if (!checksum) return EPISDET_ERR_INVALID;
    return dump_or_checksum(ds, order, path, tile, nullptr, 0, checksum);
}

}  // extern "C"
