// kernels_mfma_pairs2.hpp -- fused 2-way search on the matrix cores, two
// workgroups per CU, classes in sequence.
//
// Same contraction, FP4 encoding and pair tables as k_pairs_mfma.  That
// kernel's 512-thread workgroup and 128 KB of LDS leave one workgroup per
// CU, so the matrix cores idle while it builds and scores the tables of a
// unit; and since its cases and controls waves run side by side, the waves
// of the smaller class finish early when the classes differ in size.  This
// version:
//  * work unit: 64 A SNPs x 64 B SNPs (A tile <= B tile), in triangular
//    order, or from 16 tiles up in XCD blocks taken from per-XCD queues
//    (blocked_unrank, fetch_xcd), so that the units one XCD runs at once
//    share their rows in its L2;
//  * 256 threads = 4 waves; wave w owns A SNPs 32(w/2)..+31 (64 rows, 2 row
//    tiles) x B SNPs 32(w%2)..+31 (64 rows, 2 column tiles), for both
//    classes: 2 x 2 x 2 MFMA tiles, 128 accumulators;
//  * the chunks of the cases, then those of the controls, form one
//    sequence that all four waves contract together, so every wave does the
//    same work whatever the class sizes;
//  * a 1024-sample chunk is 128 A rows + 128 B rows of 128 bytes (32 KB),
//    loaded straight to LDS through the scalar buffer descriptor of its
//    class, double-buffered: chunk t + 1 is issued after the barrier that
//    starts chunk t;
//  * the B rows of a wave lie by plane, so its column tile cb is plane cb of 32
//    B SNPs and a lane ends up with all eight counts of its 16 pairs (one B,
//    16 A).  It bounds their scores in FP32 straight from its registers
//    (quick_bound, about 85 vector instructions a pair); only the pairs that
//    leaves go through LDS to integer tables and FP32 scores.  Before, every
//    pair's counts went through LDS and both its classes' tables were derived
//    first: pairs at 3001 x 9973 took 167 us a search, now 143, and 8192 x
//    2000 0.67 ms of kernel time, now 0.25.
// LDS: 64 KB stage / dump area, the ln m! table and the unit's single counts,
// so two workgroups fit a CU and one's scoring runs beside the other's
// counting.
#pragma once
#include "kernels_mfma_pairs.hpp"
#include "kernels_mfma4.hpp"

namespace episdet {

constexpr int P3_TA = 64, P3_TB = 64;
constexpr int P3_KW = 32;                                   // words per chunk (1024 samples)
constexpr int P3_AROWS = 2 * P3_TA;                         // 128
constexpr int P3_ROWS = P3_AROWS + 2 * P3_TB;               // 256 rows of a chunk
constexpr int P3_ROWS_PER_LOAD = 8;                         // 128-byte rows: one load = 1 KB
constexpr int P3_LOADS = P3_ROWS / P3_ROWS_PER_LOAD;        // 32 per chunk
constexpr int P3_LOADS_PER_WAVE = P3_LOADS / 4;             // 8
constexpr int P3_BUF_WORDS = P3_ROWS * P3_KW;               // 8192 (32 KB)
constexpr int P3_STAGE_WORDS = 2 * P3_BUF_WORDS;            // double-buffered (64 KB)
constexpr int P3_CLASS_WORDS = 2 * 8 * 64 * 2;              // a row tile's counts of a class: plane of B x A x lane x plane of A
constexpr int P3_DUMP_WORDS = 4 * 2 * P3_CLASS_WORDS;       // wave x class (64 KB)
constexpr int P3_SMEM_WORDS = P3_STAGE_WORDS > P3_DUMP_WORDS ? P3_STAGE_WORDS : P3_DUMP_WORDS;
static_assert(P3_KW == M2_KW, "128-byte rows use the swizzle of m2_at");

// Byte offsets, within a class's planes, of slot q of each LDS row this
// lane loads (load k of wave w fills rows 8(w + 4k) .. +7); one set per
// class, since the classes' word counts differ.
__device__ __forceinline__ void p3_row_offsets(int W, int a0, int b0, int w, int lane,
                                               unsigned (&roff)[P3_LOADS_PER_WAVE])
{
    const int rl = lane >> 3, q = (lane & 7) ^ rl;
#pragma unroll
    for (int k = 0; k < P3_LOADS_PER_WAVE; k++) {
        const int r = (w + 4 * k) * P3_ROWS_PER_LOAD + rl;
        const int rb = r - P3_AROWS;         // 64 (b / 32) + 32 plane + b % 32
        const int row = r < P3_AROWS ? 2 * a0 + r : 2 * (b0 + (rb >> 6) * 32 + (rb & 31)) + ((rb >> 5) & 1);
        roff[k] = ((unsigned)row * (unsigned)W + (unsigned)(q * 4)) * 4u;
    }
}

__device__ __forceinline__ void p3_issue_buf(i32x4_t rsrc, const unsigned (&roff)[P3_LOADS_PER_WAVE], int w0,
                                             unsigned buf, int w)
{
#pragma unroll
    for (int k = 0; k < P3_LOADS_PER_WAVE; k++)
        lds_dma16(rsrc, buf + (unsigned)((w + 4 * k) * P3_ROWS_PER_LOAD * P3_KW * 4), roff[k], (unsigned)(w0 * 4));
}

template <int C>
__device__ __forceinline__ void p3_step(const uint4 (&aw)[2], const uint4 (&bw)[2], v16f_t (&acc)[2][2])
{
    constexpr int s = mf_scale<C>();
    const v8i_t A0 = mf_operand<C>(aw[0]), A1 = mf_operand<C>(aw[1]);
#pragma unroll
    for (int cb = 0; cb < 2; cb++) {
        const v8i_t B = mf_operand<C>(bw[cb]);
        acc[0][cb] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A0, B, acc[0][cb], 4, 4, 0, s, 0, s);
        acc[1][cb] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A1, B, acc[1][cb], 4, 4, 0, s, 0, s);
    }
}

// Contracts one staged chunk into one class's accumulators.
__device__ __forceinline__ void p3_chunk(const uint32_t *cur, int ar0, int ar1, int br0, int br1, int h,
                                         v16f_t (&acc)[2][2])
{
#pragma unroll
    for (int s = 0; s < P3_KW / 8; s++) {
        const int q = 2 * s + h;
        uint4 aw[2], bw[2];
        aw[0] = *(const uint4 *)&cur[m2_at(ar0, q)];
        aw[1] = *(const uint4 *)&cur[m2_at(ar1, q)];
        bw[0] = *(const uint4 *)&cur[m2_at(br0, q)];
        bw[1] = *(const uint4 *)&cur[m2_at(br1, q)];
        p3_step<0>(aw, bw, acc);
        p3_step<1>(aw, bw, acc);
        p3_step<2>(aw, bw, acc);
        p3_step<3>(aw, bw, acc);
    }
}

// A unit number with a pair in it, and its tiles: units of XCD blocks that lie
// outside the triangle are passed over here, by the one thread that fetches.
struct P3Unit {
    unsigned long long uu;
    int tA, tB;
};
__device__ __forceinline__ P3Unit p3_fetch(const BatchPair &bp)
{
    P3Unit r;
    for (;;) {
        r.uu = bp.xcd ? fetch_xcd(bp.queue, bp.total) : atomicAdd(bp.queue, 1ull);
        if (r.uu >= bp.total) return r;
        int j = 0;
        while (j + 1 < bp.njobs && bp.job_start[j + 1] <= r.uu) j++;
        const unsigned long long u = r.uu - bp.job_start[j];
        if (!bp.jobs[j].blocked) {
            unrank_tri(u, r.tA, r.tB);
            return r;
        }
        if (blocked_unrank(u, bp.jobs[j].ntiles, r.tA, r.tB)) return r;
    }
}

// Single counts of a unit's SNPs for quick_bound: T of genotypes 0, 1, 2 and
// their D = cases - pi T, eight words each (two unused).
__device__ __forceinline__ void p3_single(const PairArgs &p, int v, float *o)
{
    const Singles s = ld_global(p.singles, min(v, p.n - 1));
    const uint32_t c2 = (uint32_t)p.N0 - s.x - s.y, t2 = (uint32_t)p.N1 - s.z - s.w;
    const float T0 = (float)(s.x + s.z), T1 = (float)(s.y + s.w), T2 = (float)(c2 + t2), pi = p.sc.lb_pi;
    *(float4 *)o = make_float4(T0, T1, T2, fmaf(-pi, T0, (float)s.x));
    *(float4 *)(o + 4) = make_float4(fmaf(-pi, T1, (float)s.y), fmaf(-pi, T2, (float)c2), 0.f, 0.f);
}

// Quick bound of one pair from its counts c[class][plane of A][plane of B].
__device__ __forceinline__ bool p3_quick(const ScoreCtx &sc, const float (&c)[2][2][2], const float4 &a0,
                                         const float4 &a1, const float4 &b0, const float4 &b1, float thr, bool valid)
{
    float T[9], D[9];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            T[i * 3 + j] = c[0][i][j] + c[1][i][j];
            D[i * 3 + j] = fmaf(-sc.lb_pi, T[i * 3 + j], c[0][i][j]);
        }
    auto derive = [](float (&t)[9], float A0, float A1, float A2, float B0, float B1) {
        t[2] = (A0 - t[0]) - t[1];
        t[5] = (A1 - t[3]) - t[4];
        t[6] = (B0 - t[0]) - t[3];
        t[7] = (B1 - t[1]) - t[4];
        t[8] = (A2 - t[6]) - t[7];
    };
    derive(T, a0.x, a0.y, a0.z, b0.x, b0.y);
    derive(D, a0.w, a1.x, a1.y, b0.w, b1.x);
    return quick_bound<9>(sc, T, D, thr, valid);
}

template <int MODE>
__global__ __launch_bounds__(256, 2) void k_pairs_mfma2(BatchPair bp)
{
    static_assert(MODE != MODE_PAIRTABLE, "the pair table is built by k_pairs_mfma");
    __shared__ __attribute__((aligned(16))) uint32_t smem[P3_SMEM_WORDS];
    __shared__ __attribute__((aligned(16))) float s_one[scores_sets(MODE) ? 128 * 8 : 4];    // 64 A, 64 B
    __shared__ P3Unit s_u;
    __shared__ unsigned s_best;
    __shared__ float s_lnf[scores_sets(MODE) ? LNF_SMALL : 1];
    if constexpr (scores_sets(MODE)) load_lnf(s_lnf);
    const int tid = threadIdx.x;
    const int w = uniform(tid >> 6), rp = w >> 1, cp = w & 1;

    unsigned long long jfirst = 0, jend = 0;
    PairArgs p;
    // The unit is fetched here, not while the last chunk is contracted: wave 0
    // would hold the others up there, and searches of few units bind them too early
    // (5284 x 113538 took 2.40 ms that way, 2.32 this way).
    if (tid == 0) s_u = p3_fetch(bp);
    for (int it = 0;; it++) {
        __syncthreads();
        if (it && tid == 0) s_u = p3_fetch(bp);
        __syncthreads();
        const unsigned long long uu = uniform(s_u.uu);
        if (uu >= bp.total) break;
        const int a0 = uniform(s_u.tA) * P3_TA, b0 = uniform(s_u.tB) * P3_TB;
        if (uu < jfirst || uu >= jend) {                  // per-XCD queues go out of order
            int j = 0;
            while (j + 1 < bp.njobs && ld_const(bp.job_start, (size_t)(j + 1)) <= uu) j++;
            p = ld_const(bp.jobs, (size_t)j);
            jfirst = ld_const(bp.job_start, (size_t)j);
            jend = ld_const(bp.job_start, (size_t)(j + 1));
        }
        // LDS rows read by this lane: A rows of its two row tiles (tile row i =
        // 2 snp + plane), B rows of its two planes (made per unit: they are not
        // to hold registers through the scoring)
        const int lane = opaque(tid & 63), h = lane >> 5, i = lane & 31;
        const int ar0 = 64 * rp + i, ar1 = 64 * rp + 32 + i;
        const int br0 = P3_AROWS + 64 * cp + i, br1 = P3_AROWS + 64 * cp + 32 + i;
        const int nch0 = p.W0 / P3_KW, nch = nch0 + p.W1 / P3_KW;
        const i32x4_t rs0 = m2_rsrc(p.p0, p.bytes0), rs1 = m2_rsrc(p.p1, p.bytes1);
        unsigned roff0[P3_LOADS_PER_WAVE], roff1[P3_LOADS_PER_WAVE];
        p3_row_offsets(p.W0, a0, b0, w, lane, roff0);
        p3_row_offsets(p.W1, a0, b0, w, lane, roff1);

        v16f_t acc[2][2][2];                                // [class][row tile][plane of B]
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int rb = 0; rb < 2; rb++)
#pragma unroll
                for (int cb = 0; cb < 2; cb++)
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[c][rb][cb][r] = 0.f;

        // chunk t of the sequence: cases chunk t, or controls chunk t - nch0
        if (nch > 0) {
            if (nch0 > 0) p3_issue_buf(rs0, roff0, 0, lds_addr(smem), w);
            else p3_issue_buf(rs1, roff1, 0, lds_addr(smem), w);
        }
        if constexpr (scores_sets(MODE)) {
            const int e = opaque(tid);
            if (e < 128) p3_single(p, e < 64 ? a0 + e : b0 + e - 64, s_one + e * 8);
        }
        unsigned best = 0;
        // two loops, one per class, so each contracts into one fixed set of
        // accumulators
#pragma unroll
        for (int c = 0; c < 2; c++) {
            for (int t = c ? nch0 : 0; t < (c ? nch : nch0); t++) {
                // this wave's loads of chunk t are its only outstanding ones
                __builtin_amdgcn_s_waitcnt(m4_wait_vm(0));
                __syncthreads();
                const int tn = t + 1;
                if (tn < nch) {
                    uint32_t *nb = smem + (tn & 1) * P3_BUF_WORDS;
                    if (tn < nch0) p3_issue_buf(rs0, roff0, tn * P3_KW, lds_addr(nb), w);
                    else p3_issue_buf(rs1, roff1, (tn - nch0) * P3_KW, lds_addr(nb), w);
                } else if (tid == 0) {
                    // the score bound arrives while the last chunk is contracted
                    if constexpr (scores_sets(MODE))
                        best = __hip_atomic_load(p.co.best_key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                p3_chunk(smem + (t & 1) * P3_BUF_WORDS, ar0, ar1, br0, br1, h, acc[c]);
            }
        }
        __builtin_amdgcn_s_waitcnt(0);
        if (tid == 0) s_best = best;
        __syncthreads();

        // Each wave scores what it counted.  Output register r = 4 q + 2 s + i
        // of row tile rb holds, in lane 32 h + b, A = 16 rb + 4 q + 2 h + s,
        // plane i, against B = b.
        const int ln = opaque(tid & 63), eh = ln >> 5, eb = ln & 31;
        const int A0 = a0 + 32 * rp + 2 * eh, B = b0 + 32 * cp + eb;
        unsigned long long hsum = 0;
        // sets whose badness lower bound is above this cannot become
        // candidates; their FP32 score is skipped (skip_threshold)
        float thr = INFINITY;
        if constexpr (scores_sets(MODE)) thr = skip_threshold(p.sc, s_best);
        // counts of a row tile -> LDS [class][plane of B][m][lane][plane of A], m = 2 q + s;
        // read by this wave alone
        float *dump = (float *)smem + w * 2 * P3_CLASS_WORDS;
        auto put = [&](const v16f_t &v, int cls, int cb) {
#pragma unroll
            for (int m = 0; m < 8; m++) {
                const int r = 4 * (m >> 1) + 2 * (m & 1);
                *(float2 *)&dump[cls * P3_CLASS_WORDS + ((cb * 8 + m) * 64 + ln) * 2] = make_float2(v[r], v[r + 1]);
            }
        };
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int cb = 0; cb < 2; cb++) put(acc[c][0][cb], c, cb);
        __builtin_amdgcn_wave_barrier();
        const float4 *oneB = (const float4 *)(s_one + (64 + 32 * cp + eb) * 8);
        // rolled, so the kernel holds the scoring code once
#pragma unroll 1
        for (int rb = 0;; rb++) {
            const int A1 = A0 + 16 * rb;
            auto read = [&](int m, float2 (&v)[2][2]) {     // [class][plane of B]
#pragma unroll
                for (int c = 0; c < 2; c++)
#pragma unroll
                    for (int j = 0; j < 2; j++)
                        v[c][j] = *(const float2 *)&dump[c * P3_CLASS_WORDS + ((j * 8 + m) * 64 + ln) * 2];
            };
            // bit m: this lane's pair with A1 + 4 q + s is not ruled out
            unsigned todo = 0;
#pragma unroll
            for (int m = 0; m < 8; m++) {
                const int A = A1 + 4 * (m >> 1) + (m & 1);
                todo |= (A < B && B < p.n) ? 1u << m : 0u;
            }
            // While no bound is known (a search's first units: half of them at
            // 3001 x 9973), one pair per lane is scored and the bound read again
            // before the rest is bounded.
            bool quick = scores_sets(MODE) && thr < INFINITY;
#pragma unroll 1
            for (;;) {
                if constexpr (scores_sets(MODE)) {
                    if (quick && p.sc.fb_scale > 0.f && __ballot(todo != 0)) {
                        const float4 b0v = oneB[0], b1v = oneB[1];
                        const float4 *oneA = (const float4 *)(s_one + (32 * rp + 16 * rb + 2 * eh) * 8);
                        unsigned keep = 0;
#pragma unroll 2
                        for (int m = 0; m < 8; m++) {
                            float2 v[2][2];
                            read(m, v);
                            const float4 *o = oneA + (4 * (m >> 1) + (m & 1)) * 2;
                            const float c[2][2][2] = {{{v[0][0].x, v[0][1].x}, {v[0][0].y, v[0][1].y}},
                                                      {{v[1][0].x, v[1][1].x}, {v[1][0].y, v[1][1].y}}};
                            keep |= p3_quick(p.sc, c, o[0], o[1], b0v, b1v, thr, (todo >> m) & 1u) ? 0u : 1u << m;
                        }
                        todo &= keep;
                    }
                    quick = false;
                }
                if (!__ballot(todo != 0)) break;
                float bad = INFINITY;
                unsigned long long packed = 0;
                if (todo) {
                    const int m = __ffs(todo) - 1;
                    todo &= todo - 1;
                    const int A = A1 + 4 * (m >> 1) + (m & 1);
                    float2 v[2][2];
                    read(m, v);
                    uint32_t n4[2][4];
#pragma unroll
                    for (int c = 0; c < 2; c++)
#pragma unroll
                        for (int j = 0; j < 2; j++) {
                            n4[c][j] = (uint32_t)v[c][j].x;
                            n4[c][2 + j] = (uint32_t)v[c][j].y;
                        }
                    const Singles sa = ld_global(p.singles, A), sb = ld_global(p.singles, B);
                    uint32_t cas[9], ctl[9];
                    pair9(n4[0][0], n4[0][1], n4[0][2], n4[0][3], sa.x, sa.y, sb.x, sb.y, (uint32_t)p.N0, cas);
                    pair9(n4[1][0], n4[1][1], n4[1][2], n4[1][3], sa.z, sa.w, sb.z, sb.w, (uint32_t)p.N1, ctl);
                    packed = (unsigned long long)A | ((unsigned long long)B << 32);
                    if constexpr (scores_sets(MODE)) {
                        if (!(thr < INFINITY && p.sc.fb_scale == 0.f && bound_exceeds<9>(p.sc, cas, ctl, thr)))
                            bad = badness_f32_flat<9>(p.sc, cas, ctl, s_lnf);
                    } else if constexpr (MODE == MODE_DUMP) {
                        uint32_t *o = p.dump + rank2(A, B) * 18;
                        for (int c = 0; c < 9; c++) {
                            o[c] = cas[c];
                            o[9 + c] = ctl[c];
                        }
                    } else if constexpr (MODE == MODE_CHECKSUM) {
                        hsum += table_hash(rank2(A, B), cas, ctl, 9);
                    }
                }
                if constexpr (MODE == MODE_SEARCH) publish_wave(p.co, p.sc.margin, bad, packed);
                if constexpr (MODE == MODE_TOPK) publish_wave_topk(p.co, p.sc.margin, bad, packed);
                if constexpr (scores_sets(MODE)) {
                    if (!(thr < INFINITY)) {
                        thr = skip_threshold(p.sc, __hip_atomic_load(p.co.best_key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                        quick = thr < INFINITY;
                    }
                }
            }
            if (rb) break;
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
                for (int cb = 0; cb < 2; cb++) put(acc[c][1][cb], c, cb);
            __builtin_amdgcn_wave_barrier();
        }
        if constexpr (MODE == MODE_CHECKSUM) {
            if (hsum) atomicAdd(p.checksum, hsum);
        }
    }
}

}  // namespace episdet
