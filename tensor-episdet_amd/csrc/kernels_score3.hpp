// kernels_score3.hpp -- scoring of a 3-way work unit's sets (versions 4 and
// 5): the counts of half a unit lie in LDS, one wave scores one X against
// 8 Y x 32 Z of them.
//
// Scoring, not counting, bounds searches of few samples: at 1000 SNPs x 4000
// samples the matrix cores need 1.4 ms, and a search that derived both
// classes' 27 integer cells of every triplet before it bounded its score took
// 4.45 ms (540 vector instructions per triplet beside the contraction's).
// Nearly every triplet only has to be shown not to matter, so that is what the
// first pass does, in FP32 from what the accumulators already hold:
//  * a lane keeps one Z, so its (X, Z) pair tables are registers of the whole
//    unit, the (X, Y) ones broadcast LDS words made once per unit, and only
//    the (Y, Z) ones are read per triplet, one triplet ahead;
//  * every cell is derived for the cell total T and for D = cases - pi T,
//    not for the two classes, since D^2 / T is all the bound needs;
//  * 1 / T is one integer subtraction (recip_above).
// That is about 250 instructions per triplet: a search at 1000 x 4000 (MI)
// took 3.67 ms with it, 777 x 20001 (K2, no signal, 30% cases) 6.46 instead of
// 7.21, 2048 x 262144 809 instead of 811.  Lanes whose triplet it cannot rule
// out are collected in a bit mask, and a second, rolled loop takes the exact
// integer tables and the FP32 score for those alone; with the scores
// branch-free (badness_f32_flat) and the search seeded (kernels_seed.hpp)
// the first is at 3.23 ms, the second at 6.05.
#pragma once
#include "kernels_valu.hpp"

namespace episdet {

// 1/t <= recip_above(t) <= 1.125/t for a normal t >= 1: with t = 2^e (1 + m),
// the float whose bits are 0x7F000000 - bits(t) is 2^-e (2 - m) / 2, and
// (1 + m)(2 - m) / 2 runs from 1 (m = 0 and 1) to 1.125 (m = 1/2).
__device__ __forceinline__ float recip_above(float t) { return __uint_as_float(0x7F000000u - __float_as_uint(t)); }

// 27 cells of one table in FP32 from the eight counts with genotypes 0 and 1
// (already in t) and the pair marginals: triplet27's derivation.  xy holds
// {00, 01, 10, 11, 20, 21}, xz all nine cells, yz {00, 01, 10, 11}.
__device__ __forceinline__ void derive27(float (&t)[27], const float (&xy)[6], const float (&xz)[9],
                                         const float (&yz)[4])
{
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
            t[EPI_C3(i, j, 2)] = (xy[i * 2 + j] - t[EPI_C3(i, j, 0)]) - t[EPI_C3(i, j, 1)];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int k = 0; k < 3; k++)
            t[EPI_C3(i, 2, k)] = (xz[i * 3 + k] - t[EPI_C3(i, 0, k)]) - t[EPI_C3(i, 1, k)];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int k = 0; k < 2; k++)
            t[EPI_C3(2, j, k)] = (yz[j * 2 + k] - t[EPI_C3(0, j, k)]) - t[EPI_C3(1, j, k)];
#pragma unroll
    for (int j = 0; j < 2; j++) t[EPI_C3(2, j, 2)] = (xy[4 + j] - t[EPI_C3(2, j, 0)]) - t[EPI_C3(2, j, 1)];
#pragma unroll
    for (int k = 0; k < 3; k++) t[EPI_C3(2, 2, k)] = (xz[6 + k] - t[EPI_C3(2, 0, k)]) - t[EPI_C3(2, 1, k)];
}

// Whether a table's quick badness bound exceeds thr, from the cell totals T
// and D = cases - pi T.  With recip_above for 1/T, S' = sum D^2 r is between
// S and 1.125 S (up to roundings, which fb_scale covers), so
//   lb_max - fb_scale S'  (+ for K2 fb_lnw L + lb_off)
// is bound_exceeds's bound or lower.  L sums the bits of max(T, 1) above
// those of 1.0f: bits(t) / 2^23 - 127 = e + m <= e + log2(1 + m) = log2 t, so
// L / 2^23 is at most sum log2 max(T, 1) (27 of them stay below 2^9 for
// fewer than 2^23 samples, so the 32-bit sum does not wrap).
// Where a lane of the wave (of those with `valid`) is left, a second bound
// replaces the constant K of fb_scale, which holds for cells of cases or
// controls alone, by one that follows the cell:  KL(p || pi) = d^2 k(p), d =
// p - pi, with k(p) = integral over u in [0, 1] of (1 - u) / (t (1 - t)), t =
// pi + u d, an average of convex functions of p, so k is convex and
// k(p) <= k(pi) + a |d|, a the larger slope of the chords to p = 0 and p = 1.
// The sums become sum D e (tb_k + tb_a |e|) with e = D r, |e| >= |d|.  On
// data without signal (777 x 20001, 30% cases, K2) the first bound leaves 3% of the triplets.
template <int NC>
__device__ __forceinline__ bool quick_bound(const ScoreCtx &sc, const float (&T)[NC], const float (&D)[NC], float thr,
                                            bool valid)
{
    float s = 0.f;
    unsigned l = 0u - (unsigned)NC * 0x3F800000u;
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const float t = fmaxf(T[c], 1.f);
        s = fmaf(D[c], D[c] * recip_above(t), s);
        l += __float_as_uint(t);
    }
    // (fb_lnw is 0 and lb_off 0 for MI)
    const float top = fmaf(sc.fb_lnw, (float)l, sc.lb_max + sc.lb_off);
    bool out = fmaf(-sc.fb_scale, s, top) > thr;
    if (__ballot(valid && !out)) {
        s = 0.f;
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const float e = D[c] * recip_above(fmaxf(T[c], 1.f));
            s = fmaf(D[c] * e, fmaf(sc.tb_a, fabsf(e), sc.tb_k), s);
        }
        out = out || top - s > thr;
    }
    return out;
}

// Pair marginals of (a, b) for quick_bound: totals and D of the nine cells.
__device__ __forceinline__ void pair_td9(const uint4 *pairs, int n, const Singles &sa, const Singles &sb, int a, int b,
                                         uint32_t N0, uint32_t N1, float pi, float (&T)[9], float (&D)[9])
{
    uint32_t cas[9], ctl[9];
    pair9_lookup(pairs, n, sa, sb, a, b, 0, N0, cas);
    pair9_lookup(pairs, n, sa, sb, a, b, 1, N1, ctl);
#pragma unroll
    for (int c = 0; c < 9; c++) {
        T[c] = (float)(cas[c] + ctl[c]);
        D[c] = fmaf(-pi, T[c], (float)cas[c]);
    }
}

// Pair marginals of a unit in LDS, made by its first 128 threads while its
// first chunk loads.  (X, Y), both X and the 32 Y: 12 words each, [T 00 01 10
// 11] [T 20 21, D 20 21] [D 00 01 10 11].  (X, Z), both X and the 32 Z: nine
// T and nine D, [word][entry], read by a lane once for all its triplets.
constexpr int S3_XY_WORDS = 64 * 12, S3_XZ_WORDS = 18 * 64;
struct S3Pairs {
    __attribute__((aligned(16))) float xy[S3_XY_WORDS];
    float xz[S3_XZ_WORDS];
};
__device__ __forceinline__ void s3_fill(const TriArgs &p, int X0, int y0, int z0, int tid, S3Pairs &s)
{
    if (tid >= 128) return;
    const int e = tid & 63;
    // entries past the last SNP or with the other SNP <= X belong to no set:
    // any table that exists will do
    const int X = min(X0 + (e >> 5), p.n - 2);
    const int o = max(min((tid < 64 ? y0 : z0) + (e & 31), p.n - 1), X + 1);
    float T[9], D[9];
    pair_td9(p.pairs, p.n, ld_global(p.singles, X), ld_global(p.singles, o), X, o, (uint32_t)p.N0, (uint32_t)p.N1,
             p.sc.lb_pi, T, D);
    if (tid < 64) {
        float4 *w = (float4 *)(s.xy + e * 12);
        w[0] = make_float4(T[0], T[1], T[3], T[4]);
        w[1] = make_float4(T[6], T[7], D[6], D[7]);
        w[2] = make_float4(D[0], D[1], D[3], D[4]);
    } else {
#pragma unroll
        for (int k = 0; k < 9; k++) {
            s.xz[k * 64 + e] = T[k];
            s.xz[(9 + k) * 64 + e] = D[k];
        }
    }
}

// (X, Z) marginals of a lane (entry e).
struct S3Lane {
    float T[9], D[9];
};
__device__ __forceinline__ void s3_lane(const S3Pairs &s, int e, S3Lane &l)
{
#pragma unroll
    for (int k = 0; k < 9; k++) {
        l.T[k] = s.xz[k * 64 + e];
        l.D[k] = s.xz[(9 + k) * 64 + e];
    }
}

// AND-counts of (Y, Z), cases and controls, read one triplet ahead.  A lane
// with no set at Y reads some entry of the table.
struct S3Yz {
    uint4 c0, c1;
};
__device__ __forceinline__ void s3_yz(const TriArgs &p, int Y, int Z, S3Yz &v)
{
    const int z = max(min(Z, p.n - 1), 1);
    const size_t at = ((size_t)min(Y, z - 1) * p.n + z) * 2;
    v.c0 = ld_global(p.pairs, at);
    v.c1 = ld_global(p.pairs, at + 1);
}

// Appends the sets of the lanes with `want`: one counter update per wave.
// Returns the candidate count before (-1: nothing appended); *n: how many.
// The scores go out as device-scope stores, which tighten_topk of any wave
// can read.
__device__ __forceinline__ long long append_wave(const CandOut &co, bool want, float bad, unsigned long long packed,
                                                 unsigned *n)
{
    const unsigned long long m = __ballot(want);
    if (!m) return -1;
    const int lane = threadIdx.x & 63;
    *n = (unsigned)__popcll(m);
    unsigned base = 0;
    if (lane == 0) base = atomicAdd(co.cand_count, *n);
    base = (unsigned)__builtin_amdgcn_readfirstlane((int)base);
    if (want) {
        const unsigned slot = base + (unsigned)__popcll(m & ((1ull << lane) - 1ull));
        if (slot < co.cand_cap) {
            co.cand[slot] = packed;
            __hip_atomic_store(co.cand_s32 + slot, bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            co.cand_count[1] = 1u;
        }
    }
    return (long long)base;
}

// Publication of one set per lane (bad = +inf: none) by one wave: the wave's
// minimum joins the global one, and every set within `margin` of the smaller
// of the two is appended (the argument of publish_candidates, whose
// workgroup minimum this replaces by a wave's).
__device__ __forceinline__ void publish_wave(const CandOut &co, float margin, float bad, unsigned long long packed)
{
    const float wmin = wave_min(bad);
    if (!(wmin < INFINITY)) return;
    unsigned g = __hip_atomic_load(co.best_key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned key = f2key(wmin);
    if (key < g) {
        unsigned old = g;
        if ((threadIdx.x & 63) == 0) old = atomicMin(co.best_key, key);
        old = (unsigned)__builtin_amdgcn_readfirstlane((int)old);
        g = old < key ? old : key;
    }
    unsigned n;
    append_wave(co, bad <= key2f(g) + margin, bad, packed, &n);
}

// Lowers the top-k bound to the k-th smallest score among the last
// TK_WINDOW candidates appended before `count` (one wave).  They are scores
// of distinct sets, so their k-th smallest bounds the k-th best of the search
// from above; slots that are reserved but not written yet hold the +inf the
// host filled them with, which only loosens the result.  A candidate was
// within the bound when it was appended, so the bound moves to about the
// k / TK_WINDOW quantile of what it let through, and a search appends about
// TK_STEP log(sets / k) / log(TK_WINDOW / k) candidates.  The selection is an
// MSB-first radix select over 32 keys per lane, about 14,000 cycles, once per
// TK_STEP candidates.
constexpr unsigned TK_WINDOW = 2048, TK_STEP = 1024;
static_assert(TK_WINDOW >= 2 * 1024, "at least twice the largest k");
__device__ __forceinline__ void tighten_topk(const CandOut &co, unsigned count)
{
    constexpr int R = TK_WINDOW / 64;
    const unsigned lane = threadIdx.x & 63u, first = count > TK_WINDOW ? count - TK_WINDOW : 0u;
    unsigned key[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const unsigned at = first + 64u * r + lane;
        key[r] = at < count ? f2key(__hip_atomic_load(co.cand_s32 + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                            : 0xFF800000u;
    }
    unsigned prefix = 0, k = co.topk;
#pragma unroll 1
    for (int b = 31; b >= 0; b--) {
        const unsigned hi = b == 31 ? 0u : (~0u << (b + 1));
        unsigned z = 0;
#pragma unroll
        for (int r = 0; r < R; r++) z += ((key[r] ^ prefix) & hi) == 0 && ((key[r] >> b) & 1u) == 0;
        z = wave_sum_u(z);
        if (k > z) {
            k -= z;
            prefix |= 1u << b;
        }
    }
    if (lane == 0 && prefix < 0xFF800000u) atomicMin(co.best_key, prefix);
}

// Top-k publication of one set per lane: every set within `margin` of the
// running bound on the k-th best is appended (the bound only decreases, so
// each of the k best sets is appended when it is evaluated), and the wave
// whose candidates cross a multiple of TK_STEP lowers the bound.
__device__ __forceinline__ void publish_wave_topk(const CandOut &co, float margin, float bad,
                                                  unsigned long long packed)
{
    const unsigned g = __hip_atomic_load(co.best_key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const float thr = g >= 0xFF800000u ? INFINITY : key2f(g) + margin;
    unsigned n = 0;
    const long long base = append_wave(co, bad <= thr && bad < INFINITY, bad, packed, &n);
    if (base < 0) return;
    const unsigned long long end = (unsigned long long)base + n;
    if (end <= co.cand_cap && end / TK_STEP != (unsigned long long)base / TK_STEP) tighten_topk(co, (unsigned)end);
}

// Words of a wave's counts in LDS: [class][q][k][lane][ij], q = 0..3, for
// genotype k of Z and ij = 2 i + j of (X, Y).  Lane 32 h + z holds Z = z0 + z
// and, at q, Y = y + 2 q + h: what MFMA output registers 4q..4q+3 of the
// tile with the Z rows of plane k hold in that lane.
constexpr int S3_CLASS_WORDS = 4 * 2 * 64 * 4;

// The same value, out of the compiler's sight: what is computed from it per
// unit is not moved out of the unit loop, where it would hold registers (and,
// with 128 accumulators, spill others) through the contraction.
__device__ __forceinline__ int opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// The counts of (class, wave region, q) as float4 per k.
__device__ __forceinline__ void s3_read(const float *cnt, int cls_stride, int q, int lane, float4 (&c)[2][2])
{
#pragma unroll
    for (int cls = 0; cls < 2; cls++)
#pragma unroll
        for (int k = 0; k < 2; k++)
            c[cls][k] = *(const float4 *)&cnt[cls * cls_stride + ((q * 2 + k) * 64 + lane) * 4];
}

// One wave's share of half a unit: X against Y = y + 2q + h (q = 0..3, h the
// lane half) and Z (one per lane of a half), whose counts start at cnt (cases;
// controls cls_stride words on).  xy: the unit's (X, Y) marginals from
// (X, y) on; e: the lane's entry of its (X, Z) marginals; yz: the (Y, Z) counts
// of q = 0; thr: skip_threshold, read again while it is +inf.
template <int MODE>
__device__ __forceinline__ void s3_score(const TriArgs &p, const float *cnt, int cls_stride, const S3Pairs &s,
                                         const float *xy, int e, S3Yz yz, int X, int y, int Z, int lane, float &thr,
                                         const float *s_lnf, unsigned long long &hsum)
{
    const int h = lane >> 5;
    unsigned todo = 0;                 // bit q: this lane's triplet of q is not ruled out
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int Y = y + 2 * q + h;
        todo |= (X < Y && Y < Z && Z < p.n) ? 1u << q : 0u;
    }
    // While no bound is known (the first units of a search that is not seeded),
    // one triplet per lane is scored and the bound read again before the rest
    // is bounded.
    bool quick = scores_sets(MODE) && thr < INFINITY;
#pragma unroll 1
    for (;;) {
        if constexpr (scores_sets(MODE)) {
            if (quick && p.sc.fb_scale > 0.f && __ballot(todo != 0)) {
                S3Lane xz;
                s3_lane(s, e, xz);
                unsigned keep = 0;
#pragma unroll 1
                for (int q = 0; q < 4; q++) {
                    const uint4 c0 = yz.c0, c1 = yz.c1;
                    if (q < 3) s3_yz(p, y + 2 * q + 2 + h, Z, yz);
                    float4 c[2][2];
                    s3_read(cnt, cls_stride, q, lane, c);
                    const float4 *xyq = (const float4 *)(xy + (2 * q + h) * 12);
                    const float4 e0 = xyq[0], e1 = xyq[1], e2 = xyq[2];
                    const float xyT[6] = {e0.x, e0.y, e0.z, e0.w, e1.x, e1.y};
                    const float xyD[6] = {e2.x, e2.y, e2.z, e2.w, e1.z, e1.w};
                    const float pi = p.sc.lb_pi;
                    const float yzT[4] = {(float)(c0.x + c1.x), (float)(c0.y + c1.y), (float)(c0.z + c1.z),
                                          (float)(c0.w + c1.w)};
                    const float yzD[4] = {fmaf(-pi, yzT[0], (float)c0.x), fmaf(-pi, yzT[1], (float)c0.y),
                                          fmaf(-pi, yzT[2], (float)c0.z), fmaf(-pi, yzT[3], (float)c0.w)};
                    float T[27], D[27];
#pragma unroll
                    for (int k = 0; k < 2; k++) {
                        const float a[4] = {c[0][k].x, c[0][k].y, c[0][k].z, c[0][k].w};
                        const float b[4] = {c[1][k].x, c[1][k].y, c[1][k].z, c[1][k].w};
#pragma unroll
                        for (int ij = 0; ij < 4; ij++) {
                            const int cell = EPI_C3(ij >> 1, ij & 1, k);
                            T[cell] = a[ij] + b[ij];
                            D[cell] = fmaf(-pi, T[cell], a[ij]);
                        }
                    }
                    derive27(T, xyT, xz.T, yzT);
                    derive27(D, xyD, xz.D, yzD);
                    keep |= quick_bound<27>(p.sc, T, D, thr, (todo >> q) & 1u) ? 0u : 1u << q;
                }
                todo &= keep;
            }
            quick = false;
        }
        // what is left, one triplet per lane and turn
        if (!__ballot(todo != 0)) break;
        float bad = INFINITY;
        unsigned long long packed = 0;
        if (todo) {
            const int q = __ffs(todo) - 1;
            todo &= todo - 1;
            const int Y = y + 2 * q + h;
            float4 c[2][2];
            s3_read(cnt, cls_stride, q, lane, c);
            uint32_t n8[2][8];
#pragma unroll
            for (int cls = 0; cls < 2; cls++)
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    n8[cls][0 + k] = (uint32_t)c[cls][k].x;
                    n8[cls][2 + k] = (uint32_t)c[cls][k].y;
                    n8[cls][4 + k] = (uint32_t)c[cls][k].z;
                    n8[cls][6 + k] = (uint32_t)c[cls][k].w;
                }
            uint32_t cas[27], ctl[27];
            triplet_tables(p, X, Y, Z, ld_global(p.singles, X), ld_global(p.singles, Y), n8[0], n8[1], cas, ctl);
            packed = (unsigned long long)X | ((unsigned long long)Y << 21) | ((unsigned long long)Z << 42);
            if constexpr (scores_sets(MODE)) {
                if (!(thr < INFINITY && p.sc.fb_scale == 0.f && bound_exceeds<27>(p.sc, cas, ctl, thr)))
                    bad = badness_f32_flat<27>(p.sc, cas, ctl, s_lnf);
            } else if constexpr (MODE == MODE_DUMP) {
                uint32_t *o = p.dump + rank3(X, Y, Z) * 54;
                for (int c2 = 0; c2 < 27; c2++) {
                    o[c2] = cas[c2];
                    o[27 + c2] = ctl[c2];
                }
            } else if constexpr (MODE == MODE_CHECKSUM) {
                hsum += table_hash(rank3(X, Y, Z), cas, ctl, 27);
            }
        }
        if constexpr (MODE == MODE_SEARCH) publish_wave(p.co, p.sc.margin, bad, packed);
        if constexpr (MODE == MODE_TOPK) publish_wave_topk(p.co, p.sc.margin, bad, packed);
        if constexpr (scores_sets(MODE)) {
            if (!(thr < INFINITY)) {
                thr = skip_threshold(p.sc, __hip_atomic_load(p.co.best_key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                quick = thr < INFINITY;
            }
            if (quick) s3_yz(p, y + h, Z, yz);
            else yz = S3Yz{};               // not held through the scoring above
        }
    }
}

}  // namespace episdet
