// kernels_seed.hpp -- a starting score bound for 3-way searches.
//
// The score bounds skip FP32 scores only once the global bound is low.
// Strongly associated triplets often hold an associated pair, so before the
// search the best few pairs are taken from the pair table and every triplet
// that contains one of them is scored:
//   k_seed_pairs     each workgroup's best pair, ranked by its chi-square sum (and,
//                    for K2, the cells' Stirling terms);
//   k_seed_pick      the best of those;
//   k_seed_triplets  FP32 badness of the triplets that contain one: the lowest
//                    joins the global bound, as a wave of the search would
//                    publish it (or all are kept, for top-k);
//   k_seed_kth       top-k: the k-th lowest, over distinct triplets.
// All follow the pair table on the search's stream, and the host waits once
// per search.  With the bound from a 2-way top-4 search of its own, whose
// result the host turned into triplets, and with argument blocks copied, not
// written by the kernel that resets the control words, the host waited six
// times: a search at 400 SNPs x 10000 samples (upload included) took 1.25 ms
// against 1.03, one at 1000 x 4000 3.67 against 3.44, and the top 100
// triplets at 1024 x 8192, which were not seeded, 6.8 against 5.0.
#pragma once
#include "kernels_score3.hpp"

namespace episdet {

constexpr int SEED_BLOCKS = 1024, SEED_MAX_PAIRS = 32;

struct SeedArgs {
    RescoreArgs r;                      // planes, counts and tables of the data
    ScoreCtx sc;                        // 3-way scoring
    unsigned long long *blk;            // [blocks][2]: rank key, packed pair (a | b << 32)
    unsigned long long *pick;           // [npairs] packed pairs, ~0: none
    int blocks, npairs;
    unsigned *best_key;                 // global bound
    float *s32;                         // top-k: badness of triplet (pair, c) at pair * n + c, else null
};

// The 3-way jobs of a batch are seeded together, job by blockIdx.y, in grids
// sized for the largest.  Without a bound, every workgroup that reaches a
// job's first units scores all their triplets.  8 2-way and 8 3-way jobs
// of 233 to 700 SNPs and 6667 to 20000 samples took 11.8 ms; with the seeds
// (75 us for the 8 jobs), candidates staged by the re-scoring kernel and
// group lists kept on the device 8.9 ms.
struct SeedMany {
    const SeedArgs *jobs;
};
__device__ __forceinline__ const SeedArgs &seed_args(const SeedArgs &a) { return a; }
__device__ __forceinline__ SeedArgs seed_args(const SeedMany &m) { return ld_const(m.jobs, (size_t)blockIdx.y); }

template <class Args>
__global__ __launch_bounds__(256) void k_seed_pairs(Args args)
{
    const SeedArgs &a = seed_args(args);
    __shared__ unsigned long long s_k[4], s_p[4];
    const int n = a.r.n, tid = threadIdx.x;
    const float pi = a.sc.lb_pi;
    const float kpi = 0.5f / (pi * (1.f - pi));
    unsigned long long key = ~0ull, pk = ~0ull;
    for (int A = blockIdx.x; A < n - 1; A += gridDim.x) {
        const Singles sa = ld_global(a.r.singles, A);
        for (int B = A + 1 + tid; B < n; B += 256) {
            float T[9], D[9];
            pair_td9(a.r.pairs, n, sa, ld_global(a.r.singles, B), A, B, (uint32_t)a.r.N0, (uint32_t)a.r.N1, pi, T, D);
            float s = 0.f, l = 0.f;
#pragma unroll
            for (int c = 0; c < 9; c++) {
                const float t = fmaxf(T[c], 1.f);
                s = fmaf(D[c], D[c] * __builtin_amdgcn_rcpf(t), s);
                l += __builtin_amdgcn_logf(t);
            }
            const float rank = a.sc.score == SCORE_K2 ? fmaf(0.5f * LN2_F, l, -kpi * s) : -s;
            const unsigned long long k = f2key(rank), q = (unsigned long long)A | ((unsigned long long)B << 32);
            if (lex_less(k, q, key, pk)) {
                key = k;
                pk = q;
            }
        }
    }
    wave_lexmin(key, pk);
    if ((tid & 63) == 0) {
        s_k[tid >> 6] = key;
        s_p[tid >> 6] = pk;
    }
    __syncthreads();
    if (tid == 0 && (int)blockIdx.x < a.blocks) {
        for (int w = 1; w < 4; w++)
            if (lex_less(s_k[w], s_p[w], key, pk)) {
                key = s_k[w];
                pk = s_p[w];
            }
        a.blk[2 * blockIdx.x] = key;
        a.blk[2 * blockIdx.x + 1] = pk;
    }
}

template <class Args>
__global__ __launch_bounds__(SEED_BLOCKS) void k_seed_pick(Args args)
{
    const SeedArgs &a = seed_args(args);
    __shared__ unsigned long long s_k[16], s_p[16];
    const int t = threadIdx.x, w = t >> 6;
    unsigned long long key = ~0ull, pk = ~0ull;
    if (t < a.blocks) {
        key = a.blk[2 * t];
        pk = a.blk[2 * t + 1];
    }
    for (int r = 0; r < a.npairs; r++) {
        unsigned long long k = key, q = pk;
        wave_lexmin(k, q);
        if ((t & 63) == 0) {
            s_k[w] = k;
            s_p[w] = q;
        }
        __syncthreads();
        k = s_k[0];
        q = s_p[0];
        for (int i = 1; i < SEED_BLOCKS / 64; i++)
            if (lex_less(s_k[i], s_p[i], k, q)) {
                k = s_k[i];
                q = s_p[i];
            }
        __syncthreads();
        if (t == 0) a.pick[r] = q;
        if (pk == q) key = pk = ~0ull;          // taken
    }
}

// One wave per (pair, c); c runs over all SNPs, so pair * n + c below npairs * n.
template <class Args>
__global__ __launch_bounds__(256) void k_seed_triplets(Args args)
{
    const SeedArgs &a = seed_args(args);
    __shared__ float s_lnf[LNF_SMALL];
    __shared__ float s_min[4];
    load_lnf(s_lnf);
    __syncthreads();
    const int lane = threadIdx.x & 63, w = uniform((int)(threadIdx.x >> 6)), n = a.r.n;
    const int t = blockIdx.x * 4 + w;
    float bad = INFINITY;
    const bool in = t < a.npairs * n;
    const int pair = in ? t / n : 0, c = in ? t % n : 0;
    const unsigned long long pk = uniform(a.pick[pair]);
    const int A = (int)(pk & 0xFFFFFFFFu), B = (int)(pk >> 32);
    bool use = in && pk != ~0ull && c != A && c != B;
    // a triplet of two of the pairs counts once, for the first of them
    for (int q = 0; q < pair && use; q++) {
        const unsigned long long o = uniform(a.pick[q]);
        const int oa = (int)(o & 0xFFFFFFFFu), ob = (int)(o >> 32);
        if ((oa == A || oa == B || oa == c) && (ob == A || ob == B || ob == c)) use = false;
    }
    if (use) {
        int s[3];
        s[0] = c < A ? c : A;
        s[1] = c < A ? A : (c < B ? c : B);
        s[2] = c < B ? B : c;
        uint32_t cas[27], ctl[27];
        wave_cells<3, 27>(a.r, s, lane, cas, ctl);
        bad = badness_f32_flat<27>(a.sc, cas, ctl, s_lnf);
    }
    if (a.s32) {
        if (in && lane == 0) a.s32[t] = bad;
        return;
    }
    if (lane == 0) s_min[w] = bad;
    __syncthreads();
    if (threadIdx.x == 0) {
        const float m = fminf(fminf(s_min[0], s_min[1]), fminf(s_min[2], s_min[3]));
        if (m < INFINITY &&
            f2key(m) < __hip_atomic_load(a.best_key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMin(a.best_key, f2key(m));
    }
}

// The k-th lowest of the m scores in s32 (+inf: none) joins the global bound:
// MSB-first radix select, one workgroup.
__global__ __launch_bounds__(1024) void k_seed_kth(const float *s32, int m, unsigned k, unsigned *best_key)
{
    __shared__ unsigned s_cnt[2][16];
    const int t = threadIdx.x, w = t >> 6;
    unsigned prefix = 0;
    for (int b = 31; b >= 0; b--) {
        const unsigned hi = b == 31 ? 0u : (~0u << (b + 1));
        unsigned z = 0;
        for (int i = t; i < m; i += 1024) {
            const unsigned key = f2key(s32[i]);
            z += ((key ^ prefix) & hi) == 0 && ((key >> b) & 1u) == 0;
        }
        z = wave_sum_u(z);
        if ((t & 63) == 0) s_cnt[b & 1][w] = z;
        __syncthreads();
        unsigned cnt = 0;
        for (int i = 0; i < 16; i++) cnt += s_cnt[b & 1][i];
        if (k > cnt) {
            k -= cnt;
            prefix |= 1u << b;
        }
    }
    if (t == 0 && prefix < 0xFF800000u) atomicMin(best_key, prefix);
}

}  // namespace episdet
