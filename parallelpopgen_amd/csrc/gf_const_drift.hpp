/*
 * gf_const_drift.hpp -- drift of one population whose model (chromosomes,
 * selection, dominance, inbreeding) is the same in every generation of a
 * launch, the usual case of a single-population run and every block of a
 * batched simulation.
 *
 * There a mutation's state is an integer, its count j of Nc chromosomes, and
 * the mean of its next draw depends on j alone.  The kernels carry j, and the
 * draws whose mean is at most 6 (a quarter of the mutations of a large run at
 * equilibrium, most of the new ones) are looked up: PoisTable holds, for each
 * count of 1..8 whose mean is in [0, 6], the 24 partial sums the truncated
 * Poisson inversion (gf_math.hpp: poiscdfinv_from) compares its uniform with,
 * as the random words at which they are passed.  The inversion's result is
 * the number of thresholds below the word: two 16-byte LDS reads and eight
 * comparisons instead of exp(-m) and two to three trips of four terms.
 *
 * Bound: vector-ALU issue.  2.0e6 mutations of N = 1e5, gamma = -10, ten
 * generations a launch: 6.9e7 vector instructions by k_advance_fused, 5.2e7
 * with the table, 4.5e7 with the arithmetic of gf_math.hpp (div_mid,
 * sqrt_pos, round_count) and the scalar gather (frag_slot) besides.  The
 * 5,000-generation run: 64.1 -> 51.2 -> 46.3 ms (44.4 with 16 generations a
 * launch); a run of 8.4e3 mutations
 * 2.14 -> 1.81 -> 1.74 ms; a batch of 64 uneven simulations 428 -> 261 ms.
 */
#ifndef GF_CONST_DRIFT_HPP_
#define GF_CONST_DRIFT_HPP_

#include "gf_drift.hpp"

namespace gf {

constexpr int POIS_ROWS = 8;    /* counts 1..8 */
constexpr int POIS_TERMS = 24;  /* the inversion stops at term 24 at the latest for means up to 6 */
constexpr int POIS_ROW_VECS = 8; /* 6 in use: a power of two, so a row's address is a shift */

/* Row j - 1, with T[k] = the largest random word w with u01(w) <= S_k (the
 * k-th partial sum), 2^32 - 1 past the row's early exit: vector 0 = T[4],
 * T[9], T[14], T[19]; vector 1 + c = T[5c .. 5c + 3]. */
struct alignas(16) PoisTable {
    uint4 v[POIS_ROWS * POIS_ROW_VECS];
    int jn;          /* rows hold the counts 1 <= j < jn */
    int pad[3];
};

/* the model of a launch, uniform over a tile */
struct ConstModel {
    int Nc;
    float N, r;      /* (float)Nc, RN(1/N) */
    float sa, sb, c1, c2;
    int neutral, mid;   /* mid: selected_freq's */
};

/* chromosome numbers the count form covers: from 100 (below, the tails are
 * binomial inversions) to 2^21 (so that x * N recovers j from x = RN(j/N):
 * both roundings together stay below 1/2) */
GF_HD bool const_drift_range(int Nc) { return Nc >= 100 && Nc <= (1 << 21); }

GF_HD float const_selected(float x, const ConstModel &C) {
    GF_STRICT_FP
    if (C.neutral) return x;   /* s == 0: Eq. 13 reduces exactly to x */
    float s = C.sb;
    if (C.sa != 0.0f) s = C.sa * x + C.sb;   /* 0 * x + sb is sb */
    s = s > -1.0f ? s : -1.0f;
    return selected_freq(x, s, C.c1, C.c2, C.mid != 0);
}

/* mean of the next draw of count j */
GF_HD float const_mean(int j, const ConstModel &C) {
    GF_STRICT_FP
    return const_selected(quot_count((float)j, C.N, C.r), C) * C.N;
}

/* T[k] of the row with mean `mean` in [0, 6] */
GF_HD uint32_t pois_threshold(float mean, int k) {
    GF_STRICT_FP
    const int km = mean <= 1.0f ? 1 : (int)__builtin_ceilf(mean);
    if (k >= 8 + 3 * km - (km > 4 ? km - 4 : 0)) return 0xffffffffu;   /* exit_index of a mean up to 14 */
    float e = expneg_tab(expneg_table(), mean), cdf = e;
    for (int i = 1; i <= k; i++) {
        e = e * (mean * kRecip[i - 1]);
        cdf = cdf + e;
    }
    uint32_t lo = 0, hi = 0xffffffffu;   /* u01(0) = 2^-33 < exp(-6) <= cdf */
    while (lo < hi) {
        const uint32_t mid = lo + (hi - lo) / 2 + 1;
        if (u01(mid) <= cdf) lo = mid; else hi = mid - 1;
    }
    return lo;
}

/* word of T[k] in its row's vectors */
GF_HD constexpr int pois_word(int k) { return k % 5 == 4 ? k / 5 : 4 * (1 + k / 5) + k % 5; }

/* Entry `id` of the table of one model, id in [0, POIS_BUILD): row id / 32,
 * threshold id % 32, one thread each (a single lane per row took 37 us, as
 * long as the first launch it was built for; 4 us). */
constexpr int POIS_BUILD = POIS_ROWS * 32;

GF_HD void pois_table_entry(int id, const ConstModel &C, PoisTable *t) {
    const int row = id >> 5, k = id & 31;
    const float mean = const_mean(row + 1, C);
    if (k < POIS_TERMS && mean >= 0.0f && mean <= 6.0f)
        reinterpret_cast<uint32_t *>(t->v + row * POIS_ROW_VECS)[pois_word(k)] = pois_threshold(mean, k);
    if (id == 0) {
        int jn = 1;
        while (jn <= POIS_ROWS && const_mean(jn, C) >= 0.0f && const_mean(jn, C) <= 6.0f) jn++;
        t->jn = const_drift_range(C.Nc) ? jn : 1;
    }
}

/* number of thresholds of row `row` below `bits` */
GF_HD int pois_lookup(const uint4 *tab, int row, uint32_t bits) {
    const uint4 *q = tab + row * POIS_ROW_VECS;
    const uint4 a = q[0];
    const int c = (int)(bits > a.x) + (int)(bits > a.y) + (int)(bits > a.z) + (int)(bits > a.w);
    const uint4 b = q[1 + c];
    return 5 * c + (int)(bits > b.x) + (int)(bits > b.y) + (int)(bits > b.z) + (int)(bits > b.w);
}

/* Advances one slot per lane through generations g0 + 1 .. g0 + K.  j: its
 * count (0 or Nc: absorbed); born: index of its birth generation in the
 * block, -1 for a slot that was there before (ascending over the lanes);
 * klast: the last generation in which it segregates, -1 if none (a slot's
 * birth generation counts).  first_freq: the first generation draws from the
 * frequency x instead of j / Nc (the state was counted in another number of
 * chromosomes). */
__device__ __forceinline__ void const_drift(int &j, int &klast, float x, bool first_freq, int born, int K, int g0,
                                            uint32_t k0, uint32_t k1, uint32_t tid, int ogen, int opop,
                                            const ConstModel &C, int jn, const uint4 *tab, const NcdfSeg *ncdf,
                                            const ExpSeg *etab) {
    GF_STRICT_FP
    u32x4 rc = {0, 0, 0, 0};
    const unsigned inner = (unsigned)(C.Nc - 1);
    klast = born;
    for (int t = __builtin_amdgcn_readfirstlane(born) + 1; t < K; t++) {
        const int g = g0 + 1 + t;
        if ((unsigned)(j - 1) < inner && born < t) {
            if ((g & 3) == 0 || t == born + 1) rc = drift_block(k0, k1, tid, ogen, opop, 0, g);
            const uint32_t bits = lane_of(rc, g & 3);
            const bool from_x = first_freq && t == 0;
            if (!from_x && j < jn) {
                j = pois_lookup(tab, j - 1, bits);
            } else {
                const float xs = const_selected(from_x ? x : quot_count((float)j, C.N, C.r), C);
                const float mean = xs * C.N;
                const float var = (1.0f - xs) * mean;
                const float u = u01(bits);
                const bool lo = mean <= 6.0f;
                if (lo || mean >= C.N - 6.0f) {   /* outside the table: close to fixation, or from a frequency */
                    const float m = lo ? mean : C.N - mean;
                    const int k = m != 0.0f ? poiscdfinv_tail(u, m, etab) : 0;   /* N >= 100 */
                    const int d = lo ? k : f2i_sat(C.N - (float)k);
                    j = min(max(d, 0), C.Nc);
                } else {
                    j = round_count(binom_normal(u, mean, var, ncdf), C.N);
                }
            }
            if ((unsigned)(j - 1) < inner) klast = t;
        }
    }
}

/* count of a slot read from the state, and its frequency if the first
 * generation needs it (const_drift's x): any count strictly between 0 and Nc
 * stands for a segregating frequency then */
__device__ __forceinline__ int const_count(float x, bool first_freq, const ConstModel &C) {
    GF_STRICT_FP
    if (!first_freq) return (int)__builtin_rintf(x * C.N);
    return x <= 0.0f ? 0 : (x >= 1.0f ? C.Nc : 1);
}

/* the table of rows[0]'s model */
static __global__ __launch_bounds__(POIS_BUILD) void k_pois_table(const GenRow<1> *__restrict__ row, int mid,
                                                           PoisTable *__restrict__ out) {
    const auto &R = *as_const(row);
    pois_table_entry(threadIdx.x, ConstModel{R.Nc[0], R.fN[0], R.newfreq[0], R.sa[0], R.sb[0], R.c1[0], R.c2[0], R.neutral_mask & 1, mid}, out);
}

/* k_advance_fused for one population and a launch whose model rows are all
 * alike (same arguments, layout and results) */
static __global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(8))) void k_advance_const(const FusedLaunch F,
                                                                                              const SegLaunch<1> S,
                                                                                              const PoisTable *__restrict__ ptab,
                                                                                              int mid, int first_freq) {
    const int lane = threadIdx.x & 63;
    const int w = wave_index();
    __shared__ unsigned int sh_wcount[WG / 64];
    __shared__ int sh_diff[KMAX + 1];
    __shared__ NcdfSeg sh_ncdf[GF_NCDF_SEGMENTS];
    __shared__ ExpSeg sh_eneg[GF_EXPNEG_SEGMENTS];
    __shared__ uint4 sh_pois[POIS_ROWS * POIS_ROW_VECS];
    load_draw_tables(sh_ncdf, sh_eneg);   /* published by the tile loop's first barrier */
    if (threadIdx.x < POIS_ROWS * POIS_ROW_VECS) sh_pois[threadIdx.x] = ptab->v[threadIdx.x];
    if (threadIdx.x <= KMAX) sh_diff[threadIdx.x] = 0;
    const int jn = as_const(ptab)->jn;
    const int M0 = *F.M_in;
    const int Mend = M0 + F.new_in_block;
    const int need_tiles = (Mend + WG - 1) / WG;
    const int T_in = F.dense ? 0 : *F.T_in;
    if (blockIdx.x == 0 && threadIdx.x == 0 && need_tiles > F.ntiles) *F.error = 2;   /* slots would be dropped */
    const GenRow<1> *rows = S.rows;
    const auto &R = *as_const(rows);
    const ConstModel C{R.Nc[0], R.fN[0], R.newfreq[0], R.sa[0], R.sb[0], R.c1[0], R.c2[0], R.neutral_mask & 1, mid};
    const int K = S.K;
    const int last_tile = need_tiles < F.ntiles ? need_tiles : F.ntiles;
    for (int tile = (int)blockIdx.x;; tile += (int)gridDim.x) {
        __syncthreads();
        if (tile >= last_tile) break;
        const int li = tile * WG + (int)threadIdx.x;
        const bool valid = li < Mend;
        const int first = tile * WG + w * 64;   /* the wave's first index */
        int64_t src = li;
        if (!F.dense && first < M0) src = frag_slot(li, first, tile, F.src0_in, F.pre_in, T_in);
        float x = 0.0f;
        int j = 0, born = -1;
        uint32_t tid = 0;
        gf_mutid id;
        id.origin_generation = 0; id.origin_population = 0; id.origin_threadID = 0; id.reserved = 0;
        if (valid) {
            if (li < M0) {
                x = F.freq_in[src];
                id = F.ids_in[src];
                tid = (uint32_t)(id.origin_threadID < 0 ? -id.origin_threadID : id.origin_threadID);
                j = const_count(x, first_freq, C);
            } else {
                const int rel = li - M0 + S.cum_base;
                int tb, pb;
                find_birth<1>(rows, K, rel, tb, pb);
                born = tb;
                tid = (uint32_t)(rel - rows[tb].newcum[0] + 1);
                id.origin_generation = S.g0 + 1 + tb;
                id.origin_threadID = (int32_t)tid;
                j = 1;
            }
        }
        int klast;
        const_drift(j, klast, x, first_freq, born, K, S.g0, S.k0, S.k1, tid, id.origin_generation, id.origin_population,
                    C, jn, sh_pois, sh_ncdf, sh_eneg);
        if (id.origin_threadID < 0) klast = K - 1;   /* preserved: kept in every generation */
        /* per-generation live counts as a difference array: +1 at the first
         * generation a slot is kept, -1 after its last one */
        const uint64_t old = __ballot(klast >= 0 && born < 0);
        if (lane == 0 && old) atomicAdd(&sh_diff[0], (int)__popcll(old));
        if (born >= 0) atomicAdd(&sh_diff[born], 1);
        if (klast >= 0 && klast + 1 < K) atomicAdd(&sh_diff[klast + 1], -1);
        const bool keep = F.compact ? klast == K - 1 : valid;
        /* tile-local stable packing */
        const uint64_t kb = __ballot(keep);
        if (lane == 0) sh_wcount[w] = (unsigned int)__popcll(kb);
        __syncthreads();
        unsigned int pos = 0;
        for (int k = 0; k < w; k++) pos += sh_wcount[k];
        pos += __builtin_amdgcn_mbcnt_hi((uint32_t)(kb >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)kb, 0u));
        if (keep) {
            const int64_t o = (int64_t)tile * WG + pos;
            __builtin_nontemporal_store(quot_count((float)j, C.N, C.r), &F.freq_out[o]);
            if (F.preserve) {
                const int z = id.origin_threadID;
                id.origin_threadID = -(z < 0 ? -z : z);
            }
            typedef int i4v __attribute__((ext_vector_type(4)));
            const i4v v = {id.origin_generation, id.origin_population, id.origin_threadID, id.reserved};
            __builtin_nontemporal_store(v, reinterpret_cast<i4v *>(&F.ids_out[o]));
        }
        if (threadIdx.x == 0) {
            unsigned int c = 0;
            for (int k = 0; k < WG / 64; k++) c += sh_wcount[k];
            F.cnt_out[tile] = c;
        }
    }
    __syncthreads();
    if (w == 0) {   /* prefix of the difference array: lane t holds generation t */
        int run = lane < K ? sh_diff[lane] : 0;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int y = __shfl_up(run, off);
            if (lane >= off) run += y;
        }
        if (lane < K && run) atomicAdd(&S.live[(size_t)(S.t0 + lane) * 64 + (blockIdx.x & 63)], (unsigned long long)run);
    }
}

} /* namespace gf */

#endif /* GF_CONST_DRIFT_HPP_ */
