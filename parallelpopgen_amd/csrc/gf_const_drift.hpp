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
 * A slot's generations go four at a time, one Philox block (drift_four): the
 * word of each is fixed and nothing but the count and the end is checked in
 * between.  The mutations born in the launch go in spans (drift_span).
 *
 * Bound: vector-ALU issue.  2.0e6 mutations of N = 1e5, gamma = -10, ten
 * generations a launch: 6.9e7 vector instructions by k_advance_fused, 5.2e7
 * with the table, 4.5e7 with the arithmetic of gf_math.hpp (div_mid,
 * sqrt_pos, round_count) and the scalar gather (frag_slot) besides.  The
 * 5,000-generation run: 64.1 -> 51.2 -> 46.3 ms, 42.5 with 16 generations a
 * launch and shorter Philox blocks, 38.6 with spans, 33.1 with 40
 * generations a launch; a run of
 * 8.4e3 mutations 1.30 -> 1.21 ms by
 * drift_four; a batch of 64 uneven simulations 228 -> 214 by drift_four, 205
 * with spans; training draws (8,192 growing simulations) 29.8 -> 28.9 -> 24.3.
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

/* whether a fixed mutation stays fixed, as the count form takes for granted
 * (drift_four leaves a count of Nc alone): not where Eq. 13 is no number at a
 * frequency of 1, whose draw is 0 (s(1) <= -1: 0/0).  A lost one stays lost in
 * every model: 0, or no number, there.  (A batch drops both at every block.) */
GF_HD bool const_keeps_fixed(const ConstModel &C) { return const_selected(1.0f, C) == 1.0f; }

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

/* One Philox block, four generations, of one slot per lane: generation
 * indices base .. base + 3 (base: philox_base of any of them; lanes need not
 * agree on it), those before `start` (FIRST) and from K on left out.  j: the
 * slot's count (0 or Nc: absorbed, nothing happens); lived: grows by one per
 * generation the slot still segregates in.  first_freq (FIRST): generation
 * index 0 draws from the frequency x instead of j / Nc (the state was counted
 * in another number of chromosomes). */
template <bool FIRST>
__device__ __forceinline__ void drift_four(int &j, int &lived, int base, int start, int K, bool first_freq, float x, int g0,
                                           uint32_t k0, uint32_t k1, uint32_t tid, int ogen, int opop, const ConstModel &C,
                                           int jn, const uint4 *tab, const NcdfSeg *ncdf, const ExpSeg *etab) {
    GF_STRICT_FP
    const unsigned inner = (unsigned)(C.Nc - 1);
    const int left = K - base;
    if (!((unsigned)(j - 1) < inner && left > 0)) return;
    const u32x4 rc = drift_block(k0, k1, tid, ogen, opop, 0, g0 + 1 + base);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if ((unsigned)(j - 1) < inner && i < left && (!FIRST || base + i >= start)) {
            const uint32_t bits = lane_of(rc, i);
            const bool from_x = FIRST && first_freq && base + i == 0;
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
            lived += (unsigned)(j - 1) < inner ? 1 : 0;
        }
    }
}

/* Birth generation of the block's new mutation rel (counted from the run's
 * start, as newcum) for every lane of a wave, whose lanes hold consecutive
 * ones from first_rel up, and the cumulative count before it.  t_at: a
 * generation not after the first lane's, moved up to it (scalar loads; a
 * binary search per lane took six dependent vector loads). */
__device__ __forceinline__ int wave_birth(const GenRow<1> *rows, int K, int rel, int first_rel, int &t_at, int &before) {
    const auto *c = as_const(rows);
    while (t_at + 1 < K && c[t_at + 1].newcum[0] <= first_rel) t_at++;
    int t = t_at;
    before = c[t].newcum[0];
    for (int k = t_at + 1; k < K; k++) {
        const int v = c[k].newcum[0];
        if (v > first_rel + 63) break;
        const bool passed = v <= rel;
        t = passed ? k : t;
        before = passed ? v : before;
    }
    return t;
}

/* ---------------- the mutations born in a block ----------------
 * More than half of a block's new mutations are lost within two
 * generations, three quarters within four; in a slot per lane they left 40 %
 * of all lanes of a run of 2.0e6 mutations idle, and 65 % of a batch of
 * growing simulations.  A wave therefore takes a span of several hundred of
 * them through three stages with a queue in LDS between two, each stage with
 * full waves: the rest of the Philox block they are born in; the next
 * Philox block; the rest of the launch's generations.  The queues keep the
 * mutations' order, which the state's layout and the results rest on.  No
 * barrier: a span is one wave's.  A lane's generation is its own (the model
 * is the same in all), so a stage mixes mutations of different ages. */
constexpr int SPAN_QUEUE = 128;  /* a stage starts with 64 waiting, or with the last */

/* queue entry: the count (<= 2^21) and the birth generation (< 64) in one
 * word, the thread ID in the other */
struct SpanQueues { uint2 q[2][SPAN_QUEUE]; };

/* New mutations n0 .. n1 - 1 (counted in the block; n0's slot starts a tile)
 * of a block of K generations after g0.  count(born, last) is called for
 * every lane whose mutation is gone, last = its last generation index, and
 * for the survivors with last = K - 1; write(tid, ogen, count, pos) for each
 * survivor, pos counting up from 0.  Returns the number of survivors. */
template <typename Count, typename Write>
__device__ __forceinline__ int drift_span(int n0, int n1, const GenRow<1> *rows, int cum_base, int K, int g0, uint32_t k0,
                                          uint32_t k1, const ConstModel &C, int jn, const uint4 *tab, const NcdfSeg *ncdf,
                                          const ExpSeg *etab, SpanQueues &sq, const Count &count, const Write &write) {
    const int lane = threadIdx.x & 63;
    const unsigned inner = (unsigned)(C.Nc - 1);
    int waiting[2] = {0, 0}, head[2] = {0, 0};
    int at = n0, out = 0;
    int t_at = first_birth(rows, K, n0 + cum_base);
    auto push = [&](int q, bool stays, int j, int born, int tid) {
        const uint64_t b = __ballot(stays);
        if (stays)
            sq.q[q][(head[q] + waiting[q] + rank_in(b)) & (SPAN_QUEUE - 1)] =
                uint2{(uint32_t)j | ((uint32_t)born << 22), (uint32_t)tid};
        waiting[q] += (int)__popcll(b);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   /* the queue is this wave's alone */
    };
    for (;;) {
        const bool more = at < n1;
        int j = 0, born = 0, tid = 0, lived = 0;
        if (waiting[1] >= 64 || (!more && waiting[0] == 0)) {   /* the remaining generations */
            const int m = min(waiting[1], 64);
            if (m == 0) break;
            const bool valid = lane < m;
            if (valid) {
                const uint2 e = sq.q[1][(head[1] + lane) & (SPAN_QUEUE - 1)];
                j = (int)(e.x & 0x3fffffu);
                born = (int)(e.x >> 22);
                tid = (int)e.y;
            }
            head[1] += m;
            waiting[1] -= m;
            const int from = min(philox_base(born + 1, g0) + 8, K);
            int base = philox_base(born + 1, g0) + 8;
            for (int b = __builtin_amdgcn_readfirstlane(base); b < K; b += 4, base += 4)
                drift_four<false>(j, lived, base, 0, K, false, 0.0f, g0, k0, k1, (uint32_t)tid, g0 + 1 + born, 0, C, jn, tab,
                                  ncdf, etab);
            if (valid) count(born, from - 1 + lived);
            const bool keep = valid && (unsigned)(j - 1) < inner;
            const uint64_t b = __ballot(keep);
            if (keep) write(tid, g0 + 1 + born, j, out + rank_in(b));
            out += (int)__popcll(b);
        } else if (waiting[0] >= 64 || !more) {   /* one Philox block */
            const int m = min(waiting[0], 64);
            const bool valid = lane < m;
            if (valid) {
                const uint2 e = sq.q[0][(head[0] + lane) & (SPAN_QUEUE - 1)];
                j = (int)(e.x & 0x3fffffu);
                born = (int)(e.x >> 22);
                tid = (int)e.y;
            }
            head[0] += m;
            waiting[0] -= m;
            const int base = philox_base(born + 1, g0) + 4;
            drift_four<false>(j, lived, base, 0, K, false, 0.0f, g0, k0, k1, (uint32_t)tid, g0 + 1 + born, 0, C, jn, tab, ncdf,
                              etab);
            const bool stays = valid && (unsigned)(j - 1) < inner;
            if (valid && !stays) count(born, base - 1 + lived);
            push(1, stays, j, born, tid);
        } else {   /* birth, and the rest of its Philox block */
            const bool valid = at + lane < n1;
            const int rel = at + lane + cum_base;
            int before;
            born = wave_birth(rows, K, rel, at + cum_base, t_at, before);
            tid = rel - before + 1;
            j = valid ? 1 : 0;
            at += 64;
            drift_four<true>(j, lived, philox_base(born + 1, g0), born + 1, K, false, 0.0f, g0, k0, k1, (uint32_t)tid,
                             g0 + 1 + born, 0, C, jn, tab, ncdf, etab);
            const bool stays = valid && (unsigned)(j - 1) < inner;
            if (valid && !stays) count(born, born + lived);
            push(0, stays, j, born, tid);
        }
    }
    return out;
}

/* survivors in tile `k` of a span of which n are left, packed from its first slot */
__device__ __forceinline__ unsigned int span_count(int n, int k) { return (unsigned int)min(max(n - k * WG, 0), WG); }

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
 * alike (same arguments, layout and results).  spans: tiles of new mutations a
 * wave takes as one span, 0: new mutations have a slot per lane like the old
 * ones. */
static __global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(8))) void k_advance_const(const FusedLaunch F,
                                                                                              const SegLaunch<1> S,
                                                                                              const PoisTable *__restrict__ ptab,
                                                                                              int mid, int first_freq, int spans) {
    const int lane = threadIdx.x & 63;
    const int w = wave_index();
    __shared__ unsigned int sh_wcount[WG / 64];
    __shared__ int sh_diff[KMAX + 1];
    __shared__ NcdfSeg sh_ncdf[GF_NCDF_SEGMENTS];
    __shared__ ExpSeg sh_eneg[GF_EXPNEG_SEGMENTS];
    __shared__ uint4 sh_pois[POIS_ROWS * POIS_ROW_VECS];
    __shared__ SpanQueues sh_span[WG / 64];
    load_draw_tables(sh_ncdf, sh_eneg);   /* published by the tile loop's first barrier */
    if (threadIdx.x < POIS_ROWS * POIS_ROW_VECS) sh_pois[threadIdx.x] = ptab->v[threadIdx.x];
    if (threadIdx.x <= KMAX) sh_diff[threadIdx.x] = 0;
    const int jn = as_const(ptab)->jn;
    const int M0 = __builtin_amdgcn_readfirstlane(*F.M_in);
    const int Mend = M0 + F.new_in_block;
    const int need_tiles = (Mend + WG - 1) / WG;
    const int T_in = F.dense ? 0 : *F.T_in;
    if (blockIdx.x == 0 && threadIdx.x == 0 && need_tiles > F.ntiles) *F.error = 2;   /* slots would be dropped */
    const GenRow<1> *rows = S.rows;
    const auto &R = *as_const(rows);
    const ConstModel C{R.Nc[0], R.fN[0], R.newfreq[0], R.sa[0], R.sb[0], R.c1[0], R.c2[0], R.neutral_mask & 1, mid};
    const int K = S.K;
    const int last_tile = need_tiles < F.ntiles ? need_tiles : F.ntiles;
    /* the tiles that hold only new slots go in spans, ahead of the others */
    const int old_tiles = spans ? min((M0 + WG - 1) / WG, last_tile) : last_tile;
    const int per_item = spans * (WG / 64);
    const int groups = spans ? (last_tile - old_tiles + per_item - 1) / per_item : 0;
    auto store = [&](int64_t o, int j, int tid, int ogen, int opop, int rest) {
        __builtin_nontemporal_store(quot_count((float)j, C.N, C.r), &F.freq_out[o]);
        if (F.preserve) tid = -(tid < 0 ? -tid : tid);
        typedef int i4v __attribute__((ext_vector_type(4)));
        const i4v v = {ogen, opop, tid, rest};
        __builtin_nontemporal_store(v, reinterpret_cast<i4v *>(&F.ids_out[o]));
    };
    /* per-generation live counts as a difference array: +1 at the start for
     * an old slot, -1 after a slot's last generation; the births, whose
     * numbers the rows hold, are added at the end */
    auto count = [&](int, int last) {
        if (last + 1 < K) atomicAdd(&sh_diff[last + 1], -1);
    };
    for (int item = (int)blockIdx.x;; item += (int)gridDim.x) {
        sync_lds();
        if (item >= groups + old_tiles) break;
        if (item < groups) {
            const int first = old_tiles + item * per_item + w * spans;   /* tile */
            const int tiles = min(last_tile - first, spans);
            if (tiles > 0) {
                const int64_t slot = (int64_t)first * WG;
                const int n = drift_span(first * WG - M0, min((first + tiles) * WG, Mend) - M0, rows, S.cum_base, K, S.g0, S.k0, S.k1,
                                         C, jn, sh_pois, sh_ncdf, sh_eneg, sh_span[w], count,
                                         [&](int tid, int ogen, int j, int pos) { store(slot + pos, j, tid, ogen, 0, 0); });
                if (lane < tiles) F.cnt_out[first + lane] = span_count(n, lane);
            }
            continue;
        }
        const int tile = item - groups;
        const int li = tile * WG + (int)threadIdx.x;
        const bool valid = li < Mend;
        const int first = tile * WG + w * 64;   /* the wave's first index */
        int64_t src = li;
        if (!F.dense && first < M0) src = frag_slot(li, first, tile, F.src0_in, F.pre_in, T_in);
        float x = 0.0f;
        int j = 0, born = -1;
        gf_mutid id;
        id.origin_generation = 0; id.origin_population = 0; id.origin_threadID = 0; id.reserved = 0;
        if (li < M0) {
            x = F.freq_in[src];
            id = F.ids_in[src];
            j = const_count(x, first_freq, C);
        }
        if (first + 63 >= M0 && first < Mend) {
            const int first_rel = max(first - M0, 0) + S.cum_base;
            int t_at = first_birth(rows, K, first_rel), before;
            const int tb = wave_birth(rows, K, li - M0 + S.cum_base, first_rel, t_at, before);
            if (li >= M0 && valid) {
                born = tb;
                id.origin_generation = S.g0 + 1 + tb;
                id.origin_threadID = li - M0 + S.cum_base - before + 1;
                j = 1;
            }
        }
        const uint32_t tid = (uint32_t)(id.origin_threadID < 0 ? -id.origin_threadID : id.origin_threadID);
        int lived = 0, base = philox_base(born + 1, S.g0);
        int b = __builtin_amdgcn_readfirstlane(base);   /* the earliest: births ascend over the lanes */
        drift_four<true>(j, lived, base, born + 1, K, first_freq, x, S.g0, S.k0, S.k1, tid, id.origin_generation,
                         id.origin_population, C, jn, sh_pois, sh_ncdf, sh_eneg);
        for (b += 4, base += 4; b < K; b += 4, base += 4)
            drift_four<false>(j, lived, base, 0, K, false, 0.0f, S.g0, S.k0, S.k1, tid, id.origin_generation,
                              id.origin_population, C, jn, sh_pois, sh_ncdf, sh_eneg);
        /* the last generation the slot is kept in; preserved: every one */
        const int last = !valid ? -1 : (id.origin_threadID < 0 ? K - 1 : born + lived);
        const uint64_t old = __ballot(last >= 0 && born < 0);
        if (lane == 0 && old) atomicAdd(&sh_diff[0], (int)__popcll(old));
        if (last >= 0 && last + 1 < K) atomicAdd(&sh_diff[last + 1], -1);
        const bool keep = F.compact ? last == K - 1 : valid;
        /* tile-local stable packing */
        const uint64_t kb = __ballot(keep);
        if (lane == 0) sh_wcount[w] = (unsigned int)__popcll(kb);
        sync_lds();
        unsigned int pos = 0;
        for (int k = 0; k < w; k++) pos += sh_wcount[k];
        if (keep) store((int64_t)tile * WG + pos + rank_in(kb), j, id.origin_threadID, id.origin_generation, id.origin_population, id.reserved);
        if (threadIdx.x == 0) {
            unsigned int c = 0;
            for (int k = 0; k < WG / 64; k++) c += sh_wcount[k];
            F.cnt_out[tile] = c;
        }
    }
    sync_lds();
    if (w == 0) {   /* prefix of the difference array: lane t holds generation t */
        int run = lane < K ? sh_diff[lane] : 0;
        const int births = blockIdx.x == 0 && lane < K ? rows[lane].newcum[1] - S.cum_base : 0;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int y = __shfl_up(run, off);
            if (lane >= off) run += y;
        }
        run += births;
        if (lane < K && run) atomicAdd(&S.live[(size_t)(S.t0 + lane) * 64 + (blockIdx.x & 63)], (unsigned long long)run);
    }
}

} /* namespace gf */

#endif /* GF_CONST_DRIFT_HPP_ */
