/*
 * gf_packed_drift.hpp -- drift of two to four populations where many slots
 * hold nothing: k_advance_fused with the slots that hold something gathered
 * from several tiles.
 *
 * A slot that is zero in every population never changes again.  The state is
 * full of them where mutations are preserved (those preserved every 100
 * generations and lost since: 89 % of the slots of the three-population run
 * in the end, so that seven lanes of a wave's 64 did something), and a
 * launch's new mutations turn into them (three quarters within four
 * generations).  A workgroup takes a chunk of up to 8 tiles, lists the slots
 * that hold something in LDS, a tile after the other (a tile of new mutations
 * after the first four to seven generations of its own), and advances them
 * 256 at a time; every slot is then written in its old order, packed in its
 * tile.
 *
 * Bound: vector-ALU issue, and the latency of a chunk's lists, which follow
 * one another.  Three populations over 2,000 generations, 1.4e7 slots in the
 * end: 90.9 -> 64.4 ms with 20 generations a launch, 56.7 with 35 (83.6
 * without packing).  Packing within each tile alone gave 80: one busy wave in
 * a workgroup of four.  Six waves per SIMD (80 VGPRs, of which two
 * populations with simple rows spill none, three 7, four 19), not eight with
 * more spills: 66.8 -> 64.3.
 */
#ifndef GF_PACKED_DRIFT_HPP_
#define GF_PACKED_DRIFT_HPP_

#include "gf_const_drift.hpp"

namespace gf {

constexpr int PACK_TILES = 8;   /* tiles of a chunk at most */

/* slots on their way to other lanes: state, mutation ID, and where they
 * belong (place in the chunk; birth generation + 1 from bit 16) */
template <int P>
struct PackList {
    float x[P][WG];
    int id[4][WG];
    int place[WG];
    unsigned int n[2][WG / 64];
    /* by place: slots to write, from a lane / with zeros */
    unsigned int keep[PACK_TILES * (WG / 32)], gone[PACK_TILES * (WG / 32)];
};

/* tiles_per_chunk: 1 .. PACK_TILES */
template <int P, bool SIMPLE>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(6))) void k_advance_packed(const FusedLaunch F, const SegLaunch<P> S,
                                                                                           int tiles_per_chunk) {
    const int lane = threadIdx.x & 63;
    const int w = wave_index();
    __shared__ int sh_chunk;
    __shared__ unsigned long long sh_live[64];
    __shared__ NcdfSeg sh_ncdf[GF_NCDF_SEGMENTS];
    __shared__ ExpSeg sh_eneg[GF_EXPNEG_SEGMENTS];
    __shared__ PackList<P> L;
    load_draw_tables(sh_ncdf, sh_eneg);   /* published by the chunk loop's first barrier */
    if (threadIdx.x < 64) sh_live[threadIdx.x] = 0;
    const int M0 = __builtin_amdgcn_readfirstlane(*F.M_in);
    const int Mend = M0 + F.new_in_block;
    const int need_tiles = (Mend + WG - 1) / WG;
    const int T_in = F.dense ? 0 : *F.T_in;
    if (blockIdx.x == 0 && threadIdx.x == 0 && need_tiles > F.ntiles) *F.error = 2;   /* slots would be dropped */
    uint64_t cnt = 0;   /* lane t: live slots of generation t */
    const GenRow<P> *rows = S.rows;
    const auto *crows = as_const(rows);
    const int K = S.K;
    const int last_tile = need_tiles < F.ntiles ? need_tiles : F.ntiles;

    /* generations b0 .. b1 - 1 (b0 a Philox block's first), a slot per lane */
    auto advance = [&](float *x, bool here, int born, const gf_mutid &id, int b0, int b1, bool &keep) {
        const bool preserved = id.origin_threadID < 0;
        const uint32_t tid = (uint32_t)(preserved ? -id.origin_threadID : id.origin_threadID);
        for (int base = b0; base < b1; base += 4) {
            u32x4 rc[P];
            if (here && born < base + 3) {
#pragma unroll
                for (int p = 0; p < P; p++)
                    rc[p] = drift_block(S.k0, S.k1, tid, id.origin_generation, id.origin_population, p, S.g0 + 1 + base);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int t = base + i;
                if (t < 0 || t >= K) continue;
                const auto &R = crows[t];
                if (here && born < t) {
                    uint32_t bits[P];
#pragma unroll
                    for (int p = 0; p < P; p++) bits[p] = lane_of(rc[p], i);
                    generation_update<P, SIMPLE>(x, R, S.g0 + 1 + t, bits, LinearSel(), sh_ncdf, sh_eneg);
                }
                keep = here && born <= t && keep_rule<P>(x, R.present_mask, preserved);
                const uint64_t b = __ballot(keep);
                if (lane == t) cnt += (uint64_t)__popcll(b);
            }
        }
    };
    /* output slot of place `at` of a chunk: its rank among its tile's slots written */
    auto position = [&](int chunk_tile, int at) {
        int pos = 0;
#pragma unroll
        for (int k = 0; k < WG / 32; k++) {
            const unsigned int m = L.keep[(at >> 8) * (WG / 32) + k] | L.gone[(at >> 8) * (WG / 32) + k];
            const int in = (at & 255) - k * 32;
            pos += __popc(in >= 32 ? m : (in <= 0 ? 0u : m & ((1u << in) - 1u)));
        }
        return (int64_t)(chunk_tile + (at >> 8)) * WG + pos;
    };
    auto store = [&](int64_t o, const float *x, const gf_mutid &id) {
#pragma unroll
        for (int p = 0; p < P; p++) __builtin_nontemporal_store(x[p], &F.freq_out[p * F.pitch + o]);
        int z = id.origin_threadID;
        if (F.preserve) z = -(z < 0 ? -z : z);
        typedef int i4v __attribute__((ext_vector_type(4)));
        __builtin_nontemporal_store(i4v{id.origin_generation, id.origin_population, z, id.reserved},
                                    reinterpret_cast<i4v *>(&F.ids_out[o]));
    };
    /* state slot of this thread's place in a tile of old slots */
    auto source = [&](int tile) {
        const int first = tile * WG + w * 64;
        int64_t src = tile * WG + (int)threadIdx.x;
        if (!F.dense && first < M0) src = frag_slot((int)src, first, tile, F.src0_in, F.pre_in, T_in);
        return src;
    };

    int parity = 0;
    for (bool own = true;; own = false) {   /* its own chunk, then tickets */
        sync_lds();
        if (threadIdx.x == 0) sh_chunk = (int)(own ? blockIdx.x : gridDim.x + atomicAdd(F.ticket, 1u));
        if (threadIdx.x < PACK_TILES * (WG / 32)) L.keep[threadIdx.x] = L.gone[threadIdx.x] = 0;
        sync_lds();
        const int chunk = __builtin_amdgcn_readfirstlane(sh_chunk) * tiles_per_chunk;   /* its first tile */
        if (chunk >= last_tile) break;
        const int tiles = min(tiles_per_chunk, last_tile - chunk);
        int listed = 0, resume = 0;
        /* advances the listed slots from generation `resume` to the end and
         * writes those to keep */
        auto run_list = [&]() {
            sync_lds();   /* the list is complete */
            /* a wave keeps to its SIMD: which ones a short list leaves idle varies */
            const int r = ((w + chunk / tiles_per_chunk) & (WG / 64 - 1)) * 64 + lane;
            const bool here = r < listed;
            float x[P];
            gf_mutid id;
            id.origin_generation = 0; id.origin_population = 0; id.origin_threadID = 0; id.reserved = 0;
            int place = 0, born = -1;
            bool keep = false;
#pragma unroll
            for (int p = 0; p < P; p++) x[p] = 0.0f;
            if (here) {
#pragma unroll
                for (int p = 0; p < P; p++) x[p] = L.x[p][r];
                id.origin_generation = L.id[0][r];
                id.origin_population = L.id[1][r];
                id.origin_threadID = L.id[2][r];
                id.reserved = L.id[3][r];
                place = L.place[r] & 0xffff;
                born = (L.place[r] >> 16) - 1;
            }
            if (resume >= K) keep = here && keep_rule<P>(x, crows[K - 1].present_mask, id.origin_threadID < 0);
            else if (__ballot(here)) advance(x, here, born, id, philox_base(resume, S.g0), K, keep);
            if (!F.compact) keep = here;
            if (keep) atomicOr(&L.keep[place >> 5], 1u << (place & 31));
            sync_lds();
            if (keep) store(position(chunk, place), x, id);
        };
        for (int k = 0; k <= tiles; k++) {   /* the last time round only the list runs */
            const int tile = chunk + k;
            const int li = tile * WG + (int)threadIdx.x;
            const bool here = k < tiles && li < Mend;
            float x[P];
            gf_mutid id;
            id.origin_generation = 0; id.origin_population = 0; id.origin_threadID = 0; id.reserved = 0;
            int born = -1, from = 0, total = 0, rank = 0;
            bool some = false;
#pragma unroll
            for (int p = 0; p < P; p++) x[p] = 0.0f;
            if (k < tiles) {
                const int64_t src = source(tile);
                if (here) {
                    if (li < M0) {
#pragma unroll
                        for (int p = 0; p < P; p++) x[p] = F.freq_in[p * F.pitch + src];
                        id = F.ids_in[src];
                    } else {
                        const int rel = li - M0 + S.cum_base;
                        int pb;
                        find_birth<P>(rows, K, rel, born, pb);
                        id.origin_generation = S.g0 + 1 + born;
                        id.origin_population = pb;
                        id.origin_threadID = rel - rows[born].newcum[pb] + 1;
#pragma unroll
                        for (int p = 0; p < P; p++) x[p] = (p == pb) ? rows[born].newfreq[p] : 0.0f;
                    }
                }
                if (F.compact && tile * WG >= M0) {
                    /* new mutations only: four to seven generations by themselves */
                    bool keep = false;
                    const int fb = first_birth<P>(rows, K, tile * WG - M0 + S.cum_base);
                    from = min(philox_base(fb + 7, S.g0), K);
                    advance(x, here, born, id, philox_base(fb, S.g0), from, keep);
                }
                some = born >= from;
#pragma unroll
                for (int p = 0; p < P; p++) some = some || x[p] != 0.0f;
                some = some && here;
                const uint64_t b = __ballot(some);
                unsigned int *n = L.n[parity];
                parity ^= 1;
                if (lane == 0) n[w] = (unsigned int)__popcll(b);
                sync_lds();
                const int n0 = (int)n[0], n1 = (int)n[1], n2 = (int)n[2], n3 = (int)n[3];
                total = __builtin_amdgcn_readfirstlane(n0 + n1 + n2 + n3);
                rank = (w > 0 ? n0 : 0) + (w > 1 ? n1 : 0) + (w > 2 ? n2 : 0) + rank_in(b);
            }
            if (k == tiles || (listed > 0 && (listed + total > WG || from != resume))) {
                run_list();
                listed = 0;
            }
            if (listed == 0) resume = from;
            const int place = k << 8 | (int)threadIdx.x;
            const bool preserved = id.origin_threadID < 0;
            const bool leaves = here && !some;
            if (leaves && (preserved || !F.compact)) atomicOr(&L.gone[place >> 5], 1u << (place & 31));
            const uint64_t left = __ballot(leaves && preserved);   /* live in every generation */
            if (lane < K) cnt += (uint64_t)__popcll(left);
            if (some) {
                const int r = listed + rank;
#pragma unroll
                for (int p = 0; p < P; p++) L.x[p][r] = x[p];
                L.id[0][r] = id.origin_generation;
                L.id[1][r] = id.origin_population;
                L.id[2][r] = id.origin_threadID;
                L.id[3][r] = id.reserved;
                L.place[r] = place | (born + 1) << 16;
            }
            listed += total;
        }
        /* the old slots that hold nothing, and the tiles' counts */
        for (int k = 0; k < tiles; k++) {
            const int place = k << 8 | (int)threadIdx.x;
            const bool zero = L.gone[place >> 5] >> (place & 31) & 1u;
            if (__ballot(zero)) {
                const int64_t src = source(chunk + k);
                if (zero) {
                    float x[P];
#pragma unroll
                    for (int p = 0; p < P; p++) x[p] = 0.0f;
                    store(position(chunk, place), x, F.ids_in[src]);
                }
            }
        }
        if ((int)threadIdx.x < tiles) {
            unsigned int c = 0;
            for (int k = 0; k < WG / 32; k++) c += (unsigned int)__popc(L.keep[threadIdx.x * (WG / 32) + k] | L.gone[threadIdx.x * (WG / 32) + k]);
            F.cnt_out[chunk + threadIdx.x] = c;
        }
    }
    if (cnt) atomicAdd(&sh_live[lane], (unsigned long long)cnt);
    sync_lds();
    if ((int)threadIdx.x < K && sh_live[threadIdx.x])
        atomicAdd(&S.live[(size_t)(S.t0 + threadIdx.x) * 64 + (blockIdx.x & 63)], sh_live[threadIdx.x]);
}

} /* namespace gf */

#endif /* GF_PACKED_DRIFT_HPP_ */
