/*
 * surrogate.hip -- learned surrogate of the simulator's sample SFS
 * (no reference counterpart).
 *
 * An ensemble of E multilayer perceptrons, each
 *     6 inputs (padded to 64) -> 4 hidden layers of 512 (GELU) -> 100 outputs
 * (99 softmax logits for the n = 100 SFS bins 1..99, one log-total head),
 * BF16 weights and activations, FP32 accumulation, trained by this file's
 * forward, backward and Adam kernels.  Every matrix product runs on the
 * gfx950 matrix cores (v_mfma_f32_32x32x16_bf16) from operands kept in
 * fragment order, so that a wave's load is one contiguous KB:
 *   k_mlp            prediction: the whole network, inputs to logits, in one
 *                    kernel (k_predict_stats: the ensemble's statistics)
 *   k_train_rows     training: forward, loss and the backward chain of 16
 *                    rows in one kernel
 *   k_train_weights  training: every layer's weight and bias gradients and
 *                    their Adam update in one kernel
 */
#include "gf_runtime.hpp"
#include "gf_sync.hpp"

#include <cmath>
#include <cstring>
#include <memory>
#include <vector>

namespace gf {
namespace sg {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int IN_PAD = 64;    /* input features padded to one K tile */
constexpr int HID = 512;
constexpr int NHID = 4;
constexpr int OUT = 100;      /* 99 bins + log-total */
constexpr int OUT_PAD = 128;
constexpr int NBINS = 99;
constexpr int POUT = NBINS + 2;   /* floats of one prediction: bins, log-total, disagreement */

/* parameter layout of one model, in floats */
struct Layout {
    size_t W[NHID + 1], b[NHID + 1];
    int in[NHID + 1], out[NHID + 1];
    size_t total;
    Layout() {
        size_t o = 0;
        for (int l = 0; l <= NHID; l++) {
            in[l] = l == 0 ? IN_PAD : HID;
            out[l] = l == NHID ? OUT_PAD : HID;
            W[l] = o; o += (size_t)in[l] * out[l];
            b[l] = o; o += out[l];
        }
        total = o;
    }
};

/* GELU, tanh form: 0.5 x (1 + tanh(u)), u = c (x + 0.044715 x^3), c =
 * sqrt(2/pi).  With sigma(v) = 1 / (1 + e^-v), 0.5 (1 + tanh(u)) =
 * sigma(2u), so gelu(x) = x sigma(2u), evaluated with the hardware exp2 and
 * reciprocal (about 1e-6 relative; the activations are then rounded to
 * bfloat16).  e^-2u = 2^(x (k1 + k2 x^2)) with k1 = -2 c log2(e) and k2 =
 * 0.044715 k1: five operations besides exp2 and the reciprocal.  e^-2u
 * overflows to inf for u << 0, where sigma -> 0. */
__device__ __forceinline__ float sigma2u(float x) {
    const float k1 = -2.302208198f, k2 = -0.1029432396f;
    const float t = x * __builtin_fmaf(k2, x * x, k1);
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(t));
}

__device__ __forceinline__ float gelu(float x) { return x * sigma2u(x); }

/* d/dx x sigma(2u) = sigma + 2 x sigma (1 - sigma) u' */
__device__ __forceinline__ float gelu_grad(float x) {
    const float c = 0.7978845608028654f;
    const float sg = sigma2u(x);
    const float du = c * (1.0f + 3.0f * 0.044715f * x * x);
    return sg + 2.0f * x * sg * (1.0f - sg) * du;
}

/* ---- the whole network in one kernel (prediction) ----
 * One workgroup takes 64 inputs (32 where that is enough for every CU to have
 * one) through every layer of one ensemble member: the activations stay in
 * LDS (64 rows of 512 bf16, 66 KB; two workgroups a CU), and the weights
 * stream from L2 straight into the registers that feed the matrix cores.
 * Each of the 8 waves owns 64 of a layer's 512 columns for all rows (2 x 2
 * blocks of v_mfma_f32_32x32x16_bf16), so no weight is read twice by a
 * workgroup and the K loop has no barrier; the weights are the first operand,
 * so a lane's accumulators run along the columns of one row and go back to
 * LDS as 8-byte pieces.  The two workgroups of a CU are independent: one's
 * GELU runs on the vector unit while the other's products run on the matrix
 * cores.
 *
 * The weights are read in fragment order (frag_w below).
 *
 * Tiles are dealt XCD-aware (xcd_order): consecutive tiles of one member go
 * to one XCD, whose L2 then holds that member's 1.7 MB of weights.
 *
 * Each output accumulates its k = 0, 16, 32, ... products in that order, as
 * k_train_rows does: the same bits.
 *
 * Bound: 262,144 inputs and 4 members take 1.94 ms, 930 TFLOP/s, of 0.9 ms
 * the matrix cores need at the 1.95 GHz they run at here.  Timing variants:
 * without the weights' L2 traffic (13 TB/s) 1.5 ms, with the identity for
 * GELU 1.75 ms, without both 1.3 ms: what is left are the layers' ends, where
 * the two workgroups cannot cover each other's latencies.  Tried: 4 waves of
 * 128 columns 2.03 ms, 128 rows and one workgroup a CU 1.98 ms (half the L2
 * traffic, nothing beside GELU), wave priorities and a staggered start no
 * change.  The layer-by-layer products it replaced (128 x 128 tiles through
 * LDS, activations through HBM) took 3.6 ms.
 * 16 inputs: 20 us with 32-row tiles and 8 k-steps of weights in flight, 44
 * with 64 rows and 4; five products one after the other took 62. */
constexpr int MR = 64;            /* rows a prediction batch is padded to */
constexpr int MLDS = HID + 8;     /* padded LDS row: conflict-free 16-byte fragment reads */
constexpr int BIASES = NHID * HID + OUT_PAD;

struct MlpArgs {
    const float *x;               /* [n][6] */
    int n;                        /* rows past it read as zero */
    const bf16 *wp; int64_t sP;   /* weights in fragment order, per member */
    const float *w; int64_t sW;   /* master parameters (biases) */
    int64_t woff[NHID + 1], boff[NHID + 1];
    float *logits; int64_t sL;    /* [E][rows][OUT_PAD] */
    int MT, T;                    /* row tiles, row tiles x members */
};

/* Fragment order of a matrix operand: 512 elements for 32 rows (or columns)
 * `r` and 16 contraction indices `c`, lane (r & 31) + 32 ((c >> 3) & 1)
 * holding the 8 elements c & 7 = 0..7 contiguously: what one lane feeds
 * v_mfma_f32_32x32x16_bf16 for either operand.  cs: contraction steps (of
 * 16) of the whole matrix. */
__host__ __device__ __forceinline__ int64_t frag(int r, int c, int cs) {
    return ((int64_t)(r >> 5) * cs + (c >> 4)) * 512 + ((r & 31) + 32 * ((c >> 3) & 1)) * 8 + (c & 7);
}

/* BF16 copies of the weights W_l [out][in], per member at W_l's offset: wp
 * contracts the inputs (forward), wt the outputs (backward) */
__global__ void k_pack_weights(const float *__restrict__ w, bf16 *__restrict__ wp, bf16 *__restrict__ wt, const Layout lay, int E) {
    const int64_t n = (int64_t)lay.total * E;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t z = i / (int64_t)lay.total, q = i % (int64_t)lay.total;
        int l = 0;
        while (l < NHID && q >= (int64_t)lay.W[l + 1]) l++;
        const int r = (int)(q - (int64_t)lay.W[l]), in = lay.in[l], out = lay.out[l];
        if (r >= in * out) continue;   /* biases */
        const int64_t base = z * (int64_t)lay.total + (int64_t)lay.W[l];
        wp[base + frag(r / in, r % in, in / 16)] = (bf16)w[i];
        wt[base + frag(r % in, r / in, out / 16)] = (bf16)w[i];
    }
}

/* Index of workgroup b of T such that consecutive indices run on one XCD:
 * the hardware hands workgroup b to XCD b % 8 */
__device__ __forceinline__ int xcd_order(int b, int T) {
    const int xcd = b & 7, r = b >> 3, per = T >> 3, rem = T & 7;
    return xcd < rem ? xcd * (per + 1) + r : rem * (per + 1) + (xcd - rem) * per + r;
}

/* RB: blocks of 32 rows per workgroup; DEPTH: k-steps of weights in flight
 * per wave */
template <int RB, int DEPTH, int EU>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(EU))) void k_mlp(const MlpArgs g) {
    constexpr int WAVES = 8, JB = 16 / WAVES, ROWS = 32 * RB, KS = HID / 16;
    __shared__ __attribute__((aligned(16))) bf16 act[ROWS][MLDS];
    __shared__ __attribute__((aligned(16))) float bias[BIASES];
    const int L = xcd_order((int)blockIdx.x, g.T);
    const int z = L / g.MT, m0 = (L % g.MT) * ROWS;
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int fr = lane & 31, hi = lane >> 5;
    const bf16 *wp = g.wp + z * g.sP;
    const float *par = g.w + z * g.sW;
    /* weight operands of this wave's column blocks JB w .. JB w + JB - 1 */
    bf16x8 fb[DEPTH][JB];
    auto fetch = [&](const bf16x8 *p, int ks, int steps, int u) {
#pragma unroll
        for (int j = 0; j < JB; j++) fb[u][j] = p[((int64_t)j * steps + ks) * 64];
    };
    auto weights = [&](int l, int steps) { return (const bf16x8 *)(wp + g.woff[l]) + (int64_t)(JB * w) * steps * 64 + lane; };
    fetch(weights(0, IN_PAD / 16), 0, IN_PAD / 16, 0);
    {
        float bv[NHID + 1];
#pragma unroll
        for (int i = 0; i <= NHID; i++) bv[i] = i < NHID || t < OUT_PAD ? par[g.boff[i] + t] : 0.0f;
#pragma unroll
        for (int i = 0; i <= NHID; i++)
            if (i < NHID || t < OUT_PAD) bias[i * HID + t] = bv[i];
    }
    for (int k = t; k < ROWS * 4; k += 64 * WAVES) {   /* inputs: 6 features in the first k-step, the rest of it zero */
        const int r = k >> 2, c = (k & 3) * 4;
        bf16x4 v;
#pragma unroll
        for (int q = 0; q < 4; q++) v[q] = (bf16)(c + q < 6 && m0 + r < g.n ? g.x[(int64_t)(m0 + r) * 6 + c + q] : 0.0f);
        *(bf16x4 *)&act[r][c] = v;
    }
    f32x16 acc[RB][JB];
    bf16x8 fa[2][RB];
    auto rows = [&](int ks, int v) {
#pragma unroll
        for (int i = 0; i < RB; i++) fa[v][i] = *(const bf16x8 *)&act[i * 32 + fr][ks * 16 + 8 * hi];
    };
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < RB; i++)
#pragma unroll
            for (int j = 0; j < JB; j++) acc[i][j] = f32x16{};
    };
    auto step = [&](int u, int v) {
#pragma unroll
        for (int j = 0; j < JB; j++)
#pragma unroll
            for (int i = 0; i < RB; i++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[u][j], fa[v][i], acc[i][j], 0, 0, 0);
    };
    /* acc -> bias, GELU, bf16 -> act.  Accumulator r of lane l of block (i, j)
     * is row 32 i + l % 32, column 32 (JB w + j) + 8 (r/4) + 4 (l/32) + r%4. */
    auto activate = [&](int l) {
        bf16x4 pk[RB][JB][4];
#pragma unroll
        for (int j = 0; j < JB; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const f32x4 bv = *(const f32x4 *)&bias[l * HID + 32 * (JB * w + j) + 8 * q + 4 * hi];
#pragma unroll
                for (int i = 0; i < RB; i++)
#pragma unroll
                    for (int k = 0; k < 4; k++) pk[i][j][q][k] = (bf16)gelu(acc[i][j][4 * q + k] + bv[k]);
            }
        sync_lds();   /* every wave has read this layer's inputs */
#pragma unroll
        for (int i = 0; i < RB; i++)
#pragma unroll
            for (int j = 0; j < JB; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) *(bf16x4 *)&act[i * 32 + fr][32 * (JB * w + j) + 8 * q + 4 * hi] = pk[i][j][q];
        sync_lds();
    };
    sync_lds();
    /* layer 1: one k-step holds all six inputs */
    clear();
    rows(0, 0);
    step(0, 0);
#pragma unroll
    for (int u = 0; u < DEPTH; u++) fetch(weights(1, KS), u, KS, u);
    activate(0);
    for (int l = 1; l < NHID; l++) {
        const bf16x8 *p = weights(l, KS);
        clear();
        rows(0, 0);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            if (ks + 1 < KS) rows(ks + 1, (ks + 1) & 1);
            step(ks % DEPTH, ks & 1);
            if (ks + DEPTH < KS) fetch(p, ks + DEPTH, KS, ks % DEPTH);
        }
        /* the next hidden layer's first operands arrive during this one's epilogue */
        if (l + 1 < NHID) {
#pragma unroll
            for (int u = 0; u < DEPTH; u++) fetch(weights(l + 1, KS), u, KS, u);
        }
        activate(l);
    }
    /* output layer: four column blocks, one each for the first four waves */
    if (w < 4) {
        const bf16x8 *po = (const bf16x8 *)(wp + g.woff[NHID]) + (int64_t)w * KS * 64 + lane;
        f32x16 o[RB];
#pragma unroll
        for (int i = 0; i < RB; i++) o[i] = f32x16{};
        bf16x8 fo[16];
#pragma unroll
        for (int k = 0; k < 16; k++) fo[k] = po[k * 64];
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            rows(ks, 0);
#pragma unroll
            for (int i = 0; i < RB; i++) o[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fo[ks % 16], fa[0][i], o[i], 0, 0, 0);
            if (ks + 16 < KS) fo[ks % 16] = po[(ks + 16) * 64];
        }
        float *dst = g.logits + z * g.sL + (int64_t)m0 * OUT_PAD;
#pragma unroll
        for (int i = 0; i < RB; i++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int c = 32 * w + 8 * q + 4 * hi;
                const f32x4 bv = *(const f32x4 *)&bias[NHID * HID + c];
                f32x4 v;
#pragma unroll
                for (int k = 0; k < 4; k++) v[k] = o[i][4 * q + k] + bv[k];
                *(f32x4 *)&dst[(int64_t)(i * 32 + fr) * OUT_PAD + c] = v;
            }
    }
}

/* ---- training: forward, loss and backward of 16 rows in one kernel ----
 * One workgroup takes 16 rows of the batch through one member's layers, the
 * loss and back, the activations (then the gradients) in LDS, the weights
 * streamed from L2 in fragment order: wp on the way up, wt on the way down.
 * It leaves what the weight gradients contract over the batch, in fragment
 * order with the batch as contraction: the layer inputs (xt, ht) and the
 * gradients of the pre-activations and logits (dt, lt).  The
 * pre-activations a lane produced come back to that lane (Z, 1 KB per wave
 * and store).  Here the rows are the first MFMA operand, so a lane holds four
 * consecutive rows of one column: 8 contiguous bytes of a batch fragment.
 *
 * Bound: the latency of the weight stream (2 x 1.7 MB per workgroup, most of
 * it just written by k_train_weights on other XCDs: 40 to 50 B a clock) and the GELU derivative's vector
 * work, with one workgroup on half of the CUs (512 rows, 4 members).  16 rows
 * instead of 32 halve the vector work of a CU for the same stream, and 16
 * k-steps in flight instead of 8: 62 -> 49 us.  Rounding points and the order
 * of every sum (products by k, the softmax sum by bin) are those of the
 * layer-by-layer kernels it replaced: compared with them, the gradients were
 * the same bits; the loss, which those summed with one atomic per row, differs
 * in its last bits.
 * One step (512 rows, 4 members) was 14 products of 6 to 20 us, loss 15,
 * column sums 5 x 4.6, Adam 17, gather and packing 9, together 300 us; now
 * this kernel and k_train_weights, 80 us. */
constexpr int TR = 16;            /* rows per workgroup: half an MFMA block (its other rows repeat them and are not used) */
constexpr int TDEPTH = 16;        /* k-steps of weights in flight per wave */
constexpr int LGS = OUT_PAD + 4;  /* LDS row of the logits */

struct TrainArgs {
    const float *X, *Y, *T;       /* [rows][6], [rows][99], [rows] */
    const int32_t *ord;           /* batch row b is row ord[b]; NULL: row b */
    int B;
    float w_tot;
    const bf16 *wp, *wt;
    const float *w;
    int64_t sW;                   /* member stride of wp, wt and w */
    int64_t woff[NHID + 1], boff[NHID + 1];
    float *Z;                     /* [E][NHID][B / TR][8 waves][4][64 lanes][4] */
    bf16 *xt, *ht, *dt, *lt;      /* batch fragments: [2], [E][NHID][16], [E][NHID][16], [E][4] x [B / 16][512] */
    float *loss;                  /* [E] */
};

__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void k_train_rows(const TrainArgs g) {
    constexpr int KS = HID / 16;
    __shared__ __attribute__((aligned(16))) bf16 act[TR][MLDS];
    __shared__ __attribute__((aligned(16))) float bias[BIASES];
    __shared__ float lg[TR][LGS], ex[TR][LGS];
    __shared__ float wloss[8];
    const int tiles = g.B / TR, L = xcd_order((int)blockIdx.x, (int)gridDim.x);   /* a member's tiles on one or two XCDs */
    const int tile = L % tiles, z = L / tiles;
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int fr = lane & 31, hi = lane >> 5;
    const int cs = g.B / 16;   /* contraction steps of the batch: one per tile */
    const bf16 *wp = g.wp + z * g.sW, *wt = g.wt + z * g.sW;
    const float *par = g.w + z * g.sW;
    auto row_of = [&](int r) { const int b = tile * TR + r; return (int64_t)(g.ord ? g.ord[b] : b); };
    bf16x8 fb[TDEPTH][2];
    auto fetch = [&](const bf16x8 *p, int ks, int steps, int u) {
        fb[u][0] = p[(int64_t)ks * 64];
        fb[u][1] = p[((int64_t)steps + ks) * 64];
    };
    auto up = [&](int l, int steps) { return (const bf16x8 *)(wp + g.woff[l]) + (int64_t)(2 * w) * steps * 64 + lane; };
    auto down = [&](int l, int steps) { return (const bf16x8 *)(wt + g.woff[l]) + (int64_t)(2 * w) * steps * 64 + lane; };
    fetch(up(0, IN_PAD / 16), 0, IN_PAD / 16, 0);
    /* targets of the loss: 32 threads per row, 4 bins each */
    const int lr = t >> 5, lc = t & 31;
    const int64_t src = row_of(lr);
    float y[4];
#pragma unroll
    for (int i = 0; i < 4; i++) y[i] = lc + 32 * i < NBINS ? g.Y[src * NBINS + lc + 32 * i] : g.T[src];
    const float x = lc < 6 ? g.X[src * 6 + lc] : 0.0f;
    float bv[NHID + 1];
#pragma unroll
    for (int i = 0; i <= NHID; i++) bv[i] = i < NHID || t < OUT_PAD ? par[g.boff[i] + t] : 0.0f;
    if (lc < 16) act[lr][lc] = (bf16)x;   /* 6 features, zero up to 16 (one k-step; the others only add zeros) */
#pragma unroll
    for (int i = 0; i <= NHID; i++)
        if (i < NHID || t < OUT_PAD) bias[i * HID + t] = bv[i];
    sync_lds();
    if (z == 0 && w < 2) {   /* the inputs' batch fragments: 2 column blocks */
        bf16x8 v;
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = w == 0 && fr < 16 ? act[8 * hi + e][fr] : (bf16)0.0f;
        *(bf16x8 *)(g.xt + ((int64_t)w * cs + tile) * 512 + lane * 8) = v;
    }
    f32x16 acc[2];
    bf16x8 fa[2];
    auto rows = [&](int ks, int v) { fa[v] = *(const bf16x8 *)&act[fr % TR][ks * 16 + 8 * hi]; };
    auto step = [&](int u, int v) {
#pragma unroll
        for (int j = 0; j < 2; j++) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[v], fb[u][j], acc[j], 0, 0, 0);
    };
    /* acc = act x operand over 32 k-steps, the first TDEPTH already in fb */
    auto product = [&](const bf16x8 *p) {
        acc[0] = f32x16{};
        acc[1] = f32x16{};
        rows(0, 0);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            if (ks + 1 < KS) rows(ks + 1, (ks + 1) & 1);
            step(ks % TDEPTH, ks & 1);
            if (ks + TDEPTH < KS) fetch(p, ks + TDEPTH, KS, ks % TDEPTH);
        }
    };
    auto prefetch = [&](const bf16x8 *p, int steps) {
#pragma unroll
        for (int u = 0; u < TDEPTH; u++) fetch(p, u, steps, u);
    };
    /* accumulator r < 8 of lane l of block j is row 8 (r/4) + 4 (l/32) + r%4,
     * column 64 w + 32 j + l%32 */
    auto zpos = [&](int l) { return (f32x4 *)g.Z + ((((int64_t)z * NHID + l) * tiles + tile) * 8 + w) * 256 + lane; };
    /* four rows of column block cb of a batch fragment array */
    auto put = [&](bf16 *base, int cb, int q, bf16x4 v) {
        *(bf16x4 *)(base + ((int64_t)cb * cs + tile) * 512 + (fr + 32 * q) * 8 + 4 * hi) = v;
    };
    auto to_act = [&](const bf16x4 (&v)[2][2]) {
        sync_lds();   /* every wave has read this layer's rows */
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int q = 0; q < 2; q++)
#pragma unroll
                for (int k = 0; k < 4; k++) act[8 * q + 4 * hi + k][64 * w + 32 * j + fr] = v[j][q][k];
        sync_lds();
    };
    auto activate = [&](int l) {
        bf16x4 v[2][2];
        f32x4 *zp = zpos(l);
        bf16 *ht = g.ht + ((int64_t)z * NHID + l) * g.B * HID;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const float b = bias[l * HID + 64 * w + 32 * j + fr];
#pragma unroll
            for (int q = 0; q < 2; q++) {
                f32x4 zz;
#pragma unroll
                for (int k = 0; k < 4; k++) { zz[k] = acc[j][4 * q + k] + b; v[j][q][k] = (bf16)gelu(zz[k]); }
                zp[(j * 2 + q) * 64] = zz;
                put(ht, 2 * w + j, q, v[j][q]);
            }
        }
        to_act(v);
    };
    acc[0] = f32x16{};
    acc[1] = f32x16{};
    rows(0, 0);
    step(0, 0);
    prefetch(up(1, KS), KS);
    activate(0);
    for (int l = 1; l < NHID; l++) {
        product(up(l, KS));
        if (l + 1 < NHID) {
            prefetch(up(l + 1, KS), KS);
        } else if (w < 4) {   /* the output layer's column block w, whole */
            const bf16x8 *po = (const bf16x8 *)(wp + g.woff[NHID]) + (int64_t)w * KS * 64 + lane;
#pragma unroll
            for (int ks = 0; ks < KS; ks++) fb[ks / 2][ks % 2] = po[ks * 64];
        }
        activate(l);
    }
    static_assert(KS == 2 * TDEPTH, "an output column block fills the operand registers");
    if (w < 4) {   /* logits: column block w */
        f32x16 o = f32x16{};
        rows(0, 0);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            if (ks + 1 < KS) rows(ks + 1, (ks + 1) & 1);
            o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[ks & 1], fb[ks / 2][ks % 2], o, 0, 0, 0);
        }
        const float b = bias[NHID * HID + 32 * w + fr];
#pragma unroll
        for (int r = 0; r < 8; r++) lg[8 * (r >> 2) + 4 * hi + (r & 3)][32 * w + fr] = o[r] + b;
    }
    /* the first backward product's operands arrive during the loss */
    constexpr int OS = OUT_PAD / 16;
    static_assert(OS <= TDEPTH, "the output layer's contraction is prefetched whole");
#pragma unroll
    for (int u = 0; u < OS; u++) fetch(down(NHID, OS), u, OS, u);
    sync_lds();
    {   /* softmax cross-entropy + w_tot (log-total - target)^2: 32 threads per row */
        float lv[4], mx = lg[lr][0];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            lv[i] = lg[lr][lc + 32 * i];
            if (lc + 32 * i < NBINS) mx = fmaxf(mx, lv[i]);
        }
#pragma unroll
        for (int off = 16; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (lc + 32 * i < NBINS) ex[lr][lc + 32 * i] = __expf(lv[i] - mx);
        sync_lds();
        float ls = 0.0f;
        if (lc == 0) {   /* the sum in bin order */
            float sum = 0.0f;
#pragma unroll
            for (int k = 0; k < NBINS; k++) sum += ex[lr][k];
            ls = logf(sum) + mx;
        }
        ls = __shfl(ls, lane & 32);
        const float invB = 1.0f / (float)g.B;
        float ce = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int k = lc + 32 * i;
            float d = 0.0f;
            if (k < NBINS) {
                const float p = __expf(lv[i] - ls);
                ce -= y[i] * (lv[i] - ls);
                d = (p - y[i]) * invB;
            } else if (k == NBINS) {   /* y holds the log-total target there */
                const float e = lv[i] - y[i];
                ce += g.w_tot * e * e;
                d = 2.0f * g.w_tot * e * invB;
            }
            act[lr][k] = (bf16)d;   /* the logits' inputs have been read by all waves */
        }
        ce *= invB;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) ce += __shfl_xor(ce, off);
        if (lane == 0) wloss[w] = ce;
    }
    sync_lds();
    if (t == 0) {
        float sum = 0.0f;
        for (int k = 0; k < 8; k++) sum += wloss[k];
        atomicAdd(&g.loss[z], sum);
    }
    if (w < 4) {   /* the logit gradients' batch fragments: column block w */
        bf16x8 v;
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = act[8 * hi + e][w * 32 + fr];
        *(bf16x8 *)(g.lt + (((int64_t)z * 4 + w) * cs + tile) * 512 + lane * 8) = v;
    }
    /* gradient of layer l's pre-activation from acc = dY W_(l+1) */
    auto back = [&](int l, const f32x4 (&zz)[4]) {
        bf16x4 v[2][2];
        bf16 *dt = g.dt + ((int64_t)z * NHID + l) * g.B * HID;
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int q = 0; q < 2; q++) {
#pragma unroll
                for (int k = 0; k < 4; k++) v[j][q][k] = (bf16)(acc[j][4 * q + k] * gelu_grad(zz[j * 2 + q][k]));
                put(dt, 2 * w + j, q, v[j][q]);
            }
        if (l > 0) to_act(v);
    };
    f32x4 zz[4];
    auto load_z = [&](int l) {
        const f32x4 *zp = zpos(l);
#pragma unroll
        for (int k = 0; k < 4; k++) zz[k] = zp[k * 64];
    };
    load_z(NHID - 1);
    acc[0] = f32x16{};
    acc[1] = f32x16{};
#pragma unroll
    for (int ks = 0; ks < OS; ks++) {
        rows(ks, 0);
        step(ks, 0);
    }
    prefetch(down(NHID - 1, KS), KS);
    back(NHID - 1, zz);
    for (int l = NHID - 1; l > 0; l--) {
        load_z(l - 1);
        product(down(l, KS));
        if (l > 1) prefetch(down(l - 1, KS), KS);
        back(l - 1, zz);
    }
}

/* ---- training: weight and bias gradients of every layer and Adam ----
 * dW_l = dY_l^T X_l contracts the batch: both operands are k_train_rows'
 * batch fragments, loaded straight into the registers of the matrix cores.
 * A workgroup of 4 waves covers 128 x 128 weights of one layer and member
 * (each wave 64 x 64), and the accumulators go through Adam where they are
 * (UPDATE), which also refreshes the two BF16 copies, or into the gradient
 * array.  The waves over a layer's first input columns also sum the gradient's
 * rows (the bias gradient) from the same fragments: 32 sums over every 32nd
 * row, then those in order.
 * Bound: Adam's 32 B per parameter (110 MB at 4 members: 18 us at 6 TB/s) after
 * 8 us of products: 31 us; 51 before a block's loads were issued together. */
struct WeightArgs {
    const bf16 *xt, *ht, *dt, *lt;
    int B;
    float *w, *m, *v, *gr;
    bf16 *wp, *wt;
    int64_t sW;
    int64_t woff[NHID + 1], boff[NHID + 1];
    float lr, b1, b2, eps, c1, c2;
};

constexpr int WBLOCKS = 3 * 16 + 4 + 4;   /* 128 x 128 blocks of a member: layers 1..3, 4, 0 */

template <bool UPDATE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_train_weights(const WeightArgs g) {
    __shared__ __attribute__((aligned(16))) bf16 sh[4][64][64 + 8];
    const int L = xcd_order((int)blockIdx.x, (int)gridDim.x);
    const int z = L / WBLOCKS, blk = L % WBLOCKS;
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int fr = lane & 31, hi = lane >> 5;
    int l, bo, bi;
    if (blk < 48) { l = 1 + blk / 16; bo = blk % 16 / 4; bi = blk % 4; }
    else if (blk < 52) { l = NHID; bo = 0; bi = blk - 48; }
    else { l = 0; bo = blk - 52; bi = 0; }
    const int o0 = bo * 128 + (w >> 1) * 64, i0 = bi * 128 + (w & 1) * 64;
    const int in = l == 0 ? IN_PAD : HID, out = l == NHID ? OUT_PAD : HID;
    if (i0 >= in) return;
    const int cs = g.B / 16;
    const bf16 *dy = l == NHID ? g.lt + (int64_t)z * 4 * cs * 512 : g.dt + ((int64_t)z * NHID + l) * g.B * HID;
    const bf16 *xx = l == 0 ? g.xt : g.ht + ((int64_t)z * NHID + l - 1) * g.B * HID;
    const bf16x8 *pa = (const bf16x8 *)dy + (int64_t)(o0 / 32) * cs * 64 + lane;
    const bf16x8 *pb = (const bf16x8 *)xx + (int64_t)(i0 / 32) * cs * 64 + lane;
    constexpr int D = 4;
    bf16x8 fa[D][2], fb[D][2];
    auto fetch = [&](int ks, int u) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            fa[u][k] = pa[((int64_t)k * cs + ks) * 64];
            fb[u][k] = pb[((int64_t)k * cs + ks) * 64];
        }
    };
    f32x16 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) acc[a][b] = f32x16{};
    /* sums[a][s][e]: rows 16 s + 8 hi + e modulo 32 of column o0 + 32 a + fr */
    const bool bias_sums = i0 == 0;
    float sums[2][2][8] = {};
    auto step = [&](int u) {
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int b = 0; b < 2; b++) acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[u][a], fb[u][b], acc[a][b], 0, 0, 0);
        if (bias_sums) {
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int e = 0; e < 8; e++) sums[a][u & 1][e] += (float)fa[u][a][e];
        }
    };
#pragma unroll
    for (int u = 0; u < D; u++) fetch(u, u);   /* B is a multiple of 64: at least D steps */
    for (int ks = 0; ks + D < cs; ks += D) {
#pragma unroll
        for (int u = 0; u < D; u++) {
            step(u);
            fetch(ks + D + u, u);
        }
    }
#pragma unroll
    for (int u = 0; u < D; u++) step(u);
    const int64_t base = z * g.sW;
    auto adam = [&](float &w, float &m, float &v, float gr) {
        m = g.b1 * m + (1.0f - g.b1) * gr;
        v = g.b2 * v + (1.0f - g.b2) * gr * gr;
        w = w - g.lr * (m / g.c1) / (sqrtf(v / g.c2) + g.eps);
    };
    if (bias_sums) {
#pragma unroll
        for (int a = 0; a < 2; a++) {
            float s = 0.0f;   /* rows 0..7 in the lower half, 8..15 in the upper, 16..23, 24..31 */
#pragma unroll
            for (int part = 0; part < 4; part++) {
                float x = s;
#pragma unroll
                for (int e = 0; e < 8; e++) x += sums[a][part >> 1][e];
                s = __shfl(x, fr + 32 * (part & 1));
            }
            const int64_t i = base + g.boff[l] + o0 + 32 * a + fr;
            if (hi == 0) {
                if (UPDATE) adam(g.w[i], g.m[i], g.v[i], s);
                else g.gr[i] = s;
            }
        }
    }
    /* accumulator r of lane l of block (a, b): weight row o0 + 32 a + 8 (r/4)
     * + 4 (l/32) + r%4, column i0 + 32 b + l%32.  A block's 48 loads are issued
     * together, ahead of its 48 stores. */
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const int i = i0 + 32 * b + fr;
            const int64_t at = base + g.woff[l] + (int64_t)(o0 + 32 * a + 4 * hi) * in + i;
            if (UPDATE) {
                float wv[16], mv[16], vv[16];
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int64_t p = at + (int64_t)(8 * (r >> 2) + (r & 3)) * in;
                    wv[r] = g.w[p];
                    mv[r] = g.m[p];
                    vv[r] = g.v[p];
                }
#pragma unroll
                for (int r = 0; r < 16; r++) adam(wv[r], mv[r], vv[r], acc[a][b][r]);
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int64_t p = at + (int64_t)(8 * (r >> 2) + (r & 3)) * in;
                    g.w[p] = wv[r];
                    g.m[p] = mv[r];
                    g.v[p] = vv[r];
                }
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int ob = 32 * a + 8 * q + 4 * hi;
                    bf16x4 v;
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        v[k] = (bf16)wv[4 * q + k];
                        sh[w][ob + k][32 * b + fr] = v[k];
                    }
                    *(bf16x4 *)(g.wt + base + g.woff[l] + frag(i, o0 + ob, out / 16)) = v;
                }
            } else {
#pragma unroll
                for (int r = 0; r < 16; r++) g.gr[at + (int64_t)(8 * (r >> 2) + (r & 3)) * in] = acc[a][b][r];
            }
        }
    if (UPDATE) {   /* wp's pieces of 8 inputs, through this wave's LDS tile */
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int ol = (lane & 31) + 32 * (k & 1), il = 16 * (k >> 1) + 8 * hi;
            *(bf16x8 *)(g.wp + base + g.woff[l] + frag(o0 + ol, i0 + il, in / 16)) = *(const bf16x8 *)&sh[w][ol][il];
        }
    }
}

/* ensemble statistics of the predictions: per-model softmax, mean SFS,
 * mean log-total and the ensemble disagreement (largest relative standard
 * deviation across models over the bins with mean mass >= 1e-3).  One wave
 * per input: lane l holds bins l and l + 64, so each model's logit row is
 * read once, coalesced, and the row's max and sum are wave reductions. */
__global__ __launch_bounds__(256) void k_predict_stats(const float *__restrict__ logits, int64_t sL, int E, int B,
                                                       float *__restrict__ sfs, float *__restrict__ tot,
                                                       float *__restrict__ dis) {
    const int lane = threadIdx.x & 63;
    const int b = (int)blockIdx.x * 4 + ((int)threadIdx.x >> 6);
    if (b >= B) return;   /* the whole wave */
    const int k1 = lane + 64;
    const bool h1 = k1 < NBINS;
    float mean0 = 0.f, mean1 = 0.f, sq0 = 0.f, sq1 = 0.f, tsum = 0.f;
    for (int z = 0; z < E; z++) {
        const float *L = logits + z * sL + (int64_t)b * OUT_PAD;
        const float l0 = L[lane];
        const float l1 = h1 ? L[k1] : l0;
        float mx = fmaxf(l0, l1);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
        const float e0 = __expf(l0 - mx), e1 = h1 ? __expf(l1 - mx) : 0.f;
        float sum = e0 + e1;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
        const float p0 = e0 / sum, p1 = e1 / sum;
        mean0 += p0; sq0 += p0 * p0;
        mean1 += p1; sq1 += p1 * p1;
        tsum += L[NBINS];
    }
    float worst = 0.f;
    {
        const float mu = mean0 / E, var = fmaxf(sq0 / E - mu * mu, 0.f);
        sfs[(int64_t)b * NBINS + lane] = mu;
        if (mu >= 1e-3f) worst = sqrtf(var) / mu;
    }
    if (h1) {
        const float mu = mean1 / E, var = fmaxf(sq1 / E - mu * mu, 0.f);
        sfs[(int64_t)b * NBINS + k1] = mu;
        if (mu >= 1e-3f) worst = fmaxf(worst, sqrtf(var) / mu);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) worst = fmaxf(worst, __shfl_xor(worst, off));
    if (lane == 0) {
        if (tot) tot[b] = tsum / E;
        if (dis) dis[b] = worst;
    }
}

} /* namespace sg */
} /* namespace gf */

using namespace gf;
using namespace gf::sg;

struct gf_sg_model {
    int E = 4, Bmax = 0;
    Layout lay;
    OwnedStream st;   /* before the buffers: they are released while it is alive */
    OwnedStream cst;  /* prediction read-back, beside the next batch's compute on st */
    DevBuf<float> w, g, m, v;       /* [E][total] */
    DevBuf<bf16> wp, wt;            /* BF16 weights in fragment order */
    /* training, Bmax rows */
    DevBuf<float> Z;
    DevBuf<bf16> xt, ht, dt, lt;
    DevBuf<float> loss;
    /* prediction */
    DevBuf<float> logits;           /* [E][B][128] */
    DevBuf<float> xin;
    DevBuf<float> pout;             /* two batches' prediction outputs */
    int64_t step = 0;
    float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
};

namespace gf {
namespace sg {

static int ensure_batch(gf_sg_model &S, int B) {
    if (B <= S.Bmax) return GF_OK;
    const size_t E = (size_t)S.E, act = E * NHID * (size_t)B * HID;
    GF_TRY(S.Z.alloc(act));
    GF_TRY(S.ht.alloc(act));
    GF_TRY(S.dt.alloc(act));
    GF_TRY(S.xt.alloc((size_t)B * IN_PAD));
    GF_TRY(S.lt.alloc(E * B * OUT_PAD));
    S.Bmax = B;
    return GF_OK;
}

/* both BF16 copies from the master weights */
static int pack_weights(gf_sg_model &S) {
    hipLaunchKernelGGL(k_pack_weights, dim3(2048), dim3(256), 0, S.st, S.w.p, S.wp.p, S.wt.p, S.lay, S.E);
    GF_HIP(hipGetLastError());
    return GF_OK;
}

/* buffers of prediction batches of up to B rows; host: also two batches'
 * inputs and outputs */
static int ensure_predict(gf_sg_model &S, int B, bool host) {
    GF_TRY(S.logits.alloc((size_t)S.E * B * OUT_PAD));
    if (host) {
        GF_TRY(S.xin.alloc((size_t)B * 6));
        GF_TRY(S.pout.alloc((size_t)2 * B * POUT));
    }
    return GF_OK;
}

/* logits of the whole ensemble for n rows of x (device, [n][6]), B = n
 * rounded up to MR rows: S.logits [E][B][128] */
static int predict_logits(gf_sg_model &S, const float *x, int n, int B) {
    const Layout &L = S.lay;
    MlpArgs a{};
    a.x = x;
    a.n = n;
    a.wp = S.wp.p; a.sP = (int64_t)L.total;
    a.w = S.w.p; a.sW = (int64_t)L.total;
    for (int l = 0; l <= NHID; l++) { a.woff[l] = (int64_t)L.W[l]; a.boff[l] = (int64_t)L.b[l]; }
    a.logits = S.logits.p; a.sL = (int64_t)B * OUT_PAD;
    /* 32-row tiles as long as they give each CU at most one workgroup (whole
     * call, 4 members: 1,024 inputs 40 us against 52, 2,048 44 against 54,
     * 4,096 62 against 59) */
    const int tiles32 = (n + 31) / 32;
    if ((int64_t)tiles32 * S.E <= num_cus()) {
        a.MT = tiles32;
        a.T = a.MT * S.E;
        hipLaunchKernelGGL((k_mlp<1, 8, 2>), dim3(a.T), dim3(512), 0, S.st, a);
    } else {
        a.MT = B / MR;
        a.T = a.MT * S.E;
        hipLaunchKernelGGL((k_mlp<2, 4, 4>), dim3(a.T), dim3(512), 0, S.st, a);
    }
    GF_HIP(hipGetLastError());
    return GF_OK;
}

/* ensemble statistics of the cnt rows predict_logits left in S.logits */
static int predict_stats(gf_sg_model &S, int cnt, float *sfs, float *tot, float *dis) {
    const int64_t sL = (int64_t)((cnt + MR - 1) / MR * MR) * OUT_PAD;
    hipLaunchKernelGGL(k_predict_stats, dim3((cnt + 3) / 4), dim3(256), 0, S.st, S.logits.p, sL, S.E, cnt, sfs, tot, dis);
    GF_HIP(hipGetLastError());
    return GF_OK;
}

/* n rows of host inputs and targets on the device (the caller synchronises
 * the stream before it returns) */
static int stage_rows(gf_sg_model &S, const float *x, const float *y, const float *t, int n, DevBuf<float> &dx,
                      DevBuf<float> &dy, DevBuf<float> &dt) {
    GF_TRY(dx.alloc((size_t)n * 6));
    GF_TRY(dy.alloc((size_t)n * NBINS));
    GF_TRY(dt.alloc(n));
    GF_HIP(hipMemcpyAsync(dx.p, x, (size_t)n * 6 * sizeof(float), hipMemcpyHostToDevice, S.st));
    GF_HIP(hipMemcpyAsync(dy.p, y, (size_t)n * NBINS * sizeof(float), hipMemcpyHostToDevice, S.st));
    GF_HIP(hipMemcpyAsync(dt.p, t, (size_t)n * sizeof(float), hipMemcpyHostToDevice, S.st));
    return GF_OK;
}

/* forward, backward and (update) Adam for a batch of B rows of X, Y, T
 * (device): rows ord[0..B), or 0..B where ord is NULL */
static int train_step(gf_sg_model &S, const float *X, const float *Y, const float *T, const int32_t *ord, int B, float lr,
                      float w_tot, bool update) {
    const Layout &L = S.lay;
    TrainArgs a{};
    a.X = X; a.Y = Y; a.T = T; a.ord = ord;
    a.B = B;
    a.w_tot = w_tot;
    a.wp = S.wp.p; a.wt = S.wt.p; a.w = S.w.p;
    a.Z = S.Z.p;
    a.xt = S.xt.p; a.ht = S.ht.p; a.dt = S.dt.p; a.lt = S.lt.p;
    a.loss = S.loss.p;
    WeightArgs b{};
    b.xt = S.xt.p; b.ht = S.ht.p; b.dt = S.dt.p; b.lt = S.lt.p;
    b.B = B;
    b.w = S.w.p; b.m = S.m.p; b.v = S.v.p; b.gr = S.g.p;
    b.wp = S.wp.p; b.wt = S.wt.p;
    a.sW = b.sW = (int64_t)L.total;
    for (int l = 0; l <= NHID; l++) {
        a.woff[l] = b.woff[l] = (int64_t)L.W[l];
        a.boff[l] = b.boff[l] = (int64_t)L.b[l];
    }
    hipLaunchKernelGGL(k_train_rows, dim3(B / TR * S.E), dim3(512), 0, S.st, a);
    GF_HIP(hipGetLastError());
    if (update) {
        S.step++;
        b.lr = lr; b.b1 = S.b1; b.b2 = S.b2; b.eps = S.eps;
        b.c1 = 1.0f - std::pow(S.b1, (float)S.step);
        b.c2 = 1.0f - std::pow(S.b2, (float)S.step);
        hipLaunchKernelGGL(k_train_weights<true>, dim3(WBLOCKS * S.E), dim3(256), 0, S.st, b);
    } else {
        hipLaunchKernelGGL(k_train_weights<false>, dim3(WBLOCKS * S.E), dim3(256), 0, S.st, b);
    }
    GF_HIP(hipGetLastError());
    return GF_OK;
}

} /* namespace sg */
} /* namespace gf */

extern "C" {

int32_t gf_sg_create(int32_t ensemble, uint64_t seed, int32_t device, gf_sg_model **out) {
    if (!out || ensemble < 1 || ensemble > 16) { set_error("gf_sg_create: invalid arguments"); return GF_ERR_ARG; }
    *out = nullptr;
    GF_TRY(select_device(device));
    std::unique_ptr<gf_sg_model> S(new gf_sg_model);
    S->E = ensemble;
    GF_HIP(S->st.create());
    StreamScope scope(S->st);
    const size_t n = (size_t)S->E * S->lay.total;
    GF_TRY(S->w.alloc(n));
    GF_TRY(S->g.alloc(n));
    GF_TRY(S->m.alloc(n));
    GF_TRY(S->v.alloc(n));
    GF_TRY(S->wp.alloc(n));
    GF_TRY(S->wt.alloc(n));
    GF_TRY(S->loss.alloc(S->E));
    /* He-style initialisation from a seeded host generator: W ~ U(-a, a),
     * a = sqrt(6 / fan_in); biases 0; padded input columns and output rows 0 */
    std::vector<float> h(n, 0.0f);
    uint64_t st = seed * 6364136223846793005ull + 1442695040888963407ull;
    auto next = [&st]() {
        st = st * 6364136223846793005ull + 1442695040888963407ull;
        return (float)((st >> 40) & 0xffffff) / 16777216.0f;
    };
    for (int e = 0; e < S->E; e++) {
        for (int l = 0; l <= NHID; l++) {
            const int I = S->lay.in[l], O = S->lay.out[l];
            const int real_in = l == 0 ? 6 : I, real_out = l == NHID ? OUT : O;
            const float a = std::sqrt(6.0f / (float)real_in);
            for (int o = 0; o < O; o++)
                for (int i = 0; i < I; i++) {
                    float v = (2.0f * next() - 1.0f) * a;
                    if (i >= real_in || o >= real_out) v = 0.0f;
                    h[(size_t)e * S->lay.total + S->lay.W[l] + (size_t)o * I + i] = v;
                }
        }
    }
    GF_HIP(hipMemcpy(S->w.p, h.data(), n * sizeof(float), hipMemcpyHostToDevice));
    GF_HIP(hipMemset(S->m.p, 0, n * sizeof(float)));
    GF_HIP(hipMemset(S->v.p, 0, n * sizeof(float)));
    GF_TRY(pack_weights(*S));
    GF_HIP(hipStreamSynchronize(S->st));
    *out = S.release();
    return GF_OK;
}

void gf_sg_free(gf_sg_model *S) { delete S; }

int32_t gf_sg_num_params(const gf_sg_model *S) { return S ? (int32_t)S->lay.total : GF_ERR_ARG; }

int32_t gf_sg_get_params(gf_sg_model *S, float *out) {
    if (!S || !out) return GF_ERR_ARG;
    return readback(out, S->w.p, (size_t)S->E * S->lay.total * sizeof(float), S->st);
}

int32_t gf_sg_set_params(gf_sg_model *S, const float *in) {
    if (!S || !in) return GF_ERR_ARG;
    const size_t n = (size_t)S->E * S->lay.total;
    GF_HIP(hipMemcpy(S->w.p, in, n * sizeof(float), hipMemcpyHostToDevice));
    GF_TRY(pack_weights(*S));
    GF_HIP(hipStreamSynchronize(S->st));
    return GF_OK;
}

/* one forward + backward on a batch (B a multiple of 64) without updating:
 * gradients [E][total] and per-model loss, for gradient checks */
int32_t gf_sg_gradients(gf_sg_model *S, const float *x, const float *y, const float *t, int32_t B, float w_tot,
                        float *grad_out, float *loss_out) {
    if (!S || !x || !y || !t || B <= 0 || B % 64) { set_error("gf_sg_gradients: invalid arguments"); return GF_ERR_ARG; }
    StreamScope scope(S->st);   /* buffers (re)allocated here belong to the model's stream */
    GF_TRY(ensure_batch(*S, B));
    DevBuf<float> dx, dy, dt;
    GF_TRY(stage_rows(*S, x, y, t, B, dx, dy, dt));
    GF_HIP(hipMemsetAsync(S->loss.p, 0, S->E * sizeof(float), S->st));
    GF_TRY(train_step(*S, dx.p, dy.p, dt.p, nullptr, B, 0.0f, w_tot, false));
    if (grad_out) GF_TRY(readback(grad_out, S->g.p, (size_t)S->E * S->lay.total * sizeof(float), S->st));
    if (loss_out) GF_TRY(readback(loss_out, S->loss.p, S->E * sizeof(float), S->st));
    GF_HIP(hipStreamSynchronize(S->st));
    return GF_OK;
}

/* epochs over n examples (host arrays), mini-batches of B drawn in the
 * order given by `order` (n ints per epoch, or NULL for 0..n-1); returns
 * the mean loss per epoch (averaged over models) */
int32_t gf_sg_train(gf_sg_model *S, const float *x, const float *y, const float *t, int32_t n, int32_t epochs,
                    int32_t B, float lr, float w_tot, const int32_t *order, float *epoch_loss) {
    if (!S || !x || !y || !t || n < B || B <= 0 || B % 64 || epochs <= 0) { set_error("gf_sg_train: invalid arguments"); return GF_ERR_ARG; }
    StreamScope scope(S->st);   /* buffers (re)allocated here belong to the model's stream */
    GF_TRY(ensure_batch(*S, B));
    /* stage the whole training set on the device once */
    DevBuf<float> dx, dy, dt;
    DevBuf<int32_t> dord;
    GF_TRY(stage_rows(*S, x, y, t, n, dx, dy, dt));
    const int nb = n / B;
    std::vector<float> lossv(S->E);
    if (order) {
        GF_TRY(dord.alloc((size_t)epochs * n));
        GF_HIP(hipMemcpyAsync(dord.p, order, (size_t)epochs * n * sizeof(int32_t), hipMemcpyHostToDevice, S->st));
    }
    for (int e = 0; e < epochs; e++) {
        GF_HIP(hipMemsetAsync(S->loss.p, 0, S->E * sizeof(float), S->st));
        for (int b = 0; b < nb; b++) {
            if (order)
                GF_TRY(train_step(*S, dx.p, dy.p, dt.p, dord.p + (size_t)e * n + (size_t)b * B, B, lr, w_tot, true));
            else
                GF_TRY(train_step(*S, dx.p + (size_t)b * B * 6, dy.p + (size_t)b * B * NBINS, dt.p + (size_t)b * B, nullptr, B,
                                  lr, w_tot, true));
        }
        GF_HIP(hipMemcpyAsync(lossv.data(), S->loss.p, S->E * sizeof(float), hipMemcpyDeviceToHost, S->st));
        GF_HIP(hipStreamSynchronize(S->st));
        if (epoch_loss) {
            float s = 0.f;
            for (float v : lossv) s += v;
            epoch_loss[e] = s / S->E / nb;
        }
    }
    GF_HIP(hipStreamSynchronize(S->st));
    return GF_OK;
}

/* ensemble prediction for n inputs: mean normalised SFS (bins 1..99),
 * mean log-total and the ensemble disagreement per input.  A batch's outputs
 * ([cnt][99], [cnt], [cnt], contiguous) come back in one copy.  Batches of up
 * to 65,536 inputs alternate between two output buffers: while batch i is
 * computed on the model's stream, batch i - 1 is read back on the copy
 * stream (each waits for the other through events); a single batch is read
 * back on the model's stream itself. */
int32_t gf_sg_predict(gf_sg_model *S, const float *x, int32_t n, float *sfs, float *tot, float *dis) {
    if (!S || !x || n <= 0 || !sfs) { set_error("gf_sg_predict: invalid arguments"); return GF_ERR_ARG; }
    StreamScope scope(S->st);   /* buffers (re)allocated here belong to the model's stream */
    const int B = std::min(65536, ((n + MR - 1) / MR) * MR);
    GF_TRY(ensure_predict(*S, B, true));
    const int nb = (n + B - 1) / B;
    struct Events {   /* [0..1] computed, [2..3] read back, per output buffer */
        hipEvent_t e[4] = {nullptr, nullptr, nullptr, nullptr};
        ~Events() { for (auto v : e) if (v) (void)hipEventDestroy(v); }
    } ev;
    if (nb > 1) {
        GF_HIP(S->cst.create());
        for (auto &v : ev.e) GF_HIP(hipEventCreateWithFlags(&v, hipEventDisableTiming));
    }
    for (int i = 0; i <= nb; i++) {
        if (i < nb) {
            const int off = i * B, cnt = std::min(B, n - off), u = i & 1;
            float *out = S->pout.p + (size_t)u * B * POUT;
            if (i >= 2) GF_HIP(hipStreamWaitEvent(S->st, ev.e[2 + u], 0));   /* buffer u read back */
            GF_HIP(hipMemcpyAsync(S->xin.p, x + (size_t)off * 6, (size_t)cnt * 6 * sizeof(float), hipMemcpyHostToDevice, S->st));
            GF_TRY(predict_logits(*S, S->xin.p, cnt, (cnt + MR - 1) / MR * MR));
            GF_TRY(predict_stats(*S, cnt, out, out + (size_t)cnt * NBINS, out + (size_t)cnt * (NBINS + 1)));
            if (nb > 1) GF_HIP(hipEventRecord(ev.e[u], S->st));
        }
        if (i >= 1) {
            const int j = i - 1, off = j * B, cnt = std::min(B, n - off), u = j & 1;
            hipStream_t st = nb > 1 ? (hipStream_t)S->cst : (hipStream_t)S->st;
            if (nb > 1) GF_HIP(hipStreamWaitEvent(st, ev.e[u], 0));
            const ReadPart parts[3] = {{sfs + (size_t)off * NBINS, (size_t)cnt * NBINS * sizeof(float)},
                                       {tot ? tot + off : nullptr, (size_t)cnt * sizeof(float)},
                                       {dis ? dis + off : nullptr, (size_t)cnt * sizeof(float)}};
            GF_TRY(readback_parts(parts, 3, S->pout.p + (size_t)u * B * POUT, st));
            if (nb > 1) GF_HIP(hipEventRecord(ev.e[2 + u], st));
        }
    }
    if (nb > 1) GF_HIP(hipStreamSynchronize(S->cst));
    GF_HIP(hipStreamSynchronize(S->st));
    return GF_OK;
}

/* gf_sg_predict on device memory: x, sfs, log_total and disagreement are
 * device pointers on the model's device (the last two may be NULL); the
 * batches run back to back on the model's stream, each writing its rows of
 * the outputs, and the call returns when they are done. */
int32_t gf_sg_predict_device(gf_sg_model *S, const float *x, int32_t n, float *sfs, float *tot, float *dis) {
    if (!S || !x || n <= 0 || !sfs) { set_error("gf_sg_predict_device: invalid arguments"); return GF_ERR_ARG; }
    int dev = -1;
    GF_HIP(hipGetDevice(&dev));
    for (const void *p : {(const void *)x, (const void *)sfs, (const void *)tot, (const void *)dis}) {
        if (!p) continue;
        hipPointerAttribute_t at{};
        if (hipPointerGetAttributes(&at, p) != hipSuccess || at.type != hipMemoryTypeDevice || at.device != dev) {
            (void)hipGetLastError();
            set_error("gf_sg_predict_device: x, sfs, log_total and disagreement must be memory of the current device");
            return GF_ERR_ARG;
        }
    }
    StreamScope scope(S->st);
    const int B = std::min(65536, ((n + MR - 1) / MR) * MR);
    GF_TRY(ensure_predict(*S, B, false));
    for (int off = 0; off < n; off += B) {
        const int cnt = std::min(B, n - off);
        GF_TRY(predict_logits(*S, x + (size_t)off * 6, cnt, (cnt + MR - 1) / MR * MR));
        GF_TRY(predict_stats(*S, cnt, sfs + (size_t)off * NBINS, tot ? tot + off : nullptr, dis ? dis + off : nullptr));
    }
    GF_HIP(hipStreamSynchronize(S->st));
    return GF_OK;
}

/* raw ensemble logits for n inputs (n a multiple of 64): [E][n][128] */
int32_t gf_sg_forward(gf_sg_model *S, const float *x, int32_t n, float *logits) {
    if (!S || !x || !logits || n <= 0 || n % MR) { set_error("gf_sg_forward: invalid arguments"); return GF_ERR_ARG; }
    StreamScope scope(S->st);   /* buffers (re)allocated here belong to the model's stream */
    GF_TRY(ensure_predict(*S, n, true));
    GF_HIP(hipMemcpyAsync(S->xin.p, x, (size_t)n * 6 * sizeof(float), hipMemcpyHostToDevice, S->st));
    GF_TRY(predict_logits(*S, S->xin.p, n, n));
    GF_TRY(readback(logits, S->logits.p, (size_t)S->E * n * OUT_PAD * sizeof(float), S->st));
    GF_HIP(hipStreamSynchronize(S->st));
    return GF_OK;
}

} /* extern "C" */
