// Skinny bf16 GEMM (the mixer projections) on gfx950 MFMA.
//
// y[b][n] = sum_k W[n][k] * x[b][k] for B activation vectors (decode: one
// token per sequence), W bf16 [N][K] (the reference's weight tensors,
// vx27_pmat.h:6-8), x and y fp32.
//
// The fp32 activations enter the MFMA exactly: each x is split into three
// bf16 parts hi + mid + lo (8 mantissa bits each, 24 in all), and the parts
// of up to 5 vectors are the columns of one MFMA B operand (3*5 <= 15 of the
// 16 columns): one v_mfma_f32_16x16x32_bf16 multiplies 16 weight rows by
// every part of 5 vectors; the products are exact in fp32 and the only
// rounding is the fp32 accumulation, as in a plain fp32 dot product.  More
// vectors go in more such groups: a weight tile loaded once feeds one MFMA
// per group, up to 13 groups (65 vectors) per pass over the weights.
// Output column n of an MFMA depends only on operand column n, so operand
// columns >= 3*B may hold anything: they feed output columns nobody reads.
//
// Layouts:
//   packed activations  [K/32 k-steps][groups][64 lanes][8] bf16: lane (g,n)
//                       of group j (its Bj <= 5 vectors 5j..) at k-step s
//                       holds part n/Bj of vector 5j + n%Bj at k = 32s + 8g + 0..7
//   tiled weights       [K/(32 KG) k-groups][N/16 row blocks][KG][64 lanes][8]
//                       bf16 (KG = 1 by default): lane (g,m) of tile (s, rb)
//                       holds W[16*rb + m][32s + 8g + 0..7].  A wave's A
//                       operand is 1 KiB contiguous and the row blocks of a
//                       k-step are adjacent (a 1 MiB slab for N = 16K rows)
//                       (vx27_hip_pack_weights_bf16 converts row-major W)
//
// More vectors than fit a few groups go in token tiles instead
// (vx_gemv_tok.h), with the same products and sums.  Both weight layouts go
// through gemv_wk_store (vx_gemv_body.h) below that: whole-K
// workgroups with the wave partials reduced in LDS, reading the weights once
// for up to 65 vectors.  Row-major weights (the plain vx27_hip_gemv_bf16
// call) are read as 16 rows x 64 bytes per tile.
#include <algorithm>

#include "vx_gemv_tok.h"

namespace {


// pack activations: grid (K/32, groups), block 64; lane (g,n) of group j
// writes its 8 elements
__global__ __launch_bounds__(64) void pack_x(const float *x, size_t x_stride, int B, uint16_t *out) {
    const int s = blockIdx.x, j = blockIdx.y, lane = threadIdx.x, g = lane >> 4, n = lane & 15;
    const int Bj = min(VX_PACK_GV, B - VX_PACK_GV * j);
    if (n >= 3 * Bj) return;   // padding columns feed unread output columns
    const int p = n / Bj, b = VX_PACK_GV * j + n % Bj;
    const float *xr = x + (size_t)b * x_stride + 32 * s + 8 * g;
    uint16_t v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = vx_bf16_part(xr[e], p);

    uint4 w;
    w.x = v[0] | ((uint32_t)v[1] << 16);
    w.y = v[2] | ((uint32_t)v[3] << 16);
    w.z = v[4] | ((uint32_t)v[5] << 16);
    w.w = v[6] | ((uint32_t)v[7] << 16);
    *(uint4 *)(out + (((size_t)s * gridDim.y + j) * 64 + lane) * 8) = w;
}

// the token layout: grid (K/32, token blocks), block 64; lane (g,n) splits
// its 8 elements of vector 16 j + n into the three tiles
__global__ __launch_bounds__(64) void pack_x_tok(const float *x, size_t x_stride, int B, uint16_t *out) {
    const int s = blockIdx.x, j = blockIdx.y, lane = threadIdx.x, g = lane >> 4, b = 16 * j + (lane & 15);
    if (b >= B) return;   // padding columns feed unread output columns
    const float *xr = x + (size_t)b * x_stride + 32 * s + 8 * g;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = xr[e];
#pragma unroll
    for (int p = 0; p < 3; p++) {
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const uint16_t u = vx_f32_to_bf16(v[e]);
            v[e] = v[e] - vx_bf16_to_f32(u);
            w[e / 2] = e & 1 ? w[e / 2] | ((uint32_t)u << 16) : u;
        }
        *(uint4 *)(out + ((((size_t)s * gridDim.y + j) * 3 + p) * 64 + lane) * 8) = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

// row-major W [N][K] -> tiled; grid (N/16, K/32), block 64
__global__ __launch_bounds__(64) void pack_w(const uint16_t *W, int K, uint16_t *Wt) {
    const int rb = blockIdx.x, s = blockIdx.y, lane = threadIdx.x, g = lane >> 4, m = lane & 15;
    const uint4 v = *(const uint4 *)(W + (size_t)(16 * rb + m) * K + 32 * s + 8 * g);
    *(uint4 *)(Wt + vx_tile_off(s, rb, gridDim.x, vx_gemv_kg(K)) + lane * 8) = v;
}

template <int RB, int G>
__global__ __launch_bounds__(VX_WK_NW * 64) void gemv_wk_store(WkWeights wt, int N, int K, const uint16_t *xp,
                                                              int B, int halves, WkStore epi) {
    vx_gemv_wk_body<RB, G>(wt, N, K, xp, B, halves, epi);
}

template <int RB, int G>
__global__ __launch_bounds__(VX_WK_NW * 64) void gemv_wk_store_x(WkWeights wt, int N, int K, WkRawX x, int B,
                                                                WkStore epi) {
    vx_gemv_wk_body<RB, G>(wt, N, K, x, B, 1, epi);
}

// Epilogue of the token-tile form: the rows into their output segment
// (fp32 or bf16; vec: 16-byte (bf16: 8-byte) aligned).
struct TokStore {
    GemmOut out;
    int vec;
    struct Pre {};
    __device__ __forceinline__ void begin() const {}
    __device__ __forceinline__ Pre load(int, int) const { return {}; }
    __device__ __forceinline__ void store(int n, int b, vx_floatx4_t y, const Pre &) const {
        GemmSeg sg = out.s[0];
#pragma unroll
        for (int t = 1; t < VX_GEMM_SEGS; t++)
            if (t < out.n && n >= 16 * out.s[t].rb0) sg = out.s[t];
        const size_t o = (size_t)b * sg.stride + (n - 16 * sg.rb0);
        if (sg.bf16) {
            uint16_t *yp = (uint16_t *)sg.p + o;
            uint32_t h[4];
#pragma unroll
            for (int e = 0; e < 4; e++) h[e] = vx_f32_to_bf16(y[e]);
            if (vec) *(uint2 *)yp = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
            else
#pragma unroll
                for (int e = 0; e < 4; e++) yp[e] = (uint16_t)h[e];
        } else {
            float *yp = (float *)sg.p + o;
            if (vec) *(vx_floatx4_t *)yp = y;
            else
#pragma unroll
                for (int e = 0; e < 4; e++) yp[e] = y[e];
        }
    }
};

template <int RB>
__global__ __launch_bounds__(512) void gemv_tok_store(TtArgs a, TokStore epi) {
    vx_gemv_tok_body<RB>(a, epi);
}

int gemv_tok(vx27_hip_ctx *ctx, const uint16_t *W, int N, int K, const uint16_t *packed, int B, const GemmOut &out) {
    bool vec = true;   // every segment takes 16-byte (bf16: 8-byte) stores
    for (int q = 0; q < out.n; q++)
        vec = vec && out.s[q].stride % 4 == 0 && ((uintptr_t)out.s[q].p & (out.s[q].bf16 ? 7 : 15)) == 0;
    const TtPlan p = vx_gemv_tok_plan(W, packed, N, K, B, ctx->n_cu);
    VX_TT_DISPATCH(ctx, gemv_tok_store, p, (TokStore{out, vec}));
    return 0;
}

}  // namespace

TtPlan vx_gemv_tok_plan(const uint16_t *W, const uint16_t *xp, int N, int K, int B, int n_cu) {
    TtPlan p = {};
    TtArgs &a = p.a;
    a.W = W; a.xp = xp; a.N = N; a.K = K; a.B = B;
    a.n_tt = (B + VX_TT_B - 1) / VX_TT_B;
    const int nb = N / 16;
    double best = 0.0;
    for (int rb = 1; rb <= VX_TT_MAX_RB; rb++) {
        const int tiles = (nb + rb - 1) / rb * a.n_tt;
        const double t = (double)((tiles + n_cu - 1) / n_cu) * (0.36 + 0.055 * rb);
        if (p.rb == 0 || t < best) {
            best = t;
            p.rb = rb;
            a.n_tiles = tiles;
        }
    }
    a.per_xcd = (a.n_tiles + 7) / 8;
    p.grid = 8 * a.per_xcd;
    return p;
}

WkPlan vx_gemv_wk_plan(int N, int K, int n_cu, int G, bool allow_halves) {
    (void)K;
    const int nb = N / 16;
    WkPlan best = {0, G, 0, 1};
    double best_t = 0.0;
    for (int single = 1; single >= 0 && best.rb == 0; single--)
        for (int halves = 1; halves <= (allow_halves ? 2 : 1); halves++)
            for (int rb = 1; rb <= vx_wk_max_rb(G); rb++) {
                const int wgs = halves * ((nb + rb - 1) / rb);
                if (single && wgs > n_cu) continue;
                // CU time ~ rounds x (rb weight tiles + G operand tiles per
                // k-step, an operand tile from L2 costing about a quarter of
                // a weight tile from HBM) x the share of the k-steps; ties
                // keep whole workgroups, then the smaller rb
                const double t = (double)((wgs + n_cu - 1) / n_cu) * (rb + 0.25 * G) / halves;
                if (best.rb == 0 || t < best_t - 1e-9) {
                    best_t = t;
                    best = {rb, G, wgs, halves};
                }
            }
    return best;
}

int vx_gemv_store_seg(vx27_hip_ctx *ctx, const uint16_t *W, int N, int K, const uint16_t *packed, int B, bool tok,
                      const GemmOut &out, bool zeroed) {
    VX_REQUIRE(N > 0 && N % 16 == 0 && K > 0 && K % 32 == 0 && B >= 1,
               "gemv: N must be a multiple of 16, K of 32, B >= 1 (N=%d K=%d B=%d)", N, K, B);
    if (tok) return gemv_tok(ctx, W, N, K, packed, B, out);
    VX_REQUIRE(B <= VX_PASS_G * VX_PACK_GV, "internal: %d vectors in operand groups", B);
    const WkPlan p = vx_gemv_wk_plan(N, K, ctx->n_cu, vx_pack_groups(B), zeroed && out.n == 1 && !out.s[0].bf16);
    VX_WK_DISPATCH(VX_WK_ALL, ctx, gemv_wk_store, p, (WkWeights{W, 0}), N, K, packed, B, p.halves, (WkStore{out, 0}));
    return 0;
}

bool vx_gemv_takes_x(int B, const float *x, size_t x_stride) {
    return B <= WK_RAW_G * VX_PACK_GV && ((uintptr_t)x & 15) == 0 && x_stride % 4 == 0;
}

int vx_gemv_store_x(vx27_hip_ctx *ctx, const uint16_t *W, int N, int K, const float *x, size_t x_stride, int B,
                    const GemmOut &out) {
    VX_REQUIRE(N > 0 && N % 16 == 0 && K > 0 && K % 32 == 0 && B >= 1 && vx_gemv_takes_x(B, x, x_stride),
               "gemv: bad call on rows (N=%d K=%d B=%d)", N, K, B);
    const WkPlan p = vx_gemv_wk_plan(N, K, ctx->n_cu, vx_pack_groups(B));
    VX_WK_DISPATCH(VX_WK_RB_G1, ctx, gemv_wk_store_x, p, (WkWeights{W, 0}), N, K, (WkRawX{x, x_stride}), B,
                   (WkStore{out, 0}));
    return 0;
}

int vx_gemv_store(vx27_hip_ctx *ctx, const uint16_t *W, int N, int K, const uint16_t *packed, int B, bool tok,
                  float *y, size_t y_stride, bool zeroed) {
    return vx_gemv_store_seg(ctx, W, N, K, packed, B, tok, vx_gemm_out1(y, y_stride), zeroed);
}

size_t vx_pack_bytes(int K, int B, bool tok) {
    if (tok) return (size_t)(K / 32) * ((B + 15) / 16) * 3 * 1024;
    return (size_t)(K / 32) * vx_pack_groups(B) * 64 * 8 * sizeof(uint16_t);
}

int vx_pack(vx27_hip_ctx *ctx, const float *x, size_t x_stride, int B, int K, bool tok, uint16_t *packed) {
    VX_REQUIRE(B >= 1 && K % 32 == 0, "pack: need B >= 1, K %% 32 == 0");
    if (tok)
        VX_LAUNCH(ctx, pack_x_tok, dim3(K / 32, (B + 15) / 16), dim3(64), x, x_stride, B, packed);
    else
        VX_LAUNCH(ctx, pack_x, dim3(K / 32, vx_pack_groups(B)), dim3(64), x, x_stride, B, packed);
    return 0;
}

extern "C" int vx27_hip_pack_weights_bf16(vx27_hip_ctx *ctx, const uint16_t *W, int N, int K, uint16_t *Wt) {
    if (vx_ctx_enter(ctx)) return -1;
    VX_REQUIRE(W && Wt && W != Wt, "vx27_hip_pack_weights_bf16: need distinct source and destination");
    VX_REQUIRE(N > 0 && N % 16 == 0 && K > 0 && K % 32 == 0,
               "vx27_hip_pack_weights_bf16: N must be a multiple of 16 and K of 32");
    VX_LAUNCH(ctx, pack_w, dim3(N / 16, K / 32), dim3(64), W, K, Wt);
    return 0;
}

extern "C" int vx27_hip_gemv_bf16(vx27_hip_ctx *ctx, const uint16_t *W, int N, int K, const float *x,
                                  size_t x_stride, int B, float *y, size_t y_stride) {
    if (vx_ctx_enter(ctx)) return -1;
    VX_REQUIRE(W && x && y, "vx27_hip_gemv_bf16: null pointer");
    VX_REQUIRE(B >= 1, "vx27_hip_gemv_bf16: B must be >= 1 (got %d)", B);
    VX_REQUIRE(N > 0 && N % 16 == 0 && K > 0 && K % 32 == 0,
               "vx27_hip_gemv_bf16: N must be a multiple of 16 and K of 32 (N=%d K=%d)", N, K);
    // one pass over W per 13 groups (65 vectors), each packing its vectors
    const int Bp0 = std::min(B, VX_PASS_G * VX_PACK_GV);
    void *scr;
    // (row-major weights go through the whole-K form at any B: operand groups)
    if (vx_ctx_scratch(ctx, vx_pack_bytes(K, Bp0, false), &scr)) return -1;
    uint16_t *packed = (uint16_t *)scr;
    for (int b0 = 0; b0 < B; b0 += VX_PASS_G * VX_PACK_GV) {
        const int Bp = std::min(B - b0, VX_PASS_G * VX_PACK_GV);
        if (vx_pack(ctx, x + (size_t)b0 * x_stride, x_stride, Bp, K, false, packed)) return -1;
        const WkPlan p = vx_gemv_wk_plan(N, K, ctx->n_cu, vx_pack_groups(Bp));
        VX_WK_DISPATCH(VX_WK_ALL, ctx, gemv_wk_store, p, (WkWeights{W, 1}), N, K, packed, Bp, p.halves,
                       (WkStore{vx_gemm_out1(y, y_stride), b0}));
    }
    return 0;
}
