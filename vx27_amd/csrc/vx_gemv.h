// Internal interface of the skinny bf16 GEMM (vx_gemv.hip), shared with the
// kernels that produce its packed operand or fuse its reduction epilogue.
#pragma once
#include "vx_common.h"

// Packed activations: vectors go in groups of VX_PACK_GV, each group one
// 16-column MFMA B operand (the three parts of its <= 5 vectors): layout
// [K/32 k-steps][groups][64 lanes][8] bf16.
// Above three groups the count is rounded up to 4, 7, 10 or 13 (65 vectors, one
// pass over the weights): the padding groups are never written and feed output
// columns nobody reads.
constexpr int VX_PACK_GV = 5;
constexpr int VX_PASS_G = 13;   // most groups: 65 vectors
__host__ __device__ __forceinline__ int vx_pack_groups(int B) {
    const int g = (B + VX_PACK_GV - 1) / VX_PACK_GV;
    return g <= 3 ? g : g <= 4 ? 4 : g <= 7 ? 7 : g <= 10 ? 10 : 13;
}
// The token layout (tok) holds 16 vectors a tile, each part a tile of its own
// (vx_gemv_tok.h): [K/32][ceil(B/16)][3 parts][64 lanes][8] bf16, lane (g, n)
// of block j: vector 16 j + n, k 8g .. 8g+7.
// The wide input projections take it from 36 vectors, where the operand groups
// are padded from 8 to 10 and the GQA qkv's whole-K workgroups (2 row blocks)
// no longer fit one round of CUs (in_proj's run two rounds from 5 groups on and
// three with 13).  The narrow output projections, whose whole-K grid fits one round at any
// group count, take it where the groups would need a second pass over the
// weights.  Kernel trace, us, weights streamed from HBM, groups / token tiles:
//   vectors       36        40        64         65         66         129
//   in_proj    95 / 64   97 / 65  127 / 75  127 / 124  153 / 124  220 / 172
//   GQA qkv    65 / 47   66 / 46   82 / 50   82 / 84   104 / 83   144 / 111
//   out_proj                                            59 / 45    83 / 48
// (65 pads to two 64-vector tiles and only breaks even there; the layer calls at
// 65 still gain, 252 -> 243 us and 164 -> 157.)  With 7 groups, 21 to 35
// vectors, in_proj takes 65 to 69 us and qkv 42; token tiles were not timed
// there.  out_proj at 64 vectors, one layer's weights in the last-level cache:
// 36 us against 40 in token tiles.
constexpr int VX_TOK_IN = 36, VX_TOK_OUT = VX_PASS_G * VX_PACK_GV + 1;
__host__ __device__ __forceinline__ bool vx_tok_in(int B) { return B >= VX_TOK_IN; }
__host__ __device__ __forceinline__ bool vx_tok_out(int B) { return B >= VX_TOK_OUT; }
size_t vx_pack_bytes(int K, int B, bool tok);
// x [B][K] (row stride x_stride) -> packed MFMA B operand (three bf16 parts).
int vx_pack(vx27_hip_ctx *ctx, const float *x, size_t x_stride, int B, int K, bool tok, uint16_t *packed);
// Output in segments: rows n >= 16 rb0 of segment s (up to the next
// segment's) go to p[r * stride + n - 16 rb0], as fp32 or as bf16 (round to
// nearest even, vx_f32_to_bf16).  Segment 0 starts at rb0 = 0.
struct GemmSeg {
    int rb0, bf16;
    size_t stride;
    void *p;
};
constexpr int VX_GEMM_SEGS = 4;
struct GemmOut {
    int n;
    GemmSeg s[VX_GEMM_SEGS];
};
// y_b[n] = sum over k of W[n][k] x_b[k] for tiled W and a packed x of B
// vectors into output segments (operand groups of up to 65 vectors: one pass
// over W; tok: token tiles, one per 64 vectors).  Each row's sum order
// is the same for any B and either layout.  zeroed: the output (fp32) holds
// zeros, written by an earlier kernel on the stream, so the rows may be added
// in two halves.
int vx_gemv_store_seg(vx27_hip_ctx *ctx, const uint16_t *W, int N, int K, const uint16_t *packed, int B, bool tok,
                      const GemmOut &out, bool zeroed = false);
// whether vx_gemv_store_x takes B vectors of K elements, x_stride apart
bool vx_gemv_takes_x(int B, const float *x, size_t x_stride);
// the same products and bits from the fp32 rows themselves, with no packed operand
int vx_gemv_store_x(vx27_hip_ctx *ctx, const uint16_t *W, int N, int K, const float *x, size_t x_stride, int B,
                    const GemmOut &out);
// the same to y[b*y_stride + n]
int vx_gemv_store(vx27_hip_ctx *ctx, const uint16_t *W, int N, int K, const uint16_t *packed, int B, bool tok,
                  float *y, size_t y_stride, bool zeroed = false);

// The projection of R tokens at once (vx_gemm.hip): y[r][n] = sum over k of
// W[n][k] x_r[k] for tiled W, fp32 x rows (x as two bf16 parts; K % 64 == 0,
// 16-byte aligned rows).
// ws: vx_gemm_ws_bytes of device scratch (the tokens packed for the MFMAs,
// and the partial sums of a last round of tiles split along k)
int vx_gemm_store(vx27_hip_ctx *ctx, const uint16_t *W, int N, int K, const float *x, size_t x_stride, int R,
                  float *y, size_t y_stride, void *ws);
size_t vx_gemm_ws_bytes(int N, int K, int R, int n_cu);
// whether vx_gemm_store takes this shape (else the GEMV passes)
bool vx_gemm_fits(int N, int K, int R, const float *x, size_t x_stride, const float *y, size_t y_stride);
int vx_gemm_store_seg(vx27_hip_ctx *ctx, const uint16_t *W, int N, int K, const float *x, size_t x_stride, int R,
                      const GemmOut &out, void *ws);
bool vx_gemm_fits_seg(int N, int K, int R, const float *x, size_t x_stride, const GemmOut &out);
constexpr int VX_GEMM_MIN_ROWS = 256;   // layer prefills use the GEMM from this many tokens (one token tile)
// The GEMM's packed tokens: one 32 KiB image per (256-token tile, 32-wide
// k-step), [token tiles][K/32][32 KiB].  In an image, part p (0: hi =
// bf16(x), 1: lo = bf16(x - hi)) of token t's elements 8g .. 8g+7 sit in
// 1 KiB block ((t % 256) / 16) * 2 + p, 16-byte unit g * 16 + ((t % 16) ^ 2g)
// (the XOR spreads a token column over the LDS banks).  Byte offset of the
// hi unit holding element k of token t (its lo unit: + 1024):
__host__ __device__ __forceinline__ size_t vx_gemm_pack_unit(int t, int k, int K) {
    const int tb = (t >> 4) & 15, n = t & 15, g = (k >> 3) & 3;
    return ((size_t)(t >> 8) * (K >> 5) + (k >> 5)) * 32768 + (size_t)tb * 2048 + (size_t)(g * 16 + (n ^ (g << 1))) * 16;
}
size_t vx_gemm_pack_bytes(int K, int R);
// vx_gemm_store_seg on tokens already packed (xp: vx_gemm_pack_bytes, rows
// past R may hold anything: they feed only outputs that are not stored);
// ws: vx_gemm_ws_bytes.
int vx_gemm_store_packed(vx27_hip_ctx *ctx, const uint16_t *W, int N, int K, const char *xp, int R,
                         const GemmOut &out, void *ws);

// Part p (0 = hi, 1 = mid, 2 = lo) of the exact three-way bf16 split of x:
// hi = bf16(x), mid = bf16(x - hi), lo = bf16(x - hi - mid); each difference
// is exact in fp32.
__device__ __forceinline__ uint16_t vx_bf16_part(float x, int p) {
    uint16_t h = vx_f32_to_bf16(x);
    for (int q = 0; q < p; q++) {
        x = x - vx_bf16_to_f32(h);
        h = vx_f32_to_bf16(x);
    }
    return h;
}

// Element k of vector b (of B) as the three parts of the packed operand:
// group j = b / 5 holds its Bj <= 5 vectors' part p of vector b' at column
// p*Bj + b' (token layout: tile p of token block b / 16 at column b % 16).
__device__ __forceinline__ void vx_pack_store(uint16_t *packed, int B, bool tok, int b, int k, float x) {
    size_t base;   // of part 0
    int step;      // elements between parts
    if (tok) {
        base = (((size_t)(k >> 5) * ((B + 15) >> 4) + (b >> 4)) * 3 * 64 + ((k >> 3) & 3) * 16 + (b & 15)) * 8 + (k & 7);
        step = 512;
    } else {
        const int G = vx_pack_groups(B), j = b / VX_PACK_GV, bl = b - VX_PACK_GV * j;
        base = (((size_t)(k >> 5) * G + j) * 64 + ((k >> 3) & 3) * 16 + bl) * 8 + (k & 7);
        step = min(VX_PACK_GV, B - VX_PACK_GV * j) * 8;
    }
    uint16_t h = vx_f32_to_bf16(x);
    packed[base] = h;
    x = x - vx_bf16_to_f32(h);
    h = vx_f32_to_bf16(x);
    packed[base + step] = h;
    x = x - vx_bf16_to_f32(h);
    packed[base + 2 * step] = vx_f32_to_bf16(x);
}
