// Whole-K workgroup GEMV body for the skinny projections (vx_gemv.hip),
// shared with the kernels that put their own epilogue after it
// (vx_layer.hip).
//
// A workgroup of 8 waves owns RB row blocks (16 RB rows) over all of K:
// wave w takes the k-steps w, w + 8, ... (so the waves of a workgroup read
// neighbouring k-step slabs of the tiled weights at any moment) and
// multiplies each weight tile it loads by all G operand groups of the pass
// (one pass over the weights for up to 65 vectors).  Each wave keeps a ring
// of D operand sets: the loads of its next D - 1 k-steps are in flight
// while the MFMAs of the current one run, so that a workgroup keeps about
// 8 D (RB + G) KiB of loads outstanding.  A row's value is fixed as
//   y = y0 + y1,   yh = (hi_h + mid_h) + lo_h,
// where hi_h, mid_h, lo_h are the column sums of waves 4h .. 4h+3 in wave
// order: the 8 partials are summed in LDS as two halves.  A plain-store
// epilogue may instead run the two halves as two workgroups of 4 waves
// that add y0 and y1 into a zeroed output with fp32 atomics: two addends
// commute, so the bits are the same, and the finer grid fills the CUs
// where whole rows would leave some idle.  The sum order is the same
// whatever RB, D, the halves or the number of vectors in the pass.
// (A split of K over workgroups, whose last arrival sums the slices, was
// measured slower on every projection shape of the model, with or without
// device-scope fences.)
#pragma once
#include <type_traits>

#include "vx_gemv.h"

typedef __bf16 vx_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float vx_floatx4_t __attribute__((ext_vector_type(4)));

constexpr int VX_WK_NW = 8;   // waves per workgroup
#ifndef VX_WK_DMAX
#define VX_WK_DMAX 4              // most operand sets in a wave's ring
#endif
#ifndef VX_GEMV_KG
#define VX_GEMV_KG 1              // k-steps per group of the tiled layout (1, 2 or 4)
#endif

static __device__ vx_bf16x8_t vx_wk_zero[64];   // zero operand tile (static storage)

// largest RB for G groups: RB x G accumulator tiles and the operand sets
// within the register budget of 8-wave workgroups
__host__ __device__ constexpr int vx_wk_max_rb(int G) {
    return G == 1 ? 20 : G == 2 ? 16 : G == 3 ? 10 : G == 4 ? 8 : G == 7 ? 4 : G == 10 ? 3 : 2;
}
// operand sets in a wave's ring: as many as fit beside the 4 RB G
// accumulator registers in about 200 (an operand set takes 4 (RB + G); of
// fp32 rows 4 (RB + 2 G), and the split about 40 registers more), 1 ..
// VX_WK_DMAX
__host__ __device__ constexpr int vx_wk_depth(int RB, int G, bool rows) {
    const int d = (200 - 4 * RB * G - (rows ? 40 : 0)) / (4 * (RB + (rows ? 2 : 1) * G));
    return d < 1 ? 1 : d > VX_WK_DMAX ? VX_WK_DMAX : d;
}

// k-steps per group of the tiled weight layout
__host__ __device__ __forceinline__ int vx_gemv_kg(int K) {
    const int nks = K / 32;
    return nks % VX_GEMV_KG == 0 ? VX_GEMV_KG : 1;
}
// element offset of tile (k-step s, row block rb) in the tiled layout
__host__ __device__ __forceinline__ size_t vx_tile_off(int s, int rb, int nb, int kg) {
    return ((size_t)(s / kg) * nb + rb) * kg * 512 + (size_t)(s % kg) * 512;
}

// Weights: tiled (vx27_hip_pack_weights_bf16) or row-major [N][K].
struct WkWeights {
    const uint16_t *W;
    int row_major;
    // this lane's 8 elements of tile (0, rb)
    __device__ __forceinline__ const uint16_t *base(int rb, int nb, int K, int kg, int lane) const {
        return row_major ? W + (size_t)(16 * rb + (lane & 15)) * K + 8 * (lane >> 4)
                         : W + vx_tile_off(0, rb, nb, kg) + lane * 8;
    }
    // offset of k-step s from tile (0, rb)
    __device__ __forceinline__ size_t off(int s, int nb, int kg) const {
        return row_major ? (size_t)s * 32 : (size_t)(s / kg) * nb * kg * 512 + (size_t)(s % kg) * 512;
    }
};

// Summed rows handed to an epilogue: y(r, b) for local row r < rows and
// vector b < B of the pass (groups 0 .. G-1 of the packed operand):
// the nh halves' values added in order (nh = 1 in a half workgroup).
template <int RB, int G>
struct WkRows {
    const float (*c)[16 * RB][16 * G + 1];   // [2][16 RB][16 G + 1]: each half's MFMA output columns
    int B;                                   // vectors in this pass (<= 5 G)
    int nh;                                  // halves summed here (2, or 1 in a half workgroup)
    __device__ __forceinline__ float y(int r, int b) const {
        const int j = b / VX_PACK_GV, bl = b - VX_PACK_GV * j, Bj = min(VX_PACK_GV, B - VX_PACK_GV * j);
        const float *c0 = c[0][r] + 16 * j;
        const float y0 = (c0[bl] + c0[Bj + bl]) + c0[2 * Bj + bl];
        if (nh == 1) return y0;
        const float *c1 = c[1][r] + 16 * j;
        return y0 + ((c1[bl] + c1[Bj + bl]) + c1[2 * Bj + bl]);
    }
};

// Epilogue interface, both called by all threads of the workgroup (rows =
// valid rows from row0, <= 16 RB):
//   Pre prefetch(int row0, int rows, int tid) const      before the K loop:
//       issues the loads the epilogue needs besides the sums (their latency
//       then hides under the loop instead of trailing it)
//   void operator()(int row0, int rows, const WkRows<RB, G> &, int tid, const Pre &) const
// The operand of a pass, as a wave's ring holds it: tiles of the packed
// operand, or (WkRaw, WK_RAW_G groups) the fp32 rows themselves, each lane
// splitting its 8 elements of a k-step into the part that its operand column
// holds.  Reading the rows spares the pack launch; the split is VALU work
// beside the loads that bound the kernel, but every workgroup repeats it and
// it grows with the groups: in_proj 27.6 us against 26.7 + 4.1 of the pack
// with one group, 34.4 against 26.4 + 4.0 with two.
struct WkPacked {
    struct Tile { vx_bf16x8_t v; };
    const vx_bf16x8_t *xb;
    int G;
    __device__ __forceinline__ WkPacked(const uint16_t *xp, int G, int, int lane)
        : xb((const vx_bf16x8_t *)xp + lane), G(G) {}
    __device__ __forceinline__ Tile load(int s, int j, bool live, const vx_bf16x8_t *zt) const {
        return Tile{*(live ? xb + ((size_t)s * G + j) * 64 : zt)};
    }
    __device__ __forceinline__ vx_bf16x8_t get(const Tile &t, int) const { return t.v; }
};
constexpr int WK_RAW_G = 1;
struct WkRawX {           // fp32 rows, 16-byte aligned, a multiple of 4 floats apart
    const float *x;
    size_t stride;
};
struct WkRaw {
    struct Tile { vx_floatx4_t a, b; };
    const float *xr[WK_RAW_G];   // this lane's vector of each group, from k = 8 (lane / 16)
    int part[WK_RAW_G];
    __device__ __forceinline__ WkRaw(const WkRawX &x, int, int B, int lane) {
#pragma unroll
        for (int j = 0; j < WK_RAW_G; j++) {   // (column n: part n / Bj of vector n % Bj; the others feed unread columns)
            const int Bj = min(VX_PACK_GV, max(B - VX_PACK_GV * j, 1)), n = min(lane & 15, 3 * Bj - 1);
            part[j] = n / Bj;
            xr[j] = x.x + (size_t)min(VX_PACK_GV * j + n % Bj, B - 1) * x.stride + 8 * (lane >> 4);
        }
    }
    __device__ __forceinline__ Tile load(int s, int j, bool live, const vx_bf16x8_t *zt) const {
        const vx_floatx4_t *p = live ? (const vx_floatx4_t *)(xr[j] + 32 * (size_t)s) : (const vx_floatx4_t *)zt;
        return Tile{p[0], live ? p[1] : p[0]};
    }
    __device__ __forceinline__ vx_bf16x8_t get(const Tile &t, int j) const {
        typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
        uint32_t u[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float v[2] = {e < 2 ? t.a[2 * e] : t.b[2 * e - 4], e < 2 ? t.a[2 * e + 1] : t.b[2 * e - 3]};
#pragma unroll
            for (int p = 0; p < 3; p++) {   // part p = bf16 of what the earlier parts leave (exact in fp32)
                const uint32_t h = __builtin_bit_cast(uint32_t, (bf16x2_t){(__bf16)v[0], (__bf16)v[1]});
                u[e] = p == 0 || part[j] == p ? h : u[e];
                v[0] = v[0] - __uint_as_float(h << 16);
                v[1] = v[1] - __uint_as_float(h & 0xffff0000u);
            }
        }
        vx_bf16x8_t r;
        __builtin_memcpy(&r, u, 16);
        return r;
    }
};

// One pass covers the B vectors of a packed operand of G groups.  halves = 1: grid ceil(N / 16 RB), block 512;
// halves = 2: grid 2 ceil(N / 16 RB), block 256, workgroup 2i + h running
// waves 4h .. 4h+3 of row group i (the epilogue then gets only its half).
// (The fp32 rows come as X = WkRawX.)
template <int RB, int G, class Epi, class X>
__device__ __forceinline__ void vx_gemv_wk_body(const WkWeights &wt, int N, int K, const X &xp, int B, int halves,
                                                const Epi &epi) {
    typedef typename std::conditional<std::is_same<X, WkRawX>::value, WkRaw, WkPacked>::type Src;
    constexpr int NW = VX_WK_NW, D = vx_wk_depth(RB, G, std::is_same<X, WkRawX>::value);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = halves == 2 ? (int)(blockIdx.x & 1) : 0;
    const int nwp = halves == 2 ? NW / 2 : NW;   // waves in this workgroup
    const int vw = h * (NW / 2) + wave;          // the wave's place in the 8-wave split
    const int rb0 = (halves == 2 ? (int)(blockIdx.x >> 1) : (int)blockIdx.x) * RB, nb = N / 16;
    const int nks = K / 32, kg = vx_gemv_kg(K);
    const int k0 = 0, k1 = nks;
    const int row0 = rb0 * 16;
    const int rows = min(16 * RB, N - row0);
    const auto pre = epi.prefetch(row0, rows, tid);
    vx_floatx4_t acc[RB][G];
#pragma unroll
    for (int r = 0; r < RB; r++)
#pragma unroll
        for (int j = 0; j < G; j++) acc[r][j] = (vx_floatx4_t){0.f, 0.f, 0.f, 0.f};
    const uint16_t *wp[RB];
#pragma unroll
    for (int r = 0; r < RB; r++)   // dead blocks re-read block 0, never stored
        wp[r] = wt.base(rb0 + r < nb ? rb0 + r : 0, nb, K, kg, lane);
    const Src src(xp, G, B, lane);
    // operands of k-step s; past the end (s >= k1) both operands come from
    // a zero tile, so that every path issues the same loads and MFMAs (the
    // waits before each MFMA then leave the later sets in flight) and the
    // extra products add exact zeros
    const vx_bf16x8_t *zt = vx_wk_zero + lane;
    auto load = [&](int s, vx_bf16x8_t(&ao)[RB], typename Src::Tile(&bo)[G]) {
        const bool live = s < k1;
#pragma unroll
        for (int j = 0; j < G; j++) bo[j] = src.load(s, j, live, zt);
        const size_t off = wt.off(s, nb, kg);
#pragma unroll
        for (int r = 0; r < RB; r++) ao[r] = *(live ? (const vx_bf16x8_t *)(wp[r] + off) : zt);
    };
    auto mma = [&](const vx_bf16x8_t(&ao)[RB], const typename Src::Tile(&bo)[G]) {
        vx_bf16x8_t o[G];
#pragma unroll
        for (int j = 0; j < G; j++) o[j] = src.get(bo[j], j);
#pragma unroll
        for (int r = 0; r < RB; r++)
#pragma unroll
            for (int j = 0; j < G; j++)
                acc[r][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ao[r], o[j], acc[r][j], 0, 0, 0);
    };
    // D operand sets in a ring: the loads of the next D - 1 k-steps of this
    // wave are in flight during the MFMAs of the current one (the branches
    // are uniform: s is a wave constant)
    vx_bf16x8_t a[D][RB];
    typename Src::Tile b[D][G];
#pragma unroll
    for (int d = 0; d < D; d++) load(k0 + vw + d * NW, a[d], b[d]);
    for (int s = k0 + vw; s < k1; s += D * NW) {   // whole rounds of D k-steps
#pragma unroll
        for (int d = 0; d < D; d++) {
            mma(a[d], b[d]);
            load(s + (d + D) * NW, a[d], b[d]);
        }
    }
    constexpr int NTL = RB * G;                         // accumulator tiles
    constexpr int RC = NTL < 64 / NW ? NTL : 64 / NW;   // tiles reduced per round (64 KiB of LDS)
    __shared__ vx_floatx4_t red[NW][RC][64];
    __shared__ float ct[2][16 * RB][16 * G + 1];
    const int nh = nwp / 4;   // halves summed in this workgroup
#pragma unroll
    for (int t0 = 0; t0 < NTL; t0 += RC) {
        if (t0) __syncthreads();   // the previous round's partials are read out
#pragma unroll
        for (int q = 0; q < RC; q++)
            if (t0 + q < NTL) red[wave][q][lane] = acc[(t0 + q) / G][(t0 + q) % G];
        __syncthreads();
        for (int t = tid; t < RC * 64; t += nwp * 64) {   // (tile t0 + q, lane l): each half's 4 partials in order
            const int q = t >> 6, l = t & 63, g = l >> 4, m = l & 15;
            const int rj = t0 + q;
            if (rj >= NTL) continue;
            const int r = rj / G, j = rj % G;
            for (int hh = 0; hh < nh; hh++) {
                const vx_floatx4_t v = ((red[4 * hh][q][l] + red[4 * hh + 1][q][l]) + red[4 * hh + 2][q][l]) +
                                       red[4 * hh + 3][q][l];
                // lane (g,m) holds C[4g+i][m]: row 16r + 4g + i, column 16j + m
#pragma unroll
                for (int i = 0; i < 4; i++) ct[hh][16 * r + 4 * g + i][16 * j + m] = v[i];
            }
        }
    }
    __syncthreads();
    epi(row0, rows, WkRows<RB, G>{ct, B, nh}, tid, pre);
}

// Epilogue: row n of vector b0 + b into the output segment that holds row n
// (added with an atomic in a half workgroup: the output, fp32, must then
// start at zero).
struct WkStore {
    GemmOut out;
    int b0;
    struct Pre {};
    __device__ __forceinline__ Pre prefetch(int, int, int) const { return {}; }
    template <int RB, int G>
    __device__ __forceinline__ void operator()(int row0, int rows, const WkRows<RB, G> &c, int tid, const Pre &) const {
        if (out.n == 1 && !out.s[0].bf16) {
            for (int t = tid; t < rows * c.B; t += c.nh * 4 * 64) {
                const int r = t % rows, b = t / rows;
                float *yp = (float *)out.s[0].p + (size_t)(b0 + b) * out.s[0].stride + row0 + r;
                if (c.nh == 1) atomicAdd(yp, c.y(r, b));
                else *yp = c.y(r, b);
            }
            return;
        }
        for (int t = tid; t < rows * c.B; t += c.nh * 4 * 64) {   // (whole workgroups)
            const int r = t % rows, b = t / rows, n = row0 + r;
            GemmSeg sg = out.s[0];
#pragma unroll
            for (int q = 1; q < VX_GEMM_SEGS; q++)
                if (q < out.n && n >= 16 * out.s[q].rb0) sg = out.s[q];
            const size_t o = (size_t)(b0 + b) * sg.stride + (n - 16 * sg.rb0);
            if (sg.bf16) ((uint16_t *)sg.p)[o] = vx_f32_to_bf16(c.y(r, b));
            else ((float *)sg.p)[o] = c.y(r, b);
        }
    }
};
// one fp32 segment
static inline GemmOut vx_gemm_out1(float *y, size_t stride) {
    GemmOut o = {};
    o.n = 1;
    o.s[0] = GemmSeg{0, 0, stride, y};
    return o;
}

// Launch plan for an N x K matrix and a pass of G groups: RB row blocks per
// workgroup, whole (halves = 1, grid ceil(N / 16 RB)) or split in two half
// workgroups (halves = 2, twice the grid, only when allow_halves: an
// epilogue that adds into a zeroed output).  The plan takes the shape that
// best balances the CUs in one round of workgroups (several rounds only
// when no single-round plan exists).
struct WkPlan {
    int rb, g, grid, halves;
};
WkPlan vx_gemv_wk_plan(int N, int K, int n_cu, int G, bool allow_halves = false);

// every (RB, G) instance: RB = 1 .. vx_wk_max_rb(G)
#define VX_WK_RB_G1(X, ...)                                                                                      \
    X(1, 1, __VA_ARGS__) X(2, 1, __VA_ARGS__) X(3, 1, __VA_ARGS__) X(4, 1, __VA_ARGS__) X(5, 1, __VA_ARGS__)    \
    X(6, 1, __VA_ARGS__) X(7, 1, __VA_ARGS__) X(8, 1, __VA_ARGS__) X(9, 1, __VA_ARGS__) X(10, 1, __VA_ARGS__)   \
    X(11, 1, __VA_ARGS__) X(12, 1, __VA_ARGS__) X(13, 1, __VA_ARGS__) X(14, 1, __VA_ARGS__)                     \
    X(15, 1, __VA_ARGS__) X(16, 1, __VA_ARGS__) X(17, 1, __VA_ARGS__) X(18, 1, __VA_ARGS__)                     \
    X(19, 1, __VA_ARGS__) X(20, 1, __VA_ARGS__)
#define VX_WK_RB_G2(X, ...)                                                                                      \
    X(1, 2, __VA_ARGS__) X(2, 2, __VA_ARGS__) X(3, 2, __VA_ARGS__) X(4, 2, __VA_ARGS__) X(5, 2, __VA_ARGS__)    \
    X(6, 2, __VA_ARGS__) X(7, 2, __VA_ARGS__) X(8, 2, __VA_ARGS__) X(9, 2, __VA_ARGS__) X(10, 2, __VA_ARGS__)   \
    X(11, 2, __VA_ARGS__) X(12, 2, __VA_ARGS__) X(13, 2, __VA_ARGS__) X(14, 2, __VA_ARGS__)                     \
    X(15, 2, __VA_ARGS__) X(16, 2, __VA_ARGS__)
#define VX_WK_RB_G3(X, ...)                                                                                      \
    X(1, 3, __VA_ARGS__) X(2, 3, __VA_ARGS__) X(3, 3, __VA_ARGS__) X(4, 3, __VA_ARGS__) X(5, 3, __VA_ARGS__)    \
    X(6, 3, __VA_ARGS__) X(7, 3, __VA_ARGS__) X(8, 3, __VA_ARGS__) X(9, 3, __VA_ARGS__) X(10, 3, __VA_ARGS__)
#define VX_WK_RB_G47(X, ...)                                                                                     \
    X(1, 4, __VA_ARGS__) X(2, 4, __VA_ARGS__) X(3, 4, __VA_ARGS__) X(4, 4, __VA_ARGS__) X(5, 4, __VA_ARGS__)    \
    X(6, 4, __VA_ARGS__) X(7, 4, __VA_ARGS__) X(8, 4, __VA_ARGS__) X(1, 7, __VA_ARGS__) X(2, 7, __VA_ARGS__)    \
    X(3, 7, __VA_ARGS__) X(4, 7, __VA_ARGS__)
#define VX_WK_RB_BIG(X, ...)                                                                                     \
    X(1, 10, __VA_ARGS__) X(2, 10, __VA_ARGS__) X(3, 10, __VA_ARGS__) X(1, 13, __VA_ARGS__) X(2, 13, __VA_ARGS__)
// (up to 7 groups: all that an input projection hands over as operand groups)
#define VX_WK_G7(X, ...)                                                                                         \
    VX_WK_RB_G1(X, __VA_ARGS__) VX_WK_RB_G2(X, __VA_ARGS__) VX_WK_RB_G3(X, __VA_ARGS__) VX_WK_RB_G47(X, __VA_ARGS__)
#define VX_WK_ALL(X, ...) VX_WK_G7(X, __VA_ARGS__) VX_WK_RB_BIG(X, __VA_ARGS__)

// Launch KERNEL<rb, g>(args...) for a plan (grid plan.grid, block 512 or
// 256 for half workgroups), of the instances LIST.
#define VX_WK_CASE(R, GG, ctx, KERNEL, p, ...)                                                                 \
    case GG * 64 + R:                                                                                          \
        VX_LAUNCH_NAMED(ctx, #KERNEL, (KERNEL<R, GG>), dim3((unsigned)p.grid),                                 \
                        dim3(VX_WK_NW * 64 / p.halves), __VA_ARGS__);                                          \
        break;
#define VX_WK_DISPATCH(LIST, ctx, KERNEL, p, ...)                                             \
    do {                                                                                      \
        switch (p.g * 64 + p.rb) {                                                            \
            LIST(VX_WK_CASE, ctx, KERNEL, p, __VA_ARGS__)                                     \
            default: VX_REQUIRE(false, "internal: no GEMV instance for rb=%d g=%d", p.rb, p.g); \
        }                                                                                     \
    } while (0)
