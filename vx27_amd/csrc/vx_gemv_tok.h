// Token-tile form of the skinny projections, for more vectors than a few
// MFMA operand groups hold (VX_TOK_IN, VX_TOK_OUT: vx_gemv.h): the same exact three-part
// products and the same bits as the whole-K GEMV (vx_gemv_body.h), shared
// with the kernels that put their own epilogue after it (vx_layer.hip).
//
// The operand holds 16 vectors a tile, their three bf16 parts as three
// tiles ([K/32][token blocks][3][1 KiB], written by pack_x_tok and
// vx_pack_store), so a lane has all parts of its outputs and combines them in
// registers.  A workgroup owns RB row blocks x 64 vectors over all of K:
// per k-step, RB weight tiles and 12 operand tiles come into LDS by
// direct-to-LDS loads, and wave q of a group multiplies the RB weight tiles
// by the three parts of token block q (every operand tile is read from LDS
// once, each weight tile four times).  A step's operands are read from LDS
// during the step before, and the loads of a later step are issued between
// the step's MFMAs, which hide their scalar work.
//
// Sum order (that of the GEMV): the k-steps of class c are c, c + 8, ...;
// each class is summed in one MFMA chain, half h adds the sums of classes
// 4h .. 4h+3 in order, part by part, and y = y0 + y1 with
// yh = (hi_h + mid_h) + lo_h.  So K is walked class by class: the class sum
// sits in one accumulator set and the half's running sum in another, added
// four times a kernel.  Waves 0-3 walk half 0 and waves 4-7 half 1 (each group
// with its own k-step, their parts of a ring slot side by side), and y1 meets
// y0 in LDS.
//
// Measured (kernel trace): in_proj 16480 x 5120 of 64 vectors 70 us against
// 93 as whole-K workgroups (515 of them, of 2 row blocks: three rounds) with one
// layer's weights in the last-level cache, 75 against 127 from HBM; of 187
// vectors 153 us against 284 in three passes, out_proj 5120 x 6144 of 187
// vectors 53 us against 117.  A step takes about 0.36 + 0.055 RB us over the
// three rounds of 187 vectors, 0.042 RB of it MFMA; one round of 64 vectors
// takes 20 us more than its 80 steps would, unaccounted for.  Timing-only
// copies of the 187-token layer (252 us): without the loads 209, without the
// MFMAs 235, without the LDS reads 245.  The operand as fp32 tiles split in registers (a third less L2
// traffic) was slower, 85 us at 64 vectors: the split's VALU work adds to a
// step.  Separate, deeper rings for the weights changed nothing.
#pragma once
#include "vx_gemv_body.h"
#include "vx_lds.h"

typedef uint32_t vx_u32x4_t __attribute__((ext_vector_type(4)));
constexpr int VX_TT_B = 64;          // vectors per workgroup
constexpr int VX_TT_MAX_RB = 6;
// steps in the LDS ring (160 KiB in all)
__host__ __device__ constexpr int vx_tt_nst(int RB) { return 160 / (2 * (RB + 12)); }

// Epilogue interface:
//   void begin() const                          every thread, before the loop
//   Pre load(int n, int b) const                waves 0-3, before the sums are complete
//   void store(int n, int b, vx_floatx4_t y, const Pre &) const
// y: rows n .. n + 3 of vector b (n % 4 == 0, n < N, b < B).
// grid 8 per_xcd, block 512.  Tile t: vectors 64 (t % n_tt) .., row blocks
// RB (t / n_tt) ..; a contiguous range of tiles runs on each XCD (workgroup
// i on XCD i % 8), so the token tiles of a row range share its weights in
// that XCD's L2.
struct TtArgs {
    const uint16_t *W;    // tiled
    const uint16_t *xp;   // packed, token layout
    int N, K, B;
    int n_tt, n_tiles, per_xcd;
};

template <int RB, class Epi>
__device__ __forceinline__ void vx_gemv_tok_body(const TtArgs &a, const Epi &epi) {
    constexpr int NST = vx_tt_nst(RB);
    constexpr int TILES = RB + 12;                  // 1 KiB tiles per group and step
    constexpr int STAGE = 2 * TILES * 1024;
    constexpr int DB = TILES / 4, DX = TILES % 4;   // loads of a wave and step: DB, one more for waves < DX
    constexpr int ND = DB + (DX ? 1 : 0);
    __shared__ __attribute__((aligned(16))) char smem[NST * STAGE];
    epi.begin();
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), q = wave & 3, h = wave >> 2;
    const int tile = (int)(blockIdx.x & 7) * a.per_xcd + (int)(blockIdx.x >> 3);
    if (tile >= a.n_tiles) return;   // (the whole workgroup)
    const int rb0 = tile / a.n_tt * RB, tb0 = tile % a.n_tt * 4;
    const int nb = a.N / 16, ntb = (a.B + 15) / 16, nks = a.K / 32, nmax = (nks + 7) / 8, T = 4 * nmax;

    // this wave's loads of a step: tiles q, q + 4, ... of [RB weight tiles,
    // 12 operand tiles].  k-steps past the end re-read the last one, row and
    // token blocks past the end the last ones (loaded, never used).
    uint32_t off[ND];
#pragma unroll
    for (int d = 0; d < ND; d++) {
        const int t = q + 4 * d, u = t < RB ? 0 : t - RB, j = min(u / 3, 3), p = u - 3 * j;
        off[d] = lane * 16 + 1024 * (t < RB ? min(rb0 + t, nb - 1) * vx_gemv_kg(a.K) : min(tb0 + j, ntb - 1) * 3 + min(p, 2));
    }
    const uint32_t ring0 = vx_lds_addr(smem) + (h * TILES + q) * 1024;
    const int kg = vx_gemv_kg(a.K);
    const uint32_t wstep = (uint32_t)(nb * kg) * 1024, xstep = (uint32_t)ntb * 3072;   // bytes of kg, of one k-step
    int dc = 0, di = 0, slot = 0;   // class (of the half) and index of the next step to load, its ring slot
    struct Next {                   // where that step's tiles are and go
        const char *w, *x;
        uint32_t dst;
    };
    auto next = [&] {
        const uint32_t s = min(4 * h + dc + 8 * di, nks - 1);
        return Next{(const char *)a.W + (uint64_t)(s / kg) * wstep + (s % kg) * 1024, (const char *)a.xp + (uint64_t)s * xstep,
                    ring0 + slot * STAGE};
    };
    auto dma = [&](const Next &nx, int d) {   // load d of the step
        if (d == DB && q >= DX) return;
        vx_dma16(q + 4 * d < RB ? nx.w : nx.x, off[d], nx.dst + d * 4096);
    };
    auto dma_next = [&] {
        slot = slot == NST - 1 ? 0 : slot + 1;
        if (++di == nmax) {   // (past the last step: the loads land in slots nobody reads)
            di = 0;
            if (dc < 3) dc++;
        }
    };
    auto landed = [&] {   // the step after the next one's loads: only the later ones' in flight
        if (DX && q < DX) __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"((DB + 1) * (NST - 2)) : "memory");
        else __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(DB * (NST - 2)) : "memory");
    };

    vx_floatx4_t acc[RB][3], sum[RB][3];
#pragma unroll
    for (int r = 0; r < RB; r++)
#pragma unroll
        for (int p = 0; p < 3; p++) sum[r][p] = acc[r][p] = (vx_floatx4_t){0.f, 0.f, 0.f, 0.f};
    const char *rd = smem + h * (TILES * 1024) + lane * 16;
    int cur = 0;
    auto read = [&](vx_u32x4_t(&x)[3], vx_u32x4_t(&w)[RB]) {   // the next unread step's operands
        const char *sb = rd + cur * STAGE;
#pragma unroll
        for (int p = 0; p < 3; p++) x[p] = *(const vx_u32x4_t *)(sb + (RB + 3 * q + p) * 1024);
#pragma unroll
        for (int r = 0; r < RB; r++) w[r] = *(const vx_u32x4_t *)(sb + r * 1024);
        cur = cur == NST - 1 ? 0 : cur + 1;
    };
    int c = 0, i = 0;
    // one step on operands read during the step before; meanwhile the next
    // step's are read and a later step's loads go into the slot whose
    // operands every wave holds
    auto step = [&](const vx_u32x4_t(&x)[3], const vx_u32x4_t(&w)[RB], vx_u32x4_t(&xn)[3], vx_u32x4_t(&wn)[RB]) {
        read(xn, wn);
        const Next nx = next();
        if (4 * h + c + 8 * i < nks) {   // (wave-uniform)
#pragma unroll
            for (int r = 0; r < (RB > ND ? RB : ND); r++) {
                __builtin_amdgcn_sched_barrier(0);
                if (r < RB)
#pragma unroll
                    for (int p = 0; p < 3; p++)
                        acc[r][p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(vx_bf16x8_t, w[r]), __builtin_bit_cast(vx_bf16x8_t, x[p]), acc[r][p], 0,
                            0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (r < ND) dma(nx, r);
            }
        } else {
#pragma unroll
            for (int d = 0; d < ND; d++) dma(nx, d);
        }
        dma_next();
        if (++i == nmax) {   // the class's sums into the half's
            i = 0;
#pragma unroll
            for (int r = 0; r < RB; r++)
#pragma unroll
                for (int p = 0; p < 3; p++) {
                    sum[r][p] = c == 0 ? acc[r][p] : sum[r][p] + acc[r][p];
                    acc[r][p] = (vx_floatx4_t){0.f, 0.f, 0.f, 0.f};
                }
            c++;
        }
        __builtin_amdgcn_sched_barrier(0);
        landed();
        vx_lds_barrier();
    };
    for (int st = 0; st < NST; st++) {
#pragma unroll
        for (int d = 0; d < ND; d++) dma(next(), d);
        dma_next();
    }
    landed();
    vx_lds_barrier();
    vx_u32x4_t xa[3], xb[3], wa[RB], wb[RB];
    read(xa, wa);
    vx_lds_barrier();
    for (int t = 0; t < T; t += 2) {   // (T is a multiple of 4)
        step(xa, wa, xb, wb);
        step(xb, wb, xa, wa);
    }
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the last, unused loads)
    const int b = tb0 * 16 + 16 * q + (lane & 15), n0 = 16 * rb0 + 4 * (lane >> 4);
    typename Epi::Pre pre[RB];
    if (h == 0 && b < a.B)
#pragma unroll
        for (int r = 0; r < RB; r++)
            if (rb0 + r < nb) pre[r] = epi.load(n0 + 16 * r, b);
    vx_floatx4_t y[RB];
#pragma unroll
    for (int r = 0; r < RB; r++) y[r] = (sum[r][0] + sum[r][1]) + sum[r][2];
    __syncthreads();   // every wave's loads have landed: the ring is free
    vx_floatx4_t *ex = (vx_floatx4_t *)smem;
    if (h == 1)
#pragma unroll
        for (int r = 0; r < RB; r++) ex[(r * 4 + q) * 64 + lane] = y[r];
    __syncthreads();
    if (h == 1) return;
#pragma unroll
    for (int r = 0; r < RB; r++) y[r] += ex[(r * 4 + q) * 64 + lane];
    if (b >= a.B) return;
#pragma unroll
    for (int r = 0; r < RB; r++)
        if (rb0 + r < nb) epi.store(n0 + 16 * r, b, y[r], pre[r]);
}

// Row blocks per workgroup for an N x K projection of B vectors: the RB with
// the least rounds of workgroups x time of a step (0.36 + 0.055 RB us).
struct TtPlan {
    int rb, grid;
    TtArgs a;
};
TtPlan vx_gemv_tok_plan(const uint16_t *W, const uint16_t *xp, int N, int K, int B, int n_cu);

#define VX_TT_CASE(R, ctx, KERNEL, p, ...)                                                                     \
    case R: VX_LAUNCH_NAMED(ctx, #KERNEL, (KERNEL<R>), dim3((unsigned)p.grid), dim3(512), p.a, __VA_ARGS__); break;
#define VX_TT_DISPATCH(ctx, KERNEL, p, ...)                                                                    \
    do {                                                                                                       \
        switch (p.rb) {                                                                                        \
            VX_TT_CASE(1, ctx, KERNEL, p, __VA_ARGS__) VX_TT_CASE(2, ctx, KERNEL, p, __VA_ARGS__)              \
            VX_TT_CASE(3, ctx, KERNEL, p, __VA_ARGS__) VX_TT_CASE(4, ctx, KERNEL, p, __VA_ARGS__)              \
            VX_TT_CASE(5, ctx, KERNEL, p, __VA_ARGS__) VX_TT_CASE(6, ctx, KERNEL, p, __VA_ARGS__)              \
            default: VX_REQUIRE(false, "internal: no token-tile instance for rb=%d", p.rb);                    \
        }                                                                                                      \
    } while (0)
