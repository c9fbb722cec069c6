// gfx950 weight-streaming GEMM of few rows: y[M,N] = x[M,K] @ W[N,K]^T, M <= 64
// (128 with x in fragment layout).
//
// The decode projections are pure weight streaming (each weight byte is
// used M times; compute is nothing next to the 8 TB/s HBM pull), and
// hipBLASLt reaches 1.8-4.6 TB/s on these shapes with a ~19 us floor on
// qkv/o (profiles/r01_decode_step_budget.md).  Two other hand-written
// kernels lose too:
//  * fragment-direct (skinny_gemm.hip): MFMA-layout loads are 16 B/lane at
//    8 KB row stride -> cold misses over-fetched ~4x;
//  * LDS-staged: full-line loads, but __syncthreads() carries a vmcnt(0),
//    draining the prefetch ring every chunk -> 87% SQ_WAIT_ANY.
//
// This kernel removes the conflict at the source: the weights are OURS,
// so they are stored pre-packed in MFMA fragment order (ops/hip.py
// pack_weight).  Element W[n][k] with n = t*32+r, k = b*64 + j*16 + h*8 + e
// lives at packed uint4 index ((t*NB + b)*4 + j)*64 + (h*32 + r), e inside.
// The stream is then PERFECTLY linear: each wave reads consecutive 1 KiB
// vectors (full 128 B line use per instruction), tagged non-temporal
// (a stream read once: -18% landed traffic), with no LDS staging, no barriers, and a register prefetch of
// one to four 4 KiB iterations per wave.
//
// Geometry: grid (N/32, ksplit) x 512 threads (8 waves).  The K/64
// k-blocks are range-partitioned over ksplit*8 waves (uneven ranges OK:
// any K%64==0, N%32==0).  Wave partials meet in a single
// end-of-kernel LDS reduce (the ONE barrier, after all streaming).
// ksplit>1 writes fp32 partials; the consumer folds them, or the block that
// arrives last at a tile (x in fragment layout, or with a fused epilogue), or
// k_wstream_combine (+bias).
#include <algorithm>
#include "act.h"
#include "tile_mma.h"

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

union u4bf8 { u32x4 u; bf16x8 v; };

// Pure-stream diagnostic: same grid/geometry/addressing as the GEMM but
// only the nt weight loads (no x, no MFMA) — measures this geometry's
// load-path ceiling so kernel iterations know what they are chasing.
__global__ __launch_bounds__(512) void k_wstream_pure(
    float* __restrict__ sink, const u32x4* __restrict__ wp,
    int N, int K, int ksplit)
{
    const int t = blockIdx.x;
    const int ks = blockIdx.y;
    const int wid = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    const int NB = K >> 6;
    const int GW = ksplit * 8;
    const int gw = ks * 8 + wid;
    const int b_lo = (int)(((int64_t)gw * NB) / GW);
    const int b_hi = (int)(((int64_t)(gw + 1) * NB) / GW);
    unsigned acc = 0;
    const u32x4* wq = wp + (((int64_t)t * NB + b_lo) * 4) * 64 + lane;
    for (int b = b_lo; b < b_hi; ++b, wq += 256) {
        u32x4 v0 = __builtin_nontemporal_load(wq);
        u32x4 v1 = __builtin_nontemporal_load(wq + 64);
        u32x4 v2 = __builtin_nontemporal_load(wq + 128);
        u32x4 v3 = __builtin_nontemporal_load(wq + 192);
        acc ^= v0.x ^ v0.w ^ v1.x ^ v1.w ^ v2.x ^ v2.w ^ v3.x ^ v3.w;
    }
    if (acc == 0xDEADBEEFu) sink[0] = 1.f;   // never: keeps loads alive
}

extern "C" int wstream_pure_bf16(void* sink, const void* wp, int N, int K,
                                 int ksplit, hipStream_t stream)
{
    dim3 grid(N / 32, ksplit);
    k_wstream_pure<<<grid, 512, 0, stream>>>(
        (float*)sink, (const u32x4*)wp, N, K, ksplit);
    return (int)hipGetLastError();
}

// MT: m-tiles of 32 rows (up to 64 rows, 128 in fragment layout).
// DEPTH: weights under way per wave, in 4 KiB iterations.
// XLDS == 2: x in fragment layout (the decode chain).  A CU's loads are what
// bounds it, x counted: rows past M repeat row M - 1, so few rows cost few
// cache lines.  1, 2 or 4 iterations ahead for 32 rows (frag_depth), in registers
// for two blocks a CU; 2 for 64, where one block a CU with two of x under way
// beats two with one (37888 x 3584: 70 us against 79).  28672 x 4096 with its
// norm and activation: 46 us before for any M, now 44 for 32 rows, 39 for 1.
// XLDS (requires MT==1): stage the x fragments through a wave-PRIVATE
// LDS tile instead of loading them in MFMA layout.  The direct x
// fragment load is 32 rows x 16 B at an 8 KB stride = 32 cache-line
// requests per instruction x 4 per iteration; staged, the global x read
// is 4 coalesced instructions (8 lines each), a dense ds_write and a
// minimum-phase swizzled ds_read (u = r*8 + (c ^ (r&7))).  Wave-private
// double-buffered tiles -> NO barrier anywhere in the stream (a
// __syncthreads would drain vmcnt and kill the weight prefetch).
// GU (requires ksplit==1): fused gate_up@SwiGLU.  The weights are
// packed with gate and up INTERLEAVED (tile t = 16 gate rows f=t*16..+16
// then the 16 matching up rows — ops/hip.py pack_weight_gu), so each
// block's 32-column output tile holds the (gate, up) pairs of 16 ffn
// columns; the epilogue computes silu(g)*u (GU == 2: gelu_tanh(g)*u) and stores [M, 16] of the
// activation directly.  Kills the separate swiglu kernel (9.7 us x 32
// layers/step) and the gate_up intermediate round-trip.
// Fused-rmsnorm chain extensions (all nullable; tp=1 decode path):
//  * rstd_parts/rstd_nt: per-tile sum-of-squares partials of the RAW
//    residual state x (written by the producing GEMM's epilogue).  The
//    epilogue scales row m by rstd[m] = rsqrt(sum*inv_h + eps) — the
//    norm WEIGHT is folded into the packed W at pack time, so
//    y = rmsnorm(x)@W' without any rmsnorm kernel in the step.
//  * res_in/sq_parts: epilogue adds the residual stream (in-place safe:
//    each (m,n) is read+written by exactly one block) and emits this
//    block's sum-of-squares partials for the NEXT GEMM's rstd.
// RoPE/KV-append epilogue bundle (RP=1 qkv GEMM): the packed qkv
// weight is PAIR-ORDERED per head (16 lo-dims then their 16 hi-dims,
// ops/hip.py pack_weight_qkv_rope), so each 32-col output tile holds
// complete rotation pairs; the epilogue rotates q/k with the host
// cos/sin tables and writes k/v straight into the paged KV pool —
// the separate rope_append kernel (8.6 us x layers/step) disappears from the decode step.
struct RopeEpi {
    const float* cos_t;   // [max_ctx, 64]
    const float* sin_t;
    const int* pos;       // [M] position of this step's token
    const int* slot;      // [M] kv slot per row
    const int* ptab;      // page table [slots, maxp]
    bf16* kp;             // this layer's K pool base
    bf16* vp;
    int nl, nkl, psz, maxp;
};

template <int MT, int DEPTH = 1, int XLDS = 0, int GU = 0, int RP = 0>
__global__ __launch_bounds__(512, XLDS == 2 && MT == 1 ? 4 : 1)
void k_wstream_gemm(
    bf16* __restrict__ y,            // [M, N] (ksplit == 1)
    float* __restrict__ part,        // [ksplit, M, N] (ksplit > 1)
    const bf16* __restrict__ x,      // [M, K], row stride xs
    const u32x4* __restrict__ wp,    // packed W (see header)
    const bf16* __restrict__ bias,   // [N] or null (ksplit==1 path)
    int M, int N, int K, int64_t xs, int ksplit,
    const float* __restrict__ rstd_parts, int rstd_nt, float inv_h,
    float eps, const bf16* __restrict__ res_in,
    float* __restrict__ sq_parts, RopeEpi rp = {}, int yfrag = 0,
    int* __restrict__ sem = nullptr) // ksplit > 1: tickets per tile, zero
{
    const int t = blockIdx.x;              // n-tile (32 cols of y)
    const int ks = blockIdx.y;
    const int tid = threadIdx.x;
    const int wid = tid >> 6;
    const int lane = tid & 63;
    const int row = lane & 31;
    const int khalf = (lane >> 5) * 8;

    const int NB = K >> 6;                 // 64-elem k-blocks
    const int GW = ksplit * 8;             // waves across k
    const int gw = ks * 8 + wid;
    const int b_lo = (int)(((int64_t)gw * NB) / GW);
    const int b_hi = (int)(((int64_t)(gw + 1) * NB) / GW);

    // clamp so every lane loads valid x rows (rows >= M never stored;
    // per-lane conditional loads would branch+vmcnt(0) per chunk)
    const int ar0 = row < M ? row : (M > 0 ? M - 1 : 0);
    const bf16* xr0 = x + (int64_t)ar0 * xs + khalf;
    const bf16* xr1 = nullptr;
    if (MT == 2) {
        const int r1 = 32 + row;
        const int ar1 = r1 < M ? r1 : (M - 1);
        xr1 = x + (int64_t)ar1 * xs + khalf;
    }

    // dynamic LDS: 32 KiB (wave-partial reduce) or 64 KiB (XLDS adds 8
    // double-buffered 4 KiB wave-private x tiles, reduce space aliased —
    // a __syncthreads separates the stream epoch from the reduce epoch)
    extern __shared__ __align__(16) char smem[];

    f32x16 acc[MT] = {};
    // rmsnorm scale of the raw-residual input: this row's sq partials from
    // the producing GEMM, FL lanes a row, several loads at a time.  The frag
    // path loads them beside its first weights: behind the stream they cost
    // every block another memory latency (gate-up 46.7 us for 32 rows, 41.6
    // for 1; now 43.8 and 38.9).
    constexpr int FL = MT == 1 ? 16 : MT == 2 ? 8 : 4;
    float rsum = 0.f;
    auto fold = [&]() {
        const int m = tid / FL;
        if (!rstd_parts || m >= M) return;
        const float* p = rstd_parts + (int64_t)m * rstd_nt;
        int i = tid % FL;
        for (; i + 7 * FL < rstd_nt; i += 8 * FL) {
            float v[8];
            #pragma unroll
            for (int k = 0; k < 8; k++) v[k] = p[i + k * FL];
            #pragma unroll
            for (int k = 0; k < 8; k++) rsum += v[k];
        }
        for (; i + FL < rstd_nt; i += 2 * FL) rsum += p[i] + p[i + FL];
        if (i < rstd_nt) rsum += p[i];
    };
    if (XLDS == 2 && b_lo < b_hi) {
        // x in fragment layout: DEPTH iterations of weights and up to two of x
        // are under way.  The first round may begin before b_lo: those slots
        // repeat the first block and are not used.
        const u32x4* wq = wp + (int64_t)t * NB * 256 + lane;
        const u32x4* xq[MT];
        #pragma unroll
        for (int m = 0; m < MT; m++)
            xq[m] = reinterpret_cast<const u32x4*>(x) + (int64_t)m * K * 4
                    + (lane & 32) + min(row, max(M - m * 32, 1) - 1);
        constexpr int XS = DEPTH < 2 ? 1 : 2;
        u4bf8 w[DEPTH][4], xr[XS][MT][4];
        auto ldw = [&](int s, int b) {
            #pragma unroll
            for (int j = 0; j < 4; j++)
                w[s][j].u = __builtin_nontemporal_load(
                    wq + (int64_t)b * 256 + j * 64);
        };
        auto ldx = [&](int s, int b) {
            #pragma unroll
            for (int m = 0; m < MT; m++)
                #pragma unroll
                for (int j = 0; j < 4; j++)
                    xr[s][m][j].u = xq[m][(int64_t)b * 256 + j * 64];
        };
        auto mul = [&](int s) {
            #pragma unroll
            for (int j = 0; j < 4; j++)
                #pragma unroll
                for (int m = 0; m < MT; m++)
                    acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        xr[s % XS][m][j].v, w[s][j].v, acc[m], 0, 0, 0);
        };
        int b = b_hi - (b_hi - b_lo + DEPTH - 1) / DEPTH * DEPTH;
        #pragma unroll
        for (int s = 0; s < DEPTH; s++) ldw(s, max(b + s, b_lo));
        #pragma unroll
        for (int s = 0; s < XS; s++) ldx(s, max(b + s, b_lo));
        fold();
        for (; b + DEPTH < b_hi; b += DEPTH) {
            #pragma unroll
            for (int s = 0; s < DEPTH; s++) {
                if (b + s >= b_lo) mul(s);
                ldw(s, b + s + DEPTH);
                ldx(s % XS, max(b + s + XS, b_lo));
            }
        }
        #pragma unroll
        for (int s = 0; s < DEPTH; s++) {
            if (b + s >= b_lo) mul(s);
            if (s + XS < DEPTH) ldx(s % XS, max(b + s + XS, b_lo));
        }
    }
    f32x16 &acc0 = acc[0], &acc1 = acc[MT - 1];     // XLDS < 2: MT <= 2
    if (XLDS != 2 && b_lo < b_hi) {
        const u32x4* wbase = wp + ((int64_t)t * NB * 4) * 64 + lane;
        u4bf8 br[DEPTH][4];
        bf16x8 a0[2], a1[2], a2[2], a3[2];
        auto lda16 = [&](bf16x8* d, int b, int off) {
            const int64_t k = ((int64_t)b << 6) + off;
            d[0] = *reinterpret_cast<const bf16x8*>(xr0 + k);
            if (MT == 2) d[1] = *reinterpret_cast<const bf16x8*>(xr1 + k);
        };
        auto lda = [&](int b) {
            lda16(a0, b, 0);
            lda16(a1, b, 16);
            lda16(a2, b, 32);
            lda16(a3, b, 48);
        };
        // clamped prefetch: an over-the-end refill re-reads a valid block
        // instead of branching per lane (the tail never computes it)
        auto ldb = [&](int s, int b) {
            const u32x4* q = wbase + (int64_t)(b < b_hi ? b : b_hi - 1)
                                     * 256;
            br[s][0].u = __builtin_nontemporal_load(q);
            br[s][1].u = __builtin_nontemporal_load(q + 64);
            br[s][2].u = __builtin_nontemporal_load(q + 128);
            br[s][3].u = __builtin_nontemporal_load(q + 192);
        };
        auto compute = [&](int s) {
            bf16x8 vb0 = br[s][0].v, vb1 = br[s][1].v;
            bf16x8 vb2 = br[s][2].v, vb3 = br[s][3].v;
            acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                a0[0], vb0, acc0, 0, 0, 0);
            acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                a1[0], vb1, acc0, 0, 0, 0);
            acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                a2[0], vb2, acc0, 0, 0, 0);
            acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                a3[0], vb3, acc0, 0, 0, 0);
            if (MT == 2) {
                acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    a0[1], vb0, acc1, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    a1[1], vb1, acc1, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    a2[1], vb2, acc1, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    a3[1], vb3, acc1, 0, 0, 0);
            }
        };
        if (XLDS == 1) {
            // --- LDS-staged x fragments (MT==1 only) ---
            bf16x8 xs4[4];
            auto glbx = [&](int b) {       // 4 coalesced reads: 8 rows
                const int64_t kk = (int64_t)b << 6;   // x 128 B each
                #pragma unroll
                for (int i2 = 0; i2 < 4; i2++) {
                    const int r = 8 * i2 + (lane >> 3);
                    const int ar = r < M ? r : (M - 1);
                    xs4[i2] = *reinterpret_cast<const bf16x8*>(
                        x + (int64_t)ar * xs + kk + (lane & 7) * 8);
                }
            };
            auto dswx = [&](int s) {       // dense swizzled tile write
                bf16* tile = reinterpret_cast<bf16*>(smem)
                             + (wid * 2 + s) * 2048;
                #pragma unroll
                for (int i2 = 0; i2 < 4; i2++) {
                    const int u = (8 * i2 + (lane >> 3)) * 8
                                  + ((lane & 7) ^ (lane >> 3));
                    *reinterpret_cast<bf16x8*>(tile + u * 8) = xs4[i2];
                }
            };
            auto dsrx = [&](int s) {       // min-phase fragment reads
                const bf16* tile = reinterpret_cast<const bf16*>(smem)
                                   + (wid * 2 + s) * 2048;
                const int r = lane & 31;
                #pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int c = j * 2 + (lane >> 5);
                    const int u = r * 8 + (c ^ (r & 7));
                    bf16x8 v = *reinterpret_cast<const bf16x8*>(
                        tile + u * 8);
                    if (j == 0) a0[0] = v;
                    else if (j == 1) a1[0] = v;
                    else if (j == 2) a2[0] = v;
                    else a3[0] = v;
                }
            };
            ldb(0, b_lo);
            glbx(b_lo);
            dswx(0);
            int b = b_lo;
            for (; b < b_hi - 1; ++b) {
                const int s = (b - b_lo) & 1;
                dsrx(s);
                compute(0);
                ldb(0, b + 1);
                glbx(b + 1);
                dswx(s ^ 1);
            }
            dsrx((b - b_lo) & 1);
            compute(0);
        } else {
            ldb(0, b_lo);
            if (DEPTH == 2) ldb(1, b_lo + 1);
            lda(b_lo);
            int b = b_lo;
            if (DEPTH == 1) {
                for (; b < b_hi - 1; ++b) {
                    compute(0);
                    ldb(0, b + 1);
                    lda(b + 1);
                }
                compute(0);
            } else {
                for (; b + 2 < b_hi; b += 2) {
                    compute(0);
                    ldb(0, b + 2);
                    lda(b + 1);
                    compute(1);
                    ldb(1, b + 3);
                    lda(b + 2);
                }
                compute(0);
                if (b + 1 < b_hi) {
                    lda(b + 1);
                    compute(1);
                }
            }
        }
    }

    // ---- reduce 8 wave partials through LDS (aliases the x tiles: the
    // barrier closes the streaming epoch before anyone writes) ----
    float (*red8)[32][32] = reinterpret_cast<float (*)[32][32]>(smem);
    float* rstd_sh = reinterpret_cast<float*>(
        smem + (XLDS == 1 ? 16 * 4096 : 8 * 32 * 32 * 4));
    if (rstd_parts) {
        if (XLDS != 2 || b_lo >= b_hi) fold();
        #pragma unroll
        for (int off = FL / 2; off; off >>= 1)
            rsum += __shfl_down(rsum, off, 64);
        if (tid % FL == 0 && tid / FL < MT * 32)
            rstd_sh[tid / FL] = rsqrtf(rsum * inv_h + eps);
    }
    if (GU) {
        const int F = N >> 1;                  // ffn width
        #pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            __syncthreads();
            #pragma unroll
            for (int r = 0; r < 16; r++) {
                const int crow = (r & 3) + 8 * (r >> 2) + 4 * (lane >> 5);
                red8[wid][crow][lane & 31] = acc[mt][r];
            }
            __syncthreads();
            const int m = tid >> 4, c = tid & 15;  // 512 thr = 32 x 16
            const int gm = m + mt * 32;
            if (gm < M) {
                float sg = 0.f, su = 0.f;
                #pragma unroll
                for (int wv = 0; wv < 8; wv++) {
                    sg += red8[wv][m][c];
                    su += red8[wv][m][c + 16];
                }
                if (rstd_parts) {              // pre-silu: nonlinear
                    const float rs = rstd_sh[gm];
                    sg *= rs;
                    su *= rs;
                }
                const float z = GU == 2 ? gelu_arg(sg) : sg;
                const float act = (sg / (1.f + __expf(-z))) * su;
                const int fc = t * 16 + c;
                y[yfrag ? (int64_t)mt * 32 * F + frag_off(m, fc)
                        : (int64_t)gm * F + fc] = __float2bfloat16(act);
            }
        }
        return;
    }
    if (RP) {
        const int qt = rp.nl * 4, kt = rp.nkl * 4;   // tiles per section
        #pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            __syncthreads();
            #pragma unroll
            for (int r = 0; r < 16; r++) {
                const int crow = (r & 3) + 8 * (r >> 2) + 4 * (lane >> 5);
                red8[wid][crow][lane & 31] = acc[mt][r];
            }
            __syncthreads();
            if (t < qt + kt) {
                // pair-packed q/k tile: cols {d0+c, d0+64+c}, c<16
                const int m = tid >> 4, c = tid & 15;
                const int gm = m + mt * 32;
                if (gm < M) {
                    const int sec_t = t < qt ? t : t - qt;
                    const int head = sec_t >> 2;
                    const int d0 = (sec_t & 3) * 16;
                    float lo = 0.f, hi = 0.f;
                    #pragma unroll
                    for (int wv = 0; wv < 8; wv++) {
                        lo += red8[wv][m][c];
                        hi += red8[wv][m][c + 16];
                    }
                    if (rstd_parts) {
                        const float rs = rstd_sh[gm];
                        lo *= rs;
                        hi *= rs;
                    }
                    if (bias) {  // bias is pair-reordered like the pack
                        lo += __bfloat162float(bias[t * 32 + c]);
                        hi += __bfloat162float(bias[t * 32 + 16 + c]);
                    }
                    const int p = rp.pos[gm];
                    const float co = rp.cos_t[p * 64 + d0 + c];
                    const float si = rp.sin_t[p * 64 + d0 + c];
                    const float rlo = lo * co - hi * si;
                    const float rhi = hi * co + lo * si;
                    if (t < qt) {          // q: standard layout in y
                        bf16* qr = y + (int64_t)gm * N + head * 128;
                        qr[d0 + c] = __float2bfloat16(rlo);
                        qr[64 + d0 + c] = __float2bfloat16(rhi);
                    } else {               // k: rotated, straight to pool
                        const int pg = rp.ptab[rp.slot[gm] * rp.maxp
                                               + p / rp.psz];
                        bf16* dst = rp.kp
                            + (((int64_t)pg * rp.nkl + head) * rp.psz
                               + p % rp.psz) * 128;
                        dst[d0 + c] = __float2bfloat16(rlo);
                        dst[64 + d0 + c] = __float2bfloat16(rhi);
                    }
                }
            } else {
                // v tile (plain 32-col order): straight to pool, no rope
                const int sec_t = t - qt - kt;
                const int head = sec_t >> 2;
                const int d0 = (sec_t & 3) * 32;
                #pragma unroll
                for (int ee = 0; ee < 2; ee++) {
                    const int e = tid + ee * 512;
                    const int mr = e >> 5, n = e & 31;
                    const int gm = mr + mt * 32;
                    if (gm < M) {
                        float sv = 0.f;
                        #pragma unroll
                        for (int wv = 0; wv < 8; wv++)
                            sv += red8[wv][mr][n];
                        if (rstd_parts) sv *= rstd_sh[gm];
                        if (bias)
                            sv += __bfloat162float(bias[t * 32 + n]);
                        const int p = rp.pos[gm];
                        const int pg = rp.ptab[rp.slot[gm] * rp.maxp
                                               + p / rp.psz];
                        bf16* dst = rp.vp
                            + (((int64_t)pg * rp.nkl + head) * rp.psz
                               + p % rp.psz) * 128;
                        dst[d0 + n] = __float2bfloat16(sv);
                    }
                }
            }
        }
        return;
    }
    __syncthreads();
    const int n0 = t * 32;
    // row mr of half mt, column n: the finished sum
    auto finish = [&](int mt, int mr, int n, float s) {
        const int m = mr + mt * 32;
        if (rstd_parts) s *= rstd_sh[m];
        if (bias) s += __bfloat162float(bias[n0 + n]);
        const int64_t yo = yfrag ? (int64_t)mt * 32 * N + frag_off(mr, n0 + n)
                                 : (int64_t)m * N + n0 + n;
        if (res_in) s += __bfloat162float(res_in[yo]);
        y[yo] = __float2bfloat16(s);
        return s * s;
    };
    // this block's sums of squares of half mt, from two values per thread
    auto squares = [&](int mt, const float* rsq) {
        __syncthreads();
        float (*sqt)[32] = reinterpret_cast<float (*)[32]>(smem);
        sqt[tid >> 5][tid & 31] = rsq[0];          // rows 0..15
        sqt[(tid >> 5) + 16][tid & 31] = rsq[1];   // rows 16..31
        __syncthreads();
        if (tid < 32) {
            float s = 0.f;
            #pragma unroll
            for (int n2 = 0; n2 < 32; n2++) s += sqt[tid][n2];
            // m-major [M][n_tiles]: the consumer's fold walks tiles
            // CONTIGUOUSLY (a tile-major layout cost 1 float per
            // 128 B line and ~3 us per consumer block)
            sq_parts[(int64_t)(tid + mt * 32) * gridDim.x + t] = s;
        }
        if (mt + 1 < MT) __syncthreads();          // sqt reused
    };
    #pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        if (mt) __syncthreads();
        #pragma unroll
        for (int r = 0; r < 16; r++) {
            const int crow = (r & 3) + 8 * (r >> 2) + 4 * (lane >> 5);
            red8[wid][crow][lane & 31] = acc[mt][r];
        }
        __syncthreads();
        float rsq[2] = {0.f, 0.f};
        #pragma unroll
        for (int ee = 0; ee < 2; ee++) {
            const int e = tid + ee * 512;
            const int mr = e >> 5, n = e & 31;
            const int m = mr + mt * 32;
            if (m >= M) continue;
            float s = 0.f;
            #pragma unroll
            for (int wv = 0; wv < 8; wv++) s += red8[wv][mr][n];
            if (ksplit == 1 && y) rsq[ee] = finish(mt, mr, n, s);
            else if (sem)
                __hip_atomic_store(
                    part + (((int64_t)ks * gridDim.x + t) * MT + mt) * 1024
                        + e, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            else part[((int64_t)ks * M + m) * N + n0 + n] = s;
        }
        if (sq_parts && ksplit == 1) squares(mt, rsq);
    }
    if (!sem) return;
    // The block that arrives last adds up the parts of its tile, in their
    // order.  Parts are written through and read past the caches (agent
    // scope), so the ticket needs no write-back of a whole L2: the stores
    // have only to be complete before it is drawn.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int* drawn = reinterpret_cast<int*>(smem);
    if (tid == 0)
        *drawn = __hip_atomic_fetch_add(sem + t, 1, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*drawn != ksplit - 1) return;
    if (tid == 0)                        // ready for the next launch
        __hip_atomic_store(sem + t, 0, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    // Two parts at a time, all of a thread's values under way together and no
    // load under a condition: each would wait for the one before it (4096 x
    // 4096, 32, 64 and 128 rows: 12.0, 16.7 and 23.5 us before, 11.2, 14.6 and
    // 19.9 now).
    float total[MT][2] = {};
    for (int k = 0; k < ksplit; k += 2) {
        float v[2][MT][2];
        #pragma unroll
        for (int q = 0; q < 2; q++)
            #pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                #pragma unroll
                for (int ee = 0; ee < 2; ee++)
                    v[q][mt][ee] = __hip_atomic_load(
                        part + (((int64_t)min(k + q, ksplit - 1) * gridDim.x
                                 + t) * MT + mt) * 1024 + tid + ee * 512,
                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        #pragma unroll
        for (int mt = 0; mt < MT; ++mt)
            #pragma unroll
            for (int ee = 0; ee < 2; ee++) {
                total[mt][ee] += v[0][mt][ee];
                if (k + 1 < ksplit) total[mt][ee] += v[1][mt][ee];
            }
    }
    #pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        float rsq[2] = {0.f, 0.f};
        #pragma unroll
        for (int ee = 0; ee < 2; ee++) {
            const int e = tid + ee * 512;
            if ((e >> 5) + mt * 32 < M)
                rsq[ee] = finish(mt, e >> 5, e & 31, total[mt][ee]);
        }
        if (sq_parts) squares(mt, rsq);
    }
}

// ---------------------------------------------------------------------------
// Many columns for rows in fragment layout: gate-up and logits.  A CU has 32 KB
// of loads under way, in order: rows that L2 has queue behind weights from
// memory, 50 GB/s of both together, 136 of what L2 has alone.  So k_wstream_gemm,
// which reads all rows for every 32 columns, loads three units of 4 KB a step of
// 64 with 64 rows, five with 128, of which one is weights.  Here a block takes CW
// tiles of 32 columns and its waves share the activations through LDS, CW + rows
// / 32 units for CW of weights: groups of CW waves walk parts of K, a step of
// every group staged at a time, the next one on its way in registers.  The
// barrier leaves loads in flight.  With norm and activation, us for 64 and 128
// rows:
//   16384 x 4096   35 and 43 (k_wstream_gemm 35 and 48)
//   28672 x 4096   46 and 53 (63 and 88; library product, norm and activation 63)
//   37888 x 3584   52 and 58 (78 and 109; four and eight tiles 69 and 70)
//  128256 x 4096  185 and 209 (265 and 380)
// Products in parts stay with k_wstream_gemm: adding up the parts of several
// tiles costs one block more than the loads saved (4096 x 14336, 128 rows:
// 56 us against 49).  More weights or activations under way give nothing.

// parts of K that a block's waves walk side by side: eight to twelve waves, of
// seven tiles fourteen
static constexpr __host__ __device__ int wide_parts(int cw)
{
    return cw == 3 ? 3 : cw == 2 ? 4 : cw == 8 ? 1 : 2;
}
// bytes for two stages of activations, or the sums that follow them
static constexpr __host__ __device__ int wide_lds(int mt, int cw)
{
    const int kw = wide_parts(cw);
    const int x = 2 * kw * mt * 4096, sums = cw * kw * 32 * 33 * 4;
    return x > sums ? x : sums;
}

template <int MT, int CW, int GU>
__global__ __launch_bounds__(CW * wide_parts(CW) * 64, 1) void k_wide(
    bf16* __restrict__ y,            // [M, N], with GU [M, N / 2]
    const u32x4* __restrict__ x,     // [M, K] in fragment layout
    const u32x4* __restrict__ wp, int M, int N, int K,
    const float* __restrict__ rstd_parts, int rstd_nt, float inv_h,
    float eps, int yfrag)
{
    constexpr int KW = wide_parts(CW), BS = CW * KW * 64;
    constexpr int DEPTH = CW > 2 && CW < 8 ? 2 : 4;
    static_assert(BS >= 512);                  // lanes for the rows' sums
    constexpr int STAGE = KW * MT * 256;               // 16-byte units
    constexpr int NX = (STAGE + BS - 1) / BS;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cw = wid % CW, kw = wid / CW;
    const int NB = K >> 6, tiles = N >> 5;
    auto from = [&](int k) { return k * NB / KW; };
    const int lo = from(kw), hi = from(kw + 1), steps = (NB + KW - 1) / KW;
    // tiles past the last repeat it and are not stored
    const int t0 = blockIdx.x * CW;
    const u32x4* wq = wp + (int64_t)min(t0 + cw, tiles - 1) * NB * 256 + lane;
    extern __shared__ __align__(16) char smem[];
    u32x4* x_s = reinterpret_cast<u32x4*>(smem);       // [2][KW][MT][256]
    float* rstd_s = reinterpret_cast<float*>(smem + wide_lds(MT, CW));

    u4bf8 w[DEPTH][4];
    u32x4 xr[NX];
    f32x16 acc[MT] = {};
    auto ldw = [&](int s, int b) {
        #pragma unroll
        for (int j = 0; j < 4; j++)
            w[s][j].u = __builtin_nontemporal_load(
                wq + (int64_t)min(b, max(hi, 1) - 1) * 256 + j * 64);
    };
    // Where a wave's 64 come from is the same for all of them, so it is worked out
    // in scalar registers.  Pointers kept per lane took 0.5 us of 14 before the
    // first weights (11008 x 1024) and with 128 rows 170 us instead of 160 (57344 x
    // 8192).
    auto ldx = [&](int r) {
        #pragma unroll
        for (int i = 0; i < NX; i++) {
            const int e = i * BS + wid * 64, u = e >> 8;   // group and row tile
            if (STAGE % BS && i == NX - 1 && u >= KW * MT) break;
            const int b = min(from(u / MT) + r, NB - 1);
            xr[i] = x[(int64_t)(u % MT) * K * 4 + (int64_t)b * 256 + (e & 255)
                      + lane];
        }
    };
    auto stx = [&](int r) {
        #pragma unroll
        for (int i = 0; i < NX; i++)
            if (i * BS + tid < STAGE)
                x_s[(r & 1) * STAGE + i * BS + tid] = xr[i];
    };
    #pragma unroll
    for (int s = 0; s < DEPTH; s++) ldw(s, lo + s);
    // where four parts begin takes longer than the weights' (1 to 3 % of 11008 x
    // 1024); of fewer the compiler's order is better, by 2 us of 490 in four layers
    // of 37 rows
    if constexpr (KW == 4) __builtin_amdgcn_sched_barrier(0);
    ldx(0);
    // the norm's partial sums, FL lanes a row
    constexpr int FL = MT == 1 ? 16 : MT == 2 ? 8 : 4;
    float rsum = 0.f;
    if (rstd_parts && tid / FL < M) {
        const float* p = rstd_parts + (int64_t)(tid / FL) * rstd_nt;
        int i = tid % FL;
        for (; i + 7 * FL < rstd_nt; i += 8 * FL) {
            float v[8];
            #pragma unroll
            for (int k = 0; k < 8; k++) v[k] = p[i + k * FL];
            #pragma unroll
            for (int k = 0; k < 8; k++) rsum += v[k];
        }
        for (; i < rstd_nt; i += FL) rsum += p[i];
    }
    stx(0);
    ldx(1);
    lds_barrier();
    for (int r0 = 0; r0 < steps; r0 += DEPTH) {
        #pragma unroll
        for (int s = 0; s < DEPTH; s++) {
            const int r = r0 + s;
            if (r >= steps) break;
            if (r + 1 < steps) stx(r + 1);
            ldx(r + 2);
            const u32x4* xb = x_s + (r & 1) * STAGE + kw * MT * 256 + lane;
            if (lo + r < hi) {
                #pragma unroll
                for (int j = 0; j < 4; j++)
                    #pragma unroll
                    for (int m = 0; m < MT; m++)
                        acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            __builtin_bit_cast(bf16x8, xb[m * 256 + j * 64]),
                            w[s][j].v, acc[m], 0, 0, 0);
            }
            ldw(s, lo + r + DEPTH);
            lds_barrier();
        }
    }
    #pragma unroll
    for (int off = FL / 2; off; off >>= 1) rsum += __shfl_down(rsum, off, 64);
    if (tid % FL == 0 && tid / FL < MT * 32)
        rstd_s[tid / FL] = rstd_parts ? rsqrtf(rsum * inv_h + eps) : 1.f;

    // 32 rows at a time: the groups' sums meet in LDS
    float (*sum)[32][33] = reinterpret_cast<float (*)[32][33]>(smem);
    #pragma unroll
    for (int m = 0; m < MT; m++) {
        __syncthreads();
        #pragma unroll
        for (int r = 0; r < 16; r++)
            sum[wid][(r & 3) + 8 * (r >> 2) + 4 * (lane >> 5)][lane & 31] =
                acc[m][r];
        __syncthreads();
        auto total = [&](int c, int mr, int n) {
            float s = 0.f;
            #pragma unroll
            for (int k = 0; k < KW; k++) s += sum[k * CW + c][mr][n];
            return s;
        };
        constexpr int C = GU ? 16 : 32;                // columns of a tile
        const int cols = GU ? N / 2 : N;
        for (int e = tid; e < CW * 32 * C; e += BS) {
            const int n = e % C, c = e / C % CW, mr = e / (C * CW);
            const int row = m * 32 + mr, col = (t0 + c) * C + n;
            if (row >= M || t0 + c >= tiles) continue;
            float v = total(c, mr, n) * rstd_s[row];
            if (GU) {
                const float up = total(c, mr, n + 16) * rstd_s[row];
                const float z = GU == 2 ? gelu_arg(v) : v;
                v = v / (1.f + __expf(-z)) * up;
            }
            y[yfrag ? (int64_t)m * 32 * cols + frag_off(mr, col)
                    : (int64_t)row * cols + col] = __float2bfloat16(v);
        }
    }
}

// Tiles a block: those with which the busiest of 256 CUs is done first, in units
// of 4 KB a step of K.  A block of k_wide loads its tiles and all rows, or waits: two
// tiles take what 4.8 + mt / 2 units take.  A tile of k_wstream_gemm (1), of
// which a CU has several at a time, takes 0.8 (1 + mt), its rows coming from
// L1 at times.  All weights take 0.0068 units a tile at the memory's rate, so
// where that is more, eight tiles load fewer rows for them; not for K of 1024,
// which ends sooner in two parts side by side.  Numbers other than 2, 4 and 8 are
// for one round of blocks: of several rounds the weights' reads are what is left;
// three, whose parts of K do not divide it, from K of 2048 on.  us:
//                     rows    1    2    3    4    5    6    7    8
//   16384 x 4096        64   34        34   36   42   45   50   55
//                      128   46   41   41   45   51   53   60   68
//   22016 x 4096        64   47        37   38   44   47   52   57
//                      128   64   68   44   47   53   55   62   69
//   28672 x 4096        64   60        64   44   47   50   55   59
//   37888 x 3584        64   75        61   66   49   50   54   56
//                      128  105   92   75   82   55   57   62   68
//   49152 x 4096        64   95        76   83   94   72   69   69
//   57344 x 3584        64  107        90   72   86   96   72   69
//                      128  151  127  113   94  102  109   77   78
//   24576 x 1536        64   26        19   19   22   23   25   26
//   32000 x 2048        64   37        39   32   28   30   32   34
// Over 21 numbers of columns, 9 of K from 512 to 4096 and 33 to 128 rows the
// choice takes 0.6 % more than the best one, with 2, 4 and 8 alone 4.8 %; 14 % for
// the last line, where one round of five would do.
// Up to 32 rows the stream's own blocks, two a CU, read at the memory's rate; 25
// rows and more are all the cache lines that 32 are, and blocks that fill half
// of a last round wait for them (32 rows, stream and k_wide: 22016 x 4096 34.6
// and 31.7, 37888 x 3584 49.5 and 46.0; 28672 x 4096 43.3 and 43.8, 24576 x 3072
// 27.6 and 28.2).  Eight tiles a block take rounds of a block a CU, and a last
// round takes as long whatever it has, so it has to be nearly full: the more
// so where the stream's waves have whole rounds of four (frag_depth).  Stream
// and eight tiles, 32 rows:
//   blocks            257      352      400      512      544      594
//   x 4096         96  111  129  136  146  148  190  177  200  216  218  223
//   x 3584         88   99  115  116  132  122  172  150  184  187  201  193
// With norm and activation the stream writes less: 352 blocks x 4096 117 and 135,
// 512 170 and 171, 594 x 3584 177 and 188.
static int wide_tiles(int M, int N, int K, bool gated)
{
    const int tiles = N / 32, mt = (M + 31) / 32;
    const int whole = (tiles + 255) / 256;     // of one round of blocks
    if (M <= 32) {
        if (M <= 24 || K < 3072) return 1;
        if (tiles >= 2048) {
            const int blocks = (tiles + 7) / 8, rounds = (blocks + 255) / 256;
            const double full = blocks / (256. * rounds);
            return (gated ? rounds == 1 : full >= (K % 2048 ? 0.77 : 0.85))
                       ? 8 : 1;
        }
        return tiles > 512 && (-tiles & 511) > 256 ? whole : 1;
    }
    // two tiles of 64 rows are 5.8 units, one after the other 4.8 at most
    auto units = [&](int cw) {
        const int blocks = (tiles + cw - 1) / cw;
        return (blocks + 255) / 256
               * std::max<double>(cw + mt, cw < 4 ? 4.8 + 0.5 * mt : 0);
    };
    int best = 1;
    double least = whole * 0.8 * (1 + mt);
    for (int cw = mt == 2 ? 4 : 2; cw <= 8; cw *= 2)
        if (units(cw) < least) least = units(best = cw);
    const double reads = K > 1024 ? tiles * 0.0068 : 0;
    for (int cw : {3, 5, 6, 7}) {
        if (cw < whole || (cw == 3 && K < 2048)) continue;
        const double u = std::max(units(cw), reads);
        if (u < least) {
            least = u;
            best = cw;
        }
    }
    return best;
}

// tiles a block that a product takes, 1: k_wstream_gemm
extern "C" int wstream_wide_tiles(int M, int N, int K, int gated)
{
    return M < 1 || M > 128 || N < 32 || K < 64 ? -104
                                                : wide_tiles(M, N, K, gated);
}

template <int GU>
static int wide(int cw, void* y, const void* x, const void* wp, int M, int N,
                int K, const void* rstd_parts, int rstd_nt, float inv_h,
                float eps, int yfrag, hipStream_t stream)
{
    const int mt = (M + 31) / 32;
    const int lds = wide_lds(mt, cw) + 512;            // + a scale per row
    auto go = [&](auto k) {
        const hipError_t e = hipFuncSetAttribute(
            (const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return (int)e;
        k<<<(N / 32 + cw - 1) / cw, cw * wide_parts(cw) * 64, lds, stream>>>(
            (bf16*)y, (const u32x4*)x, (const u32x4*)wp, M, N, K,
            (const float*)rstd_parts, rstd_nt, inv_h, eps, yfrag);
        return (int)hipGetLastError();
    };
    #define WIDE(CW)                                                       \
        if (cw == CW)                                                      \
            return mt == 1   ? go(k_wide<1, CW, GU>)                       \
                   : mt == 2 ? go(k_wide<2, CW, GU>)                       \
                   : mt == 3 ? go(k_wide<3, CW, GU>)                       \
                             : go(k_wide<4, CW, GU>)
    if (cw == 2 && mt > 2)
        return mt == 3 ? go(k_wide<3, 2, GU>) : go(k_wide<4, 2, GU>);
    WIDE(3);
    WIDE(4);
    WIDE(5);
    WIDE(6);
    WIDE(7);
    WIDE(8);
    #undef WIDE
    return -105;                                       // no such tiles
}

// ---------------------------------------------------------------------------
// Blocks of 16 columns and all of K for few rows in fragment layout.
// k_wstream_gemm's 32 columns make 128 blocks of 4096, so such products go in
// parts of K, and adding those up (stores through to memory, a ticket, loads
// back) takes 2.4 us at the end of each.  Half as wide, 256 blocks load the same
// weights without parts; but each loads all rows, so the more rows, the less it
// is worth (wstream_residual).  us in parts and here, with residual and sums:
//               rows     1            8           16           24           32
//   4096 x 4096      9.8  7.2     9.9  7.2    10.0  7.7    10.4  8.5    10.6  9.7
//   3584 x 3584      8.9  6.4     8.6  6.4     8.8  6.9     9.4  8.1     9.9  9.2
//   2048 x 2048      6.5  4.4     6.5  4.4     6.5  4.7     6.9  5.4     7.0  5.9
//   4096 x 14336    22.6 21.5    22.8 21.3    23.0 22.8    23.9 25.9    25.7 31.3
// and over tiles from 49 rows on:
//               rows    40           48           56                64
//   4096 x 4096     13.0 12.1    13.9 12.3    13.3 15.7 12.6    13.6 15.7 13.7
//   3584 x 3584     11.9 11.0    11.7 10.7    12.3 14.3 11.8    12.6 14.2 12.4
//   2048 x 2048      8.5  6.7     8.6  7.0     8.9 12.1  7.8     9.1 12.2  8.4
// (7.2 us are 4.7 TB/s.)  A line of 128 bytes of the pack has eight columns, so a
// wave's load takes whole lines here too: columns 16 h to 16 h + 15 of a tile, or,
// where a rotation pairs columns, 8 h to 8 h + 7 of both its halves.
// Rows are asked for as far ahead as weights, as loads return in order; four
// steps are as fast as six or eight.  Registers are for two blocks a CU, with
// rotation for three, and from 33 rows on, and of 17 on up to 4096 columns (no
// more blocks than CUs), for one.
// ROPE: norm (none without rstd_parts), rotation and append as k_wstream_gemm has
// them, else residual and sums of squares.
// A sums a wave, of every A-th step: with those of eight waves no fewer than the
// parts of a stream have, as a longer sum rounds more.  rms of what sums of K
// products of size one are off by, 4096 columns, streamed, with one sum a wave and
// with four: K of 4096 6.0e-6, 7.8e-6, 4.8e-6; of 14336 2.0e-5, 2.8e-5, 1.5e-5.
// Neither is faster than the other.
template <int RT, int A, bool ROPE>
__global__ __launch_bounds__(512, ROPE ? 6 : RT == 1 || A == 2 ? 4 : 2) void k_narrow(
    bf16* y, const u32x4* __restrict__ x, const u32x4* __restrict__ wp,
    const bf16* __restrict__ bias, int M, int N, int K,
    const float* __restrict__ rstd_parts, int rstd_nt, float inv_h, float eps,
    const bf16* res_in, float* __restrict__ sq_parts, RopeEpi rp = {})
{
    constexpr int D = 4;                      // steps of 64 under way
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = blockIdx.x >> 1, half = blockIdx.x & 1;
    const int NB = K >> 6, lo = wid * NB / 8, hi = (wid + 1) * NB / 8;
    const int last = max(hi - 1, lo);
    const int qt = rp.nl * 4, kt = rp.nkl * 4;         // tiles per section
    const bool pairs = ROPE && t < qt + kt;
    // a lane's unit of 16 bytes: eight of k of one column, or row
    const unsigned unit = (g >> 1) * 64 + (g & 1) * 32;
    const int c = pairs ? (r & 8) * 2 + half * 8 + (r & 7) : half * 16 + r;
    typedef __attribute__((address_space(1))) const char* Global;
    const uint64_t lw = (unit + c) * 16u;
    uint64_t lx[RT];
    #pragma unroll
    for (int m = 0; m < RT; m++) {
        const int at = min(m * 16 + r, M - 1);
        lx[m] = (uint64_t)(at >> 5) * K * 64 + (unit + (at & 31)) * 16u;
    }
    const Global wq = (Global)(wp + (int64_t)t * NB * 256), xq = (Global)x;
    u4bf8 w[D][2], xr[D][RT][2];
    f32x4 acc[A][RT] = {};
    auto step = [](Global p, int b) {
        Global q = p + (int64_t)b * 4096;
        asm("" : "+s"(q));                    // no address per lane
        return q;
    };
    auto load = [&](int s, int b) {
        const Global q = step(wq, b), p = step(xq, b);
        #pragma unroll
        for (int a = 0; a < 2; a++)
            w[s][a].u = __builtin_nontemporal_load(
                (const u32x4*)(q + lw + a * 2048));
        #pragma unroll
        for (int m = 0; m < RT; m++)
            #pragma unroll
            for (int a = 0; a < 2; a++)
                xr[s][m][a].u = *(const u32x4*)(p + lx[m] + a * 2048);
    };
    auto mul = [&](int s) {
        #pragma unroll
        for (int a = 0; a < 2; a++)
            #pragma unroll
            for (int m = 0; m < RT; m++)
                acc[s % A][m] = mma(xr[s][m][a].v, w[s][a].v,
                                    acc[s % A][m]);
    };
    #pragma unroll
    for (int s = 0; s < D; s++) load(s, min(lo + s, last));
    // this thread's results, of rows 32 apart, and what they need besides the sums
    static_assert(RT == 1 || !ROPE);
    constexpr int RR = (RT + 1) / 2, FL = 32;
    const int row = threadIdx.x >> 4, col = threadIdx.x & 15;
    const int n16 = blockIdx.x * 16 + col;
    float add[RR] = {}, rsum = 0.f;
    if (!ROPE) {
        #pragma unroll
        for (int i = 0; i < RR; i++)
            if (row + i * 32 < min(M, RT * 16))
                add[i] = __bfloat162float(
                    res_in[frag_row_off(row + i * 32, n16, N)]);
    } else {
        // the norm's partial sums, FL lanes a row; eight at a time do not fit 80
        // registers beside the loads under way (12288 x 4096, one row: 22.9 us with 12
        // of them spilled, 17.9 so)
        const int m = threadIdx.x / FL;
        if (rstd_parts && m < M) {
            const float* p = rstd_parts + (int64_t)m * rstd_nt;
            int i = threadIdx.x % FL;
            for (; i + 3 * FL < rstd_nt; i += 4 * FL) {
                float v[4];
                #pragma unroll
                for (int k = 0; k < 4; k++) v[k] = p[i + k * FL];
                #pragma unroll
                for (int k = 0; k < 4; k++) rsum += v[k];
            }
            for (; i + FL < rstd_nt; i += 2 * FL) rsum += p[i] + p[i + FL];
            if (i < rstd_nt) rsum += p[i];
        }
    }
    int b = lo;
    for (; b + 2 * D <= hi; b += D)
        #pragma unroll
        for (int s = 0; s < D; s++) {
            mul(s);
            load(s, b + s + D);
            __builtin_amdgcn_sched_barrier(0);
        }
    #pragma unroll
    for (int s = 0; s < D; s++) {
        if (b + s < hi) mul(s);
        if (b + s + D < hi) load(s, b + s + D);
    }
    #pragma unroll
    for (int s = 0; s < D - 1; s++)
        if (b + s + D < hi) mul(s);

    // the waves' sums; rows of 20 are 16 banks apart four rows on
    __shared__ float red[8][RT * 16][20];
    __shared__ float rstd_s[RT * 16];
    #pragma unroll
    for (int m = 0; m < RT; m++) {
        #pragma unroll
        for (int n = 1; n < A; n *= 2)
            #pragma unroll
            for (int s = 0; s + n < A; s += 2 * n) acc[s][m] += acc[s + n][m];
        #pragma unroll
        for (int i = 0; i < 4; i++)
            red[wid][m * 16 + g * 4 + i][r] = acc[0][m][i];
    }
    if (ROPE) {
        #pragma unroll
        for (int o = FL / 2; o; o >>= 1) rsum += __shfl_down(rsum, o, 64);
        if (threadIdx.x % FL == 0)
            rstd_s[threadIdx.x / FL] =
                rstd_parts ? rsqrtf(rsum * inv_h + eps) : 1.f;
    }
    __syncthreads();
    auto total = [&](int m, int n) {
        float s = 0.f;
        #pragma unroll
        for (int v = 0; v < 8; v++) s += red[v][m][n];
        return s;
    };
    if (!ROPE) {
        #pragma unroll
        for (int i = 0; i < RR; i++) {
            const int m = row + i * 32;
            if (m >= RT * 16) return;
            float s = total(m, col) + add[i];
            if (m < M) y[frag_row_off(m, n16, N)] = __float2bfloat16(s);
            s *= s;
            #pragma unroll
            for (int o = 8; o; o >>= 1) s += __shfl_xor(s, o, 64);
            if (col == 0 && m < M)
                sq_parts[(int64_t)m * gridDim.x + blockIdx.x] = s;
        }
        return;
    }
    if (row >= min(M, RT * 16) || (pairs && col >= 8)) return;
    const float rs = rstd_s[row];
    float lo_v = total(row, col) * rs;
    float hi_v = pairs ? total(row, col + 8) * rs : 0.f;
    const int p = rp.pos[row], n0 = half * (pairs ? 8 : 16) + col;
    if (bias) {
        lo_v += __bfloat162float(bias[t * 32 + n0]);
        if (pairs) hi_v += __bfloat162float(bias[t * 32 + 16 + n0]);
    }
    const int sec = t < qt ? t : pairs ? t - qt : t - qt - kt, head = sec >> 2;
    bf16* dst = y + (int64_t)row * N + head * 128;
    if (t >= qt) {
        const int page = rp.ptab[rp.slot[row] * rp.maxp + p / rp.psz];
        dst = (pairs ? rp.kp : rp.vp)
              + (((int64_t)page * rp.nkl + head) * rp.psz + p % rp.psz) * 128;
    }
    if (pairs) {
        const int d = (sec & 3) * 16 + n0;
        const float co = rp.cos_t[p * 64 + d], si = rp.sin_t[p * 64 + d];
        dst[d] = __float2bfloat16(lo_v * co - hi_v * si);
        dst[64 + d] = __float2bfloat16(hi_v * co + lo_v * si);
    } else
        dst[(sec & 3) * 32 + n0] = __float2bfloat16(lo_v);
}

// y = x W^T + res_in, both in fragment layout (they may be one); sq_parts: N / 16
// sums of squares a row
extern "C" int wstream_narrow_bf16(
    void* y, const void* x, const void* wp, int M, int N, int K,
    const void* res_in, void* sq_parts, hipStream_t stream)
{
    if (M < 1 || M > 64 || N < 32 || N % 32 || K < 64 || K % 64 || !res_in
        || !sq_parts)
        return -104;
    // of more than 4096 columns, a block a CU, streams have two parts at most
    (M <= 16   ? k_narrow<1, 4, false>
     : M <= 32 ? N > 4096 ? k_narrow<2, 2, false> : k_narrow<2, 4, false>
     : M <= 48 ? k_narrow<3, 4, false>
               : k_narrow<4, 4, false>)<<<N / 16, 512, 0, stream>>>(
        (bf16*)y, (const u32x4*)x, (const u32x4*)wp, nullptr, M, N, K, nullptr,
        0, 0.f, 0.f, (const bf16*)res_in, (float*)sq_parts, RopeEpi{});
    return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// Blocks of 64 columns in parts of K, a wave two tiles of 32, for long K and 17 to
// 48 rows in fragment layout.  A block of k_wstream_gemm loads all rows of its K for
// 32 columns, with 48 rows 1.5 bytes of them for a byte of weights; here half, in
// twice as many parts, whose sums take longer to meet.  us, with residual and sums:
//               rows     16           24           32           45
//   4096 x 14336     21.9 22.7    22.7 22.7    24.3 23.1    28.4 25.8
//   3584 x 18944     26.9 25.9    27.2 26.0    29.7 26.8    35.2 30.6
//   4096 x 11008     18.9 19.5    19.7 19.7    20.5 20.1    24.4 22.3
//   5120 x 13824     34.9 27.2    35.4 26.0    38.5 26.8    48.0 30.1
//   8192 x 28672     72.5 75.5    75.0 74.7    80.7 75.3    93.4 81.6
// (117 MB in 23.1 us are 5.1 TB/s; two, three and four steps ahead are alike.)  From
// 49 rows on tiles are as fast.
template <int MT>
__global__ __launch_bounds__(512, 1) void k_duo(
    bf16* y, float* __restrict__ part, const u32x4* __restrict__ x,
    const u32x4* __restrict__ wp, int M, int N, int K, int ksplit,
    const bf16* res_in, float* __restrict__ sq_parts, int* __restrict__ sem)
{
    constexpr int D = MT == 1 ? 3 : 2;        // steps of 64 under way
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t = blockIdx.x, ks = blockIdx.y;
    const int NB = K >> 6, GW = ksplit * 8, gw = ks * 8 + wid;
    const int lo = gw * NB / GW, hi = (gw + 1) * NB / GW;
    const int last = max(hi - 1, lo);
    typedef __attribute__((address_space(1))) const char* Global;
    const Global wq = (Global)(wp + (int64_t)t * 2 * NB * 256), xq = (Global)x;
    const int64_t next = (int64_t)NB * 4096;          // the second tile
    const uint64_t lw = lane * 16u;
    uint64_t lx[MT];
    #pragma unroll
    for (int m = 0; m < MT; m++)
        lx[m] = (uint64_t)m * K * 64 + (lane & 32) * 16u
                + min(lane & 31, max(M - m * 32, 1) - 1) * 16u;
    u4bf8 w[D][2][4], xr[D][MT][4];
    f32x16 acc[2][MT] = {};
    auto step = [](Global p, int64_t at) {
        Global q = p + at;
        asm("" : "+s"(q));                    // no address per lane
        return q;
    };
    auto load = [&](int s, int b) {
        const Global p = step(xq, (int64_t)b * 4096);
        #pragma unroll
        for (int c = 0; c < 2; c++) {
            const Global q = step(wq, (int64_t)b * 4096 + c * next);
            #pragma unroll
            for (int j = 0; j < 4; j++)
                w[s][c][j].u = __builtin_nontemporal_load(
                    (const u32x4*)(q + lw + j * 1024));
        }
        #pragma unroll
        for (int m = 0; m < MT; m++)
            #pragma unroll
            for (int j = 0; j < 4; j++)
                xr[s][m][j].u = *(const u32x4*)(p + lx[m] + j * 1024);
    };
    auto mul = [&](int s) {
        #pragma unroll
        for (int j = 0; j < 4; j++)
            #pragma unroll
            for (int m = 0; m < MT; m++)
                #pragma unroll
                for (int c = 0; c < 2; c++)
                    acc[c][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        xr[s][m][j].v, w[s][c][j].v, acc[c][m], 0, 0, 0);
    };
    #pragma unroll
    for (int s = 0; s < D; s++) load(s, min(lo + s, last));
    int b = lo;
    for (; b + 2 * D <= hi; b += D)
        #pragma unroll
        for (int s = 0; s < D; s++) {
            mul(s);
            load(s, b + s + D);
            __builtin_amdgcn_sched_barrier(0);
        }
    #pragma unroll
    for (int s = 0; s < D; s++) {
        if (b + s < hi) mul(s);
        if (b + s + D < hi) load(s, b + s + D);
    }
    #pragma unroll
    for (int s = 0; s < D - 1; s++)
        if (b + s + D < hi) mul(s);

    // 32 rows of 64 columns at a time: a thread has four columns of one row
    extern __shared__ __align__(16) char smem[];
    float (*red)[32][64] = reinterpret_cast<float (*)[32][64]>(smem);
    const int row = tid >> 4, col = (tid & 15) * 4;
    f32x4 v[MT];
    #pragma unroll
    for (int m = 0; m < MT; m++) {
        if (m) __syncthreads();
        #pragma unroll
        for (int c = 0; c < 2; c++)
            #pragma unroll
            for (int r = 0; r < 16; r++)
                red[wid][(r & 3) + 8 * (r >> 2) + 4 * (lane >> 5)]
                   [c * 32 + (lane & 31)] = acc[c][m][r];
        __syncthreads();
        v[m] = f32x4{};
        #pragma unroll
        for (int u = 0; u < 8; u++)
            v[m] += *reinterpret_cast<const f32x4*>(&red[u][row][col]);
    }
    const int tiles = gridDim.x;
    if (ksplit > 1) {
        // The block that arrives last adds up the parts, in their order, as in
        // k_wstream_gemm: written through, read past the caches.
        #pragma unroll
        for (int m = 0; m < MT; m++) {
            float* p = part + (((int64_t)ks * tiles + t) * MT + m) * 2048 + tid * 4;
            #pragma unroll
            for (int e = 0; e < 4; e += 2) {
                const uint64_t u = (uint64_t)__float_as_uint(v[m][e + 1]) << 32
                                   | __float_as_uint(v[m][e]);
                __hip_atomic_store(reinterpret_cast<uint64_t*>(p + e), u,
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        int* drawn = reinterpret_cast<int*>(smem);
        if (tid == 0)
            *drawn = __hip_atomic_fetch_add(sem + t, 1, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*drawn != ksplit - 1) return;
        if (tid == 0)
            __hip_atomic_store(sem + t, 0, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        #pragma unroll
        for (int m = 0; m < MT; m++) v[m] = f32x4{};
        for (int k = 0; k < ksplit; k += 4) {
            uint64_t u[4][MT][2];
            #pragma unroll
            for (int q = 0; q < 4; q++)
                #pragma unroll
                for (int m = 0; m < MT; m++)
                    #pragma unroll
                    for (int e = 0; e < 2; e++)
                        u[q][m][e] = __hip_atomic_load(
                            reinterpret_cast<const uint64_t*>(
                                part + (((int64_t)min(k + q, ksplit - 1) * tiles
                                         + t) * MT + m) * 2048 + tid * 4) + e,
                            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            #pragma unroll
            for (int q = 0; q < 4; q++)
                if (k + q < ksplit)
                    #pragma unroll
                    for (int m = 0; m < MT; m++)
                        #pragma unroll
                        for (int e = 0; e < 4; e++)
                            v[m][e] += __uint_as_float(
                                (unsigned)(u[q][m][e >> 1] >> 32 * (e & 1)));
        }
    }
    #pragma unroll
    for (int m = 0; m < MT; m++) {
        const int at = m * 32 + row;
        const int64_t o = frag_row_off(at, t * 64 + col, N);
        float s = 0.f;
        if (at < M) {
            const bf16x4 r = *reinterpret_cast<const bf16x4*>(res_in + o);
            bf16x4 q;
            #pragma unroll
            for (int e = 0; e < 4; e++) {
                const float f = v[m][e] + (float)r[e];
                q[e] = (__bf16)f;
                s += f * f;
            }
            *reinterpret_cast<bf16x4*>(y + o) = q;
        }
        #pragma unroll
        for (int o = 8; o; o >>= 1) s += __shfl_xor(s, o, 64);
        if ((tid & 15) == 0 && at < M) sq_parts[(int64_t)at * tiles + t] = s;
    }
}

// y = x W^T + res_in, both in fragment layout (they may be one), in `ksplit` parts
// of K; part: as many times the floats of N columns of whole row tiles; sem: zeros,
// one per 64 columns, zero again at the end; sq_parts: N / 64 sums of squares a row.
// wstream_residual takes it for up to 48 rows in two parts and more.
extern "C" int wstream_duo_bf16(
    void* y, void* part, const void* x, const void* wp, int M, int N, int K,
    int ksplit, const void* res_in, void* sq_parts, void* sem,
    hipStream_t stream)
{
    if (M < 1 || M > 64 || N < 64 || N % 64 || K < 64 || K % 64 || ksplit < 1
        || !res_in || !sq_parts || (ksplit > 1 && (!part || !sem)))
        return -104;
    constexpr int lds = 8 * 32 * 64 * 4;
    auto go = M <= 32 ? k_duo<1> : k_duo<2>;
    const hipError_t e = hipFuncSetAttribute(
        (const void*)go, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return (int)e;
    go<<<dim3(N / 64, ksplit), 512, lds, stream>>>(
        (bf16*)y, (float*)part, (const u32x4*)x, (const u32x4*)wp, M, N, K,
        ksplit, (const bf16*)res_in, (float*)sq_parts, (int*)sem);
    return (int)hipGetLastError();
}

// How a residual product of few rows goes: 0 streamed in `ksplit` parts, 1 in
// blocks of 16 columns, or in blocks of 64 in as many parts as are returned, two
// or more.  What has least to load on the busiest of 256 CUs, rows counted by the
// eight of a cache line, but no less than 1.4 times its share of the weights, which
// is what memory takes (8192 x 28672, 16 rows: 69.9 us streamed, 72.4 in blocks of
// 64).  Adding up parts takes the time of 200 KB, of more than 32 rows 270, of
// blocks of 64 columns 300 and 20 more for each part beyond four (512 x 18944, 48
// rows: 15.1 us in 8 parts, 22.1 in 32 of 64 columns).  Blocks of 16 columns load
// what K of 768 takes even if it is less (4096 x 256, 32 rows: 4.5 us streamed,
// 5.1).  Over 12 numbers of columns from 512 to 8192, 16 of K from 128 to 28672 and
// 8 of rows from 1 to 64 the choice takes 1.9 % more than the best of the three,
// parts (tiles in parts from 49 rows on) alone 13 %, 16 columns alone 21 %, and at
// most 2.7 % more than parts.
// From 49 rows on the parts are of tiles, which use CUs that fewer than 2048
// columns leave without a block, and are no slower than 64 columns; at the price
// of 256 KB the choice keeps tiles for 4096 x 5632, 56 rows, of 17.1 us where 16
// columns take 15.1, and takes 16 columns nowhere that they are slower.
extern "C" int wstream_residual(int M, int N, int K, int ksplit)
{
    if (M < 1 || N < 32 || N % 32 || K < 64 || K % 64 || ksplit < 1) return -104;
    if (M > 64 || (M > 48 && N < 2048)) return 0;
    const int rows = (M + 7) / 8 * 8;
    // bytes: of a column's, and all rows'
    auto load = [&](int columns, int parts, int k) {
        const int64_t blocks = N / columns * parts;
        return std::max<int64_t>(
            (blocks + 255) / 256 * (k / parts) * 2 * (columns + rows),
            1.4 / 128 * N * K);
    };
    const int sums = M > 48 ? 256 : M > 32 ? 270 : 200;
    const int64_t whole = load(16, 1, std::max(K, 768));
    const int64_t parts = load(32, ksplit, K) + (ksplit > 1 ? sums << 10 : 0);
    int64_t least = std::min(whole, parts);
    int best = whole <= parts;
    const int ks = N % 64 ? 0 : std::min(256 / (N / 64), K / 512);
    if (M <= 48 && ks > 1
        && load(64, ks, K) + ((300 + 20 * std::max(ks - 4, 0)) << 10) < least)
        best = ks;
    return best;
}

// Iterations ahead for 32 rows in fragment layout: four where every wave has whole
// rounds of four, or one.  Slots of a first round that a wave does not have are
// loaded all the same, and 4 KB of each of 16 waves are already twice what a CU
// can have under way (32 KB, 57 GB/s of weights).  us for 1 and 32 rows:
//                    one          four
//   28672 x 4096     44.5  49.2   42.6  48.5      8 iterations a wave
//   37888 x 3584     47.8  55.9   50.3  58.8      7
//   18432 x 3072     23.5  27.6   26.9  31.9      6
//   4096 x 14336     22.4  25.1   23.4  26.4      14, in two parts
//   4096 x 11008     19.0  20.9   19.6  21.4      10 or 11
// Two of 17 rows and more where a CU has no second block to load meanwhile and
// the waves have no more than two or four iterations, or half of them three, us
// of one and two for 12 and 32 rows:
//   2048 x 2048       6.4   7.2    6.4   6.9      2, in two parts
//   4096 x 1024       4.9   5.6    4.9   5.4      2
//   3584 x 3584       8.8   9.9    8.8   9.7      3 or 4, in two parts
// With 256 blocks (8192 x 1024, norm and activation) 5.3 and 5.9, two 5.5 and 6.1;
// of 3 iterations (3072 x 3072, in two parts) 7.6 and 8.8, two 8.4 and 9.1.
static int frag_depth(int M, int N, int K, int ksplit)
{
    const int its = K / 64, waves = 8 * ksplit;
    if (its % (4 * waves) == 0) return 4;
    return M > 16 && N / 32 * ksplit < 256
                   && (its == 2 * waves
                       || (2 * its >= 7 * waves && its < 4 * waves))
               ? 2 : 1;
}

extern "C" int wstream_depth(int M, int N, int K, int ksplit)
{
    return M < 1 || M > 32 || N < 32 || K < 64 || ksplit < 1
               ? -104 : frag_depth(M, N, K, ksplit);
}

// Fused gate_up @ SwiGLU over GU-interleaved packed weights.
// N = 2F total weight rows; output is the activation [M, F].
// rstd_parts: optional fused-rmsnorm scale of the raw-residual input.
template <int GU>
static int wstream_gu(
    void* act, const void* x, const void* wp, int M, int N, int K,
    int64_t xs, int xlds, const void* rstd_parts, int rstd_nt,
    float inv_h, float eps, int yfrag, hipStream_t stream)
{
    dim3 grid(N / 32, 1);
    const int lds = (xlds == 1 ? 16 * 4096 : 8 * 32 * 32 * 4) + 512;
    if (M > (xlds == 2 ? 128 : 64)) return -104;   // rows of a block
    if (xlds == 2) {           // frag chain
        const int cw = wide_tiles(M, N, K, true);
        if (cw > 1)
            return wide<GU>(cw, act, x, wp, M, N, K, rstd_parts, rstd_nt,
                            inv_h, eps, yfrag, stream);
    }
    if (M > 32) {
        if (xlds == 2) {
            (M <= 64   ? k_wstream_gemm<2, 2, 2, GU>
             : M <= 96 ? k_wstream_gemm<3, 2, 2, GU>
                       : k_wstream_gemm<4, 2, 2, GU>)
                <<<grid, 512, lds, stream>>>(
                (bf16*)act, nullptr, (const bf16*)x, (const u32x4*)wp,
                nullptr, M, N, K, xs, 1, (const float*)rstd_parts,
                rstd_nt, inv_h, eps, nullptr, nullptr, {}, yfrag, nullptr);
            return (int)hipGetLastError();
        }
        // generic-path fused product and activation, direct x loads (unused
        // by default: measured below lib at 64 users)
        if (rstd_parts || yfrag) return -102;
        k_wstream_gemm<2, 1, 0, GU><<<grid, 512, lds, stream>>>(
            (bf16*)act, nullptr, (const bf16*)x, (const u32x4*)wp,
            nullptr, M, N, K, xs, 1, nullptr, 0, 0.f, 0.f,
            nullptr, nullptr, {}, 0);
        return (int)hipGetLastError();
    }
    const int d = frag_depth(M, N, K, 1);
    auto go = xlds == 2 ? (d == 4   ? k_wstream_gemm<1, 4, 2, GU>
                           : d == 2 ? k_wstream_gemm<1, 2, 2, GU>
                                    : k_wstream_gemm<1, 1, 2, GU>)
              : xlds == 1 ? k_wstream_gemm<1, 1, 1, GU>
                          : k_wstream_gemm<1, 1, 0, GU>;
    go<<<grid, 512, lds, stream>>>(
        (bf16*)act, nullptr, (const bf16*)x, (const u32x4*)wp,
        nullptr, M, N, K, xs, 1, (const float*)rstd_parts, rstd_nt,
        inv_h, eps, nullptr, nullptr, {}, yfrag, nullptr);
    return (int)hipGetLastError();
}

extern "C" int wstream_gu_bf16(
    void* act, const void* x, const void* wp, int M, int N, int K,
    int64_t xs, int xlds, const void* rstd_parts, int rstd_nt,
    float inv_h, float eps, int yfrag, int gelu, hipStream_t stream)
{
    return (gelu ? wstream_gu<2> : wstream_gu<1>)(
        act, x, wp, M, N, K, xs, xlds, rstd_parts, rstd_nt, inv_h, eps,
        yfrag, stream);
}


__global__ __launch_bounds__(256) void k_wstream_combine(
    bf16* __restrict__ y, const float* __restrict__ part,
    const bf16* __restrict__ bias, int64_t total, int64_t mn, int N,
    int ksplit)
{
    for (int64_t i = blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        float s = 0.f;
        for (int k = 0; k < ksplit; k++) s += part[k * mn + i];
        if (bias) s += __bfloat162float(bias[i % N]);
        y[i] = __float2bfloat16(s);
    }
}

// y == null: the partial sums, fp32, are the result.  sem (x in fragment
// layout, or up to 32 rows): zeros, one per 32 columns; the product adds up its
// own parts, then part holds ksplit * N * 32 floats for every 32 rows.
extern "C" int wstream_gemm_bf16(
    void* y, void* part, const void* x, const void* wp, const void* bias,
    int M, int N, int K, int64_t xs, int ksplit, int depth, int xlds,
    const void* rstd_parts, int rstd_nt, float inv_h, float eps,
    const void* res_in, void* sq_parts, int yfrag, void* sem_,
    hipStream_t stream)
{
    dim3 grid(N / 32, ksplit);
    int* sem = ksplit > 1 && y ? (int*)sem_ : nullptr;
    if (M > (xlds == 2 ? 128 : 64)) return -104;   // rows of a block
    if (sem && xlds != 2 && M > 32) return -103;
    const int lds_red = 8 * 32 * 32 * 4 + 512;     // reduce + rstd tail
    const int lds_x = 16 * 4096 + 512;             // + 8x2 x tiles
    const float* rp = (const float*)rstd_parts;
    const bf16* ri = (const bf16*)res_in;
    float* sq = (float*)sq_parts;
    // what is fused needs the finished sums, and k_wstream_combine writes rows
    if (ksplit > 1 && !sem && (rstd_parts || res_in || sq_parts || yfrag))
        return -100;
    const int d = frag_depth(M, N, K, ksplit);
    if (xlds == 2 && ksplit == 1 && y && !bias && !ri && !sq) {
        const int cw = wide_tiles(M, N, K, false);
        if (cw > 1)
            return wide<0>(cw, y, x, wp, M, N, K, rp, rstd_nt, inv_h, eps,
                           yfrag, stream);
    }
    if (M <= 32) {
        if (xlds == 2)
            (d == 4   ? k_wstream_gemm<1, 4, 2>
             : d == 2 ? k_wstream_gemm<1, 2, 2>
                      : k_wstream_gemm<1, 1, 2>)
                <<<grid, 512, lds_red, stream>>>(
                (bf16*)y, (float*)part, (const bf16*)x, (const u32x4*)wp,
                (const bf16*)bias, M, N, K, xs, ksplit, rp, rstd_nt,
                inv_h, eps, ri, sq, {}, yfrag, sem);
        else if (xlds == 1)
            k_wstream_gemm<1, 1, 1><<<grid, 512, lds_x, stream>>>(
                (bf16*)y, (float*)part, (const bf16*)x, (const u32x4*)wp,
                (const bf16*)bias, M, N, K, xs, ksplit, rp, rstd_nt,
                inv_h, eps, ri, sq, {}, yfrag, sem);
        else if (depth == 2)
            k_wstream_gemm<1, 2><<<grid, 512, lds_red, stream>>>(
                (bf16*)y, (float*)part, (const bf16*)x, (const u32x4*)wp,
                (const bf16*)bias, M, N, K, xs, ksplit, rp, rstd_nt,
                inv_h, eps, ri, sq, {}, yfrag, sem);
        else
            k_wstream_gemm<1, 1><<<grid, 512, lds_red, stream>>>(
                (bf16*)y, (float*)part, (const bf16*)x, (const u32x4*)wp,
                (const bf16*)bias, M, N, K, xs, ksplit, rp, rstd_nt,
                inv_h, eps, ri, sq, {}, yfrag, sem);
    } else {
        if (xlds == 2) {
            (M <= 64   ? k_wstream_gemm<2, 2, 2>
             : M <= 96 ? k_wstream_gemm<3, 2, 2>
                       : k_wstream_gemm<4, 2, 2>)
                <<<grid, 512, lds_red, stream>>>(
                (bf16*)y, (float*)part, (const bf16*)x, (const u32x4*)wp,
                (const bf16*)bias, M, N, K, xs, ksplit, rp, rstd_nt,
                inv_h, eps, ri, sq, {}, yfrag, sem);
        } else if (rstd_parts || res_in || sq_parts || yfrag) {
            return -101;           // fusion needs the frag path at MT2
        } else if (depth == 2)
            k_wstream_gemm<2, 2><<<grid, 512, lds_red, stream>>>(
                (bf16*)y, (float*)part, (const bf16*)x, (const u32x4*)wp,
                (const bf16*)bias, M, N, K, xs, ksplit, nullptr, 0,
                0.f, 0.f, nullptr, nullptr);
        else
            k_wstream_gemm<2, 1><<<grid, 512, lds_red, stream>>>(
                (bf16*)y, (float*)part, (const bf16*)x, (const u32x4*)wp,
                (const bf16*)bias, M, N, K, xs, ksplit, nullptr, 0,
                0.f, 0.f, nullptr, nullptr);
    }
    if (ksplit > 1 && y && !sem) {
        const int64_t mn = (int64_t)M * N;
        const int64_t want = (mn + 255) / 256;
        const int blocks = (int)(want < 1024 ? want : 1024);
        k_wstream_combine<<<blocks, 256, 0, stream>>>(
            (bf16*)y, (const float*)part, (const bf16*)bias, mn, mn, N,
            ksplit);
    }
    return (int)hipGetLastError();
}



// Rotated products of up to 16 rows go in blocks of 16 columns where blocks of 32
// are more than the 256 CUs, which leaves some of them two; where those of 16 are
// no more than three a CU, all that fit at once; and where a wave has most of the
// four steps that it asks for at first.  us in blocks of 32 and of 16:
//   columns               8448       10240       12288       13312       16384
//   x 1024,  1 row      6.9  7.7    7.2  8.0    7.4  8.2    7.5  9.6    8.0 10.1
//           16          7.6  9.1    7.7  9.4    8.0  9.8    8.0 11.3    8.6 12.1
//   x 1792,  1          9.9  8.8   10.4  9.2   10.9  9.8
//           16         10.8 10.5   11.2 11.3   11.5 11.5
//   x 2048,  1         10.9  9.4   11.3  9.6   11.6 10.2   11.9 11.6   13.1 12.6
//           16         11.7 11.0   12.2 11.3   12.6 11.8   12.8 13.4   13.8 14.9
//   x 4096,  1         18.8 15.6   19.7 16.6   20.3 17.5   20.8 20.5   24.0 22.5
//           16         20.2 18.0   20.7 19.5   21.4 20.1   21.6 23.8   24.5 25.8
//   x 8192,  1         34.5 29.1   36.4 31.0   38.4 33.7   38.9 39.5   44.9 43.2
//           16         36.8 33.0   38.4 35.2   40.0 36.9   40.3 44.5   45.6 47.7
// 6144 x 4096 gains nothing.
static bool rope_narrow(int M, int N, int K)
{
    return M >= 1 && M <= 16 && N % 32 == 0 && N > 256 * 32 && N <= 3 * 256 * 16
           && K >= 1792;
}

extern "C" int wstream_rope_narrow(int M, int N, int K)
{
    return rope_narrow(M, N, K);
}

// qkv GEMM with fused RoPE + paged KV append (fused decode chain):
// q lands rotated in y's standard layout; k/v land in the paged pool.
extern "C" int wstream_qkv_rope_bf16(
    void* y, const void* x, const void* wp, const void* bias,
    int M, int N, int K, int64_t xs,
    const void* rstd_parts, int rstd_nt, float inv_h, float eps,
    const void* rcos, const void* rsin, const void* pos,
    const void* slot, const void* ptab, void* kp, void* vp,
    int nl, int nkl, int psz, int maxp, int xf, hipStream_t stream)
{
    dim3 grid(N / 32, 1);
    const int lds = 8 * 32 * 32 * 4 + 512;
    RopeEpi rp{(const float*)rcos, (const float*)rsin, (const int*)pos,
               (const int*)slot, (const int*)ptab, (bf16*)kp, (bf16*)vp,
               nl, nkl, psz, maxp};
    const int d = frag_depth(M, N, K, 1);
    if (M > (xf ? 128 : 32)) return -104;          // rows of a block
    if (xf && rope_narrow(M, N, K)) {
        k_narrow<1, 1, true><<<N / 16, 512, 0, stream>>>(
            (bf16*)y, (const u32x4*)x, (const u32x4*)wp, (const bf16*)bias, M, N,
            K, (const float*)rstd_parts, rstd_nt, inv_h, eps, nullptr, nullptr,
            rp);
        return (int)hipGetLastError();
    }
    if (xf && M > 32)
        (M <= 64   ? k_wstream_gemm<2, 2, 2, 0, 1>
         : M <= 96 ? k_wstream_gemm<3, 2, 2, 0, 1>
                   : k_wstream_gemm<4, 2, 2, 0, 1>)
            <<<grid, 512, lds, stream>>>(
            (bf16*)y, nullptr, (const bf16*)x, (const u32x4*)wp,
            (const bf16*)bias, M, N, K, xs, 1, (const float*)rstd_parts,
            rstd_nt, inv_h, eps, nullptr, nullptr, rp, 0, nullptr);
    else if (xf)
        (d == 4   ? k_wstream_gemm<1, 4, 2, 0, 1>
         : d == 2 ? k_wstream_gemm<1, 2, 2, 0, 1>
                  : k_wstream_gemm<1, 1, 2, 0, 1>)
            <<<grid, 512, lds, stream>>>(
            (bf16*)y, nullptr, (const bf16*)x, (const u32x4*)wp,
            (const bf16*)bias, M, N, K, xs, 1, (const float*)rstd_parts,
            rstd_nt, inv_h, eps, nullptr, nullptr, rp, 0,
            nullptr);
    else
        k_wstream_gemm<1, 1, 0, 0, 1><<<grid, 512, lds, stream>>>(
            (bf16*)y, nullptr, (const bf16*)x, (const u32x4*)wp,
            (const bf16*)bias, M, N, K, xs, 1, (const float*)rstd_parts,
            rstd_nt, inv_h, eps, nullptr, nullptr, rp);
    return (int)hipGetLastError();
}

