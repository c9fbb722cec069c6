// Decode attention over paged keys and values, heads of 128.
//
// One query token per sequence, G = Hq / KVH query heads per key/value head:
// the work is to read every cached key and value once, 512 bytes per token
// and key/value head.  A block of eight waves takes a (sequence, key/value
// head), or one of `split` parts of it; its G heads are the columns of a
// 16-wide matrix tile, so a byte is read once for all of them.
//
// Every wave walks its own steps of 32 keys with its own maximum and sum, and
// nothing passes through LDS before the one merge at the end:
//  * a key row is the row operand of mfma_16x16x32 as it lies in memory;
//  * values are loaded as whole rows (four of them per instruction) and
//    turned in registers: a lane holds columns 8c..8c+7 of the eight keys
//    whose weights it holds, and 32 byte permutes make of them the operands
//    of eight value tiles (tile v has the columns 8c + v);
//  * both are requested a step ahead, 16 KB in flight per wave.
// Weights stay fp32: they enter the product with the values as three bf16
// terms, which hold all 24 bits.
//
// Bound by memory: 5.2 TB/s over large caches, where a device copy makes 4.7.
// Before, keys and values went through LDS for products on the vector units,
// one head a wave (32 heads, 8 of them key/value heads, unless said):
//   32 users, 256 to 768 tokens                34.2 us, now 17.5
//   128 users, 350 to 1050                      131 us, now 70
//   12 users, 4096 to 12288                     144 us, now 83
//   45 users, 300 to 900, 28 / 4 heads           46 us, now 18.5
//   20 users, 550 to 1650, 32 / 32 heads        282 us, now 69
// Loading values through wave-private LDS tiles instead is no faster and
// costs 70 KB of LDS; non-temporal loads gain 2 us at 128 users and lose as
// much at 45.
#pragma once
#include "flash32.h"

// two floats that other blocks write or read in the same launch
DEV void put2(float* p, float a, float b) {
    const uint64_t v = (uint64_t)__float_as_uint(b) << 32
                       | __float_as_uint(a);
    __hip_atomic_store(reinterpret_cast<uint64_t*>(p), v, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
DEV float2 get2(const float* p) {
    const uint64_t v = __hip_atomic_load(
        reinterpret_cast<const uint64_t*>(p), __ATOMIC_RELAXED,
        __HIP_MEMORY_SCOPE_AGENT);
    return {__uint_as_float((unsigned)v), __uint_as_float(v >> 32)};
}

// Pages: with SH they are 1 << pshift tokens and no smaller than a tile of
// 16 keys, so a tile's page number is the same for the whole wave; otherwise
// any number of tokens, looked up key by key.
// s: DECODE_LDS bytes
constexpr int DECODE_LDS = 8 * 8 * (128 + 2) * 4;

template <bool SH>
DEV void decode_block(
    float* s, int kvh, int seq, int z, int split, int least,
    bf16* __restrict__ out,               // [S, Hq, D] (split == 1)
    float* __restrict__ o_part,           // [S, Hq, split, D]
    float* __restrict__ ml_part,          // [S, Hq, split, 2] maximum, sum
    int* __restrict__ sem,                // [S, KVH] tickets, zero
    const bf16* __restrict__ q,           // [S, Hq, D], rows qs apart
    const bf16* __restrict__ kpool,       // [P][KVH][page][D]
    const bf16* __restrict__ vpool,
    const int* __restrict__ page_table,   // [slots][max_pages]
    const int* __restrict__ slot_ids, const int* __restrict__ seq_lens,
    int G, int KVH, int page, int pshift, int max_pages, float unit,
    int64_t qs, int window, int fragout)
{
    constexpr int D = 128, NW = 8, KT = 32;
    constexpr float NEG = -3.0e38f;
    const int Hq = G * KVH;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, lr = lane & 15, g = lane >> 4;
    const int kv_len = seq_lens[seq], last = kv_len - 1;
    const int* pt = page_table + (int64_t)slot_ids[seq] * max_pages;
    // first key that the query, at kv_len - 1, sees
    const int lo = window > 0 ? max(0, kv_len - window) : 0;
    const int first = lo / KT, steps = (kv_len + KT - 1) / KT - first;
    // parts in use: each has `least` steps, at least one a wave (300 tokens of
    // one user: 7.3 us in one part, 8.2 in two)
    const int parts = max(1, min(split, steps / least));
    if (z >= parts) return;
    const int GW = parts * NW;            // a wave's steps: every GW-th

    float* o_s = s;                       // [NW * 8][D]
    float* ml_s = s + NW * 8 * D;         // [NW * 8][2]

    bf16x8 qf[4], kf[2][4];
    u32x4 vr[8];
    const bf16* qr = q + seq * qs + (kvh * G + min(lr, G - 1)) * D + g * 8;
    #pragma unroll
    for (int d = 0; d < 4; d++) qf[d] = frag8(qr + d * 32);

    // SH: pages of a step's tiles, looked up a step before they are needed
    int pg[2], next[2];
    auto pages = [&](int st) {
        #pragma unroll
        for (int t = 0; SH && t < 2; t++) {
            pg[t] = next[t];
            next[t] = pt[min((first + st) * KT + t * 16, last) >> pshift];
        }
    };
    // row of a key within one of the pools
    auto row = [&](const bf16* pool, int t, int key) {
        if (SH)
            return pool + (((int64_t)pg[t] * KVH + kvh) << pshift) * D
                   + (key & ((1 << pshift) - 1)) * D;
        return pool + (((int64_t)pt[key / page] * KVH + kvh) * page
                       + key % page) * D;
    };
    // keys past the last are the last again, with a weight of zero
    auto load_k = [&](int st) {
        #pragma unroll
        for (int t = 0; t < 2; t++) {
            const int key = min((first + st) * KT + t * 16 + lr, last);
            const bf16* r = row(kpool, t, key) + g * 8;
            #pragma unroll
            for (int d = 0; d < 4; d++) kf[t][d] = frag8(r + d * 32);
        }
    };
    auto load_v = [&](int st) {
        #pragma unroll
        for (int e = 0; e < 8; e++) {
            const int key = min((first + st) * KT + (e >> 2) * 16 + g * 4
                                + (e & 3), last);
            vr[e] = *reinterpret_cast<const u32x4*>(
                row(vpool, e >> 2, key) + lr * 8);
        }
    };

    float m = NEG, l = 0.f;
    f32x4 acc[8] = {};
    int st = z * NW + wid;
    if (st < steps) {
        pages(st);
        pages(st + GW);
        load_k(st);
        load_v(st);
    }
    for (; st < steps; st += GW) {
        const bool more = st + GW < steps;
        f32x4 s[2] = {};           // scores
        #pragma unroll
        for (int d = 0; d < 4; d++) {
            s[0] = mma(kf[0][d], qf[d], s[0]);
            s[1] = mma(kf[1][d], qf[d], s[1]);
        }
        if (more) {
            pages(st + 2 * GW);
            load_k(st + GW);
        }
        // scores of the keys base + 16 j + 4 g + i for head lr
        const int base = (first + st) * KT;
        const bool inside = base >= lo && base + KT <= kv_len;
        float mx = NEG;
        #pragma unroll
        for (int j = 0; j < 2; j++)
            #pragma unroll
            for (int i = 0; i < 4; i++) {
                const int key = base + j * 16 + g * 4 + i;
                float v = s[j][i] * unit;
                if (!inside && (key < lo || key > last)) v = NEG;
                s[j][i] = v;
                mx = fmaxf(mx, v);
            }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float mn = fmaxf(m, mx), ref = mn > NEG ? mn : 0.f;
        const float f = __builtin_amdgcn_exp2f(m - ref);
        m = mn;
        float sum = 0.f;
        bf16x8 w0, w1, w2;
        #pragma unroll
        for (int e = 0; e < 8; e++) {
            const float p = __builtin_amdgcn_exp2f(s[e >> 2][e & 3] - ref);
            sum += p;
            w0[e] = (__bf16)p;
            const float r = p - (float)w0[e];
            w1[e] = (__bf16)r;
            w2[e] = (__bf16)(r - (float)w1[e]);
        }
        l = l * f + sum;                  // of this lane's keys only
        #pragma unroll
        for (int v = 0; v < 8; v++) acc[v] *= f;
        #pragma unroll
        for (int v = 0; v < 8; v++) {
            u32x4 a;
            #pragma unroll
            for (int k = 0; k < 4; k++)
                a[k] = __builtin_amdgcn_perm(
                    vr[2 * k + 1][v >> 1], vr[2 * k][v >> 1],
                    v & 1 ? 0x07060302u : 0x05040100u);
            const bf16x8 af = __builtin_bit_cast(bf16x8, a);
            acc[v] = mma(af, w2, acc[v]);
            acc[v] = mma(af, w1, acc[v]);
            acc[v] = mma(af, w0, acc[v]);
        }
        if (more) load_v(st + GW);
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);

    // the waves meet: head lr, columns 8 (4 g + i) + v
    if (lr < G) {
        #pragma unroll
        for (int i = 0; i < 4; i++) {
            f32x4* d = reinterpret_cast<f32x4*>(
                o_s + (wid * G + lr) * D + (g * 4 + i) * 8);
            d[0] = f32x4{acc[0][i], acc[1][i], acc[2][i], acc[3][i]};
            d[1] = f32x4{acc[4][i], acc[5][i], acc[6][i], acc[7][i]};
        }
        if (g == 0) {
            ml_s[(wid * G + lr) * 2] = m;
            ml_s[(wid * G + lr) * 2 + 1] = l;
        }
    }
    __syncthreads();
    const bool live = threadIdx.x < G * (D / 4);
    const int h = live ? threadIdx.x / (D / 4) : 0;
    const int c = (threadIdx.x % (D / 4)) * 4, hq = kvh * G + h;
    float top = NEG, den = 0.f;
    #pragma unroll
    for (int w = 0; w < NW; w++) top = fmaxf(top, ml_s[(w * G + h) * 2]);
    f32x4 sum = {};
    #pragma unroll
    for (int w = 0; w < NW; w++) {
        const float f = __builtin_amdgcn_exp2f(ml_s[(w * G + h) * 2] - top);
        den += f * ml_s[(w * G + h) * 2 + 1];
        sum += f * *reinterpret_cast<const f32x4*>(o_s + (w * G + h) * D + c);
    }
    if (parts > 1) {
        // The block that arrives last merges the parts, in their order.  They
        // are written through and read past the caches (agent scope), so the
        // stores have only to be complete before the ticket is drawn.
        const int64_t at = ((int64_t)seq * Hq + hq) * split;
        if (live) {
            put2(o_part + (at + z) * D + c, sum[0], sum[1]);
            put2(o_part + (at + z) * D + c + 2, sum[2], sum[3]);
            if (c == 0) put2(ml_part + (at + z) * 2, top, den);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        int* drawn = reinterpret_cast<int*>(o_s);
        if (threadIdx.x == 0)
            *drawn = __hip_atomic_fetch_add(
                sem + seq * KVH + kvh, 1, __ATOMIC_RELAXED,
                __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*drawn != parts - 1) return;
        if (threadIdx.x == 0)             // ready for the next launch
            __hip_atomic_store(sem + seq * KVH + kvh, 0, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        top = NEG;
        den = 0.f;
        sum = f32x4{};
        for (int i = 0; i < parts; i += 8) {
            float2 ml[8], a[8], b[8];     // all under way together
            #pragma unroll
            for (int j = 0; j < 8; j++) {
                const int64_t p = at + min(i + j, parts - 1);
                ml[j] = get2(ml_part + p * 2);
                a[j] = get2(o_part + p * D + c);
                b[j] = get2(o_part + p * D + c + 2);
            }
            #pragma unroll
            for (int j = 0; j < 8; j++) {
                if (i + j >= parts) break;
                const float mn = fmaxf(top, ml[j].x);
                const float f = __builtin_amdgcn_exp2f(top - mn);
                const float w = __builtin_amdgcn_exp2f(ml[j].x - mn);
                top = mn;
                den = den * f + ml[j].y * w;
                sum = sum * f + f32x4{a[j].x, a[j].y, b[j].x, b[j].y} * w;
            }
        }
    }
    if (!live) return;
    sum *= den > 0.f ? 1.f / den : 0.f;
    put_out(out, seq, hq, c, Hq, D, sum, fragout);
}
