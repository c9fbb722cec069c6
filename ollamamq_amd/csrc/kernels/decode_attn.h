// Decode attention over paged keys and values, heads of 128.
//
// One query token per sequence, G = Hq / KVH query heads per key/value head:
// the work is to read every cached key and value once, 512 bytes per token
// and key/value head.  A block of eight waves takes a (sequence, key/value
// head), or one of `split` parts of it; its G heads are the columns of a
// 16-wide matrix tile, so a byte is read once for all of them.
//
// Every wave walks its own steps of 32 keys with its own maximum and sum, and
// nothing is shared before the one merge at the end:
//  * keys and values are loaded a step ahead, 16 KB under way per wave, in whole
//    rows, four of them an instruction: keys straight to LDS of the wave's own.  A
//    key row is the row operand of mfma_16x16x32; loaded to registers in that
//    form, 16 lanes touch 16 lines for 16 bytes each;
//  * values are turned in registers: a lane holds columns 8c..8c+7 of the eight
//    keys whose weights it holds, and 32 byte permutes make of them the operands
//    of eight value tiles (tile v has the columns 8c + v).  With pages of 16, 32,
//    64, ... tokens they come as they lie; with others through LDS as well, as
//    the compiler waits for all loads to LDS by 64 bit addresses before it uses a
//    register that was loaded;
//  * page numbers are looked up for many steps at once, a lane each.
// Weights stay fp32: they enter the product with the values as three bf16
// terms, which hold all 24 bits.
//
// Bound by memory: 4.9 to 5.4 TB/s over large caches, where a device copy makes
// 4.7.  us, with keys and values loaded to registers in operand order, and so (32
// heads, 8 of them key/value heads, unless said):
//   one user, 300 tokens                        7.4, now 5.9
//   32 users, 256 to 768                       17.8, now 16.4
//   128 users, 350 to 1050                     70.6, now 68.0
//   12 users, 4096 to 12288                    84.4, now 81.0
//   24 users, 1000 to 3000                     46.6, now 42.7
//   48 users, 300 to 900, 28 / 4 heads         18.7, now 16.9
//   24 users, 550 to 1650, 32 / 32 heads       78.4, now 77.4
//   24 users, 1000 to 3000, pages of 24 tokens  52.7, now 45.0
// With values through LDS too, 128 KB a block, the next one does not start while
// the last waves merge (128 users of 8 to 24 tokens 13.0, now 11.8, loaded to
// registers 12.3; 32 heads, 68 users of 86 to 257 53.6, 50.7, 53.3).  Contexts of
// one step are up to 0.2 us slower than with loads to registers where only few
// blocks have them (28 / 4 heads, one user 3.9, now 4.1).
// A wave's steps one after the other and heads dealt to the XCDs in turn are 1 to
// 3 % slower; whole lines of 8 rows an instruction, put right in registers, no
// faster than operand order.
#pragma once
#include <type_traits>
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
// any number of tokens, and every key has its own.
// smem: decode_lds bytes, for a wave 32 keys and, without SH, values
constexpr int decode_lds(bool sh) { return 8 * (sh ? 1 : 2) * 32 * 128 * 2; }

template <bool SH>
DEV void decode_block(
    char* smem, int kvh, int seq, int z, int split, int least,
    int S, int cus,
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
    int kv_len = seq_lens[seq], slot = slot_ids[seq];
    int other = split > 1 && cus ? seq_lens[min(lane, S - 1)] : 0;
    // asked for together; scalars by themselves, or they count as a lane's own
    asm volatile("" : "+s"(kv_len), "+s"(slot));
    asm volatile("" : "+v"(other));
    const int last = kv_len - 1;
    const int* pt = page_table + (int64_t)slot * max_pages;
    // first key that the query, at kv_len - 1, sees
    const int lo = window > 0 ? max(0, kv_len - window) : 0;
    const int first = lo / KT, steps = (kv_len + KT - 1) / KT - first;
    // Parts in use: each has `least` steps, at least one a wave (two parts cost
    // 300 tokens of one user 0.9 us).  With cus, an even share, for a block a CU,
    // of what all sequences have: short contexts stay whole, where parts of 8
    // steps made up to 768 blocks with as many ends, and long ones take no longer
    // than the rest.  So the order of a sequence's sums depends on the lengths of
    // those beside it, as the most parts do on their number and longest context.
    // us with 8 steps and so (ragged, key/value heads), of batches as decode steps
    // pad them: 12 users of 800 tokens, 8 heads 16.7, 13.9; 16 of 600 16.5, 13.8;
    // 16 of 1500 27.6, 25.2; 24 of 800, 4 heads 17.1, 14.2; 32 of 1500 28.2, 25.6;
    // 3 of 1000, 32 heads 17.9, 15.1; beside prompts, where they are not padded, 20
    // of 600, 8 heads 18.0, 14.6; 45 of 600, 4 heads 19.6, 15.4.  Over 17 batches
    // and 15 lengths from 100 to 4000 5 % less on average, and more in one case
    // (4 of 500, 32 heads 12.0, 13.3).  Shares of 36 and more end too far apart: 12
    // of 8192 took 88 us for 82.  Finding the share takes 0.2 to 0.4 us, so contexts
    // of less than two parts and of 100 steps and more, whose share is seldom less
    // than that, go without.
    if (z > 0 && z >= steps / least) return;
    if (split > 1 && cus && steps >= 2 * least && steps < 100) {
        auto steps_of = [&](int n) {
            return (n + KT - 1) / KT - (window > 0 ? max(0, n - window) / KT : 0);
        };
        int all = lane < S ? steps_of(other) : 0;
        for (int i = lane + 64; i < S; i += 64) all += steps_of(seq_lens[i]);
        #pragma unroll
        for (int d = 32; d; d >>= 1) all += __shfl_xor(all, d, 64);
        all = __builtin_amdgcn_readfirstlane(all);
        const int share = (all * KVH + cus - 1) / cus;
        if (share < 36) least = max(least, share);
    }
    const int parts = max(1, min(split, steps / least));
    if (z >= parts) return;
    const int GW = parts * NW;            // a wave's steps: every GW-th

    // a wave's own: 32 keys and values, in the end its G results, maxima and sums
    constexpr int OWN = decode_lds(SH) / NW / 4;      // floats
    float* o_s = reinterpret_cast<float*>(smem);
    char* keys = smem + wid * OWN * 4;
    char* values = keys + KT * D * 2;

    bf16x8 qf[4];
    u32x4 vr[8];
    const bf16* qr = q + seq * qs + (kvh * G + min(lr, G - 1)) * D + g * 8;
    #pragma unroll
    for (int d = 0; d < 4; d++) qf[d] = frag8(qr + d * 32);

    int st = z * NW + wid;
    // the key of instruction e; past the last the last again, with no weight
    auto key_of = [&](int st, int e) {
        return min((first + st) * KT + e * 4 + g, last);
    };
    // Pages are looked up for many of a wave's steps at once, one a lane: of a
    // step's two tiles, or as many as its keys can lie in.
    const int per = SH ? 2 : (KT - 1) / page + 2, many = 64 / per;
    int book = 0, pg[SH ? 2 : 8];
    auto pages = [&](int st, int j) {
        if (j == 0) {
            const int b = lane / per, p = lane - b * per;
            const int key = (first + st + b * GW) * KT;
            book = pt[SH ? min(key + p * 16, last) >> pshift
                         : min(min(key, last) / page + p, last / page)];
            asm volatile("" : "+v"(book));    // waited for here alone
        }
        #pragma unroll
        for (int t = 0; SH && t < 2; t++)
            pg[t] = __builtin_amdgcn_readlane(book, j * 2 + t);
        #pragma unroll
        for (int e = 0; !SH && e < 8; e++)
            pg[e] = __shfl(book, j * per + key_of(st, e) / page
                                     - (first + st) * KT / page, 64);
    };
    // SH: tile t of a step, 16 keys of one page, has an address of the wave's and
    // 32 bits a lane (64 bits a lane, many users of 150 to 600 tokens: 2 %
    // slower).  One past the last key takes the last's tile.
    auto tile_of = [&](int st, int t) {
        return min((first + st) * KT + t * 16, last & ~15);
    };
    auto tile_at = [&](const bf16* pool, int st, int t) {
        return pool + ((((int64_t)pg[t] * KVH + kvh) << pshift)
                       + (tile_of(st, t) & ((1 << pshift) - 1))) * D;
    };
    auto row_of = [&](int st, int t, int i) -> unsigned {
        const int tile = tile_of(st, t);
        return min((first + st) * KT + t * 16 + i - tile, last - tile);
    };
    auto to_lds = [&](const bf16* pool, int st, int e, int piece, char* to) {
        auto* lds = (__attribute__((address_space(3))) void*)(to + e * 1024);
        if constexpr (SH)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                __builtin_amdgcn_make_buffer_rsrc(
                    (void*)tile_at(pool, st, e >> 2), 0, 16 * D * 2, 0x27000),
                lds, 16, row_of(st, e >> 2, (e & 3) * 4 + g) * 256 + piece * 16,
                0, 0, 0);
        else {
            const int key = key_of(st, e);
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void*)(
                    pool + (((int64_t)pg[e] * KVH + kvh) * page + key % page) * D
                    + piece * 8),
                lds, 16, 0, 0);
        }
    };
    // The loads of keys and of values take turns and their waits count them, so
    // none may pass another; and a buffer has been read before it is loaded again.
    auto in_order = [] {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto load_k = [&](int st) {
        in_order();
        // pieces of 16 bytes where 16 rows are read without bank conflicts
        #pragma unroll
        for (int e = 0; e < 8; e++)
            to_lds(kpool, st, e, lr ^ ((e & 3) * 4 + g), keys);
        in_order();
    };
    auto key_at = [&](int t, int d) {
        return *reinterpret_cast<const bf16x8*>(
            keys + t * 4096 + lr * 256 + ((d * 4 + g) ^ lr) * 16);
    };
    auto load_v = [&](int st) {
        in_order();
        if constexpr (SH) {
            typedef __attribute__((address_space(1))) const char* Global;
            typedef __attribute__((address_space(1))) const u32x4* Global16;
            #pragma unroll
            for (int t = 0; t < 2; t++) {
                Global from = (Global)tile_at(vpool, st, t);
                asm volatile("" : "+s"(from));        // known after the keys
                #pragma unroll
                for (int e = 0; e < 4; e++)
                    vr[t * 4 + e] = *(Global16)(
                        from + (row_of(st, t, g * 4 + e) * 256 + lr * 16));
            }
        } else {
            #pragma unroll
            for (int e = 0; e < 8; e++) to_lds(vpool, st, e, lr, values);
        }
        in_order();
    };
    // all but the last n loads have come
    #define ARRIVED(n)                                                     \
        do {                                                               \
            __builtin_amdgcn_sched_barrier(0);                             \
            asm volatile("s_waitcnt vmcnt(" #n ")" ::: "memory");          \
            __builtin_amdgcn_sched_barrier(0);                             \
        } while (0)

    float m = NEG, l = 0.f;
    f32x4 acc[8] = {};
    // The last step has code of its own, so that the compiler knows what is under
    // way behind the values: its waits for them count too.
    auto step = [&](auto another, int j) {
        constexpr bool more = decltype(another)::value;
        ARRIVED(8);                // keys
        f32x4 s[2] = {};           // scores
        #pragma unroll
        for (int d = 0; d < 4; d++) {
            s[0] = mma(key_at(0, d), qf[d], s[0]);
            s[1] = mma(key_at(1, d), qf[d], s[1]);
        }
        if constexpr (more) {
            pages(st + GW, j);
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
        if constexpr (!SH) {
            if constexpr (more) ARRIVED(8);
            else ARRIVED(0);
            #pragma unroll
            for (int e = 0; e < 8; e++)
                vr[e] = *reinterpret_cast<const u32x4*>(
                    values + ((e >> 2) * 16 + g * 4 + (e & 3)) * 256 + lr * 16);
        }
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
        if constexpr (more) load_v(st + GW);
    };
    if (st < steps) {
        if (SH) {
            // the first step's pages as scalars: a short context has no others
            #pragma unroll
            for (int t = 0; t < 2; t++)
                pg[t] = pt[min((first + st) * KT + t * 16, last) >> pshift];
        } else
            pages(st, 0);
        // what the loop takes from registers is there before its loads
        #pragma unroll
        for (int d = 0; d < 4; d++) asm volatile("" : "+v"(qf[d]));
        load_k(st);
        load_v(st);
        for (int j = SH ? 0 : 1 % many; st + GW < steps;
             st += GW, j = j + 1 < many ? j + 1 : 0)
            step(std::true_type{}, j);
        step(std::false_type{}, 0);
    }
    #undef ARRIVED
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);

    // the waves meet: head lr, columns 8 (4 g + i) + v
    if (lr < G) {
        #pragma unroll
        for (int i = 0; i < 4; i++) {
            f32x4* d = reinterpret_cast<f32x4*>(
                o_s + wid * OWN + lr * D + (g * 4 + i) * 8);
            d[0] = f32x4{acc[0][i], acc[1][i], acc[2][i], acc[3][i]};
            d[1] = f32x4{acc[4][i], acc[5][i], acc[6][i], acc[7][i]};
        }
        if (g == 0) {
            o_s[wid * OWN + 8 * D + lr * 2] = m;
            o_s[wid * OWN + 8 * D + lr * 2 + 1] = l;
        }
    }
    __syncthreads();
    const bool live = threadIdx.x < G * (D / 4);
    const int h = live ? threadIdx.x / (D / 4) : 0;
    const int c = (threadIdx.x % (D / 4)) * 4, hq = kvh * G + h;
    float top = NEG, den = 0.f;
    #pragma unroll
    for (int w = 0; w < NW; w++)
        top = fmaxf(top, o_s[w * OWN + 8 * D + h * 2]);
    f32x4 sum = {};
    #pragma unroll
    for (int w = 0; w < NW; w++) {
        const float* ml = o_s + w * OWN + 8 * D + h * 2;
        const float f = __builtin_amdgcn_exp2f(ml[0] - top);
        den += f * ml[1];
        sum += f * *reinterpret_cast<const f32x4*>(o_s + w * OWN + h * D + c);
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
