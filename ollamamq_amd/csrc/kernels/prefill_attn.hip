// gfx950 causal attention of portions of prompts over paged keys and values,
// heads of 128.
//
// The G = Hq / KVH query heads of a key/value head are rows of one tile (row =
// token * G + head), so a staged key serves all of them, whatever G is.
// Before, a wave had one head's 32 tokens, weights went through LDS and values
// were transposed by 2-byte stores (32 heads, 8 of them key/value heads):
//   8100 tokens, window 4096     1288 us (315 TF), now 460 (883)
//   2 x 2048                      334 us (205 TF), now 100 (690)
//   7 prompts, 2310 together       68 us (103 TF), now 25 (278)
//   2048, 32 / 32 heads          1781 us, now 66
// of which values without bank conflicts and pages a chunk ahead are the last
// steps, one after another on one card: 474, 103, 26 and 72 us before.
#include <algorithm>
#include "decode_attn.h"

constexpr int D = 128;

struct Item { int slot, tok0, pos0, row0, rows; };

template <bool SH, int NW>
DEV void prefill_block(
    char* smem, int kvh, const Item it,
    bf16* __restrict__ out,               // [T, Hq, D], or its fragments
    const bf16* __restrict__ q,           // [T, Hq, D], rows qs apart
    const bf16* __restrict__ kpool,       // [P][KVH][page][D]
    const bf16* __restrict__ vpool, const int* __restrict__ page_table,
    int G, int KVH, int page, int pshift, int max_pages, float unit,
    int64_t qs, int window, int fragout)
{
    const int Hq = G * KVH;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, h = lane >> 5;
    const int* pt = page_table + (int64_t)it.slot * max_pages;
    const int end = it.row0 + it.rows - 1;
    const int p_lo = it.pos0 + it.row0 / G, kv_len = it.pos0 + end / G + 1;
    auto first_seen = [&](int p) {
        return window > 0 ? max(0, p - window + 1) : 0;
    };
    // the wave's rows and their positions
    const int w0 = it.row0 + wid * 32;
    const int w_lo = it.pos0 + min(w0, end) / G;
    const int w_hi = it.pos0 + min(w0 + 31, end) / G;
    const int row = min(w0 + col, end);
    const int tok = it.tok0 + row / G, head = kvh * G + row % G;
    const int qpos = it.pos0 + row / G;

    bf16x8 qf[8];
    const bf16* qr = q + tok * qs + head * D + h * 8;
    #pragma unroll
    for (int c = 0; c < 8; c++) qf[c] = frag8(qr + c * 16);
    // a wave takes four keys at a time
    auto page_of = [&](int base, int w0) {
        return SH ? pt[min(base + w0, kv_len - 1) >> pshift] : 0;
    };
    auto at = [&](const bf16* pool, int base, int pg, int k, int c) {
        const int key = min(base + k, kv_len - 1);
        int64_t r;
        if (SH) {
            r = (((int64_t)pg * KVH + kvh) << pshift) * D
                + ((key & ((1 << pshift) - 1)) * D + c);
        } else
            r = (((int64_t)pt[key / page] * KVH + kvh) * page + key % page)
                * D + c;
        return *reinterpret_cast<const u32x4*>(pool + r);
    };
    const Seen see{first_seen(qpos), qpos, first_seen(w_lo), first_seen(w_hi),
                   w_lo, w0 > end ? -1 : w_hi};
    constexpr int KT = 64;
    float m = -3.0e38f, l = 0.f;
    f32x16 o[4] = {};
    Flash32<D, D, NW, false>::walk(
        reinterpret_cast<bf16*>(smem), qf, first_seen(p_lo) / KT,
        (kv_len + KT - 1) / KT, unit, page_of,
        [&](int base, int p, int k, int c) { return at(kpool, base, p, k, c); },
        [&](int base, int p, int k, int c) { return at(vpool, base, p, k, c); },
        see, m, l, o);
    if (w0 + col > end) return;
    const float f = l > 0.f ? 1.f / l : 0.f;
    #pragma unroll
    for (int t = 0; t < 4; t++)
        #pragma unroll
        for (int r = 0; r < 16; r += 4)
            put_out(out, tok, head, t * 32 + 2 * r + 4 * h, Hq, D,
                    f32x4{o[t][r], o[t][r + 1], o[t][r + 2], o[t][r + 3]}
                        * f, fragout);
}

template <bool SH, int NW>
__global__ __launch_bounds__(NW * 64, 2) void k_prefill_attn(
    bf16* __restrict__ out, const bf16* __restrict__ q,
    const bf16* __restrict__ kpool, const bf16* __restrict__ vpool,
    const int* __restrict__ page_table, const Item* __restrict__ items, int G,
    int KVH, int page, int pshift, int max_pages, float unit, int64_t qs,
    int window, int fragout)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    prefill_block<SH, NW>(smem, blockIdx.x, items[blockIdx.y], out, q, kpool,
                          vpool, page_table, G, KVH, page, pshift, max_pages,
                          unit, qs, window, fragout);
}

// Both kinds of a mixed batch in one launch: neither fills the chip where a
// prompt joins a few users, and each is a latency of its own (24 users of 400
// to 1200 tokens and a prompt of 517 within a step: 24 and 19 us one after the
// other, 30 together).  Blocks of prompts come first, the longest walks, and
// the later parts of a context, of which there may be none, last; registers
// leave one block of eight waves a CU, as decode alone has.
template <bool SH>
__global__ __launch_bounds__(512, 2) void k_mixed_attn(
    bf16* __restrict__ out, float* __restrict__ o_part,
    float* __restrict__ ml_part, int* __restrict__ sem,
    const bf16* __restrict__ q, const bf16* __restrict__ kpool,
    const bf16* __restrict__ vpool, const int* __restrict__ page_table,
    const Item* __restrict__ items, int n_items,
    const int* __restrict__ slot_ids, const int* __restrict__ seq_lens,
    int S, int split, int least, int cus, int G, int KVH, int page,
    int pshift, int max_pages, float unit, int64_t qs, int window, int fragout)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int b = blockIdx.y - n_items;
    if (b < 0)
        prefill_block<SH, 8>(smem, blockIdx.x, items[blockIdx.y], out, q,
                             kpool, vpool, page_table, G, KVH, page, pshift,
                             max_pages, unit, qs, window, fragout);
    else
        decode_block<SH>(smem, blockIdx.x, b % S,
                         b / S, split, least, S, cus, out, o_part, ml_part, sem, q,
                         kpool, vpool, page_table, slot_ids, seq_lens, G, KVH,
                         page, pshift, max_pages, unit, qs, window, fragout);
}

// items: int32 [n, 5]: slot, flat index and position of the portion's first
// token, first row (token * G + head) within the portion, rows; no more than
// 32 * waves rows each
extern "C" int prefill_attn_bf16(
    void* out, const void* q, const void* kpool, const void* vpool,
    const void* page_table, const void* items, int n_items, int waves,
    int Hq, int KVH, int page, int max_pages, float scale, int64_t q_stride,
    int window, int fragout, hipStream_t stream)
{
    const int G = Hq / KVH;
    if (G < 1 || G > 8 || G * KVH != Hq || page < 1
        || (reinterpret_cast<uintptr_t>(q) & 15) || q_stride % 8)
        return (int)hipErrorInvalidValue;
    const bool sh = page >= 16 && !(page & (page - 1));
    const float unit = scale * 1.4426950408889634f;
    const int lds = Flash32<D, D, 8, false>::LDS;
    #define PF(SH, NW)                                                     \
        do {                                                               \
            static const hipError_t ok = hipFuncSetAttribute(              \
                (const void*)k_prefill_attn<SH, NW>,                       \
                hipFuncAttributeMaxDynamicSharedMemorySize, lds);          \
            if (ok != hipSuccess) return (int)ok;                          \
            k_prefill_attn<SH, NW>                                         \
                <<<dim3(KVH, n_items), NW * 64, lds, stream>>>(            \
                    (bf16*)out, (const bf16*)q, (const bf16*)kpool,        \
                    (const bf16*)vpool, (const int*)page_table,            \
                    (const Item*)items, G, KVH, page,                      \
                    sh ? __builtin_ctz(page) : 0, max_pages, unit,         \
                    q_stride, window, fragout);                            \
        } while (0)
    #define PF_W(SH)                                                       \
        do {                                                               \
            switch (waves) {                                               \
                case 4: PF(SH, 4); break;                                  \
                case 8: PF(SH, 8); break;                                  \
                default: return (int)hipErrorInvalidValue;                 \
            }                                                              \
        } while (0)
    if (sh) PF_W(true); else PF_W(false);
    #undef PF_W
    #undef PF
    return (int)hipGetLastError();
}

// S single tokens, rows 0 .. S - 1, and items of 256 rows; part and sem as for
// decode_attn_bf16
extern "C" int mixed_attn_bf16(
    void* out, void* part, void* sem, const void* q, const void* kpool,
    const void* vpool, const void* page_table, const void* items, int n_items,
    const void* slot_ids, const void* seq_lens, int S, int split, int least,
    int cus, int Hq, int KVH, int page, int max_pages, float scale, int64_t q_stride,
    int window, int fragout, hipStream_t stream)
{
    const int G = Hq / KVH;
    if (G < 1 || G > 8 || G * KVH != Hq || page < 1 || S < 1 || n_items < 1
        || (reinterpret_cast<uintptr_t>(q) & 15) || q_stride % 8
        || split < 1 || least < 8 || cus < 0 || (split > 1 && (!part || !sem)))
        return (int)hipErrorInvalidValue;
    const bool sh = page >= 16 && !(page & (page - 1));
    const int flash = Flash32<D, D, 8, false>::LDS;
    const int lds = std::max(flash, decode_lds(sh));
    auto go = sh ? k_mixed_attn<true> : k_mixed_attn<false>;
    const hipError_t ok = hipFuncSetAttribute(
        (const void*)go, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (ok != hipSuccess) return (int)ok;
    go<<<dim3(KVH, n_items + S * split), 512, lds, stream>>>(
        (bf16*)out, (float*)part, (float*)part + (int64_t)S * Hq * split * D,
        (int*)sem, (const bf16*)q, (const bf16*)kpool, (const bf16*)vpool,
        (const int*)page_table, (const Item*)items, n_items,
        (const int*)slot_ids, (const int*)seq_lens, S, split, least, cus, G, KVH,
        page, sh ? __builtin_ctz(page) : 0, max_pages,
        scale * 1.4426950408889634f, q_stride, window, fragout);
    return (int)hipGetLastError();
}
