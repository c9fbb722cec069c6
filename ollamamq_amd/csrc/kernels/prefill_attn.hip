// gfx950 causal attention of portions of prompts over paged keys and values,
// heads of 128.
//
// The G = Hq / KVH query heads of a key/value head are rows of one tile (row =
// token * G + head), so a staged key serves all of them, whatever G is.  A
// block of NW waves takes 32 * NW rows and walks the keys they see in chunks
// of 64:
//   S^T[64 keys, 32 rows] = K Q^T     a row's scores are on one lane pair, so
//                                     maximum and sum need one exchange
//   O^T[128, 32 rows] += V^T P^T      the weights are operands as they are:
//                                     values are read through the LDS
//                                     transpose load in the order in which a
//                                     32x32 result holds its rows
// The next chunk is on its way to registers while this one is computed and is
// written to the other of two LDS buffers, so a chunk costs one barrier.
//
// Bound by LDS reads and the exponentials beside the matrix products: 32 rows
// a wave read 32 KB per chunk for 1024 cycles of products.  Before, a wave had
// one head's 32 tokens, weights went through LDS and values were transposed
// by 2-byte stores (32 heads, 8 of them key/value heads):
//   8100 tokens, window 4096     1301 us (312 TF), now 427 (952)
//   2 x 2048                      335 us (205 TF), now 86 (800)
//   7 prompts, 2310 together       66 us (106 TF), now 23 (300)
//   2048, 32 / 32 heads          1777 us, now 66
// Raised priority during the products loses 3 %.
#include "tile_mma.h"

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;

constexpr int D = 128, KT = 64, LD = D + 8;
constexpr float NEG = -3.0e38f;

// lane (col, h) <- column c + col of rows r0 + 4h .. and r0 + 8 + 4h ..
DEV bf16x8 value_frag32(const bf16* tile, int lane) {
    const int lr = lane & 15, sub = (lane >> 4) & 1, h = lane >> 5;
    const bf16* p = tile + (4 * h + (lr >> 2)) * LD + sub * 16 + (lr & 3) * 4;
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_s16x4*)const_cast<bf16*>(p));
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_s16x4*)const_cast<bf16*>(p + 8 * LD));
    return __builtin_bit_cast(
        bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}
DEV f32x16 mma32(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
// the other lane of a row's pair
DEV float pair_max(float x) {
    const unsigned u = __float_as_uint(x);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

struct Item { int slot, tok0, pos0, row0, rows; };

template <bool SH, int NW>
__global__ __launch_bounds__(NW * 64, 2) void k_prefill_attn(
    bf16* __restrict__ out,               // [T, Hq, D], or its fragments
    const bf16* __restrict__ q,           // [T, Hq, D], rows qs apart
    const bf16* __restrict__ kpool,       // [P][KVH][page][D]
    const bf16* __restrict__ vpool, const int* __restrict__ page_table,
    const Item* __restrict__ items, int G, int KVH, int page, int pshift,
    int max_pages, float unit, int64_t qs, int window, int fragout)
{
    const int kvh = blockIdx.x, Hq = G * KVH;
    const Item it = items[blockIdx.y];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, h = lane >> 5;
    const int* pt = page_table + (int64_t)it.slot * max_pages;
    const int end = it.row0 + it.rows - 1;
    const int p_lo = it.pos0 + it.row0 / G, kv_len = it.pos0 + end / G + 1;
    const int c_lo = window > 0 ? max(0, p_lo - window + 1) / KT : 0;
    const int c_hi = (kv_len + KT - 1) / KT;
    // the wave's rows and their positions
    const int w0 = it.row0 + wid * 32;
    const int w_lo = it.pos0 + w0 / G;
    const int w_hi = it.pos0 + min(w0 + 31, end) / G;
    const int row = min(w0 + col, end);
    const int tok = it.tok0 + row / G, head = kvh * G + row % G;
    const int qpos = it.pos0 + row / G;

    extern __shared__ __attribute__((aligned(16))) char smem[];
    bf16* lds = reinterpret_cast<bf16*>(smem);    // [2][K, V][KT][LD]

    bf16x8 qf[8];
    const bf16* qr = q + tok * qs + head * D + h * 8;
    #pragma unroll
    for (int c = 0; c < 8; c++) qf[c] = frag8(qr + c * 16);

    // staging: a wave takes four keys at a time, 16 lanes a key
    constexpr int NP = 16 / NW;
    u32x4 kp[NP], vp[NP];
    const int sk = lane >> 4, sc = (lane & 15) * 8;
    auto load = [&](int base) {
        #pragma unroll
        for (int j = 0; j < NP; j++) {
            const int k0 = base + (j * NW + wid) * 4;
            const int key = min(k0 + sk, kv_len - 1);
            int64_t r;
            if (SH) {
                const int pg = pt[min(k0, kv_len - 1) >> pshift];
                r = (((int64_t)pg * KVH + kvh) << pshift) * D
                    + ((key & ((1 << pshift) - 1)) * D + sc);
            } else
                r = (((int64_t)pt[key / page] * KVH + kvh) * page
                     + key % page) * D + sc;
            kp[j] = *reinterpret_cast<const u32x4*>(kpool + r);
            vp[j] = *reinterpret_cast<const u32x4*>(vpool + r);
        }
    };
    auto store = [&](bf16* buf) {
        #pragma unroll
        for (int j = 0; j < NP; j++) {
            bf16* d = buf + ((j * NW + wid) * 4 + sk) * LD + sc;
            *reinterpret_cast<u32x4*>(d) = kp[j];
            *reinterpret_cast<u32x4*>(d + KT * LD) = vp[j];
        }
    };

    float m = NEG, l = 0.f;
    f32x16 o[4] = {};
    load(c_lo * KT);
    store(lds);
    __syncthreads();
    for (int ch = c_lo; ch < c_hi; ch++) {
        const int base = ch * KT;
        const bf16* k_s = lds + ((ch - c_lo) & 1) * 2 * KT * LD;
        const bf16* v_s = k_s + KT * LD;
        if (ch + 1 < c_hi) load(base + KT);
        if (base <= w_hi && (window <= 0 || base + KT > w_lo - window + 1)) {
            f32x16 s[2] = {};
            #pragma unroll
            for (int c = 0; c < 8; c++)
                #pragma unroll
                for (int t = 0; t < 2; t++)
                    s[t] = mma32(frag8(k_s + (t * 32 + col) * LD + h * 8
                                       + c * 16), qf[c], s[t]);
            if (base + KT - 1 > w_lo
                || (window > 0 && base <= w_hi - window)) {
                #pragma unroll
                for (int t = 0; t < 2; t++)
                    #pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int d = qpos - (base + t * 32 + (r & 3)
                                              + 8 * (r >> 2) + 4 * h);
                        if (d < 0 || (window > 0 && d >= window))
                            s[t][r] = -INFINITY;
                    }
            }
            float mx = s[0][0];
            #pragma unroll
            for (int t = 0; t < 2; t++)
                #pragma unroll
                for (int r = 0; r < 16; r++) mx = fmaxf(mx, s[t][r]);
            mx = pair_max(mx) * unit;
            // weights are relative to a maximum at most 8 octaves old: they
            // stay below 2^8 and are rounded relative to themselves
            if (__any(mx > m + 8.f)) {
                const float mn = fmaxf(m, mx);
                const float f = __builtin_amdgcn_exp2f(m - mn);
                m = mn;
                l *= f;
                #pragma unroll
                for (int t = 0; t < 4; t++) o[t] *= f;
            }
            bf16x8 p[4];
            #pragma unroll
            for (int t = 0; t < 2; t++)
                #pragma unroll
                for (int r = 0; r < 16; r++) {
                    const float e = __builtin_amdgcn_exp2f(
                        fmaf(s[t][r], unit, -m));
                    l += e;
                    p[t * 2 + r / 8][r & 7] = (__bf16)e;
                }
            #pragma unroll
            for (int k = 0; k < 4; k++)
                #pragma unroll
                for (int t = 0; t < 4; t++)
                    o[t] = mma32(value_frag32(v_s + k * 16 * LD + t * 32,
                                              lane), p[k], o[t]);
        }
        if (ch + 1 < c_hi)
            store(lds + ((ch + 1 - c_lo) & 1) * 2 * KT * LD);
        __syncthreads();
    }
    l += __shfl_xor(l, 32, 64);
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
    const int lds = 4 * KT * LD * 2;
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
