// gfx950 decode attention: see decode_attn.h
#include "decode_attn.h"

template <bool SH>
__global__ __launch_bounds__(512, 2) void k_decode_attn(
    bf16* __restrict__ out, float* __restrict__ o_part,
    float* __restrict__ ml_part, int* __restrict__ sem,
    const bf16* __restrict__ q, const bf16* __restrict__ kpool,
    const bf16* __restrict__ vpool, const int* __restrict__ page_table,
    const int* __restrict__ slot_ids, const int* __restrict__ seq_lens,
    int G, int KVH, int page, int pshift, int max_pages, float unit,
    int64_t qs, int window, int fragout, int least, int cus)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    decode_block<SH>(smem, blockIdx.x, blockIdx.y,
                     blockIdx.z, gridDim.z, least, gridDim.y, cus, out, o_part,
                     ml_part, sem, q, kpool, vpool, page_table, slot_ids, seq_lens, G, KVH,
                     page, pshift, max_pages, unit, qs, window, fragout);
}

// part: S * Hq * split * (D + 2) floats, sem: S * KVH zeros, which are zero
// again at the end; neither is used with split 1; least, cus: see decode_block
extern "C" int decode_attn_bf16(
    void* out, void* part, void* sem, const void* q, const void* kpool,
    const void* vpool, const void* page_table, const void* slot_ids,
    const void* seq_lens, int S, int Hq, int KVH, int page, int max_pages,
    float scale, int64_t q_stride, int split, int least, int cus,
    int window, int fragout, hipStream_t stream)
{
    const int G = Hq / KVH;
    if (G < 1 || G > 8 || G * KVH != Hq || page < 1
        || (reinterpret_cast<uintptr_t>(q) & 15) || q_stride % 8
        || split < 1 || least < 8 || cus < 0 || (split > 1 && (!part || !sem)))
        return (int)hipErrorInvalidValue;
    const bool sh = page >= 16 && !(page & (page - 1));
    const float unit = scale * 1.4426950408889634f;
    auto go = sh ? k_decode_attn<true> : k_decode_attn<false>;
    const hipError_t ok = hipFuncSetAttribute(
        (const void*)go, hipFuncAttributeMaxDynamicSharedMemorySize, decode_lds(sh));
    if (ok != hipSuccess) return (int)ok;
    go<<<dim3(KVH, S, split), 512, decode_lds(sh), stream>>>(
        (bf16*)out, (float*)part, (float*)part + (int64_t)S * Hq * split * 128,
        (int*)sem, (const bf16*)q, (const bf16*)kpool, (const bf16*)vpool,
        (const int*)page_table,
        (const int*)slot_ids, (const int*)seq_lens, G, KVH, page,
        sh ? __builtin_ctz(page) : 0, max_pages, unit, q_stride, window,
        fragout, least, cus);
    return (int)hipGetLastError();
}
