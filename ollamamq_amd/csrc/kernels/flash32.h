// Core of attention over portions of prompts in bf16: 32 rows a wave, a block
// of NW waves walks the keys that its rows see in chunks of 64.
//   S^T[64 keys, 32 rows] = K Q^T     a row's scores are on one lane pair, so
//                                     maximum and sum need one exchange
//   O^T[DV, 32 rows] += V^T P^T       the weights are operands as they are:
//                                     values are read in the order in which a
//                                     32x32 result holds its rows, through the
//                                     LDS transpose load, or as they are where
//                                     the caller has them transposed (VT)
// The next chunk is on its way to registers while this one is computed and is
// written to the other of two LDS buffers, so a chunk costs one barrier.
// Bound by LDS reads and the exponentials beside the matrix products: with
// 128-wide keys and values 32 rows a wave read 32 KB per chunk for 1024 cycles
// of products.  Raised priority during the products loses 3 %.
#pragma once
#include "tile_mma.h"

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;

DEV f32x16 mma32(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
// the other lane of a row's pair
DEV float pair_max(float x) {
    const unsigned u = __float_as_uint(x);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// Keys that a lane's row sees, first and last; of the wave's first and last
// row, where neither bound ever falls.  A wave without rows: last_hi -1.
struct Seen { int first, last, first_lo, first_hi, last_lo, last_hi; };

template <int DK, int DV, int NW, bool VT> struct Flash32 {
    // Rows of K are 4 banks apart from a multiple of 64, whole rows of V 16: a
    // transpose load takes 64 bytes of each of four (with 4, 55 % of the cycles
    // of LDS were conflicts).
    static constexpr int KT = 64, KS = DK + 8, VS = VT ? KT + 4 : DV + 32;
    static constexpr int KB = KT * KS, VB = (VT ? DV : KT) * VS;
    static constexpr int LDS = 2 * (KB + VB) * 2;      // bytes
    static constexpr int NK = DK / 8 / NW, NV = DV / 8 / NW;

    // lane (col, h) <- values col of keys k0 + 4h .. and k0 + 8 + 4h ..
    DEV bf16x8 values(const bf16* v_s, int k0, int v0, int lane) {
        const int h = lane >> 5;
        if constexpr (VT) {
            const bf16* p = v_s + (v0 + (lane & 31)) * VS + k0 + 4 * h;
            return frag44(p, p + 8);
        } else {
            const int lr = lane & 15, sub = (lane >> 4) & 1;
            const bf16* p = v_s + (k0 + 4 * h + (lr >> 2)) * VS + v0
                            + sub * 16 + (lr & 3) * 4;
            const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (lds_s16x4*)const_cast<bf16*>(p));
            const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (lds_s16x4*)const_cast<bf16*>(p + 8 * VS));
            return __builtin_bit_cast(bf16x8, __builtin_shufflevector(
                a, b, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    }

    // Chunks c_lo .. c_hi - 1.  page(base, w0): of the wave's piece from row w0
    // on, also past the last key; kat(base, page, row, c), vat: eight values
    // from column c of a row on (rows are keys, for transposed values columns);
    // unit: of a score, in octaves.  m: the row's maximum; l: this lane's sum
    // of weights.  Pages are looked up a chunk before their loads, which would
    // wait for them with the products behind them.
    template <class P, class K, class V>
    DEV void walk(bf16* lds, bf16x8* qf, int c_lo, int c_hi, float unit,
                  P page, K kat, V vat, const Seen& see, float& m, float& l,
                  f32x16* o)
    {
        const int tid = threadIdx.x, lane = tid & 63;
        const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int col = lane & 31, h = lane >> 5;
        constexpr int KC = DK / 8, VC = (VT ? KT : DV) / 8;
        u32x4 kp[NK], vp[NV];
        int k_page[NK], v_page[NV];
        auto ask = [&](int base) {
            #pragma unroll
            for (int j = 0; j < NK; j++)
                k_page[j] = page(base, (wid * 64 + j * NW * 64) / KC);
            #pragma unroll
            for (int j = 0; j < NV; j++)
                v_page[j] = page(base, (wid * 64 + j * NW * 64) / VC);
        };
        // a row's maximum is taken before the unit: it has to be positive
        if (unit < 0.f)
            #pragma unroll
            for (int c = 0; c < DK / 16; c++)
                qf[c] = __builtin_bit_cast(
                    bf16x8, __builtin_bit_cast(u32x4, qf[c]) ^ 0x80008000u);
        unit = fmaxf(fabsf(unit), 1e-37f);
        auto load = [&](int base) {
            #pragma unroll
            for (int j = 0; j < NK; j++) {
                const int u = tid + j * NW * 64;
                kp[j] = kat(base, k_page[j], u / KC, u % KC * 8);
            }
            #pragma unroll
            for (int j = 0; j < NV; j++) {
                const int u = tid + j * NW * 64;
                vp[j] = vat(base, v_page[j], u / VC, u % VC * 8);
            }
        };
        auto store = [&](bf16* buf) {
            #pragma unroll
            for (int j = 0; j < NK; j++) {
                const int u = tid + j * NW * 64;
                *reinterpret_cast<u32x4*>(buf + u / KC * KS + u % KC * 8) =
                    kp[j];
            }
            #pragma unroll
            for (int j = 0; j < NV; j++) {
                const int u = tid + j * NW * 64;
                bf16* d = buf + KB + u / VC * VS + u % VC * 8;
                if constexpr (VT) {                    // rows of 8 bytes
                    typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
                    *reinterpret_cast<u32x2*>(d) = u32x2{vp[j][0], vp[j][1]};
                    *reinterpret_cast<u32x2*>(d + 4) =
                        u32x2{vp[j][2], vp[j][3]};
                } else
                    *reinterpret_cast<u32x4*>(d) = vp[j];
            }
        };
        ask(c_lo * KT);
        load(c_lo * KT);
        ask(c_lo * KT + KT);
        store(lds);
        __syncthreads();
        for (int ch = c_lo; ch < c_hi; ch++) {
            const int base = ch * KT;
            const bf16* k_s = lds + ((ch - c_lo) & 1) * (KB + VB);
            const bf16* v_s = k_s + KB;
            if (ch + 1 < c_hi) {
                load(base + KT);
                ask(base + 2 * KT);
            }
            if (base <= see.last_hi && base + KT > see.first_lo) {
                f32x16 s[2] = {};
                #pragma unroll
                for (int c = 0; c < DK / 16; c++)
                    #pragma unroll
                    for (int t = 0; t < 2; t++)
                        s[t] = mma32(frag8(k_s + (t * 32 + col) * KS + h * 8
                                           + c * 16), qf[c], s[t]);
                if (base + KT - 1 > see.last_lo || base < see.first_hi) {
                    #pragma unroll
                    for (int t = 0; t < 2; t++)
                        #pragma unroll
                        for (int r = 0; r < 16; r++) {
                            const int key = base + t * 32 + (r & 3)
                                            + 8 * (r >> 2) + 4 * h;
                            if (key > see.last || key < see.first)
                                s[t][r] = -INFINITY;
                        }
                }
                float mx = s[0][0];
                #pragma unroll
                for (int t = 0; t < 2; t++)
                    #pragma unroll
                    for (int r = 0; r < 16; r++) mx = fmaxf(mx, s[t][r]);
                mx = pair_max(mx) * unit;
                // The largest weight is exactly 1.  With a maximum of up to 8
                // octaves ago it is rounded like the others: 3 to 6 % faster,
                // but errors against float64 grow by 0.2 to 9 %.
                if (__any(mx > m)) {
                    const float mn = fmaxf(m, mx);
                    const float f = __builtin_amdgcn_exp2f(m - mn);
                    m = mn;
                    l *= f;
                    #pragma unroll
                    for (int t = 0; t < DV / 32; t++) o[t] *= f;
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
                    for (int t = 0; t < DV / 32; t++)
                        o[t] = mma32(values(v_s, k * 16, t * 32, lane), p[k],
                                     o[t]);
            }
            if (ch + 1 < c_hi) store(lds + ((ch + 1 - c_lo) & 1) * (KB + VB));
            __syncthreads();
        }
        l += __shfl_xor(l, 32, 64);
    }
};
