// gfx950 products of many rows: y[M, N] = x[M, K] @ W[N, K]^T, x in fragment
// layout (tile_mma.h), W packed the same way (ops/hip.py pack_weight and its
// kin), with what follows a product of the fused chain in the epilogue.
//
// What bounds it: at 256 CUs the matrix cores draw the card down to 1.5 to
// 1.7 GHz, where this loop keeps them 89 % busy (1.5 PFLOP/s over the rows that
// are there; 2.25 with operands that do not move).  So a product takes what its
// padded tiles take, and what is left to gain is padding, passes beside the
// product and, for few rows, CUs without a tile.
//
// * A block of four waves, one a SIMD, makes 32 HM x 32 HN of y; a wave keeps
//   its quarter, HM x HN accumulators of 16 x 16.  Large tiles because every
//   byte that a CU loads costs power and time: 256 x 256 makes 128 operations
//   of a byte.
// * K goes by in slabs of 32 through four stages of LDS.  Both operands lie in
//   fragment order, so a slab of 32 rows is 2 KB in a row, goes to LDS without
//   passing registers (16 bytes a lane) and comes back without bank conflicts.
//   Three slabs are under way while one is multiplied.
// * A wave issues one instruction every four clocks, a 16x16x32 product takes
//   16: no more than three other instructions may stand beside it.  Hence
//   pointers per piece that move only with the tile, stages known at compile
//   time, one barrier a slab, and loads and reads spread over a slab's products
//   (a slab of 63 products in 300 instructions ran at 1.30 PFLOP/s, in 183 at
//   1.43).
// * Blocks stay and take the next tile, whose first slabs are on their way
//   while the last one's results are stored.
//
// Within 32 rows or columns LDS holds groups of eight in the order 0 2 | 1 3: 16
// columns of a tile are then 8 of the first and 8 of the last 16, so the gate and
// up columns of pack_weight_gu and the rotation pairs of pack_weight_qkv_rope
// meet in one accumulator, 32 lanes apart.
//
// us for 541, 2317 and 8100 rows, one after another on one card:
//   28672 x 4096, gated   library product 140, 421, 1270 and norm and
//                         activation 15, 50, 166; here 107, 440, 1270
//   6144 x 4096, rotated  40, 88, 268 and norm and append 11, 28, 78; here 40,
//                         114, 320
//   4096 x 14336          112, 213, 610; here 76 (three parts and what adds
//                         them up), 204, 626
// Rows that are normed already (tile_rows_bf16), for 559, 1200 and 4096 rows:
//   28672 x 4096, gated   library product and activation 147, 268, 747; here 105,
//                         223, 722
//   16384 x 4096          74, 142, 405; here 71, 131, 420
//   10816 x 4096          54, 97, 399; here 52, 90, 290
//   4096 x 14336          115, 157, 325; here 64, 115 (parts, left to the reader),
//                         316
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <utility>
#include "act.h"
#include "tile_mma.h"

namespace {

enum { RESIDUAL, GATED, ROPE, PARTS, ROWS, ROW_PARTS };

// where a rotated or plain key and value go (ROPE)
struct Append {
    const float* cos_t;   // [positions, 64]
    const float* sin_t;
    const int* pos;       // [M]
    const int* slot;      // [M]
    const int* ptab;      // page table [slots, maxp]
    bf16* kp;             // this layer's pools
    bf16* vp;
    int nl, nkl, psz, maxp;
};

struct TileArgs {
    bf16* y;              // RESIDUAL, GATED: fragment layout; ROPE, ROWS: [M, N]
    float* part;          // PARTS: see k_tile_fold; ROW_PARTS: [ks, M, N];
                          // GATED, ROPE: [M] scratch
    const bf16* x;
    const bf16* w;
    const bf16* bias;     // ROPE: [N] or null, in W's order
    const bf16* res;      // RESIDUAL: the residual stream, may be y
    float* sq;            // RESIDUAL: [M, tiles of columns] sums of squares
    const float* rstd;    // GATED, ROPE: [M, rstd_nt] sums of squares of x
    int rstd_nt;          // GATED: 0 where x is normed already
    float inv_h, eps;
    int M, N, K;
    int mt, nt, ks, gm;   // tiles of rows, of columns, parts of K, rows a group
    int gelu;
    Append ap;
    int rows_at;          // bytes of LDS before what is kept of rows
};

// 1 KB pieces to LDS, a lane's 16 bytes at base + voff to lds + 16 * lane.  An
// instruction's offset moves both addresses, so one M0 serves two.
template <int O0, int O1>
DEV void to_lds2(uint64_t b0, uint64_t b1, int voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t"
                 "global_load_lds_dwordx4 %1, %2 offset:%4\n\t"
                 "global_load_lds_dwordx4 %1, %3 offset:%5"
                 :: "s"(lds), "v"(voff), "s"(b0), "s"(b1), "n"(O0), "n"(O1)
                 : "memory");        // M0: the compiler keeps nothing there
}
template <int O0>
DEV void to_lds1(uint64_t b0, int voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t"
                 "global_load_lds_dwordx4 %1, %2 offset:%3"
                 :: "s"(lds), "v"(voff), "s"(b0), "n"(O0) : "memory");
}
DEV void to_lds4(const void* b0, int voff, uint32_t lds) {   // 256 bytes
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t"
                 "global_load_lds_dword %1, %2"
                 :: "s"(lds), "v"(voff), "s"((uint64_t)b0) : "memory");
}
template <int N> DEV void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}

template <int I> using ic = std::integral_constant<int, I>;
template <int... I, class F>
DEV void each_of(std::integer_sequence<int, I...>, F f) { (f(ic<I>{}), ...); }
// f(0), .. f(N - 1), as constants
template <int N, class F> DEV void each(F f) {
    each_of(std::make_integer_sequence<int, N>{}, f);
}

// row or column of 32 that half h (16 of LDS's order) has at its place p
DEV int in_strip(int h, int p) {
    return (p >> 3) * 16 + h * 8 + (p & 7);
}
// element (row, col) of fragments of N columns
DEV int64_t frag_at(int row, int col, int N) {
    return (int64_t)(row >> 5) * 32 * N + (col >> 3) * 256 + (row & 31) * 8
           + (col & 7);
}
DEV void put4(bf16* p, const f32x4& v) {
    *reinterpret_cast<bf16x4*>(p) =
        bf16x4{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
}
DEV f32x4 get4(const bf16* p) {
    const bf16x4 v = *reinterpret_cast<const bf16x4*>(p);
    return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}
// the upper lanes of a with the lower lanes of b
DEV void swap32(f32x4& a, f32x4& b) {
    #pragma unroll
    for (int i = 0; i < 4; i++) {
        const auto r = __builtin_amdgcn_permlane32_swap(
            __float_as_uint(a[i]), __float_as_uint(b[i]), false, false);
        a[i] = __uint_as_float(r[0]);
        b[i] = __uint_as_float(r[1]);
    }
}

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
// Lanes 16 g of a and b hold four columns each; those of two such groups side by
// side: a's eight on the first of them, b's on the second
DEV u32x4 trade16(const f32x4& a, const f32x4& b) {
    typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
    const auto pack = [](const f32x4& v) {
        return __builtin_bit_cast(u32x2, bf16x4{(__bf16)v[0], (__bf16)v[1],
                                                (__bf16)v[2], (__bf16)v[3]});
    };
    const u32x2 p = pack(a), q = pack(b);
    const auto lo = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
    return u32x4{lo[0], hi[0], lo[1], hi[1]};
}

// n / (1 + e), e not negative, as close as the division is: a reciprocal and
// one step of Newton's method on the quotient, infinities and NaN as a division
// has them.  In eighths, for reciprocals of 2^126 and more are flushed.  Prompts
// take 0.4 % longer than with the reciprocal alone, 1.3 with the division.
DEV float over_1_and(float n, float e) {
    const float d = fmaf(e, 0.125f, 0.125f), r = __builtin_amdgcn_rcpf(d);
    n *= 0.125f;
    const float q = n * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, n), r, q), d, n);
}

// stages of LDS; four keep three slabs of a large tile under way, small tiles
// need more of their slabs for as many bytes
constexpr int tile_stages(int hm, int hn) { return hm + hn <= 8 ? 8 : 4; }
// bytes before three values per row: the first tile's sums of squares, nt per
// row, take the place of the last stage at first and may need more than that
constexpr int tile_rows_at(int hm, int hn, int nt) {
    const int stage = (hm + hn) * 2048, last = (tile_stages(hm, hn) - 1) * stage;
    const int sums = (hm * 128 * nt + 1023) / 1024 * 1024;
    return last + (sums > stage ? sums : stage);
}
constexpr int tile_lds(int hm, int hn, int nt) {
    return tile_rows_at(hm, hn, nt) + hm * 32 * 12;
}

template <int HM, int HN, int EPI>
__global__ __launch_bounds__(256, 1) void k_tile_gemm(const TileArgs a)
{
    constexpr int STRIPS = HM + HN, STAGE = STRIPS * 2048;
    constexpr int STAGES = tile_stages(HM, HN);
    constexpr int PER = STRIPS / 2;        // pieces per wave and slab
    constexpr int PAIRS = (PER + 1) / 2;
    static_assert(STRIPS % 2 == 0 && PER <= 8);
    extern __shared__ __align__(1024) char smem[];
    const uint32_t lds0 =
        (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    float* row_f = reinterpret_cast<float*>(smem + a.rows_at);
    int* row_pos = reinterpret_cast<int*>(row_f + HM * 32);
    int* row_kv = row_pos + HM * 32;
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wid >> 1, wn = wid & 1;
    const int r16 = lane & 15, g4 = lane >> 4;

    // A round's tiles are dealt to the XCDs in runs, so that the blocks which
    // share an L2 share rows and columns too; a last, short round as evenly.
    const int items = a.mt * a.nt * a.ks, G = gridDim.x;
    auto item_at = [&](int first) {
        const int per = (min(G, items - first) + 7) >> 3;
        const int j = blockIdx.x >> 3;
        const int id = first + (blockIdx.x & 7) * per + j;
        return first < items && j < per && id < items ? id : -1;
    };
    const int nq = a.K / (32 * STAGES);    // rounds of slabs
    int m, n, k, q0, q1;
    auto tile_at = [&](int id, int& m, int& n, int& k, int& q0, int& q1) {
        const int mn = a.mt * a.nt;
        k = id / mn;
        id -= k * mn;
        const int per = a.gm * a.nt, g = id / per, r = id - g * per;
        const int rows = min(a.gm, a.mt - g * a.gm);
        n = r / rows;
        m = g * a.gm + r - n * rows;
        q0 = nq * k / a.ks;
        q1 = nq * (k + 1) / a.ks;
    };
    int first = 0, id = item_at(0);
    if (id < 0) return;
    tile_at(id, m, n, k, q0, q1);

    // the order of LDS comes from which lane loads what
    int voff, turn;
    const int lane_off = ((lane & 32) + in_strip(lane >> 4 & 1, r16)) * 16;
    uint64_t base[PER];
    const int strip_bytes = a.K * 64;
    // strips past the last repeat it; nothing of theirs is stored
    const int ms = (a.M + 31) >> 5, ns = a.N >> 5;
    auto point = [&](int m, int n, int q0) {
        #pragma unroll
        for (int i = 0; i < PER; i++) {
            const int d = wid * PER + i, s = d >> 1;
            const uint64_t p = s < HM
                ? (uint64_t)a.x
                      + (int64_t)min(m * HM + s, ms - 1) * strip_bytes
                : (uint64_t)a.w
                      + (int64_t)min(n * HN + s - HM, ns - 1) * strip_bytes;
            base[i] = p + (d & 1) * 1024 - (i - PER / 2) * 1024;
        }
        turn = m & (STAGES - 1);
        voff = lane_off + q0 * (STAGES * 2048) + turn * 2048;
    };
    point(m, n, q0);
    const uint32_t lds_w = lds0 + (wid * PER + PER / 2) * 1024;
    auto load = [&](auto p_, auto st_) {   // two pieces into a stage
        constexpr int p = 2 * decltype(p_)::value, st = decltype(st_)::value;
        constexpr int o = (p - PER / 2) * 1024;
        if constexpr (p + 1 < PER)
            to_lds2<o, o + 1024>(base[p], base[p + 1], voff,
                                 lds_w + st * STAGE);
        else
            to_lds1<o>(base[p], voff, lds_w + st * STAGE);
    };
    // Strips are a multiple of 4 KB apart, so the same slab of every strip lies
    // in the same channels of L2: neighbouring tiles of rows take a round's
    // slabs in another order (4096 x 14336 in three parts, 541 rows: 71 us
    // against 82; 1024 rows whole: 107 against 122).
    auto step = [&](auto st_) {
        constexpr int st = decltype(st_)::value;
        voff += st < STAGES - 1 ? ((st + 1 ^ turn) - (st ^ turn)) * 2048
                                : (STAGES + turn - (st ^ turn)) * 2048;
    };
    auto load_stage = [&](auto st) {
        each<PAIRS>([&](auto p) { load(p, st); });
        step(st);
    };

    // What the results of the first tile's rows need goes straight to LDS,
    // ahead of the slabs.  Into registers it came behind all of theirs, sums
    // of squares eight rows of a wave after the other and the page after the
    // position and the slot.  K of 256, so little else, us with 1, 16 and 128
    // sums a row: 541 x 28672 over 9 x 7, gated, 21.3, 24.4 and 30.1, now 20.7,
    // 20.5 and 22.9; 1000 x 6144 over 8 x 4, rotated, 15.1, 18.3 and 22.3, now
    // 15.5, 15.7 and 18.7 (128 there by the other kernel).
    const bool sums = (EPI == GATED || EPI == ROPE) && a.rstd_nt > 0;
    const float* sums_s =
        reinterpret_cast<const float*>(smem + (STAGES - 1) * STAGE);
    if (sums) {
        const uint32_t to = lds0 + (STAGES - 1) * STAGE;
        const int64_t from = (int64_t)m * HM * 32 * a.rstd_nt;
        const float* p = a.rstd + from;
        const int end = (int)min((int64_t)HM * 128 * a.rstd_nt,
                                 ((int64_t)a.M * a.rstd_nt - from) * 4);
        // past the end the last again
        if (a.rstd_nt % 4 == 0 && (uint64_t)a.rstd % 16 == 0)
            for (int i = wid * 1024; i < end; i += 4096)
                to_lds1<0>((uint64_t)p, min(i + lane * 16, end - 16), to + i);
        else
            for (int i = wid * 256; i < end; i += 1024)
                to_lds4(p, min(i + lane * 4, end - 4), to + i);
    }
    // every wave waits for those of its own rows alone
    auto own_rows = [&](auto f) {
        if constexpr (EPI == ROPE)
            for (int i = wid; i < HM / 2; i += 4)
                f(i * 64 + lane, lds0 + a.rows_at + i * 256);
    };
    own_rows([&](int r, uint32_t to) {
        const int at = min(m * HM * 32 + r, a.M - 1) * 4;
        to_lds4(a.ap.pos, at, to + HM * 128);
        to_lds4(a.ap.slot, at, to + HM * 256);
    });
    each<STAGES - 1>(load_stage);
    if (sums || EPI == ROPE) {
        wait_loads<PER * (STAGES - 1)>();
        own_rows([&](int r, uint32_t to) {
            const int at = row_kv[r] * a.ap.maxp + row_pos[r] / a.ap.psz;
            to_lds4(a.ap.ptab, at * 4, to + HM * 256);
        });
    }
    if (sums) {
        lds_barrier();
        for (int r = threadIdx.x; r < HM * 32; r += 256) {
            const float* p = sums_s + r * a.rstd_nt;
            // eight side by side, so of n the chain is of n / 8 + 3, and the
            // bits are those of k_row_sums; loads behind conditions of their own
            // would spill 95 registers (8 x 8 tiles, 400 bytes a lane)
            f32x4 s{}, t{};
            if (a.rstd_nt % 8 == 0)
                #pragma unroll 2
                for (int e = 0; e < a.rstd_nt; e += 8) {
                    s += *reinterpret_cast<const f32x4*>(p + e);
                    t += *reinterpret_cast<const f32x4*>(p + e + 4);
                }
            else
                #pragma unroll 1
                for (int e = 0; e < a.rstd_nt; e += 8) {
                    const int last = a.rstd_nt - 1 - e;
                    #pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float u = p[e + min(i, last)];
                        const float v = p[e + min(i + 4, last)];
                        s[i] += i <= last ? u : 0.f;
                        t[i] += i + 4 <= last ? v : 0.f;
                    }
                }
            row_f[r] = rsqrtf((s[0] + s[1] + (s[2] + s[3])
                               + (t[0] + t[1] + (t[2] + t[3])))
                              * a.inv_h + a.eps);
        }
        lds_barrier();
    } else if (EPI == GATED) {
        for (int r = threadIdx.x; r < HM * 32; r += 256) row_f[r] = 1.f;
    }
    load_stage(ic<STAGES - 1>{});

    // Operands of a slab: half h of an operand's strips, lanes 16 j .. of it
    // its columns 8 j ..; a wave's halves may begin inside a strip.  Pointers
    // that the compiler cannot derive from each other, or it adds up an address
    // for each read between the products (8 x 8 tiles: 1238 clocks a slab of
    // 1024 for its products, 1174 without).
    constexpr int NF = HM + HN;
    bf16x8 f[2][NF];
    typedef const __attribute__((address_space(3))) char* lds_ptr;
    typedef const __attribute__((address_space(3))) bf16x8* lds_frag;
    // an instruction reaches 64 KB from its pointer
    constexpr int REACH = 65536 / STAGE, POINTERS = (STAGES + REACH - 1) / REACH;
    lds_ptr at[2][2][POINTERS];            // operand, parity, stages
    #pragma unroll
    for (int o = 0; o < 2; o++)
        #pragma unroll
        for (int par = 0; par < 2; par++)
            #pragma unroll
            for (int s = 0; s < POINTERS; s++) {
                const int h = (o ? wn * HN : wm * HM) + par;
                at[o][par][s] = (lds_ptr)smem + (g4 >> 1) * 1024
                                + (g4 & 1) * 512 + r16 * 16 + o * HM * 2048
                                + (h >> 1) * 2048 + (h & 1) * 256
                                + s * REACH * STAGE;
                if (par == 0 || (o ? HN : HM) & 1)
                    asm volatile("" : "+v"(at[o][par][s]));
            }
    auto read = [&](int buf, auto st_, int i) {
        constexpr int st = decltype(st_)::value;
        const int o = i >= HM, h = o ? i - HM : i;
        const bool even = (o ? HN : HM) % 2 == 0;
        f[buf][i] = *(lds_frag)(
            at[o][even ? 0 : h & 1][st / REACH] + (even ? (h & 1) * 256 : 0)
            + st % REACH * STAGE + (h >> 1) * 2048);
    };
    f32x4 acc[HM][HN] = {};

    // One slab: its operands are in registers.  Whoever passes the barrier
    // knows that every wave has read this stage, which the slab four ahead may
    // then take, and that the next slab has landed: of a wave's loads only
    // those of the two after it are still under way.
    auto slab = [&](auto st_) {
        constexpr int st = decltype(st_)::value, cur = st & 1, MF = HM * HN;
        constexpr ic<(st + 1) % STAGES> next{};
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier"
                     :: "n"(PER * (STAGES - 2)) : "memory");
        __builtin_amdgcn_sched_barrier(0);
        each<MF>([&](auto i_) {
            constexpr int i = decltype(i_)::value;
            // reads over the first three quarters, loads over all of it
            #pragma unroll
            for (int q = 0; q < NF; q++)
                if (q * MF * 3 / (4 * NF) == i) read(cur ^ 1, next, q);
            each<PAIRS>([&](auto p) {
                if constexpr ((decltype(p)::value * MF + MF / 4) / PAIRS == i)
                    load(p, st_);
            });
            // to and fro, so that one operand stays
            constexpr int r = i / HN, c = r & 1 ? HN - 1 - i % HN : i % HN;
            acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                f[cur][HM + c], f[cur][r], acc[r][c], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        });
        step(st_);
    };

    // The same for a later tile: the loads are under way before the stores of
    // the tile before, for which they would wait.  Sums of squares in parts are
    // added up by another kernel then.
    struct {
        float sq[2];
        int pos[2], slot[2];
    } of_row;
    auto ask_rows = [&](int m) {
        #pragma unroll
        for (int i = 0; i < 2; i++) {
            const int r = min(m * HM * 32 + i * 256 + (int)threadIdx.x,
                              a.M - 1);
            if (EPI == GATED || EPI == ROPE)
                if (a.rstd_nt == 1) of_row.sq[i] = a.rstd[r];
            if (EPI == ROPE) {
                of_row.pos[i] = a.ap.pos[r];
                of_row.slot[i] = a.ap.slot[r];
            }
        }
    };
    auto keep_rows = [&](int m) {
        #pragma unroll
        for (int i = 0; i < 2; i++) {
            const int r = i * 256 + threadIdx.x;
            if (r >= HM * 32) continue;
            if (EPI == GATED || EPI == ROPE)
                row_f[r] = a.rstd_nt
                    ? rsqrtf(of_row.sq[i] * a.inv_h + a.eps) : 1.f;
            if (EPI == ROPE) {
                const Append& ap = a.ap;
                const int pos = of_row.pos[i];
                const int page =
                    ap.ptab[of_row.slot[i] * ap.maxp + pos / ap.psz];
                row_pos[r] = pos;
                row_kv[r] = page * ap.nkl * ap.psz + pos % ap.psz;
            }
        }
    };
    wait_loads<PER * (STAGES - 1)>();
    asm volatile("s_barrier" ::: "memory");
    #pragma unroll
    for (int i = 0; i < NF; i++) read(0, ic<0>{}, i);

    for (;;) {
        const int next_id = item_at(first + G);
        int m1 = m, n1 = n, k1 = k, p0 = q0, p1 = q1;
        if (next_id >= 0) tile_at(next_id, m1, n1, k1, p0, p1);
        for (int q = q0; q < q1; q++) {
            if (q == q1 - 1) {
                if (next_id >= 0) point(m1, n1, p0);
                else voff -= STAGES * 2048;    // once more, for nobody
            }
            each<STAGES>(slab);
        }

        // A lane has row in_strip(.., r16) of every 16 rows and the columns
        // from in_strip(.., 4 * g4) on of every 16 columns, four of them.
        // Worked out anew for each tile: kept through the loop they would be
        // spilled, and a reload waits for every store before it.
        int here = lane;
        asm volatile("" : "+v"(here));
        const int r16 = here & 15, g4 = here >> 4;
        if (EPI == ROPE && first == 0) {   // pages to places
            for (int r = threadIdx.x; r < HM * 32; r += 256)
                row_kv[r] = row_kv[r] * a.ap.nkl * a.ap.psz
                            + row_pos[r] % a.ap.psz;
            lds_barrier();
        }
        if (next_id >= 0) ask_rows(m1);
        auto row_in = [&](int i) {         // within the tile
            const int h = wm * HM + i;
            return (h >> 1) * 32 + in_strip(h & 1, r16);
        };
        const int nh = a.N >> 4;           // halves of columns
        const int hj0 = n * HN * 2 + wn * HN;
        const int live = min(HN, nh - hj0);    // of this wave's
        if constexpr (EPI == PARTS) {
            const int mh = ms * 2, hi0 = m * HM * 2 + wm * HM;
            float* out = a.part + (((int64_t)k * mh + hi0) * nh + hj0) * 256
                         + here * 4;
            #pragma unroll
            for (int i = 0; i < HM; i++, out += nh * 256)
                if (hi0 + i < mh) {
                    #pragma unroll
                    for (int j = 0; j < HN; j++)
                        if (j < live)
                            *reinterpret_cast<f32x4*>(out + j * 256) =
                                acc[i][j];
                }
        } else if constexpr (EPI == ROW_PARTS) {
            #pragma unroll
            for (int i = 0; i < HM; i++) {
                const int row = m * HM * 32 + row_in(i);
                float* p = a.part + ((int64_t)k * a.M + row) * a.N
                           + in_strip(0, 4 * g4);
                #pragma unroll
                for (int j = 0; j < HN; j++) {
                    const int h = hj0 + j;
                    if (row < a.M && j < live)
                        *reinterpret_cast<f32x4*>(p + (h >> 1) * 32
                                                  + (h & 1) * 8) = acc[i][j];
                }
            }
        } else if constexpr (EPI == ROWS) {
            // Lanes that hold four columns of a row beside four others hold
            // eight of it, and of the next 16 rows, after trading halves.
            #pragma unroll
            for (int i = 0; i < HM; i += 2) {
                const bool two = i + 1 < HM;
                const int mine = two && g4 & 1 ? row_in(min(i + 1, HM - 1))
                                               : row_in(i);
                const int row = m * HM * 32 + mine;
                bf16* p = a.y + (int64_t)row * a.N
                          + (two ? g4 >> 1 << 4 : in_strip(0, 4 * g4));
                #pragma unroll
                for (int j = 0; j < HN; j++) {
                    const int h = hj0 + j;
                    bf16* at = p + (h >> 1) * 32 + (h & 1) * 8;
                    const bool ok = row < a.M && j < live;
                    if (two) {
                        const u32x4 v = trade16(acc[i][j],
                                                acc[min(i + 1, HM - 1)][j]);
                        if (ok) *reinterpret_cast<u32x4*>(at) = v;
                    } else if (ok) {
                        put4(at, acc[i][j]);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);     // registers
            }
        } else if constexpr (EPI == RESIDUAL) {
            // halves of columns are 256 elements apart, strips 1024
            const char* res = reinterpret_cast<const char*>(a.res);
            char* y = reinterpret_cast<char*>(a.y);
            // from a strip's first half; a wave without columns reads others'
            const int rel = live > 0 ? hj0 & 1 : 0;
            const int even = live > 0 ? hj0 - rel : 0;
            auto offset = [&](int i) {
                const int r = min(m * HM * 32 + row_in(i), a.M - 1);
                return (uint32_t)(frag_at(r, even * 16
                                          + in_strip(0, 4 * g4), a.N) * 2);
            };
            auto at = [&](int j) {
                const int h = rel + j;
                return (h >> 1) * 2048 + (h & 1) * 512;
            };
            constexpr int AHEAD = 3;
            bf16x4 old[AHEAD][HN];
            auto fetch = [&](int b, int i) {
                const char* p = res + offset(i);
                #pragma unroll
                for (int j = 0; j < HN; j++)
                    old[b][j] = *reinterpret_cast<const bf16x4*>(
                        p + at(max(min(j, live - 1), 0)));
            };
            #pragma unroll
            for (int i = 0; i + 1 < AHEAD; i++) fetch(i, i);
            float sums[HM];
            #pragma unroll
            for (int i = 0; i < HM; i++) {
                if (i + AHEAD - 1 < HM)
                    fetch((i + AHEAD - 1) % AHEAD, i + AHEAD - 1);
                const bool ok = m * HM * 32 + row_in(i) < a.M;
                char* p = y + offset(i);
                float s2 = 0.f;
                #pragma unroll
                for (int j = 0; j < HN; j++) {
                    f32x4 v = acc[i][j];
                    #pragma unroll
                    for (int e = 0; e < 4; e++) v[e] += (float)old[i % AHEAD][j][e];
                    if (ok && j < live) {
                        put4(reinterpret_cast<bf16*>(p + at(j)), v);
                        #pragma unroll
                        for (int e = 0; e < 4; e++) s2 += v[e] * v[e];
                    }
                }
                s2 += __shfl_xor(s2, 16, 64);
                sums[i] = s2 + __shfl_xor(s2, 32, 64);
                __builtin_amdgcn_sched_barrier(0);     // registers
            }
            // the two waves of a row
            if (wn && g4 == 0)
                #pragma unroll
                for (int i = 0; i < HM; i++) row_f[row_in(i)] = sums[i];
            lds_barrier();
            if (!wn && g4 == 0)
                #pragma unroll
                for (int i = 0; i < HM; i++) {
                    const int r = m * HM * 32 + row_in(i);
                    if (r < a.M)
                        a.sq[(int64_t)r * a.nt + n] =
                            sums[i] + row_f[row_in(i)];
                }
        } else {
            // Two accumulators at a time: after the swap one holds first
            // halves (gates, low dimensions), the other the second, of the
            // first accumulator on lower lanes and of the second on upper.
            const int c4 = (g4 & 1) * 4;
            const bool upper = g4 >> 1;
            float rs[HM];
            #pragma unroll
            for (int i = 0; i < HM; i++) rs[i] = row_f[row_in(i)];
            auto pair = [&](int i0, int j0, int i1, int j1, f32x4& lo,
                            f32x4& hi) {
                lo = acc[i0][j0] * rs[i0];
                hi = acc[i1][j1] * rs[i1];
                swap32(lo, hi);
            };
            // accumulators two by two: of a row, then the last of two rows
            constexpr int ROW = HN / 2, ENDS = HN & 1 ? (HM + 1) / 2 : 0;
            if constexpr (EPI == GATED) {
                char* y = reinterpret_cast<char*>(a.y);
                auto offset = [&](int i) {
                    const int r = min(m * HM * 32 + row_in(i), a.M - 1);
                    return (uint32_t)(frag_at(r, hj0 * 8 + c4, a.N >> 1) * 2);
                };
                auto put = [&](char* p, bool ok, const f32x4& lo,
                               const f32x4& hi) {
                    f32x4 v;
                    #pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float z = a.gelu ? gelu_arg(lo[e]) : lo[e];
                        v[e] = over_1_and(lo[e], __expf(-z)) * hi[e];
                    }
                    if (ok) put4(reinterpret_cast<bf16*>(p), v);
                };
                #pragma unroll
                for (int i = 0; i < HM; i++) {
                    const bool ok = m * HM * 32 + row_in(i) < a.M;
                    char* p = y + offset(i) + upper * 512;
                    #pragma unroll
                    for (int j = 0; j < 2 * ROW; j += 2) {
                        f32x4 lo, hi;
                        pair(i, j, i, j + 1, lo, hi);
                        put(p + j * 512, ok && j + upper < live, lo, hi);
                    }
                    __builtin_amdgcn_sched_barrier(0);     // registers
                }
                #pragma unroll
                for (int e = 0; e < ENDS; e++) {
                    const int i0 = 2 * e, i1 = min(i0 + 1, HM - 1);
                    f32x4 lo, hi;
                    pair(i0, HN - 1, i1, HN - 1, lo, hi);
                    const int i = upper ? i1 : i0;
                    put(y + (upper ? offset(i1) : offset(i0)) + (HN - 1) * 512,
                        m * HM * 32 + (upper ? row_in(i1) : row_in(i0)) < a.M
                            && HN <= live && !(upper && i1 == i0), lo, hi);
                }
            } else {
                // A strip is one head's: a quarter of its pairs, or of its
                // values.
                static_assert(HN % 2 == 0);
                const Append& ap = a.ap;
                const int qt = ap.nl * 4, kt = ap.nkl * 4, t0 = hj0 >> 1;
                const int c = upper * 8 + c4;
                bf16x4 bias[ROW][2];
                if (a.bias)
                    #pragma unroll
                    for (int j = 0; j < ROW; j++) {
                        const bf16* b = a.bias + min(t0 + j, ns - 1) * 32 + c;
                        bias[j][0] = *reinterpret_cast<const bf16x4*>(b);
                        bias[j][1] = *reinterpret_cast<const bf16x4*>(b + 16);
                    }
                f32x4 turn[2][ROW][2];
                auto fetch = [&](int b, int i) {
                    const uint32_t o = row_pos[row_in(i)] * 64 + c;
                    #pragma unroll
                    for (int j = 0; j < ROW; j++) {
                        const int d = (t0 + j & 3) * 16;
                        turn[b][j][0] =
                            *reinterpret_cast<const f32x4*>(ap.cos_t + d + o);
                        turn[b][j][1] =
                            *reinterpret_cast<const f32x4*>(ap.sin_t + d + o);
                    }
                };
                fetch(0, 0);
                #pragma unroll
                for (int i = 0; i < HM; i++) {
                    if (i + 1 < HM) fetch((i + 1) & 1, i + 1);
                    const int row = m * HM * 32 + row_in(i);
                    const int64_t kv = (int64_t)row_kv[row_in(i)] * 128 + c;
                    const uint32_t q = row * a.N + c;
                    #pragma unroll
                    for (int j = 0; j < ROW; j++) {
                        f32x4 lo, hi;
                        pair(i, 2 * j, i, 2 * j + 1, lo, hi);
                        if (a.bias)
                            #pragma unroll
                            for (int e = 0; e < 4; e++) {
                                lo[e] += (float)bias[j][0][e];
                                hi[e] += (float)bias[j][1][e];
                            }
                        const int t = t0 + j;
                        if (t >= ns) continue;
                        if (t >= qt + kt) {        // values as they are
                            const int s = t - qt - kt;
                            bf16* p = ap.vp + (s >> 2) * ap.psz * 128
                                      + (s & 3) * 32;
                            if (row < a.M) {
                                put4(p + kv, lo);
                                put4(p + kv + 16, hi);
                            }
                            continue;
                        }
                        const f32x4 co = turn[i & 1][j][0];
                        const f32x4 si = turn[i & 1][j][1];
                        const f32x4 u = lo * co - hi * si;
                        const f32x4 v = hi * co + lo * si;
                        const int s = t < qt ? t : t - qt, d = (s & 3) * 16;
                        if (row >= a.M) continue;
                        if (t < qt) {
                            bf16* p = a.y + (s >> 2) * 128 + d;
                            put4(p + q, u);
                            put4(p + q + 64, v);
                        } else {
                            bf16* p = ap.kp + (s >> 2) * ap.psz * 128 + d;
                            put4(p + kv, u);
                            put4(p + kv + 64, v);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);     // registers
                }
            }
        }
        if (next_id >= 0) {
            lds_barrier();                 // every wave has read its rows
            keep_rows(m1);
        }
        // Stores count as loads do: none may be under way when the next tile
        // counts its own.  By then its first slabs have landed too.
        wait_loads<0>();
        if (next_id < 0) return;
        first += G;
        m = m1, n = n1, k = k1, q0 = p0, q1 = p1;
        #pragma unroll
        for (int i = 0; i < HM; i++)
            #pragma unroll
            for (int j = 0; j < HN; j++) acc[i][j] = f32x4{};
        // read again: 4 (HM + HN) registers less to keep through the epilogue
        #pragma unroll
        for (int i = 0; i < NF; i++) read(0, ic<0>{}, i);
    }
}

// Sums of a product in parts: y = res + sum of the parts, and sums of squares.
// A part is [16 rows, in pairs to 32][16 columns] accumulators as k_tile_gemm's
// lanes hold them.  A block takes 16 rows and a `pieces`-th of the columns, a
// wave four accumulators at a time with the loads of all of them and of the
// first KS parts under way.  What bounds it is the wait for those: others' caches
// held them.  us with the product, two parts under way before and all now: 128 x
// 4096 x 4096 in 4 parts 17.8 and 16.2, 128 x 3584 x 18944 in 4 48.3 and 46.6,
// 300 x 4096 x 14336 in 3 59.8 and 58.7.  y may be res: a lane reads
// only what it writes itself afterwards, and the padding of rows past M.
template <int BS, int KS>
__global__ __launch_bounds__(BS) void k_tile_fold(
    bf16* y, const bf16* res, float* __restrict__ sq,
    const float* __restrict__ part, int M, int N, int ks)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int r16 = lane & 15, g4 = lane >> 4;
    const int hi = blockIdx.x, pieces = gridDim.y;
    const int mh = gridDim.x, nh = N >> 4;
    const int row = (hi >> 1) * 32 + in_strip(hi & 1, r16);
    const int from = nh * blockIdx.y / pieces;
    const int to = nh * (blockIdx.y + 1) / pieces;
    const int64_t step = (int64_t)mh * nh * 256;
    float s2 = 0.f;
    constexpr int J = 4, W = BS / 64;
    for (int j0 = from + wid; j0 < to; j0 += J * W) {
        f32x4 v[KS][J];
        bf16x4 old[J];
        const float* p[J];
        int64_t at[J];
        #pragma unroll
        for (int i = 0; i < J; i++) {
            const int j = j0 + i * W < to ? j0 + i * W : j0;
            p[i] = part + ((int64_t)hi * nh + j) * 256 + lane * 4;
            at[i] = frag_at(row, (j >> 1) * 32 + in_strip(j & 1, 4 * g4), N);
            #pragma unroll
            for (int k = 0; k < KS; k++)
                v[k][i] = *reinterpret_cast<const f32x4*>(p[i] + k * step);
            old[i] = *reinterpret_cast<const bf16x4*>(res + at[i]);
        }
        __builtin_amdgcn_sched_barrier(0);     // all of them before any sum
        #pragma unroll
        for (int i = 0; i < J; i++) {
            f32x4 t = v[0][i];
            #pragma unroll
            for (int k = 1; k < KS; k++) t += v[k][i];
            for (int k = KS; k < ks; k++)
                t += *reinterpret_cast<const f32x4*>(p[i] + k * step);
            if (row >= M || j0 + i * W >= to) continue;
            #pragma unroll
            for (int e = 0; e < 4; e++) {
                t[e] += (float)old[i][e];
                s2 += t[e] * t[e];
            }
            put4(y + at[i], t);
        }
    }
    s2 += __shfl_xor(s2, 16, 64);
    s2 += __shfl_xor(s2, 32, 64);
    __shared__ float sum[BS / 64][16];
    if (lane < 16) sum[wid][lane] = s2;
    __syncthreads();
    if (threadIdx.x < 16 && row < M) {
        float s = 0.f;
        #pragma unroll
        for (int w = 0; w < BS / 64; w++) s += sum[w][threadIdx.x];
        sq[(int64_t)row * pieces + blockIdx.y] = s;
    }
}

// The same for a rotated product: x W^T of normed rows with its bias, queries
// rotated to y, keys and values to their pages.  A wave takes strips of 32
// columns, two at a time: a head's 16 pairs of dimensions, or its values.  What
// the 16 rows need is asked for ahead of the parts, every lane for its own row.
// Waits bound it; with the product in parts, 128 rows, us, and k_wstream_gemm,
// which rotates by itself: 6144 x 4096 22.9 and 25.0, 4608 x 3584 18.3 and 23.9.
template <int BS, int KS>
__global__ __launch_bounds__(BS) void k_tile_fold_rope(const TileArgs a)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int r16 = lane & 15, g4 = lane >> 4;
    const bool upper = g4 >> 1;
    const int c = upper * 8 + (g4 & 1) * 4;        // after the swap
    const Append& ap = a.ap;
    const int hi = blockIdx.x, mh = gridDim.x, nh = a.N >> 4, ns = a.N >> 5;
    const int row = (hi >> 1) * 32 + in_strip(hi & 1, r16);
    const int at = min(row, a.M - 1);
    const int from = ns * blockIdx.y / gridDim.y;
    const int to = ns * (blockIdx.y + 1) / gridDim.y;
    const int64_t step = (int64_t)mh * nh * 256;
    const int pos = ap.pos[at], slot = ap.slot[at];
    // sums of a row: eight side by side, as k_row_sums adds them up
    const float* sums = a.rstd + (int64_t)at * a.rstd_nt;
    float s2[2] = {};
    #pragma unroll 2
    for (int e = g4; e < a.rstd_nt; e += 8) {
        const float v = sums[min(e + 4, a.rstd_nt - 1)];
        s2[0] += sums[e];
        s2[1] += e + 4 < a.rstd_nt ? v : 0.f;
    }
    int64_t kv = 0;
    float rs = 0.f;
    const int qt = ap.nl * 4, kt = ap.nkl * 4;
    constexpr int J = 2, W = BS / 64;
    for (int j0 = from + wid; j0 < to; j0 += J * W) {
        f32x4 v[KS][J][2], turn[J][2];
        bf16x4 bias[J][2];
        const float* p[J];
        #pragma unroll
        for (int i = 0; i < J; i++) {
            const int t = j0 + i * W < to ? j0 + i * W : j0;
            p[i] = a.part + ((int64_t)hi * nh + 2 * t) * 256 + lane * 4;
            #pragma unroll
            for (int k = 0; k < KS; k++)
                #pragma unroll
                for (int h = 0; h < 2; h++)
                    v[k][i][h] = *reinterpret_cast<const f32x4*>(
                        p[i] + k * step + h * 256);
            if (a.bias)
                #pragma unroll
                for (int h = 0; h < 2; h++)
                    bias[i][h] = *reinterpret_cast<const bf16x4*>(
                        a.bias + t * 32 + c + h * 16);
            const int o = pos * 64 + (t & 3) * 16 + c;
            turn[i][0] = *reinterpret_cast<const f32x4*>(ap.cos_t + o);
            turn[i][1] = *reinterpret_cast<const f32x4*>(ap.sin_t + o);
        }
        if (j0 == from + wid) {            // the first time
            const int page = ap.ptab[slot * ap.maxp + pos / ap.psz];
            kv = ((int64_t)page * ap.nkl * ap.psz + pos % ap.psz) * 128 + c;
            #pragma unroll
            for (int h = 0; h < 2; h++) {
                s2[h] += __shfl_xor(s2[h], 16, 64);
                s2[h] += __shfl_xor(s2[h], 32, 64);
            }
            rs = rsqrtf((s2[0] + s2[1]) * a.inv_h + a.eps);
        }
        #pragma unroll
        for (int i = 0; i < J; i++) {
            const int t = j0 + i * W;
            f32x4 lo = v[0][i][0], hi2 = v[0][i][1];
            #pragma unroll
            for (int k = 1; k < KS; k++) {
                lo += v[k][i][0];
                hi2 += v[k][i][1];
            }
            for (int k = KS; k < a.ks; k++) {
                lo += *reinterpret_cast<const f32x4*>(p[i] + k * step);
                hi2 += *reinterpret_cast<const f32x4*>(p[i] + k * step + 256);
            }
            lo *= rs;
            hi2 *= rs;
            swap32(lo, hi2);
            if (a.bias)
                #pragma unroll
                for (int e = 0; e < 4; e++) {
                    lo[e] += (float)bias[i][0][e];
                    hi2[e] += (float)bias[i][1][e];
                }
            if (t >= to || row >= a.M) continue;
            if (t >= qt + kt) {
                const int s = t - qt - kt;
                bf16* d = ap.vp + (s >> 2) * ap.psz * 128 + (s & 3) * 32 + kv;
                put4(d, lo);
                put4(d + 16, hi2);
                continue;
            }
            const f32x4 u = lo * turn[i][0] - hi2 * turn[i][1];
            const f32x4 w = hi2 * turn[i][0] + lo * turn[i][1];
            const int s = t < qt ? t : t - qt, d = (s & 3) * 16;
            bf16* q = t < qt
                ? a.y + (int64_t)row * a.N + (s >> 2) * 128 + d + c
                : ap.kp + (s >> 2) * ap.psz * 128 + d + kv;
            put4(q, u);
            put4(q + 64, w);
        }
    }
}

// parts of sums of squares of a row, added up: eight lanes a row
__global__ __launch_bounds__(256) void k_row_sums(
    float* __restrict__ out, const float* __restrict__ in, int M, int nt)
{
    const int r = blockIdx.x * 32 + (threadIdx.x >> 3);
    float s = 0.f;
    if (r < M)
        #pragma unroll 4
        for (int e = threadIdx.x & 7; e < nt; e += 8)
            s += in[(int64_t)r * nt + e];
    s += __shfl_xor(s, 1, 64);
    s += __shfl_xor(s, 2, 64);
    s += __shfl_xor(s, 4, 64);
    if (r < M && (threadIdx.x & 7) == 0) out[r] = s;
}

template <int EPI>
int launch(TileArgs a, int hm, int hn, int cus, hipStream_t stream)
{
    const int items = a.mt * a.nt * a.ks;
    constexpr bool NORMED = EPI == GATED || EPI == ROPE;
    // blocks that live together: LDS holds two of the smallest tile
    constexpr int ALL = 160 * 1024;
    const int each = 2 * tile_lds(hm, hn, 0) <= ALL ? 2 : 1;
    const int room = cus * each;
    const int grid = (items < room ? items + 7 : room) / 8 * 8;
    // A block of several tiles takes one sum per row, and so does one without
    // room for more.  The launch that adds them up takes 3 us.
    const bool add_up = NORMED && a.rstd_nt > 1
        && (items > grid || a.rstd_nt > 256
            || tile_lds(hm, hn, a.rstd_nt) > ALL / each);
    a.rows_at = tile_rows_at(hm, hn, NORMED && !add_up ? a.rstd_nt : 1);
    const int lds = a.rows_at + hm * 32 * 12;
    auto go = [&](auto k) {
        // the same for every call: another thread may be between this and the
        // launch
        const hipError_t e = hipFuncSetAttribute(
            (const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize,
            ALL / each);
        if (e != hipSuccess) return (int)e;
        if (add_up) {
            k_row_sums<<<(a.M + 31) / 32, 256, 0, stream>>>(a.part, a.rstd,
                                                            a.M, a.rstd_nt);
            a.rstd = a.part;
            a.rstd_nt = 1;
        }
        k<<<grid, 256, lds, stream>>>(a);
        return (int)hipGetLastError();
    };
    #define TILE(A, B) \
        if (hm == A && hn == B) return go(k_tile_gemm<A, B, EPI>)
    TILE(8, 8);
    if constexpr (EPI != ROPE) TILE(9, 7);
    if constexpr (EPI != ROPE) TILE(7, 7);
    TILE(8, 6);
    TILE(10, 4);
    TILE(6, 6);
    TILE(8, 4);
    TILE(6, 4);
    TILE(4, 4);
    TILE(4, 2);
    if constexpr (EPI == RESIDUAL || EPI == ROPE || EPI == PARTS) TILE(2, 2);
    #undef TILE
    return -110;                            // no such tile
}

// in units of 32 rows and columns
constexpr int TILES[][2] = {{8, 8}, {9, 7}, {7, 7}, {8, 6}, {10, 4},
                            {6, 6}, {8, 4}, {6, 4}, {4, 4}, {4, 2}};

int div_up(int a, int b) { return (a + b - 1) / b; }
double pow8(double x) { x *= x; x *= x; return x * x; }

// us that a product takes, about the largest of what the busiest CU takes, a
// slab of 32 of K being bound by its products or its loads; of what all padded
// work draws at the power limit; and of reading the weights.  Parts cost a second
// launch, which reads them; what they cost is that of an earlier k_tile_fold (541
// x 4096 in 3 parts 13.0 us, now 8.4; 128 x 4096 in 4 6.1, now 4.9).
double estimate(int M, int N, int K, int hm, int hn, int ks, int cus)
{
    const int unit = 32 * tile_stages(hm, hn), area = hm * hn;
    const int items = div_up(M, 32 * hm) * div_up(N, 32 * hn) * ks;
    const double slabs = div_up(K / unit, ks) * unit / 32;
    const double slab = std::max(area * 0.00715, hm * 0.0239 + hn * 0.0223);
    const double busiest =
        div_up(items, cus) * (slabs * slab + 2.6 + area * 0.202);
    const double power =
        (double)items * area / cus * (slabs * 0.0079 + 0.202);
    const double t = sqrt(sqrt(sqrt(pow8(busiest) + pow8(power)
                                    + pow8((double)N * K * 4e-7))));
    return ks > 1 ? t + 3.0 + (double)ks * M * N * 1.5e-6 : t;
}

bool takes(int K, int epi, int hm, int hn)
{
    return K % (32 * tile_stages(hm, hn)) == 0 && !(epi == ROPE && hn % 2);
}

struct Choice { int hm, hn, ks; double us; };

Choice choose(int M, int N, int K, int epi, int cus)
{
    Choice best{0, 0, 0, INFINITY};
    for (const auto& [hm, hn] : TILES) {
        if (!takes(K, epi, hm, hn)) continue;
        const int unit = 32 * tile_stages(hm, hn);
        const int64_t tiles =
            (int64_t)div_up(M, 32 * hm) * div_up(N, 32 * hn);
        for (int ks = 1; ks <= (epi == RESIDUAL ? 8 : 1); ks++) {
            if (ks > 1 && (tiles * ks > 2.5 * cus || K / unit < 2 * ks)) break;
            const double t = estimate(M, N, K, hm, hn, ks, cus);
            if (t < best.us) best = {hm, hn, ks, t};
        }
    }
    return best;
}

}  // namespace

// The tiles of a product and its parts, hm | hn << 8 | ks << 16: those that the
// estimate likes best.  It was fitted to 6700 times of every tile at 24 numbers
// of rows from 129 to 8192 and the 11 matrices of the presets (3584 to 37888
// columns); at 25 others what it chooses for a layer takes 0.5 % more than the
// best choice on average and 4 % at most.  From 65 to 128 rows, weights not in
// cache, o and down of 3584 to 8192 columns: down 0 to 7 % more than the best;
// o of up to 4096 columns would take 5 to 20 % less over tiles of 64 x 64, which
// are not weighed there.
// Few rows are weights' reads: the smallest tiles, in as many parts as there are
// CUs but of no fewer than 1536 of K (64 rows of 4096 x 4096 and 4096 x 14336
// in cache, parts: 1 14.4 and more than 40, 2 12.5, 3 13.2 and 33.1, 4 13.3 and
// 29.1; not in cache 2 16.5, 4 14.9 and 29.9).
// On the host a choice takes 1.5 us; in Python it took 10 to 70, and a step of a
// new number of rows 90 us longer than the next one (four layers, 301 to 399).
extern "C" int tile_gemm_plan(int M, int N, int K, int epi, int cus)
{
    if (M < 1 || N < 32 || K < 128 || K % 128 || cus < 8 || epi < RESIDUAL
        || epi > ROPE)
        return -111;
    auto plan = [](int hm, int hn, int ks) { return hm | hn << 8 | ks << 16; };
    if (M <= 64 && epi != GATED && K % 256 == 0) {
        const int parts = std::min({cus / div_up(N, 64), K / 1536, 8});
        return plan(2, 2, epi == RESIDUAL ? std::max(1, parts) : 1);
    }
    const Choice c = choose(M, N, K, epi, cus);
    return c.hm ? plan(c.hm, c.hn, c.ks) : -110;
}

// A gated or rotated product of several rounds of tiles in two: as many of its
// rows as fill whole rounds of one size of tile, and the others over tiles of
// their own.  In one a last round takes as long whatever it has (2310 rows of
// 28672 x 4096 over 7 x 7 tiles: 5.5 rounds, 449 us; 576 rows over 9 x 7, one
// round, and 1734 over 7 x 7, four: 412).  us in one and in two:
//                    rows   1600       2310       3000       4500
//   28672 x 4096          296 283    449 412    539 522
//   37888 x 3584                     510 488
//   22016 x 4096          247 232               436 417    633 610
// A second launch takes 9 us by the estimate's measure, and two are to take 1 %
// less.  Over 96 random numbers of rows from 129 to 8192 and 12 matrices, 156 go in
// two and take 4.5 % less on average; five take 0.6 to 3.7 % more.
// Rows of the first | its tile << 24 | the others' tile << 40, each hm | hn << 8,
// or 0 for one launch.
extern "C" int64_t tile_gemm_split(int M, int N, int K, int epi, int cus)
{
    if (M <= 128 || N < 32 || K < 128 || K % 128 || cus < 8
        || (epi != GATED && epi != ROPE))
        return 0;
    const Choice one = choose(M, N, K, epi, cus);
    double least = one.us / 1.01 - 9.0;
    int64_t best = 0;
    for (const auto& [hm, hn] : TILES) {
        if (hm * hn < 40) break;               // no rounds of small tiles
        if (!takes(K, epi, hm, hn)) continue;
        const int columns = div_up(N, 32 * hn);
        for (int rows = 32 * hm, n = columns; rows < M;
             rows += 32 * hm, n += columns) {
            if (n < 0.92 * div_up(n, cus) * cus) continue;
            const double t = estimate(rows, N, K, hm, hn, 1, cus);
            if (t >= least) break;
            const Choice rest = choose(M - rows, N, K, epi, cus);
            if (t + rest.us >= least) continue;
            least = t + rest.us;
            best = rows | (int64_t)(hm | hn << 8) << 24
                   | (int64_t)(rest.hm | rest.hn << 8) << 40;
        }
    }
    return best;
}

// Tiles are hm x hn times 32 rows and columns.  epi: RESIDUAL (y = res + x W^T,
// sq), GATED (y = act(gate) * up of normed x), ROPE (normed x, positions, keys
// and values appended) or PARTS (y and sq come from part, ks parts of K).
extern "C" int tile_gemm_bf16(
    void* y, void* part, const void* x, const void* w, const void* bias,
    const void* res, void* sq, const void* rstd, int rstd_nt, float inv_h,
    float eps, int M, int N, int K, int epi, int hm, int hn, int ks, int gm,
    int pieces, int gelu, int cus, const void* rcos, const void* rsin,
    const void* pos, const void* slot, const void* ptab, void* kp, void* vp,
    int nl, int nkl, int psz, int maxp, hipStream_t stream)
{
    const int unit = 32 * tile_stages(hm, hn);     // of K
    const bool normed = epi == GATED || epi == ROPE;
    // fp32 parts, or a sum per row, where it comes in several
    const bool scratch = epi == PARTS || (normed && rstd_nt > 1);
    if (epi < RESIDUAL || epi > PARTS || M < 1 || N < 32 || N % 32
        || K < unit || K % unit || ks < 1 || ks > K / unit
        || (int64_t)(M + 31) * N >= (int64_t)1 << 31
        || gm < 1 || cus < 8 || (scratch && !part)
        || (normed && (!rstd || rstd_nt < 1))
        || (epi == PARTS ? pieces < 1 : ks != 1)
        || (epi == ROPE && N != (nl + 2 * nkl) * 128))
        return -111;
    TileArgs a{(bf16*)y, (float*)part, (const bf16*)x, (const bf16*)w,
               (const bf16*)bias, (const bf16*)res, (float*)sq,
               (const float*)rstd, rstd_nt, inv_h, eps, M, N, K,
               (M + hm * 32 - 1) / (hm * 32), (N + hn * 32 - 1) / (hn * 32),
               ks, gm, gelu,
               {(const float*)rcos, (const float*)rsin, (const int*)pos,
                (const int*)slot, (const int*)ptab, (bf16*)kp, (bf16*)vp,
                nl, nkl, psz, maxp}};
    if (epi == RESIDUAL) return launch<RESIDUAL>(a, hm, hn, cus, stream);
    if (epi == GATED) return launch<GATED>(a, hm, hn, cus, stream);
    if (epi == ROPE) return launch<ROPE>(a, hm, hn, cus, stream);
    if (const int e = launch<PARTS>(a, hm, hn, cus, stream)) return e;
    const dim3 grid((M + 31) / 32 * 2, pieces);
    #define FOLD(KS) \
        case KS: k_tile_fold<256, KS><<<grid, 256, 0, stream>>>( \
            (bf16*)y, (const bf16*)res, (float*)sq, (const float*)part, M, N, \
            ks); break
    switch (std::min(ks, 8)) {
        FOLD(1); FOLD(2); FOLD(3); FOLD(4); FOLD(5); FOLD(6); FOLD(7); FOLD(8);
    }
    #undef FOLD
    return (int)hipGetLastError();
}

// The same over rows that are normed already: y = act(gate) * up in fragment
// layout (GATED), x W^T in rows (ROWS) or its ks parts in fp32 (ROW_PARTS).
extern "C" int tile_rows_bf16(
    void* y, void* part, const void* x, const void* w, int M, int N, int K,
    int epi, int hm, int hn, int ks, int gm, int gelu, int cus,
    hipStream_t stream)
{
    const int unit = 32 * tile_stages(hm, hn);     // of K
    if ((epi != GATED && epi != ROWS && epi != ROW_PARTS) || M < 1 || N < 32
        || N % 32 || K < unit || K % unit || ks < 1 || ks > K / unit
        || (int64_t)(M + 31) * N >= (int64_t)1 << 31 || gm < 1 || cus < 8
        || (epi != ROW_PARTS && ks != 1) || !(epi == ROW_PARTS ? part : y))
        return -111;
    TileArgs a{};
    a.y = (bf16*)y, a.part = (float*)part;
    a.x = (const bf16*)x, a.w = (const bf16*)w;
    a.M = M, a.N = N, a.K = K;
    a.mt = div_up(M, hm * 32), a.nt = div_up(N, hn * 32), a.ks = ks;
    a.gm = gm, a.gelu = gelu;
    if (epi == GATED) return launch<GATED>(a, hm, hn, cus, stream);
    if (epi == ROWS) return launch<ROWS>(a, hm, hn, cus, stream);
    return launch<ROW_PARTS>(a, hm, hn, cus, stream);
}

// As tile_gemm_bf16's ROPE, the product in ks parts of K.  part: ks times the
// rows, in 32s, times N.
extern "C" int tile_rope_parts_bf16(
    void* y, void* part, const void* x, const void* w, const void* bias,
    const void* rstd, int rstd_nt, float inv_h, float eps, int M, int N, int K,
    int hm, int hn, int ks, int gm, int cus, const void* rcos,
    const void* rsin, const void* pos, const void* slot, const void* ptab,
    void* kp, void* vp, int nl, int nkl, int psz, int maxp,
    hipStream_t stream)
{
    const int unit = 32 * tile_stages(hm, hn);     // of K
    if (M < 1 || N != (nl + 2 * nkl) * 128 || N < 32 || K < unit || K % unit
        || ks < 1 || ks > K / unit || (int64_t)(M + 31) * N >= (int64_t)1 << 31
        || gm < 1 || cus < 8 || !part || !rstd || rstd_nt < 1)
        return -111;
    TileArgs a{};
    a.y = (bf16*)y, a.part = (float*)part, a.x = (const bf16*)x;
    a.w = (const bf16*)w, a.bias = (const bf16*)bias;
    a.rstd = (const float*)rstd, a.rstd_nt = rstd_nt;
    a.inv_h = inv_h, a.eps = eps, a.M = M, a.N = N, a.K = K;
    a.mt = div_up(M, hm * 32), a.nt = div_up(N, hn * 32), a.ks = ks;
    a.gm = gm;
    a.ap = {(const float*)rcos, (const float*)rsin, (const int*)pos,
            (const int*)slot, (const int*)ptab, (bf16*)kp, (bf16*)vp,
            nl, nkl, psz, maxp};
    if (const int e = launch<PARTS>(a, hm, hn, cus, stream)) return e;
    // a wave's two strips at a time, once
    const dim3 grid(div_up(M, 32) * 2, std::max(1, N / 256));
    #define FOLD(KS) \
        case KS: k_tile_fold_rope<256, KS><<<grid, 256, 0, stream>>>(a); break
    switch (std::min(ks, 4)) { FOLD(1); FOLD(2); FOLD(3); FOLD(4); }
    #undef FOLD
    return (int)hipGetLastError();
}
