// MFMA GEMM for operands whose rows start anywhere (Float16, BFloat16, Float32, Int8 / UInt8):  C (+)= op(A) . op(B)
//
// The DMA-fed ring kernels (gemm_ring_impl.h) need rows of whole 16-byte chunks.  A product that misses this -- an odd k or n, a view
// that starts inside a chunk, a table of pointers nobody vouches for -- runs here, straight from where its operands lie: 16 bytes per lane
// and load at whatever element the row starts on (global memory takes unaligned vector accesses), through registers into LDS in the layouts
// of the ring kernels, and from there the same fragment reads and the same matrix instructions in the same order of k: the same bits.
//
//   * 64 x 64, 128 x 64 or 128 x 128 tiles, four wavefronts of WBM x WBN blocks of 32 x 32; a K-step is 128 bytes of k per row.
//   * DEPTH K-steps of loads in flight per thread (registers), two LDS stages, one barrier per K-step: while a K-step is multiplied the next one
//     is written to the other stage.  Every load is unconditional.  In the last K-step a chunk that the end of its row cuts off is loaded from the
//     row's last 16 bytes and shifted into place on its way to LDS, which also fills it up with zeros; before it nothing is shifted, also on the
//     edge of M and N, so one loop serves every tile (shifting there behind a test per chunk made the compiler wait for each load by itself, and
//     the tiles on the edge set the pace: 1023 x 1537 x 1985 on 128 x 128 31.3 -> 26.5 us).  Rows past the edge
//     repeat the last one; their sums are never stored.
//   * The sums go through LDS to memory, eight consecutive columns per lane.
//   * k ranges (krange_items, k_total): the last range is what is left, ranges write sums in 32 bits (C_PARTIAL).
//   * FOLD (fold_steps): a batch whose tiles fill the CUs runs the k ranges of its item inside one workgroup, which adds up each range's sums in
//     registers, from C0 or the bias on, as the second pass over partial sums does: the bits of the item alone, nothing through memory.
//
// What bounds it: the latency of the loads where few tiles have a deep k (hence the k ranges, and 64 x 64 tiles that put several workgroups
// on every CU), the LDS of the CU where there are many (64 x 64 tiles read 256 bytes of LDS per cycle of MFMA, twice what it delivers).
// Operands that no cache holds arrive at the latency of the two or three K-steps in flight: Float16 1023 x 1537 x 2049 26.8 us in cache, 28.5 cycled through
// 0.8 GB, 32.6 alone behind a sweep of the caches (padded copies, which stream them in: 29.5, 31 and 34.6).
// Measured, the register-staged kernel with element-wise loads (or the vector ALU, Int8) before -> now: BFloat16 448 x 3704 x 166 A^T.B 263 -> 10.8 us,
// 576 x 3797 x 448 226 -> 12.8, 2429 x 1536 x 157 77 -> 13.5, 3712 x 543 x 448 45 -> 9.9; Float32 128 x 6463 x 720 218 -> 24,
// 1000 x 774 x 64 35 -> 9.8, 2049^3 213 (padded copies) -> 187; Int8 256 x 1792 x 39 198 -> 8.2 us.
#pragma once
#include "gemm_ring_impl.h"

namespace ntg {

// 16 bytes at any element
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(1)));
typedef uint32_t u32x2_any __attribute__((ext_vector_type(2), aligned(1)));

// the 16 bytes moved down by `bytes` (0 .. 16), zeros from above
__device__ __forceinline__ u32x4 shift_down(u32x4 v, int bytes) {
    const uint64_t lo = (uint64_t)v[0] | ((uint64_t)v[1] << 32), hi = (uint64_t)v[2] | ((uint64_t)v[3] << 32);
    const int s = 8 * (bytes & 7);
    const uint64_t l1 = s ? (lo >> s) | (hi << (64 - s)) : lo, h1 = hi >> s;
    const uint64_t rl = bytes >= 16 ? 0 : bytes >= 8 ? h1 : l1, rh = bytes >= 8 ? 0 : h1;
    return u32x4{(uint32_t)rl, (uint32_t)(rl >> 32), (uint32_t)rh, (uint32_t)(rh >> 32)};
}

// One operand's share of a thread: NV chunks of 16 bytes per K-step of its 64 WB x (128 bytes of k) tile
template <bool KC, int WB, int ES>
struct AnyOperand {
    static constexpr int VEL = 16 / ES, BK = 128 / ES, NV = 2 * WB;
    static constexpr int ROW = 64 * WB * ES;             // bytes of one k-row of an M/N-contiguous tile
    static constexpr int CH = ROW / 16;                  // 16-byte chunks in it (4 .. 32)
    static constexpr int RSTEP = KC ? 32 : 256 / CH;     // rows (K-contiguous) / k-rows from one chunk of a thread to its next; the 16 bytes of the row stay
    const NTG_GLOBAL char* base;                         // the tile's first element at the first k
    const NTG_GLOBAL char* base_last;                    // ... at k = K - BK (K-contiguous: it may lie before the row, the offsets lead back) / last * BK
    int64_t adv;
    uint32_t pitch;                                      // bytes from a stored row to the next
    uint32_t off[KC ? NV : 1];                           // byte offsets of the chunks (M/N-contiguous: of the first, the others RSTEP rows apart)
    uint32_t last_step;                                  // what the last K-step adds to them
    int krow, kr;                                        // M/N-contiguous: k-row of the first chunk; k-rows that exist in the last K-step
    int lds, cut;                                        // LDS bytes of the first chunk; bytes to shift it down by in the last K-step (16: nothing of it exists)
    bool cut_last;                                       // (uniform) some chunk of the last K-step does not exist as a whole

    __device__ __forceinline__ void setup(const NTG_GLOBAL char* first, int64_t ld, int mn0, int MN, int K, int last, int tid) {
        kr = K - last * BK;
        pitch = (uint32_t)(ld * ES);
        if constexpr (KC) {
            base = first + (int64_t)mn0 * ld * ES;
            base_last = base + (int64_t)(K - BK) * ES;
            adv = 128;
            cut_last = kr < BK;
            const int row = tid >> 3, slot = tid & 7;
            const int k = last * BK + slot * VEL, at = k < K - VEL ? k : K - VEL;           // (K - BK <= at: what base_last lacks is not negative)
            last_step = (uint32_t)((at - (K - BK) - slot * VEL) * ES);
            cut = (k - at) * ES < 16 ? (k - at) * ES : 16;
            lds = row * 128 + ((slot ^ swz8(row)) << 4);                                    // (swz8 repeats every 16 rows)
            krow = 0;
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int r = mn0 + row + 32 * i < MN ? row + 32 * i : MN - 1 - mn0;
                off[i] = (uint32_t)r * pitch + (uint32_t)(slot * 16);
            }
        } else {
            // (the offsets carry VEL elements: the chunk may start before the tile where its columns are fewer than a chunk; the matrix has VEL of them)
            base = first + (int64_t)mn0 * ES - 16;
            base_last = base + (int64_t)last * BK * ld * ES;
            adv = (int64_t)BK * ld * ES;
            cut_last = kr < BK || mn0 + 64 * WB > MN;
            krow = tid / CH;
            // A chunk that the end of its row cuts off runs on into the next k-row, which holds a chunk at least: the columns past the edge are sums
            // of their own, which nobody stores.  Only the last k-row has none behind it: the last K-step loads that chunk from the row's last 16 bytes.
            const int c = tid % CH, mn = mn0 + c * VEL, at = mn < MN - VEL ? mn : MN - VEL, on = mn < MN ? mn : MN - VEL;
            cut = (mn - at) * ES < 16 ? (mn - at) * ES : 16;
            off[0] = (uint32_t)krow * pitch + (uint32_t)((on - mn0 + VEL) * ES);
            last_step = (uint32_t)((at - on) * ES);
            const int sw = ES == 2 ? 2 * (krow & 3) : ES == 4 ? 8 * (krow & 1) : mn8_swizzle<CH>(krow);      // (the same for krow + RSTEP)
            lds = krow * ROW + ((c ^ sw) << 4);
        }
    }
    __device__ __forceinline__ void load(u32x4& v, int i, int kt, int last) const {
        const bool l = kt >= last;                                 // (uniform; K-steps past the end load the last one again)
        const NTG_GLOBAL char* b = l ? base_last : base + (int64_t)kt * adv;
        uint32_t o;
        if constexpr (KC) o = off[i] + (l ? last_step : 0u);
        else {
            // (the last k-row once more in the place of those that do not exist)
            int k = krow + RSTEP * i;
            if (l) k = k < kr ? k : kr - 1;
            o = off[0] + (uint32_t)(k - krow) * pitch + (l ? last_step : 0u);
        }
        v = *(const NTG_GLOBAL u32x4_any*)(b + o);
    }
    // cut_off: the last K-step, and some chunk of it does not exist as a whole (uniform)
    __device__ __forceinline__ void store(char* tile, const u32x4& v, int i, bool cut_off) const {
        char* to = tile + lds + RSTEP * (KC ? 128 : ROW) * i;
        if (cut_off) *reinterpret_cast<u32x4*>(to) = shift_down(v, KC || krow + RSTEP * i < kr ? cut : 16);
        else *reinterpret_cast<u32x4*>(to) = v;
    }
};

template <int DT, bool TA, bool TB, int WBM, int WBN, bool FOLD>
__global__ void __launch_bounds__(256, WBM == 1 ? 3 : 2) gemm_any_kernel(const GemmParams p) {
    using E = Elem<DT>;
    using T = typename E::T;
    using AccV = typename E::AccV;
    using AccS = typename E::AccS;
    constexpr int ES = (int)sizeof(T), BK = 128 / ES, TM = 64 * WBM, TN = 64 * WBN, WTM = 32 * WBM, WTN = 32 * WBN, TILE_A = TM * 128, STAGE = TILE_A + TN * 128;
    constexpr int DEPTH = WBN == 1 ? 3 : 2;
    constexpr bool CHAIN = std::is_same<T, float>::value;          // Float32: the chain starts from C0 / the bias, the epilogue only stores
    using OA = AnyOperand<!TA, WBM, ES>;
    using OB = AnyOperand<TB, WBN, ES>;
    __shared__ __attribute__((aligned(1024))) char lds[2 * STAGE]; // two stages of an A and a B tile
    if (p.gate && *p.gate != p.gate_want) return;                  // (uniform: the other kernel of a gated pair does this product)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave >> 1, wn = wave & 1;
    const int lid = xcd_contiguous_id(blockIdx.x, gridDim.x);
    const int tiles = p.tiles_m * p.tiles_n, b = lid / tiles;
    int tm, tn;
    tile_coords(lid - b * tiles, p.tiles_m, p.tiles_n, 4, tm, tn);
    const int m0 = tm * TM, n0 = tn * TN;
    int K = p.K;
    if (p.k_total) {                                               // (uniform) the last k range is what is left
        const int left = p.k_total - b / p.krange_items * p.K;
        if (left < K) K = left;
    }
    const gptr<char> A = (gptr<char>)(p.Aptr ? static_cast<const char*>(((gptr<const void*>)p.Aptr)[b])
                                             : static_cast<const char*>(p.A) + operand_offset(p, b, p.sA, p.sAk) * ES);
    const gptr<char> B = (gptr<char>)(p.Bptr ? static_cast<const char*>(((gptr<const void*>)p.Bptr)[b])
                                             : static_cast<const char*>(p.B) + operand_offset(p, b, p.sB, p.sBk) * ES);
    // (C_PARTIAL: a matrix of 32-bit sums)
    const int64_t ces = p.cmode == C_PARTIAL ? 4 : ES;
    const gptr_mut<char> C = (gptr_mut<char>)(p.Cptr ? static_cast<char*>(((gptr<void*>)p.Cptr)[b]) : static_cast<char*>(p.C) + (int64_t)b * p.sC * ces);
    const NTG_GLOBAL T* bias = (const NTG_GLOBAL T*)static_cast<const T*>(p.bias) + (int64_t)b * p.bias_bs;

    AccV acc[WBM][WBN], tot[FOLD ? WBM : 1][FOLD ? WBN : 1];
#pragma unroll
    for (int i = 0; i < WBM; ++i)
#pragma unroll
        for (int j = 0; j < WBN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[i][j][r] = (AccS)0;
                if constexpr (FOLD) tot[i][j][r] = (AccS)0;
            }
    if constexpr (CHAIN || FOLD) {
        if (p.cmode == C_ACCUMULATE || p.cmode == C_BIAS) {        // (uniform)
            const bool from_c = p.cmode == C_ACCUMULATE;
#pragma unroll
            for (int i = 0; i < WBM; ++i)
#pragma unroll
                for (int j = 0; j < WBN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        // (addresses clamped into C / the bias: what lies past the edge is not stored)
                        int m = m0 + wm * WTM + 32 * i + (lane & 31), n = n0 + wn * WTN + 32 * j + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                        m = m < p.M ? m : p.M - 1;
                        n = n < p.N ? n : p.N - 1;
                        const AccS c0 = (AccS)(from_c ? ((gptr<T>)C)[(int64_t)m * p.ldc + n] : bias[(int64_t)m * p.bias_rs + (int64_t)n * p.bias_cs]);
                        if constexpr (FOLD) tot[i][j][r] = c0;
                        else acc[i][j][r] = c0;
                    }
        }
    }

    const int KT = (K + BK - 1) / BK, last = KT - 1;
    OA a;
    OB bb;
    a.setup(A, p.lda, m0, p.M, K, last, tid);
    bb.setup(B, p.ldb, n0, p.N, K, last, tid);
    constexpr int NVA = OA::NV, NVB = OB::NV;
    u32x4 ra[DEPTH][NVA], rb[DEPTH][NVB];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
#pragma unroll
        for (int i = 0; i < NVA; ++i) a.load(ra[d][i], i, d, last);
#pragma unroll
        for (int i = 0; i < NVB; ++i) bb.load(rb[d][i], i, d, last);
    }

    // fragments of 16 bytes of k per lane for quarter-step ks (0 .. 3), as the ring kernels read them
    auto read_a_or_b = [&](auto& f, const char* tile, auto kc_tag, auto wb_tag, int wbase, int ks) __attribute__((always_inline)) {
        constexpr bool KC = decltype(kc_tag)::value;
        constexpr int WB = decltype(wb_tag)::value, ROW = 64 * WB * ES;
#pragma unroll
        for (int blk = 0; blk < WB; ++blk) {
            const int mn = wbase + 32 * blk;
            if constexpr (KC && ES != 4) {
                f[blk] = *reinterpret_cast<const u32x4*>(tile + (mn + (lane & 31)) * 128 + (((2 * ks + (lane >> 5)) ^ swz8(lane & 31)) << 4));
            } else if constexpr (KC) {
                // Float32: element e is k = 2 e + lane / 32 of the quarter-step
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    f[blk][e] = *reinterpret_cast<const uint32_t*>(tile + (mn + (lane & 31)) * 128 + (((2 * ks + (e >> 1)) ^ swz8(lane & 31)) << 4) +
                                                                   8 * (e & 1) + 4 * (lane >> 5));
            } else if constexpr (ES == 4) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    f[blk][e] = *reinterpret_cast<const uint32_t*>(tile + (8 * ks + 2 * e + (lane >> 5)) * ROW + (((mn + (lane & 31)) * 4) ^ (128 * (lane >> 5))));
            } else if constexpr (ES == 2) {
                const int bl = lane >> 4, s = lane & 15, e = s >> 2, q = s & 3;
                const int mnl = mn + 16 * (bl & 1) + 4 * q;
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    const int krow = 16 * ks + 8 * (bl >> 1) + 4 * half + e;
                    const shortx4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (__attribute__((address_space(3))) shortx4*)(tile + krow * ROW + (((mnl >> 3) ^ (2 * e)) << 4) + (mnl & 7) * 2));
                    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                    const u32x2 w = __builtin_bit_cast(u32x2, v);
                    f[blk][2 * half] = w[0];
                    f[blk][2 * half + 1] = w[1];
                }
            } else {
                const int grp = lane >> 4, i = lane & 15;
                const int mnl = mn + 16 * (grp & 1) + 8 * (i & 1);
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const int krow = 32 * ks + 16 * (grp >> 1) + 8 * t + (i >> 1);
                    const intx2v v = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                        (__attribute__((address_space(3))) intx2v*)(tile + krow * ROW + (((mnl >> 4) ^ mn8_swizzle<ROW / 16>(krow)) << 4) + (mnl & 15)));
                    f[blk][2 * t] = (uint32_t)v[0];
                    f[blk][2 * t + 1] = (uint32_t)v[1];
                }
            }
        }
    };
    int fold_at = p.fold_steps - 1;                                // FOLD: the K-step that ends the range
    // K-step kt out of its stage; behind each quarter's matrix instructions a quarter of the chunks of K-step kt + 1 (set d) goes to the other
    // stage, which was last read before this K-step's barrier, and with MORE the loads of K-step kt + 1 + DEPTH take their registers
    auto step = [&](int kt, int d, auto more_tag) __attribute__((always_inline)) {
        constexpr bool MORE = decltype(more_tag)::value;         // (false: kt + 1 may be the last K-step)
        const char* sa = lds + (kt & 1) * STAGE;
        char* nx = lds + (~kt & 1) * STAGE;
        const bool lastk = !MORE && kt + 1 == last, cut_a = lastk && a.cut_last, cut_b = lastk && bb.cut_last;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        u32x4 fa[2][WBM], fb[2][WBN];
        using KCA = std::integral_constant<bool, !TA>;
        using KCB = std::integral_constant<bool, TB>;
        using WA = std::integral_constant<int, WBM>;
        using WB = std::integral_constant<int, WBN>;
        read_a_or_b(fa[0], sa, KCA{}, WA{}, wm * WTM, 0);
        read_a_or_b(fb[0], sa + TILE_A, KCB{}, WB{}, wn * WTN, 0);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            if (ks < 3) {
                read_a_or_b(fa[(ks + 1) & 1], sa, KCA{}, WA{}, wm * WTM, ks + 1);
                read_a_or_b(fb[(ks + 1) & 1], sa + TILE_A, KCB{}, WB{}, wn * WTN, ks + 1);
            }
#pragma unroll
            for (int i = 0; i < WBM; ++i)
#pragma unroll
                for (int j = 0; j < WBN; ++j) {
                    // (the operands swapped: a lane holds four consecutive columns of one row of C)
                    if constexpr (ES == 4 && CHAIN) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const uint32_t x = fb[ks & 1][j][e], y = fa[ks & 1][i][e];
                            E::mma(acc[i][j], __builtin_bit_cast(float, x), __builtin_bit_cast(float, y));
                        }
                    } else {
                        E::mma(acc[i][j], fb[ks & 1][j], fa[ks & 1][i]);
                    }
                }
            if (MORE || kt < last) {
#pragma unroll
                for (int c = ks * (NVA + NVB) / 4; c < (ks + 1) * (NVA + NVB) / 4; ++c) {       // A's chunks, then B's
                    const int i = c < NVA ? c : c - NVA;
                    if (c < NVA) {
                        a.store(nx, ra[d][i], i, cut_a);
                        if constexpr (MORE) a.load(ra[d][i], i, kt + 1 + DEPTH, last);
                    } else {
                        bb.store(nx + TILE_A, rb[d][i], i, cut_b);
                        if constexpr (MORE) bb.load(rb[d][i], i, kt + 1 + DEPTH, last);
                    }
                }
            }
        }
        if constexpr (FOLD) {
            if (kt == fold_at || kt == last) {                     // (uniform)
                fold_at += p.fold_steps;
#pragma unroll
                for (int i = 0; i < WBM; ++i)
#pragma unroll
                    for (int j = 0; j < WBN; ++j)
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            tot[i][j][r] += acc[i][j][r];
                            acc[i][j][r] = (AccS)0;
                        }
            }
        }
    };
    {
        const bool cut_a = last == 0 && a.cut_last, cut_b = last == 0 && bb.cut_last;
#pragma unroll
        for (int i = 0; i < NVA; ++i) {
            a.store(lds, ra[0][i], i, cut_a);
            a.load(ra[0][i], i, DEPTH, last);
        }
#pragma unroll
        for (int i = 0; i < NVB; ++i) {
            bb.store(lds + TILE_A, rb[0][i], i, cut_b);
            bb.load(rb[0][i], i, DEPTH, last);
        }
    }
    // (K-step kt + 1 is in set (kt + 1) % DEPTH; the rounds end before the last K-step is written to LDS)
    int kt = 0;
    for (; kt + DEPTH <= last - 1; kt += DEPTH)
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) step(kt + d, (d + 1) % DEPTH, std::true_type{});
#pragma unroll
    for (int d = 0; d < DEPTH + 1; ++d)
        if (kt + d <= last) step(kt + d, (d + 1) % DEPTH, std::false_type{});     // (uniform)

    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();                                  // all fragments read: LDS is free for the sums
    asm volatile("" ::: "memory");
    // ---- epilogue: [row][TN sums of 4 bytes], 16-byte slot s of row r at s ^ (r & 7) ----
    typedef AccS accx4 __attribute__((ext_vector_type(4)));
    typedef AccS accx4_any __attribute__((ext_vector_type(4), aligned(4)));
    constexpr int SROW = TN * 4;
    static_assert(TM * SROW <= 2 * STAGE, "the sums fit into the stages");
#pragma unroll
    for (int i = 0; i < WBM; ++i)
#pragma unroll
        for (int j = 0; j < WBN; ++j)
#pragma unroll
            for (int rq = 0; rq < 4; ++rq) {
                const int row = wm * WTM + 32 * i + (lane & 31), slot = (wn * WTN + 32 * j) / 4 + 2 * rq + (lane >> 5);
                const AccV& s = FOLD ? tot[FOLD ? i : 0][FOLD ? j : 0] : acc[i][j];
                *reinterpret_cast<accx4*>(lds + row * SROW + ((slot ^ (row & 7)) << 4)) = accx4{s[4 * rq], s[4 * rq + 1], s[4 * rq + 2], s[4 * rq + 3]};
            }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    constexpr int LPR = TN / 8;                                    // lanes per row, eight columns each
#pragma unroll
    for (int t = 0; t < TM * LPR / 256; ++t) {
        const int idx = tid + 256 * t, row = idx / LPR, g = idx % LPR;
        const int m = m0 + row, n = n0 + 8 * g;
        const accx4 lo = *reinterpret_cast<const accx4*>(lds + row * SROW + (((2 * g) ^ (row & 7)) << 4));
        const accx4 hi = *reinterpret_cast<const accx4*>(lds + row * SROW + (((2 * g + 1) ^ (row & 7)) << 4));
        AccS v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        if (m >= p.M || n >= p.N) continue;
        const bool whole = n + 8 <= p.N;
        if (p.cmode == C_PARTIAL) {                                // (rows of whole 16-byte chunks: what lies past column N is not read as a sum)
            NTG_GLOBAL AccS* wp = (NTG_GLOBAL AccS*)C + (int64_t)m * p.ldc + n;
            *(NTG_GLOBAL accx4*)wp = lo;
            if (n + 4 < p.N) *(NTG_GLOBAL accx4*)(wp + 4) = hi;
            continue;
        }
        NTG_GLOBAL T* cp = (NTG_GLOBAL T*)C + (int64_t)m * p.ldc + n;
        if constexpr (!CHAIN && !FOLD) {
            if (p.cmode == C_ACCUMULATE) {
                if (whole) {
                    if constexpr (ES == 2) {
                        const u32x4 c = *(const NTG_GLOBAL u32x4_any*)cp;
#pragma unroll
                        for (int e = 0; e < 8; ++e) v[e] += Cvt16<DT>::up((uint16_t)(c[e >> 1] >> (16 * (e & 1))));
                    } else {
                        const u32x2_any c = *(const NTG_GLOBAL u32x2_any*)cp;
#pragma unroll
                        for (int e = 0; e < 8; ++e) v[e] += (AccS)((c[e >> 2] >> (8 * (e & 3))) & 0xffu);
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (n + e < p.N) v[e] += (AccS)cp[e];
                }
            } else if (p.cmode == C_BIAS) {
                const NTG_GLOBAL T* bp = bias + (int64_t)m * p.bias_rs + (int64_t)n * p.bias_cs;
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (n + e < p.N) v[e] += (AccS)bp[(int64_t)e * p.bias_cs];
            }
        }
        if constexpr (ES != 1) {
            if (p.act == ACT_RELU) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = v[e] > (AccS)0 ? v[e] : (AccS)0;
            }
        }
        if (!whole) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (n + e < p.N) cp[e] = (T)v[e];
        } else if constexpr (ES == 2) {
            u32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (uint32_t)Cvt16<DT>::down(v[2 * e]) | ((uint32_t)Cvt16<DT>::down(v[2 * e + 1]) << 16);
            *(NTG_GLOBAL u32x4_any*)cp = o;
        } else if constexpr (ES == 1) {
            u32x2_any o;                                           // the low 8 bits of each sum
#pragma unroll
            for (int h = 0; h < 2; ++h)
                o[h] = ((uint32_t)v[4 * h] & 0xffu) | (((uint32_t)v[4 * h + 1] & 0xffu) << 8) | (((uint32_t)v[4 * h + 2] & 0xffu) << 16) | ((uint32_t)v[4 * h + 3] << 24);
            *(NTG_GLOBAL u32x2_any*)cp = o;
        } else {
            *(NTG_GLOBAL accx4_any*)cp = accx4{v[0], v[1], v[2], v[3]};
            *(NTG_GLOBAL accx4_any*)(cp + 4) = accx4{v[4], v[5], v[6], v[7]};
        }
    }
}

template <int DT, int WBM, int WBN, bool FOLD>
static hipError_t launch_any_wb(bool ta, bool tb, const GemmParams& pin, hipStream_t s) {
    GemmParams p = pin;
    p.tiles_m = (p.M + 64 * WBM - 1) / (64 * WBM);
    p.tiles_n = (p.N + 64 * WBN - 1) / (64 * WBN);
    const int64_t blocks = (int64_t)p.tiles_m * p.tiles_n * p.batch;
    if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
    const dim3 g((unsigned)blocks), t(256);
    if (ta && tb) hipLaunchKernelGGL((gemm_any_kernel<DT, true, true, WBM, WBN, FOLD>), g, t, 0, s, p);
    else if (ta) hipLaunchKernelGGL((gemm_any_kernel<DT, true, false, WBM, WBN, FOLD>), g, t, 0, s, p);
    else if (tb) hipLaunchKernelGGL((gemm_any_kernel<DT, false, true, WBM, WBN, FOLD>), g, t, 0, s, p);
    else hipLaunchKernelGGL((gemm_any_kernel<DT, false, false, WBM, WBN, FOLD>), g, t, 0, s, p);
    return hipGetLastError();
}
template <int DT, bool FOLD>
static hipError_t launch_any_tile(bool ta, bool tb, const GemmParams& p, hipStream_t s) {
    // 128 x 128 tiles where these reach three quarters of the CUs (BFloat16 3618 x 739 x 9392: 84 us against 112 on 128 x 64 and 126 on 64 x 64;
    // 2429 x 1536 x 157, 38 tiles: 23 against 12), 128 x 64 where those put one on each CU at most and 64 x 64 more than one (Float16 1023 x 1537 x
    // 1985: 18.6 us against 21.6 and 26.5 on 128 x 128), and 128 x 128 again from half of the CUs on where 128 x 64 would need a second round.  That last line
    // on 21 shapes of 128 .. 191 tiles, single and batched, every storage form, BFloat16 and Int8: the best of the three or within 2 % of it (BFloat16 1023 x
    // 1537 x 2049 26.8 us, 29.4 on 128 x 64, 29.3 on 64 x 64; 1281 x 3001 x 1667 43.6 / 52.2 / 51.4; 6 x (513 x 1537 x 641) 27.3 / 31.6 / 29.5; 2049 x 515 x 1281 14.6 / 15.2 /
    // 14.3).  Float32 always on 64 x 64: the matrix pipe is its bound on either and the smaller tile spreads evenly (2049^3: 188 us against 274).
    if constexpr (DT != DT_F32) {
        auto tiles = [&](int r, int c) { return (int64_t)((p.M + r - 1) / r) * ((p.N + c - 1) / c) * p.batch; };
        if (p.M > 64 && p.N > 64 && (tiles(128, 128) >= 192 || (tiles(128, 128) >= 128 && tiles(128, 64) > 256))) return launch_any_wb<DT, 2, 2, FOLD>(ta, tb, p, s);
        if (p.M > 64 && tiles(64, 64) > 256 && tiles(128, 64) <= 256) return launch_any_wb<DT, 2, 1, FOLD>(ta, tb, p, s);
    }
    return launch_any_wb<DT, 1, 1, FOLD>(ta, tb, p, s);
}
template <int DT>
static hipError_t launch_any(bool ta, bool tb, const GemmParams& p, hipStream_t s) {
    if constexpr (DT != DT_I8)
        if (p.fold_steps) return launch_any_tile<DT, true>(ta, tb, p, s);
    return launch_any_tile<DT, false>(ta, tb, p, s);
}

}  // namespace ntg
