// 16-, 32- and 64-bit integer products on the 8-bit matrix pipe:  C (+)= op(A) . op(B), wrapping in the element type.
//
// The reference's integer product wraps in the element type (nt/mp/simde_traits/simde_traits_avx2.h:810-812 16-bit, :444-446 32-bit,
// :523-540 64-bit), i.e. it is the exact product modulo 2^W, W = 8 P.  Write every operand as P balanced signed bytes,
// a = sum_i a_i 2^(8 i) (mod 2^W) with a_i in [-128, 127]; then
//   sum_k a b = sum_{i + j < P} 2^(8 (i + j)) sum_k a_i b_j   (mod 2^W),
// the terms with i + j >= P being multiples of 2^W: 3, 10 or 36 8-bit products.
//
//   * One kernel does all of it.  The operands are loaded as they lie (16 bytes per lane at any element, any pitch), a lane splits eight
//     consecutive elements into P eight-byte pieces on their way to LDS: the bytes of (a + 0x80..80) ^ 0x80..80 are the balanced digits (adding
//     128 to every digit carries once into the next), v_perm_b32 sorts them by digit, five vector instructions an element.
//   * LDS holds P byte tiles an operand, K-contiguous operands [row][32 k], M/N-contiguous ones [k][row] as the 8-bit ring kernel's, so the
//     fragments are its ds_read_b128 / ds_read_b64_tr_b8.  Every fragment of a K-step (32 k) is read once and meets all the digits it needs.
//   * The products of one shift i + j have accumulators of their own (P sets, 32-bit sums: P K 2^14 < 2^31), folded together at the end.
//   * 64 x 64 tiles, 128 x 64 where they are many; four wavefronts of 1 x 1 or 2 x 1 blocks of 32 x 32.  (128 x 128 with one workgroup per CU was
//     measured slower: Int32 8 x 1024^3 97.6 us.)
// Bound: vector instructions, LDS and the matrix pipe's P (P + 1) / 2 products about evenly; Int32 on 128 x 64 tiles spills 34 to 53 of its 256 registers (140 to 176
// bytes a lane, none for A.B^T): two workgroups on a CU leave no more.  Before, the digits went through memory (a pass that split each
// operand, P products writing 32-bit sums, a pass that added these) or the product ran on the vector ALU: Int32 8 x 1024^3 147 -> 84 us, 80 x 1088 x 152
// 150 -> 20; Int16 23 x 58 x 3008 x 3072 1040 -> 121; Int64 1024^3 135 -> 41, 16 x 824 x 3454 x 80 1219 -> 236 us.
#pragma once
#include "gemm_any_impl.h"

namespace ntg {

template <int P> struct IntElem;
template <> struct IntElem<2> { typedef uint16_t U; typedef uint32_t X; };
template <> struct IntElem<4> { typedef uint32_t U; typedef uint32_t X; };
template <> struct IntElem<8> { typedef uint64_t U; typedef uint64_t X; };

// eight consecutive elements (P / 2 chunks of 16 bytes) -> P pieces of eight signed digits, least significant first
template <int P>
__device__ __forceinline__ void split_digits(const u32x4 (&v)[P / 2], uint64_t (&piece)[P]) {
    constexpr uint32_t H = 0x80808080u;
    uint32_t out[P][2];
    if constexpr (P == 2) {
        typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            uint32_t t[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const uint32_t x = v[0][2 * h + e];
                const u16x2 s = __builtin_bit_cast(u16x2, x) + (u16x2){0x8080, 0x8080};
                t[e] = __builtin_bit_cast(uint32_t, s) ^ H;
            }
            out[0][h] = __builtin_amdgcn_perm(t[1], t[0], 0x06040200u);
            out[1][h] = __builtin_amdgcn_perm(t[1], t[0], 0x07050301u);
        }
    } else {
        // w[d][e]: dword d (0: the low 32 bits) of element e, as digits
        constexpr int ND = P / 4;
        uint32_t w[ND][8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if constexpr (P == 4) {
                w[0][e] = (v[e >> 2][e & 3] + H) ^ H;
            } else {
                const uint64_t x = (uint64_t)v[e >> 1][2 * (e & 1)] | ((uint64_t)v[e >> 1][2 * (e & 1) + 1] << 32);
                const uint64_t s = x + 0x8080808080808080ull;
                w[0][e] = (uint32_t)s ^ H;
                w[ND - 1][e] = (uint32_t)(s >> 32) ^ H;
            }
        }
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t* t = &w[d][4 * h];
                const uint32_t a = __builtin_amdgcn_perm(t[1], t[0], 0x05010400u), b = __builtin_amdgcn_perm(t[1], t[0], 0x07030602u);
                const uint32_t c = __builtin_amdgcn_perm(t[3], t[2], 0x05010400u), e = __builtin_amdgcn_perm(t[3], t[2], 0x07030602u);
                out[4 * d][h] = __builtin_amdgcn_perm(c, a, 0x05040100u);
                out[4 * d + 1][h] = __builtin_amdgcn_perm(c, a, 0x07060302u);
                out[4 * d + 2][h] = __builtin_amdgcn_perm(e, b, 0x05040100u);
                out[4 * d + 3][h] = __builtin_amdgcn_perm(e, b, 0x07060302u);
            }
    }
#pragma unroll
    for (int i = 0; i < P; ++i) piece[i] = (uint64_t)out[i][0] | ((uint64_t)out[i][1] << 32);
}

// One operand's share of a thread: WB groups of eight consecutive elements per K-step of its 64 WB x 32 tile.  As in AnyOperand a group that the end
// of its row cuts off is loaded from the row's last eight elements; its digits are shifted down, which puts zeros above them.
template <bool KC, int WB, int P>
struct IntOperand {
    static constexpr int ES = P, BK = 32, TE = 64 * WB, NC = P / 2;
    static constexpr int GR = KC ? 4 : TE / 8;           // groups in a row of the tile
    static constexpr int RSTEP = 256 / GR;               // rows from one group of a thread to its next
    static constexpr int PLANE = TE * BK;                // bytes of one digit's tile
    const NTG_GLOBAL char* base;
    const NTG_GLOBAL char* base_last;
    int64_t adv;
    uint32_t pitch, off[WB], last_step;
    int row, kr, lds, cut;
    bool edge;

    __device__ __forceinline__ void setup(const NTG_GLOBAL char* first, int64_t ld, int mn0, int MN, int K, int last, int tid) {
        kr = K - last * BK;
        pitch = (uint32_t)(ld * ES);
        row = tid / GR;
        const int g = tid % GR;
        if constexpr (KC) {
            base = first + (int64_t)mn0 * ld * ES;
            base_last = base + (int64_t)(K - BK) * ES;
            adv = BK * ES;
            edge = false;
            const int k = last * BK + 8 * g, at = k < K - 8 ? k : K - 8;
            last_step = (uint32_t)((at - (K - BK) - 8 * g) * ES);
            cut = k - at < 8 ? k - at : 8;
            lds = row * BK + 8 * g;
#pragma unroll
            for (int i = 0; i < WB; ++i) {
                const int r = mn0 + row + RSTEP * i < MN ? row + RSTEP * i : MN - 1 - mn0;
                off[i] = (uint32_t)r * pitch + (uint32_t)(8 * g * ES);
            }
        } else {
            base = first + (int64_t)(mn0 - 8) * ES;                // (the offsets carry eight elements)
            base_last = base + (int64_t)last * BK * ld * ES;
            adv = (int64_t)BK * ld * ES;
            edge = mn0 + TE > MN;
            const int mn = mn0 + 8 * g, at = mn < MN - 8 ? mn : MN - 8;
            cut = mn - at < 8 ? mn - at : 8;
            last_step = 0;
            lds = row * TE + (((g >> 1) ^ mn8_swizzle<TE / 16>(row)) << 4) + 8 * (g & 1);      // (the swizzle repeats every 8 rows)
#pragma unroll
            for (int i = 0; i < WB; ++i) off[i] = (uint32_t)(row + RSTEP * i) * pitch + (uint32_t)((at - mn0 + 8) * ES);
        }
    }
    __device__ __forceinline__ void load(u32x4 (&v)[NC], int i, int kt, int last) const {
        const bool l = kt >= last;                                 // (uniform; K-steps past the end load the last one again)
        const NTG_GLOBAL char* b = l ? base_last : base + (int64_t)kt * adv;
        uint32_t o = off[i];
        if constexpr (KC) o += l ? last_step : 0u;
        else {
            const int k = row + RSTEP * i;
            if (l && k >= kr) o -= (uint32_t)(k - (kr - 1)) * pitch;       // (the last k-row once more)
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) v[c] = *(const NTG_GLOBAL u32x4_any*)(b + o + 16 * c);
    }
    __device__ __forceinline__ void store(char* tile, const u32x4 (&v)[NC], int i, bool cut_off, bool lastk) const {
        uint64_t d[P];
        split_digits<P>(v, d);
        if (cut_off) {                                             // (uniform)
            const int c = KC ? (lastk ? cut : 0) : !lastk || row + RSTEP * i < kr ? cut : 8;
#pragma unroll
            for (int q = 0; q < P; ++q) d[q] = c >= 8 ? 0 : d[q] >> (8 * c);
        }
#pragma unroll
        for (int q = 0; q < P; ++q) *reinterpret_cast<uint64_t*>(tile + q * PLANE + lds + RSTEP * (KC ? BK : TE) * i) = d[q];
    }
};

template <int P, bool TA, bool TB, int WBM>
__global__ void __launch_bounds__(256, P == 8 ? 1 : 2) gemm_int_kernel(const GemmParams p) {
    typedef typename IntElem<P>::U U;
    typedef typename IntElem<P>::X X;
    constexpr int WBN = 1, BK = 32, TM = 64 * WBM, TN = 64 * WBN, WTM = 32 * WBM, WTN = 32 * WBN, PLANE_A = TM * BK, PLANE_B = TN * BK;
    constexpr int TILE_A = P * PLANE_A, STAGE = TILE_A + P * PLANE_B, DEPTH = P == 8 || WBM == 2 ? 2 : 3;
    using OA = IntOperand<!TA, WBM, P>;
    using OB = IntOperand<TB, WBN, P>;
    constexpr int NC = OA::NC;
    __shared__ __attribute__((aligned(1024))) char lds[2 * STAGE];
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
                                             : static_cast<const char*>(p.A) + operand_offset(p, b, p.sA, p.sAk) * P);
    const gptr<char> B = (gptr<char>)(p.Bptr ? static_cast<const char*>(((gptr<const void*>)p.Bptr)[b])
                                             : static_cast<const char*>(p.B) + operand_offset(p, b, p.sB, p.sBk) * P);
    const gptr_mut<U> C = (gptr_mut<U>)(p.Cptr ? static_cast<U*>(((gptr<void*>)p.Cptr)[b]) : static_cast<U*>(p.C) + (int64_t)b * p.sC);
    const NTG_GLOBAL U* bias = (const NTG_GLOBAL U*)static_cast<const U*>(p.bias) + (int64_t)b * p.bias_bs;

    intx16 acc[P][WBM][WBN];
#pragma unroll
    for (int s = 0; s < P; ++s)
#pragma unroll
        for (int i = 0; i < WBM; ++i)
#pragma unroll
            for (int j = 0; j < WBN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[s][i][j][r] = 0;

    const int KT = (K + BK - 1) / BK, last = KT - 1;
    const bool cut_k = K - last * BK < BK;
    OA a;
    OB bb;
    a.setup(A, p.lda, m0, p.M, K, last, tid);
    bb.setup(B, p.ldb, n0, p.N, K, last, tid);
    u32x4 ra[DEPTH][WBM][NC], rb[DEPTH][WBN][NC];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
#pragma unroll
        for (int i = 0; i < WBM + WBN; ++i) {
            if (i < WBM) a.load(ra[d][i < WBM ? i : 0], i, d, last);
            else bb.load(rb[d][i < WBM ? 0 : i - WBM], i - WBM, d, last);
        }

    auto read_frag = [&](intx4& f, const char* tile, auto kc_tag, auto edge_tag, int mn) __attribute__((always_inline)) {
        if constexpr (decltype(kc_tag)::value) {
            f = *reinterpret_cast<const intx4*>(tile + (mn + (lane & 31)) * BK + 16 * (lane >> 5));
        } else {
            constexpr int TE = decltype(edge_tag)::value;
            const int grp = lane >> 4, i = lane & 15;
            const int mnl = mn + 16 * (grp & 1) + 8 * (i & 1);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int krow = 16 * (grp >> 1) + 8 * t + (i >> 1);
                const intx2v v = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                    (__attribute__((address_space(3))) intx2v*)(tile + krow * TE + (((mnl >> 4) ^ mn8_swizzle<TE / 16>(krow)) << 4) + (mnl & 15)));
                f[2 * t] = v[0];
                f[2 * t + 1] = v[1];
            }
        }
    };
    // K-step kt out of its stage; between its products the digits of K-step kt + 1 (set d) go to the other stage, which was last read before this
    // K-step's barrier, and with MORE the loads of K-step kt + 1 + DEPTH take their registers
    auto step = [&](int kt, int d, auto more_tag, bool special) __attribute__((always_inline)) {
        constexpr bool MORE = decltype(more_tag)::value;
        const char* sa = lds + (kt & 1) * STAGE;
        char* nx = lds + (~kt & 1) * STAGE;
        const bool lastk = special && cut_k && kt + 1 == last, cut_a = lastk || (special && a.edge), cut_b = lastk || (special && bb.edge);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        intx4 fa[P][WBM], fb[P][WBN];
        using KCA = std::integral_constant<bool, !TA>;
        using KCB = std::integral_constant<bool, TB>;
#pragma unroll
        for (int q = 0; q < P; ++q)
#pragma unroll
            for (int i = 0; i < WBM + WBN; ++i) {
                if (i < WBM) read_frag(fa[q][i < WBM ? i : 0], sa + q * PLANE_A, KCA{}, std::integral_constant<int, TM>{}, wm * WTM + 32 * i);
                else read_frag(fb[q][i < WBM ? 0 : i - WBM], sa + TILE_A + q * PLANE_B, KCB{}, std::integral_constant<int, TN>{}, wn * WTN + 32 * (i - WBM));
            }
#pragma unroll
        for (int x = 0; x < P; ++x) {
#pragma unroll
            for (int y = 0; x + y < P; ++y)
#pragma unroll
                for (int i = 0; i < WBM; ++i)
#pragma unroll
                    for (int j = 0; j < WBN; ++j)       // (the operands swapped: a lane holds four consecutive columns of one row of C)
                        acc[x + y][i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[y][j], fa[x][i], acc[x + y][i][j], 0, 0, 0);
            if (x == 0 && (!special || kt < last)) {
#pragma unroll
                for (int i = 0; i < WBM; ++i) {
                    a.store(nx, ra[d][i], i, cut_a, lastk);
                    if constexpr (MORE) a.load(ra[d][i], i, kt + 1 + DEPTH, last);
                }
            }
            if (x == 1 && (!special || kt < last)) {
#pragma unroll
                for (int j = 0; j < WBN; ++j) {
                    bb.store(nx + TILE_A, rb[d][j], j, cut_b, lastk);
                    if constexpr (MORE) bb.load(rb[d][j], j, kt + 1 + DEPTH, last);
                }
            }
        }
    };
    {
        const bool lastk = cut_k && last == 0, cut_a = lastk || a.edge, cut_b = lastk || bb.edge;
#pragma unroll
        for (int i = 0; i < WBM; ++i) {
            a.store(lds, ra[0][i], i, cut_a, lastk);
            a.load(ra[0][i], i, DEPTH, last);
        }
#pragma unroll
        for (int j = 0; j < WBN; ++j) {
            bb.store(lds + TILE_A, rb[0][j], j, cut_b, lastk);
            bb.load(rb[0][j], j, DEPTH, last);
        }
    }
    // (K-step kt + 1 is in set (kt + 1) % DEPTH; the rounds end before the last K-step is written to LDS)
    int kt = 0;
    const bool edge = a.edge || bb.edge;                           // (uniform) a tile on the edge of an operand stored along it
    if (edge) {
        for (; kt + DEPTH <= last - 1; kt += DEPTH)
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) step(kt + d, (d + 1) % DEPTH, std::true_type{}, true);
    } else {
        for (; kt + DEPTH <= last - 1; kt += DEPTH)
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) step(kt + d, (d + 1) % DEPTH, std::true_type{}, false);
    }
#pragma unroll
    for (int d = 0; d < DEPTH + 1; ++d)
        if (kt + d <= last) step(kt + d, (d + 1) % DEPTH, std::false_type{}, true);     // (uniform)

    typedef U ux4 __attribute__((ext_vector_type(4), aligned(sizeof(U))));
#pragma unroll
    for (int i = 0; i < WBM; ++i) {
        const int m = m0 + wm * WTM + 32 * i + (lane & 31);
#pragma unroll
        for (int j = 0; j < WBN; ++j)
#pragma unroll
            for (int rq = 0; rq < 4; ++rq) {
                const int n = n0 + wn * WTN + 32 * j + 8 * rq + 4 * (lane >> 5);
                if (m >= p.M || n >= p.N) continue;
                const bool whole = n + 4 <= p.N;
                NTG_GLOBAL U* cp = C + (int64_t)m * p.ldc + n;
                X v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = 0;
#pragma unroll
                    for (int s = 0; s < P; ++s) v[e] += (X)(int64_t)acc[s][i][j][4 * rq + e] << (8 * s);
                }
                if (p.cmode == C_ACCUMULATE) {
                    if (whole) {
                        const ux4 c = *(const NTG_GLOBAL ux4*)cp;
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] += (X)c[e];
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (n + e < p.N) v[e] += (X)cp[e];
                    }
                } else if (p.cmode == C_BIAS) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (n + e < p.N) v[e] += (X)bias[(int64_t)m * p.bias_rs + (int64_t)(n + e) * p.bias_cs];
                }
                if (whole) {
                    ux4 o;
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[e] = (U)v[e];
                    *(NTG_GLOBAL ux4*)cp = o;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (n + e < p.N) cp[e] = (U)v[e];
                }
            }
    }
}

template <int P, int WBM>
static hipError_t launch_int_wb(bool ta, bool tb, const GemmParams& pin, hipStream_t s) {
    GemmParams p = pin;
    p.tiles_m = (p.M + 64 * WBM - 1) / (64 * WBM);
    p.tiles_n = (p.N + 63) / 64;
    const int64_t blocks = (int64_t)p.tiles_m * p.tiles_n * p.batch;
    if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
    const dim3 g((unsigned)blocks), t(256);
    if (ta && tb) hipLaunchKernelGGL((gemm_int_kernel<P, true, true, WBM>), g, t, 0, s, p);
    else if (ta) hipLaunchKernelGGL((gemm_int_kernel<P, true, false, WBM>), g, t, 0, s, p);
    else if (tb) hipLaunchKernelGGL((gemm_int_kernel<P, false, true, WBM>), g, t, 0, s, p);
    else hipLaunchKernelGGL((gemm_int_kernel<P, false, false, WBM>), g, t, 0, s, p);
    return hipGetLastError();
}

}  // namespace ntg
