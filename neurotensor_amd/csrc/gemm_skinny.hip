// Skinny GEMM (m <= 32): C[m, n] (+)= op(A)[m, k] . op(B)[k, n]   (Float32 first, Float16 / BFloat16 below)
//
// With so few rows the product streams B exactly once and is bound by HBM bandwidth,
// not by the matrix cores, so the tiling is chosen for the memory system: a workgroup of
// 8 wavefronts owns a strip of SW columns of C and all of K; the wavefronts take k-steps
// of 16 round-robin, feed v_mfma_f32_16x16x4_f32 straight from global memory (B is used
// once, so staging it in LDS would only add traffic), and their partial sums are added in
// a fixed order through LDS, which keeps the result deterministic (no atomics).
//
// Lane (c = lane%16, g = lane/16) holds, per k-step, A[row c][k0+4g .. k0+4g+3] and
// B[k0+4g+e][n0 + CPL*c .. +CPL-1] for e = 0..3: MFMA e uses k = k0+4g+e for lane group g
// on both operands, and MFMA column c stands for strip column CPL*c + j.
//
// Sizes and rows off every 16-byte boundary take the same loads: vectors are declared at the alignment of one element (the memory system takes them at any
// address), rows and columns past the end are clamped onto the last ones and their sums not stored, and the one k-step that K does not fill is read element by
// element, all of them in flight, by the wavefront whose turn it is.  A guard per element around every load, which such products had before, made each wait
// one for everything.  (Whole strips and steps, RAGGED = false, leave the clamps out.)  Float16 on one card, before | now, us: 3 x 4352 x 10109 (B stored [n][k]) 129 | 19.3 (with the clamp of relu, which was a pass of its own), 6 x 5229 x 331 61 | 21.5, 8 x 1536 x 472 28.5 | 4.5.
#include "ntg_common.h"

namespace ntg {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx4e __attribute__((ext_vector_type(4), aligned(4)));          // at any element

template <int MB, int CPL, bool TA, bool TB, bool RAGGED>
__global__ void __launch_bounds__(512) gemm_skinny_f32_kernel(const GemmParams p) {
    constexpr int NW = 8;
    constexpr int SW = 16 * CPL;
    __shared__ float part[NW][MB * CPL * 4][64];

    const int tid = threadIdx.x;
    // (the wavefront's number in a scalar register: the branches below must be real ones, a matrix instruction runs whatever the lane mask says)
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int b = blockIdx.y;
    const int n0 = blockIdx.x * SW;

    // (global pointers: the waits of the register ring below are per k-step only if the loads are not FLAT instructions)
    const NTG_GLOBAL float* A = (const NTG_GLOBAL float*)(p.Aptr ? static_cast<const float*>(p.Aptr[b]) : static_cast<const float*>(p.A) + operand_offset(p, b, p.sA, p.sAk));
    const NTG_GLOBAL float* B = (const NTG_GLOBAL float*)(p.Bptr ? static_cast<const float*>(p.Bptr[b]) : static_cast<const float*>(p.B) + operand_offset(p, b, p.sB, p.sBk));
    NTG_GLOBAL float* C = (NTG_GLOBAL float*)(p.Cptr ? static_cast<float*>(p.Cptr[b]) : static_cast<float*>(p.C) + (int64_t)b * p.sC);

    floatx4 acc[MB][CPL];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < CPL; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    const int steps = p.K / 16;                  // whole ones
    // D k-steps of loads are kept in flight per wavefront (a register ring), so that
    // 8 wavefronts per CU cover the HBM latency-bandwidth product.  (Up to 12 in 96 registers were slower: 8 x 4096 x 4096 22.5 | 24.5 us.)
    constexpr int D = 4;
    float a[D][MB][4];
    float bv[D][4][CPL];

    int row[MB];                                 // (rows and columns past the end: the last ones, their sums are not stored)
#pragma unroll
    for (int i = 0; i < MB; ++i) row[i] = i * 16 + c < p.M ? i * 16 + c : p.M - 1;
    // B stored [k][n]: this lane's first column (N >= CPL)
    const int nb = !RAGGED || n0 + CPL * c < p.N - CPL ? n0 + CPL * c : p.N - CPL;

    auto load_step = [&](int d, int s) {
        const int kl = s * 16 + 4 * g;          // this lane's first k
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            if constexpr (!TA) {
                const floatx4 t = i * 16 + c < p.M ? *(const NTG_GLOBAL floatx4e*)(A + (int64_t)row[i] * p.lda + kl) : floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int e = 0; e < 4; ++e) a[d][i][e] = t[e];
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) a[d][i][e] = A[(int64_t)(kl + e) * p.lda + row[i]];
            }
        }
        if constexpr (!TB) {
            typedef float fv __attribute__((ext_vector_type(CPL), aligned(4)));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const fv t = *(const NTG_GLOBAL fv*)(B + (int64_t)(kl + e) * p.ldb + nb);
#pragma unroll
                for (int j = 0; j < CPL; ++j) bv[d][e][j] = t[j];
            }
        } else {
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const int n = n0 + CPL * c + j;
                const floatx4 t = *(const NTG_GLOBAL floatx4e*)(B + (int64_t)(!RAGGED || n < p.N ? n : p.N - 1) * p.ldb + kl);
#pragma unroll
                for (int e = 0; e < 4; ++e) bv[d][e][j] = t[e];
            }
        }
    };
    auto load_rest = [&]() {                     // the k-step that K does not fill, into slot 0
        const int kl = steps * 16 + 4 * g;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k = kl + e < p.K ? kl + e : p.K - 1;
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                const float v = TA ? A[(int64_t)k * p.lda + row[i]] : A[(int64_t)row[i] * p.lda + k];
                a[0][i][e] = kl + e < p.K ? v : 0.f;
            }
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const int n = n0 + CPL * c + j;
                const float v = TB ? B[(int64_t)(!RAGGED || n < p.N ? n : p.N - 1) * p.ldb + k] : B[(int64_t)k * p.ldb + nb + j];
                bv[0][e][j] = kl + e < p.K ? v : 0.f;
            }
        }
    };

    auto compute = [&](int d) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < CPL; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[d][i][e], bv[d][e][j], acc[i][j], 0, 0, 0);
    };
    // Rounds of D k-steps.  While a whole further round exists, a round runs without a branch (multiply step d, request the
    // step that takes its registers): the number of loads in flight is then the same at every wait, and the compiler waits
    // for one step's loads and leaves the other D - 1 steps in flight.  (Where paths with different counts meet it waits
    // for everything; the guarded rounds at the end, and the whole loop for a short k, are of that kind.)
    int base = wave;
    if (wave + (2 * D - 1) * NW < steps) {               // (uniform per wavefront)
#pragma unroll
        for (int d = 0; d < D; ++d) load_step(d, wave + d * NW);
        for (; base + (2 * D - 1) * NW < steps; base += D * NW) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                compute(d);
                load_step(d, base + (d + D) * NW);
            }
        }
    } else {
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (wave + d * NW < steps) load_step(d, wave + d * NW);
    }
    for (; base < steps; base += D * NW) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int s = base + d * NW;
            if (s < steps) {
                compute(d);
                if (s + D * NW < steps) load_step(d, s + D * NW);
            }
        }
    }
    if constexpr (RAGGED) {
        if (p.K > steps * 16 && wave == (steps & (NW - 1))) {      // (uniform per wavefront)
            load_rest();
            compute(0);
        }
    }

#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < CPL; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[wave][(i * CPL + j) * 4 + r][lane] = acc[i][j][r];
    __syncthreads();

    constexpr int TOTAL = MB * CPL * 4 * 64;
    const NTG_GLOBAL float* bias = (const NTG_GLOBAL float*)static_cast<const float*>(p.bias);
    for (int idx = tid; idx < TOTAL; idx += 512) {
        const int l = idx & 63, q = idx >> 6;
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) sum += part[w][q][l];     // fixed order: deterministic
        const int r = q & 3, j = (q >> 2) % CPL, i = (q >> 2) / CPL;
        const int m = i * 16 + 4 * (l >> 4) + r;
        // (a lane whose columns were moved back from the end leaves those that others have)
        const int first = n0 + CPL * (l & 15), n = (TB || !RAGGED || first < p.N - CPL ? first : p.N - CPL) + j;
        if (m < p.M && n < p.N && n >= first) {
            NTG_GLOBAL float* cp = C + (int64_t)m * p.ldc + n;
            if (p.cmode == C_ACCUMULATE) sum += *cp;
            else if (p.cmode == C_BIAS) sum += bias[(int64_t)b * p.bias_bs + (int64_t)m * p.bias_rs + (int64_t)n * p.bias_cs];
            if (p.act == ACT_RELU) sum = sum > 0.f ? sum : 0.f;
            *cp = sum;
        }
    }
}

template <int MB, int CPL, bool TA, bool TB>
static hipError_t launch_skinny_cfg(const GemmParams& p, hipStream_t s) {
    constexpr int SW = 16 * CPL;
    const dim3 grid((unsigned)((p.N + SW - 1) / SW), (unsigned)p.batch);
    if (p.K % 16 || p.N % SW) hipLaunchKernelGGL((gemm_skinny_f32_kernel<MB, CPL, TA, TB, true>), grid, dim3(512), 0, s, p);
    else hipLaunchKernelGGL((gemm_skinny_f32_kernel<MB, CPL, TA, TB, false>), grid, dim3(512), 0, s, p);
    return hipGetLastError();
}

template <int MB, int CPL>
static hipError_t launch_skinny_t(bool ta, bool tb, const GemmParams& p, hipStream_t s) {
    if (ta) return tb ? launch_skinny_cfg<MB, CPL, true, true>(p, s) : launch_skinny_cfg<MB, CPL, true, false>(p, s);
    return tb ? launch_skinny_cfg<MB, CPL, false, true>(p, s) : launch_skinny_cfg<MB, CPL, false, false>(p, s);
}

// ---- Float16 / BFloat16, m <= 32 -----------------------------------------------------------------
// Same plan with v_mfma_f32_16x16x32: lane (c = lane%16, g = lane/16) feeds 8 consecutive k
// (k0 + 8g ..) of row c of A and of one column of B.  Per k-step of 32:
//   TB  (B stored [n][k]): the 8 k of column c + 16 j are one 16-byte load; MFMA j covers column c + 16 j.
//   !TB (B stored [k][n]): the lane loads CPL consecutive columns (n0 + CPL c ..) of each of its 8 k rows
//       (coalesced along n) and transposes the 8 x CPL block in registers (v_perm_b32); MFMA j covers
//       column CPL c + j.
// fp32 accumulation over all of K, one rounding at the end (C0 added in fp32).
typedef uint32_t su32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t su32x4e __attribute__((ext_vector_type(4), aligned(2)));        // at any element
typedef __bf16 sbf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 shalfx8 __attribute__((ext_vector_type(8)));

template <int DT> struct Skinny16;
template <> struct Skinny16<DT_F16> {
    using T = _Float16;
    static __device__ __forceinline__ floatx4 mma(su32x4 a, su32x4 b, floatx4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(shalfx8, a), __builtin_bit_cast(shalfx8, b), c, 0, 0, 0);
    }
};
template <> struct Skinny16<DT_BF16> {
    using T = __bf16;
    static __device__ __forceinline__ floatx4 mma(su32x4 a, su32x4 b, floatx4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(sbf16x8, a), __builtin_bit_cast(sbf16x8, b), c, 0, 0, 0);
    }
};

template <int DT, int MB, int CPL, bool TA, bool TB, bool RAGGED>
__global__ void __launch_bounds__(512) gemm_skinny16_kernel(const GemmParams p) {
    using S = Skinny16<DT>;
    using T = typename S::T;
    constexpr int NW = 8;
    constexpr int SW = 16 * CPL;
    constexpr int BW = TB ? 4 : (CPL + 1) / 2;          // dwords per B load
    constexpr int NB = TB ? CPL : 8;                    // B loads per k-step
    __shared__ float part[NW][MB * CPL * 4][64];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);      // (scalar: as in the Float32 kernel)
    const int c = lane & 15, g = lane >> 4;
    const int b = blockIdx.y;
    const int n0 = blockIdx.x * SW;

    const NTG_GLOBAL T* A = (const NTG_GLOBAL T*)(p.Aptr ? static_cast<const T*>(p.Aptr[b]) : static_cast<const T*>(p.A) + (int64_t)b * p.sA);
    const NTG_GLOBAL T* B = (const NTG_GLOBAL T*)(p.Bptr ? static_cast<const T*>(p.Bptr[b]) : static_cast<const T*>(p.B) + (int64_t)b * p.sB);
    NTG_GLOBAL T* C = (NTG_GLOBAL T*)(p.Cptr ? static_cast<T*>(p.Cptr[b]) : static_cast<T*>(p.C) + (int64_t)b * p.sC);

    floatx4 acc[MB][CPL];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < CPL; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    const int steps = p.K / 32;                         // whole ones
    constexpr int D = (NB * BW >= 32 || MB * CPL >= 8) ? 2 : 4;   // k-steps of loads in flight per wavefront (register budget)
    su32x4 a[D][MB];
    uint32_t bv[D][NB][BW];

    int row[MB];                                        // (rows and columns past the end: as in the Float32 kernel)
#pragma unroll
    for (int i = 0; i < MB; ++i) row[i] = i * 16 + c < p.M ? i * 16 + c : p.M - 1;
    const int nb = !RAGGED || n0 + CPL * c < p.N - CPL ? n0 + CPL * c : p.N - CPL;

    auto pack8 = [&](auto&& elem) -> su32x4 {            // 8 elements -> 4 packed dwords
        T tmp[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) tmp[e] = elem(e);
        su32x4 r;
        __builtin_memcpy(&r, tmp, 16);
        return r;
    };

    auto load_step = [&](int d, int s) {
        const int kl = s * 32 + 8 * g;                   // this lane's first k
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            // (a real branch: lanes without a row ask the cache for nothing, and the scheduler does not gather a round's requests behind its products,
            //  which cost the linear layer of 16 x 4096 x 11008 3 %)
            if constexpr (!TA) a[d][i] = i * 16 + c < p.M ? *(const NTG_GLOBAL su32x4e*)(A + (int64_t)row[i] * p.lda + kl) : su32x4{0u, 0u, 0u, 0u};
            else a[d][i] = pack8([&](int e) -> T { return A[(int64_t)(kl + e) * p.lda + row[i]]; });
        }
        if constexpr (TB) {
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const int n = n0 + c + 16 * j;
                const su32x4 t = *(const NTG_GLOBAL su32x4e*)(B + (int64_t)(!RAGGED || n < p.N ? n : p.N - 1) * p.ldb + kl);
#pragma unroll
                for (int w = 0; w < 4; ++w) bv[d][j][w] = t[w];
            }
        } else {
            typedef uint16_t bvec __attribute__((ext_vector_type(CPL), aligned(2)));
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const bvec t = *(const NTG_GLOBAL bvec*)(B + (int64_t)(kl + e) * p.ldb + nb);
                if constexpr (CPL == 1) bv[d][e][0] = t[0];
                else __builtin_memcpy(&bv[d][e][0], &t, 2 * CPL);
            }
        }
    };
    auto load_rest = [&]() {                             // the k-step that K does not fill, into slot 0
        const int kl = steps * 32 + 8 * g;
        auto at = [&](int e) { return kl + e < p.K ? kl + e : p.K - 1; };
#pragma unroll
        for (int i = 0; i < MB; ++i)
            a[0][i] = pack8([&](int e) -> T {
                const T v = TA ? A[(int64_t)at(e) * p.lda + row[i]] : A[(int64_t)row[i] * p.lda + at(e)];
                return kl + e < p.K ? v : (T)0.0f;
            });
        if constexpr (TB) {
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const int n = n0 + c + 16 * j;
                const su32x4 t = pack8([&](int e) -> T {
                    const T v = B[(int64_t)(!RAGGED || n < p.N ? n : p.N - 1) * p.ldb + at(e)];
                    return kl + e < p.K ? v : (T)0.0f;
                });
#pragma unroll
                for (int w = 0; w < 4; ++w) bv[0][j][w] = t[w];
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                T tmp[2 * BW];
#pragma unroll
                for (int j = 0; j < 2 * BW; ++j) {
                    const T v = B[(int64_t)at(e) * p.ldb + nb + (j < CPL ? j : 0)];
                    tmp[j] = kl + e < p.K ? v : (T)0.0f;
                }
                __builtin_memcpy(&bv[0][e][0], tmp, 4 * BW);
            }
        }
    };

    auto compute = [&](int d) {
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
            su32x4 bt;
            if constexpr (TB) {
#pragma unroll
                for (int w = 0; w < 4; ++w) bt[w] = bv[d][j][w];
            } else {
                // column j of the 8 x CPL block: dword w packs k rows 2w, 2w+1
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const uint32_t lo = bv[d][2 * w][j >> 1], hi = bv[d][2 * w + 1][j >> 1];
                    bt[w] = (j & 1) ? __builtin_amdgcn_perm(hi, lo, 0x07060302u) : __builtin_amdgcn_perm(hi, lo, 0x05040100u);
                }
            }
#pragma unroll
            for (int i = 0; i < MB; ++i) acc[i][j] = S::mma(a[d][i], bt, acc[i][j]);
        }
    };

    // (rounds without a branch while a whole further round exists: see the Float32 kernel above)
    int base = wave;
    if (wave + (2 * D - 1) * NW < steps) {               // (uniform per wavefront)
#pragma unroll
        for (int d = 0; d < D; ++d) load_step(d, wave + d * NW);
        for (; base + (2 * D - 1) * NW < steps; base += D * NW) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                compute(d);
                load_step(d, base + (d + D) * NW);
            }
        }
    } else {
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (wave + d * NW < steps) load_step(d, wave + d * NW);
    }
    for (; base < steps; base += D * NW) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int s = base + d * NW;
            if (s < steps) {
                compute(d);
                if (s + D * NW < steps) load_step(d, s + D * NW);
            }
        }
    }
    if constexpr (RAGGED) {
        if (p.K > steps * 32 && wave == (steps & (NW - 1))) {      // (uniform per wavefront)
            load_rest();
            compute(0);
        }
    }

#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < CPL; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[wave][(i * CPL + j) * 4 + r][lane] = acc[i][j][r];
    __syncthreads();

    constexpr int TOTAL = MB * CPL * 4 * 64;
    const NTG_GLOBAL T* bias = (const NTG_GLOBAL T*)static_cast<const T*>(p.bias);
    for (int idx = tid; idx < TOTAL; idx += 512) {
        const int l = idx & 63, q = idx >> 6;
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) sum += part[w][q][l];     // fixed order: deterministic
        const int r = q & 3, j = (q >> 2) % CPL, i = (q >> 2) / CPL;
        const int m = i * 16 + 4 * (l >> 4) + r;
        const int first = n0 + (TB ? (l & 15) : CPL * (l & 15));
        const int n = TB ? first + 16 * j : (!RAGGED || first < p.N - CPL ? first : p.N - CPL) + j;
        if (m < p.M && n < p.N && n >= first) {
            NTG_GLOBAL T* cp = C + (int64_t)m * p.ldc + n;
            if (p.cmode == C_ACCUMULATE) sum += (float)*cp;
            else if (p.cmode == C_BIAS) sum += (float)bias[(int64_t)b * p.bias_bs + (int64_t)m * p.bias_rs + (int64_t)n * p.bias_cs];
            if (p.act == ACT_RELU) sum = sum > 0.f ? sum : 0.f;      // (before the one rounding: the same bits)
            *cp = (T)sum;
        }
    }
}

template <int DT, int MB, int CPL, bool TA, bool TB>
static hipError_t launch_skinny16_cfg(const GemmParams& p, hipStream_t s) {
    constexpr int SW = 16 * CPL;
    const dim3 grid((unsigned)((p.N + SW - 1) / SW), (unsigned)p.batch);
    if (p.K % 32 || p.N % SW) hipLaunchKernelGGL((gemm_skinny16_kernel<DT, MB, CPL, TA, TB, true>), grid, dim3(512), 0, s, p);
    else hipLaunchKernelGGL((gemm_skinny16_kernel<DT, MB, CPL, TA, TB, false>), grid, dim3(512), 0, s, p);
    return hipGetLastError();
}

template <int DT, int MB, int CPL>
static hipError_t launch_skinny16_t(bool ta, bool tb, const GemmParams& p, hipStream_t s) {
    if (ta) return tb ? launch_skinny16_cfg<DT, MB, CPL, true, true>(p, s) : launch_skinny16_cfg<DT, MB, CPL, true, false>(p, s);
    return tb ? launch_skinny16_cfg<DT, MB, CPL, false, true>(p, s) : launch_skinny16_cfg<DT, MB, CPL, false, false>(p, s);
}

template <int DT>
static hipError_t launch_skinny16(bool ta, bool tb, const GemmParams& p, hipStream_t s) {
    // Columns per lane (strip = 16 x that): as many workgroups as possible without exceeding one per CU -- a second
    // round of workgroups costs more than narrower strips gain.  B stored [k][n] is loaded with (2 x columns)-byte
    // accesses, so 2 columns per lane (4-byte loads) is never worth it there; B stored [n][k] goes down to one column (a lane's load is a row's 16 bytes
    // of k, a line of its own to the cache whatever the strip, so a CU's rate is what bounds a strip: 8 x 8192 x 480 20.7 us on 15 strips, 13.4 on 30;
    // 32 x 8192 x 4096 31.0 on 128, 24.2 on 256; 6 x 5229 x 331, rows at any element, 33.8 | 21.5).
    const int widest = p.M > 16 ? 4 : 8, narrowest = tb ? 1 : 4;
    int cpl = widest;
    for (int cand = widest; cand >= narrowest; cand >>= 1) {
        const int64_t wgs = ((p.N + 16 * cand - 1) / (16 * cand)) * (int64_t)p.batch;
        if (wgs <= 256) cpl = cand;
    }
    while (!tb && cpl > p.N) cpl >>= 1;                 // (a lane's columns are one load)
    if (p.M <= 16) {
        if (cpl == 8) return launch_skinny16_t<DT, 1, 8>(ta, tb, p, s);
        if (cpl == 4) return launch_skinny16_t<DT, 1, 4>(ta, tb, p, s);
        if (cpl == 2) return launch_skinny16_t<DT, 1, 2>(ta, tb, p, s);
        return launch_skinny16_t<DT, 1, 1>(ta, tb, p, s);
    }
    if (cpl == 4) return launch_skinny16_t<DT, 2, 4>(ta, tb, p, s);
    if (cpl == 2) return launch_skinny16_t<DT, 2, 2>(ta, tb, p, s);
    return launch_skinny16_t<DT, 2, 1>(ta, tb, p, s);
}

hipError_t launch_gemm_skinny(int dtype, bool ta, bool tb, const GemmParams& p, hipStream_t s, bool* handled) {
    *handled = false;
    if (p.M > 32 || p.batch > NTG_SKINNY_MAX_ITEMS) return hipSuccess;
    if ((dtype == DT_F16 || dtype == DT_BF16) && p.K >= 128) {
        *handled = true;
        return dtype == DT_F16 ? launch_skinny16<DT_F16>(ta, tb, p, s) : launch_skinny16<DT_BF16>(ta, tb, p, s);
    }
    if (dtype != DT_F32 || p.K < 64) return hipSuccess;
    *handled = true;
    // widest strip that still gives every CU a workgroup
    const int64_t want = 256;
    int cpl = 4;
    if (p.M > 16) cpl = 2;
    while (cpl > 1 && ((p.N + 16 * cpl - 1) / (16 * cpl)) * (int64_t)p.batch < want) cpl >>= 1;
    while (!tb && cpl > p.N) cpl >>= 1;
    if (p.M <= 16) {
        if (cpl == 4) return launch_skinny_t<1, 4>(ta, tb, p, s);
        if (cpl == 2) return launch_skinny_t<1, 2>(ta, tb, p, s);
        return launch_skinny_t<1, 1>(ta, tb, p, s);
    }
    if (cpl == 2) return launch_skinny_t<2, 2>(ta, tb, p, s);
    return launch_skinny_t<2, 1>(ta, tb, p, s);
}

}  // namespace ntg
