// Small reductions and permutations around the GEMM kernels: the ordered sum of the split-K partial products, the
// ordered sum of per-image weight gradients, and the channel-swapped, tap-reversed copy of a convolution kernel.
// All are HBM bound, deterministic (fixed summation order, no atomics) and launched on the caller's stream.
#include "ntg_common.h"

#include <algorithm>
#include <cstring>

namespace ntg {

// out[i] (+)= sum over b of part[b*n + i], b ascending: the order in which per-image weight
// gradients are added up by the reference's batch loop (conv.cpp:466-469).
template <class T, class Acc>
__global__ void __launch_bounds__(256) reduce_batch_kernel(const T* __restrict__ part, T* __restrict__ out, const int64_t batch,
                                                           const int64_t n, const int accumulate) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        Acc acc = accumulate ? (Acc)out[i] : (Acc)0;
        for (int64_t b = 0; b < batch; ++b) acc += (Acc)part[b * n + i];
        out[i] = (T)acc;
    }
}


// The reference's own order for the element types whose sums are checked bit for bit (Float32, Float64, the complex types):
// conv_dkernel forms sum(0) of the per-image products first -- item 0, then += item 1, ... in the element type
// (tensor_files/sum_exp_log.cpp:112-124) -- and adds that sum to d_kernel last (conv.cpp:466-469).
template <class T>
__global__ void __launch_bounds__(256) reduce_batch_sum_first_kernel(const T* __restrict__ part, T* __restrict__ out, const int64_t batch,
                                                                     const int64_t n, const int accumulate) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        T acc = part[i];
        for (int64_t b = 1; b < batch; ++b) acc += part[b * n + i];
        if (accumulate) {
            T o = out[i];
            o += acc;
            acc = o;
        }
        out[i] = acc;
    }
}

// The same sum for partial weight gradients held channels-last, part[b][o][t][c], into the kernel's own layout out[o][c][t]: a
// thread owns 16 bytes of consecutive channels of one (row, tap) and every SLICES-th of the partial sums (four reads in flight),
// the slices of a column group are added through LDS in slice order.  Bound by the reads of the partial sums; with one slice a
// small gradient (3 x 3 x 3 x 32 x 64: 55296 elements, 54 workgroups) over hundreds of partial sums would be one long chain of
// memory latencies on a few CUs, so SLICES grows until the launch has about 1024 workgroups (28 partial sums of 589824 elements,
// 66 MB: four slices, 16.1 us).  The order of the additions depends on the sizes only.
template <class T, int SLICES>
__global__ void __launch_bounds__(256) reduce_batch_taps_last_kernel(const float* __restrict__ part, T* __restrict__ out, const int64_t batch,
                                                                     const int64_t rows, const int64_t og, const int64_t ogp, const int64_t cg, const int64_t cgp,
                                                                     const int64_t taps, const int accumulate) {
    constexpr int VEC = 4;
    typedef float PV __attribute__((ext_vector_type(VEC)));
    constexpr int COLS = 256 / SLICES;                    // column groups of VEC elements per workgroup
    __shared__ float sums[SLICES > 1 ? 256 * VEC : 1];
    const int64_t n = rows * cgp * taps, nv = n / VEC;    // (the partial sums hold cgp >= cg channels per tap, the rest padding; cgp % VEC == 0)
    const int col = (int)threadIdx.x % COLS, sl = (int)threadIdx.x / COLS;
    const int64_t v = (int64_t)blockIdx.x * COLS + col;
    const int64_t i = v * VEC;
    float acc[VEC] = {};
    if (v < nv) {
        const float* pp = part + i;
        int64_t b = sl;
        for (; b + 3 * SLICES < batch; b += 4 * SLICES) {
            PV x[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) x[u] = *reinterpret_cast<const PV*>(pp + (b + u * SLICES) * n);
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int e = 0; e < VEC; ++e) acc[e] += x[u][e];
        }
        for (; b < batch; b += SLICES) {
            const PV x = *reinterpret_cast<const PV*>(pp + b * n);
#pragma unroll
            for (int e = 0; e < VEC; ++e) acc[e] += x[e];
        }
    }
    if constexpr (SLICES > 1) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) sums[(e * SLICES + sl) * COLS + col] = acc[e];
        __syncthreads();
        if (sl != 0) return;
        for (int o = 1; o < SLICES; ++o)
#pragma unroll
            for (int e = 0; e < VEC; ++e) acc[e] += sums[(e * SLICES + o) * COLS + col];
    }
    if (v >= nv) return;
    const int64_t c = i % cgp, t = (i / cgp) % taps;
    int64_t o = i / (cgp * taps);
    if (ogp != og) {                                      // (uniform; a group's rows may be padded too)
        const int64_t g = o / ogp;
        if (o - g * ogp >= og) return;
        o -= g * (ogp - og);
    }
    T* dst = out + (o * cg + c) * taps + t;
#pragma unroll
    for (int e = 0; e < VEC; ++e)
        if (c + e < cg) dst[(int64_t)e * taps] = (T)(accumulate ? (float)dst[(int64_t)e * taps] + acc[e] : acc[e]);
}

// Split-K epilogue: C (+)= sum over the k ranges of part[s][m][n], s ascending, starting from C0 (the incoming C, the
// broadcast bias, or zero).  One rounding to T at the end.
template <class T, class P, class Acc>
__global__ void __launch_bounds__(256) splitk_reduce_kernel(const P* __restrict__ part, const int splits, const int64_t split_stride, const int64_t ldp, const GemmParams p) {
    const int64_t total = (int64_t)p.M * p.N;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t b = blockIdx.y;                                      // item of the batch: its partial sums follow the previous item's
    T* C = static_cast<T*>(p.C) + b * p.sC;
    const T* bias = static_cast<const T*>(p.bias) + b * p.bias_bs;
    part += b * ((int64_t)p.M * ldp);
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += stride) {
        const int64_t m = idx / p.N, n = idx - m * p.N;
        T* cp = C + m * p.ldc + n;
        Acc acc = (Acc)0;
        if (p.cmode == C_ACCUMULATE) acc = (Acc)*cp;
        else if (p.cmode == C_BIAS) acc = (Acc)bias[m * p.bias_rs + n * p.bias_cs];
        for (int s = 0; s < splits; ++s) acc += (Acc)part[(int64_t)s * split_stride + m * ldp + n];
        if (p.act == ACT_RELU) acc = acc > (Acc)0 ? acc : (Acc)0;
        *cp = (T)acc;
    }
}

// The same sum, four consecutive columns per thread with 16-byte accesses to the partial sums, whose rows lie ldp elements apart (a multiple
// of four); C may start anywhere.  The partial loads of four k ranges are in flight together.
template <class T, class P, class Acc>
__global__ void __launch_bounds__(256) splitk_reduce_vec_kernel(const P* __restrict__ part, const int splits, const int64_t split_stride, const uint32_t ldp, const GemmParams p) {
    typedef T TV __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    typedef P PV __attribute__((ext_vector_type(4)));
    const uint32_t nq = ldp / 4, quads = (uint32_t)p.M * nq;
    const uint32_t stride = gridDim.x * blockDim.x;
    const int64_t b = blockIdx.y;
    T* C = static_cast<T*>(p.C) + b * p.sC;
    const T* bias = static_cast<const T*>(p.bias) + b * p.bias_bs;
    part += b * ((int64_t)p.M * ldp);
    for (uint32_t q = blockIdx.x * blockDim.x + threadIdx.x; q < quads; q += stride) {
        const uint32_t m = q / nq, n = (q - m * nq) * 4;
        if (n >= (uint32_t)p.N) continue;
        const bool whole = n + 4 <= (uint32_t)p.N;
        T* ce = C + (int64_t)m * p.ldc + n;
        Acc acc[4] = {(Acc)0, (Acc)0, (Acc)0, (Acc)0};
        if (p.cmode == C_ACCUMULATE) {
            if (whole) {
                const TV c0 = *reinterpret_cast<const TV*>(ce);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] = (Acc)c0[e];
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < (uint32_t)p.N) acc[e] = (Acc)ce[e];
            }
        } else if (p.cmode == C_BIAS) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + e < (uint32_t)p.N) acc[e] = (Acc)bias[(int64_t)m * p.bias_rs + (int64_t)(n + e) * p.bias_cs];
        }
        const P* pp = part + (int64_t)q * 4;
        int s = 0;
        for (; s + 4 <= splits; s += 4) {
            PV v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = *reinterpret_cast<const PV*>(pp + (int64_t)(s + u) * split_stride);
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] += (Acc)v[u][e];
        }
        for (; s < splits; ++s) {
            const PV v = *reinterpret_cast<const PV*>(pp + (int64_t)s * split_stride);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] += (Acc)v[e];
        }
        TV o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (T)((p.act == ACT_RELU && !(acc[e] > (Acc)0)) ? (Acc)0 : acc[e]);
        if (whole) *reinterpret_cast<TV*>(ce) = o;
        else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + e < (uint32_t)p.N) ce[e] = o[e];
        }
    }
}

// p.batch items (at most 65535 per call): item b's partial sums start b * M * ldp elements into every k range's block, the
// ranges' blocks lie p.batch * M * ldp elements apart
template <class T, class P, class Acc>
static void launch_splitk_reduce_t(const void* part, int splits, const GemmParams& p, int64_t ldp, hipStream_t s) {
    const int64_t total = (int64_t)p.M * ldp, split_stride = total * p.batch;
    const bool vec = ldp % 4 == 0 && total < (1LL << 31) && (reinterpret_cast<uintptr_t>(part) % (4 * sizeof(P))) == 0;
    if (vec) hipLaunchKernelGGL((splitk_reduce_vec_kernel<T, P, Acc>), dim3(grid_for(total / 4), (unsigned)p.batch), dim3(256), 0, s, (const P*)part, splits, split_stride, (uint32_t)ldp, p);
    else hipLaunchKernelGGL((splitk_reduce_kernel<T, P, Acc>), dim3(grid_for((int64_t)p.M * p.N), (unsigned)p.batch), dim3(256), 0, s, (const P*)part, splits, split_stride, ldp, p);
}

// C[b][m][n] = C[b][m][n] > 0 ? C[b][m][n] : 0 -- relu_ = clamp_(x, 0) of the reference (activation_functions.cpp:143,
// min_max.cpp:115-121: max(x, 0) with the second operand returned for NaN and for -0)
template <class T>
__global__ void __launch_bounds__(256) relu_inplace_kernel(T* __restrict__ C, const int64_t ldc, const int64_t sC, const int64_t M, const int64_t N,
                                                           const int64_t batch) {
    const int64_t total = batch * M * N;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const int64_t n = i % N, m = (i / N) % M, b = i / (N * M);
        T* cp = C + b * sC + m * ldc + n;
        const T v = *cp;
        if (!((float)v > 0.0f) || v != v) *cp = (T)0.0f;
    }
}
template <>
__global__ void __launch_bounds__(256) relu_inplace_kernel<double>(double* __restrict__ C, const int64_t ldc, const int64_t sC, const int64_t M,
                                                                   const int64_t N, const int64_t batch) {
    const int64_t total = batch * M * N;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const int64_t n = i % N, m = (i / N) % M, b = i / (N * M);
        double* cp = C + b * sC + m * ldc + n;
        if (!(*cp > 0.0)) *cp = 0.0;
    }
}
hipError_t launch_relu_inplace(int dtype, void* C, int64_t ldc, int64_t sC, int64_t M, int64_t N, int64_t batch, hipStream_t s) {
    const int64_t total = batch * M * N;
    if (total <= 0) return hipSuccess;
    const dim3 g(grid_for(total)), t(256);
    switch (dtype) {
    case DT_F32: hipLaunchKernelGGL(relu_inplace_kernel<float>, g, t, 0, s, (float*)C, ldc, sC, M, N, batch); break;
    case DT_F64: hipLaunchKernelGGL(relu_inplace_kernel<double>, g, t, 0, s, (double*)C, ldc, sC, M, N, batch); break;
    case DT_F16: hipLaunchKernelGGL(relu_inplace_kernel<_Float16>, g, t, 0, s, (_Float16*)C, ldc, sC, M, N, batch); break;
    case DT_BF16: hipLaunchKernelGGL(relu_inplace_kernel<__bf16>, g, t, 0, s, (__bf16*)C, ldc, sC, M, N, batch); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_splitk_reduce(int dtype, const void* part, int splits, const GemmParams& p, int64_t ldp, hipStream_t s) {
    const int64_t total = (int64_t)p.M * p.N;
    if (total == 0 || p.batch < 1) return hipSuccess;
    if (p.batch > 65535) return hipErrorInvalidValue;
    switch (dtype) {
    case DT_F32: launch_splitk_reduce_t<float, float, float>(part, splits, p, ldp, s); break;
    case DT_F64: launch_splitk_reduce_t<double, double, double>(part, splits, p, ldp, s); break;
    case DT_F16: launch_splitk_reduce_t<_Float16, float, float>(part, splits, p, ldp, s); break;
    case DT_BF16: launch_splitk_reduce_t<__bf16, float, float>(part, splits, p, ldp, s); break;
    case DT_I8: case DT_U8: launch_splitk_reduce_t<uint8_t, int, int>(part, splits, p, ldp, s); break;      // (the low 8 bits, either signedness)
    case DT_I16: case DT_U16: launch_splitk_reduce_t<uint16_t, uint16_t, uint16_t>(part, splits, p, ldp, s); break;
    case DT_I32: case DT_U32: launch_splitk_reduce_t<uint32_t, uint32_t, uint32_t>(part, splits, p, ldp, s); break;
    case DT_I64: case DT_U64: launch_splitk_reduce_t<uint64_t, uint64_t, uint64_t>(part, splits, p, ldp, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}


// wt[g][c][oc][t] = w[g*og + oc][c][taps-1-t]: the kernel with input/output channels swapped
// inside each group and both tap axes reversed, i.e. the weights of the convolution that maps
// the output gradient back to the image.
template <class T>
__global__ void __launch_bounds__(256) flip_weights_kernel(const T* __restrict__ w, T* __restrict__ wt, const int64_t groups,
                                                           const int64_t og, const int64_t cg, const int64_t taps) {
    const int64_t total = groups * og * cg * taps;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += stride) {
        const int64_t t = idx % taps;
        int64_t r = idx / taps;
        const int64_t oc = r % og;
        r /= og;
        const int64_t c = r % cg;
        const int64_t g = r / cg;
        wt[idx] = w[((g * og + oc) * cg + c) * taps + (taps - 1 - t)];
    }
}


hipError_t launch_reduce_batch(int dtype, const void* part, void* out, int64_t batch, int64_t n, int accumulate, hipStream_t s) {
    if (n == 0) return hipSuccess;
    const dim3 g(grid_for(n)), b(256);
    switch (dtype) {
    case DT_F32: hipLaunchKernelGGL((reduce_batch_sum_first_kernel<float>), g, b, 0, s, (const float*)part, (float*)out, batch, n, accumulate); break;
    case DT_F64: hipLaunchKernelGGL((reduce_batch_sum_first_kernel<double>), g, b, 0, s, (const double*)part, (double*)out, batch, n, accumulate); break;
    case DT_F16: hipLaunchKernelGGL((reduce_batch_kernel<_Float16, float>), g, b, 0, s, (const _Float16*)part, (_Float16*)out, batch, n, accumulate); break;
    case DT_BF16: hipLaunchKernelGGL((reduce_batch_kernel<__bf16, float>), g, b, 0, s, (const __bf16*)part, (__bf16*)out, batch, n, accumulate); break;
    case DT_C32: hipLaunchKernelGGL((reduce_batch_sum_first_kernel<LanePair<_Float16>>), g, b, 0, s, (const LanePair<_Float16>*)part, (LanePair<_Float16>*)out, batch, n, accumulate); break;
    case DT_C64: hipLaunchKernelGGL((reduce_batch_sum_first_kernel<LanePair<float>>), g, b, 0, s, (const LanePair<float>*)part, (LanePair<float>*)out, batch, n, accumulate); break;
    case DT_C128: hipLaunchKernelGGL((reduce_batch_sum_first_kernel<LanePair<double>>), g, b, 0, s, (const LanePair<double>*)part, (LanePair<double>*)out, batch, n, accumulate); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <class T>
static void launch_reduce_taps_last_t(const void* part, void* out, int64_t batch, int64_t rows, int64_t og, int64_t ogp, int64_t cg, int64_t cgp, int64_t taps, int accumulate, hipStream_t s) {
    const int64_t nv = rows * cgp * taps / 4;
#define NTG_TAPS_LAST(S) \
    hipLaunchKernelGGL((reduce_batch_taps_last_kernel<T, S>), dim3((unsigned)((nv * S + 255) / 256)), dim3(256), 0, s, (const float*)part, (T*)out, batch, rows, og, ogp, cg, cgp, taps, accumulate)
    if (nv >= 256 * 1024 || batch < 8) NTG_TAPS_LAST(1);
    else if (nv * 4 >= 256 * 1024 || batch < 32) NTG_TAPS_LAST(4);
    else NTG_TAPS_LAST(16);
#undef NTG_TAPS_LAST
}
hipError_t launch_reduce_batch_taps_last(int dtype, const void* part, void* out, int64_t batch, int64_t rows, int64_t og, int64_t ogp, int64_t cg, int64_t cgp,
                                         int64_t taps, int accumulate, hipStream_t s) {
    const int64_t n = rows * cgp * taps;
    if (n == 0) return hipSuccess;
    if (cgp % 4 != 0 || (reinterpret_cast<uintptr_t>(part) & 15) != 0 || n / 64 >= 0x7fffffffLL) return hipErrorInvalidValue;
    switch (dtype) {
    case DT_F32: launch_reduce_taps_last_t<float>(part, out, batch, rows, og, ogp, cg, cgp, taps, accumulate, s); break;
    case DT_F16: launch_reduce_taps_last_t<_Float16>(part, out, batch, rows, og, ogp, cg, cgp, taps, accumulate, s); break;
    case DT_BF16: launch_reduce_taps_last_t<__bf16>(part, out, batch, rows, og, ogp, cg, cgp, taps, accumulate, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_flip_weights(int64_t es, const void* w, void* wt, int64_t groups, int64_t og, int64_t cg, int64_t taps, hipStream_t s) {
    const int64_t total = groups * og * cg * taps;
    if (total == 0) return hipSuccess;
    const dim3 g(grid_for(total)), b(256);
    switch (es) {
    case 2: hipLaunchKernelGGL(flip_weights_kernel<uint16_t>, g, b, 0, s, (const uint16_t*)w, (uint16_t*)wt, groups, og, cg, taps); break;
    case 4: hipLaunchKernelGGL(flip_weights_kernel<uint32_t>, g, b, 0, s, (const uint32_t*)w, (uint32_t*)wt, groups, og, cg, taps); break;
    case 8: hipLaunchKernelGGL(flip_weights_kernel<uint64_t>, g, b, 0, s, (const uint64_t*)w, (uint64_t*)wt, groups, og, cg, taps); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// im[b][c][z][y][x] (+)= the element of the phase plane that holds it: phase e = (position + p) % s per axis stores the image
// positions s (a0 + a) + e - p as its positions a; phases without taps contribute zero.  A thread does V consecutive elements of
// an image row (16 bytes in one store at any element; the last piece of a row that is no whole pieces moves back over the one before, which stores the
// same values, or adds to C element by element; rows shorter than a piece go four elements at a time): the divisions are made once per row piece and the column phase
// advances by counting (Float16 32 x 64 x 56 x 56: one element per thread with all its divisions 19.8 us, this 12.9).  At a column
// stride of two, the one in common use, a piece is half a chunk of one phase's row and half a chunk of the other's: two loads at any element
// where the counting makes one of two bytes for each of its elements, 8.5 us (25.7 MB: 5.5 at the rate of a large copy).  Rows of 52, element by element
// before: BFloat16 53 x 256 x 52 x 52 81 us, 33 now (73 MB each way: 31).
template <class T, int V, bool STORE16>
__global__ void __launch_bounds__(256) phase_interleave_kernel(const T* __restrict__ tmp, T* __restrict__ im, const PhaseLayout q, const uint32_t total,
                                                               const FastDiv div_pieces, const int accumulate) {
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= total) return;
    const uint32_t pieces = (uint32_t)(q.sz[2] + V - 1) / V;
    const uint32_t row = fast_div(idx, div_pieces);
    uint32_t x0 = (idx - row * pieces) * V;
    bool whole = STORE16;
    if constexpr (STORE16) {
        if (x0 + V > (uint32_t)q.sz[2]) {
            whole = !accumulate;
            if (whole) x0 = (uint32_t)q.sz[2] - V;
        }
    }
    const uint32_t t1 = fast_div(row, q.div_rows[1]), y = row - t1 * (uint32_t)q.sz[1];
    const uint32_t bc = fast_div(t1, q.div_rows[0]), z = t1 - bc * (uint32_t)q.sz[0];
    const uint32_t Z = z + (uint32_t)q.p[0], Y = y + (uint32_t)q.p[1], X = x0 + (uint32_t)q.p[2];
    const uint32_t az = fast_div(Z, q.div_s[0]), ez = Z - az * (uint32_t)q.s[0];
    const uint32_t ay = fast_div(Y, q.div_s[1]), ey = Y - ay * (uint32_t)q.s[1];
    uint32_t ax = fast_div(X, q.div_s[2]), ex = X - ax * (uint32_t)q.s[2];
    const int rz = (int)az - q.a0[0][ez], ry = (int)ay - q.a0[1][ey];
    const int rphase = (int)((ez * (uint32_t)q.s[1] + ey) * (uint32_t)q.s[2]);
    constexpr int64_t none = -(1LL << 62);
    // (the row's place in the planes of each column phase)
    int64_t rowoff[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
        rowoff[e] = e < q.s[2] && q.plane_off[rphase + e] >= 0
                  ? q.plane_off[rphase + e] + (int64_t)bc * phase_plane(q, (int)ez, (int)ey, e) + ((int64_t)rz * q.n[1][ey] + ry) * q.n[2][e] - q.a0[2][e] : none;
    T* dst = im + (int64_t)row * q.sz[2] + x0;
    if constexpr (STORE16) {
        if (q.s[2] == 2 && whole) {
            typedef T TV __attribute__((ext_vector_type(V), aligned(sizeof(T))));
            typedef T TH __attribute__((ext_vector_type(V / 2), aligned(sizeof(T))));
            const int64_t o0 = (ex ? rowoff[1] : rowoff[0]), o1 = (ex ? rowoff[0] : rowoff[1]);
            TH f0, f1;
#pragma unroll
            for (int i = 0; i < V / 2; ++i) f0[i] = f1[i] = (T)0.0f;
            if (o0 != none) f0 = *reinterpret_cast<const TH*>(tmp + o0 + ax);
            if (o1 != none) f1 = *reinterpret_cast<const TH*>(tmp + o1 + ax + ex);
            TV o;
#pragma unroll
            for (int i = 0; i < V; ++i) o[i] = i & 1 ? f1[i >> 1] : f0[i >> 1];
            if (accumulate) {                                          // (uniform)
                const TV c = *reinterpret_cast<const TV*>(dst);
#pragma unroll
                for (int i = 0; i < V; ++i) o[i] = (T)((float)o[i] + (float)c[i]);
            }
            *reinterpret_cast<TV*>(dst) = o;
            return;
        }
    }
    T v[V];
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const int64_t o = ex == 0u ? rowoff[0] : ex == 1u ? rowoff[1] : ex == 2u ? rowoff[2] : rowoff[3];
        const bool ok = (int)x0 + i < q.sz[2];
        float f = ok && o != none ? (float)tmp[o + ax] : 0.0f;
        if (accumulate && ok) f += (float)dst[i];
        v[i] = (T)f;
        if (++ex == (uint32_t)q.s[2]) { ex = 0u; ++ax; }
    }
    if (whole) {
        typedef T TV __attribute__((ext_vector_type(V), aligned(sizeof(T))));
        TV o;
#pragma unroll
        for (int i = 0; i < V; ++i) o[i] = v[i];
        *reinterpret_cast<TV*>(dst) = o;
    } else {
#pragma unroll
        for (int i = 0; i < V; ++i)
            if ((int)x0 + i < q.sz[2]) dst[i] = v[i];
    }
}

template <class T>
static hipError_t launch_phase_interleave_t(const void* tmp, void* im, const PhaseLayout& q, int accumulate, hipStream_t s) {
    constexpr int V16 = 16 / (int)sizeof(T), V = 4;
    const int64_t rows = (int64_t)q.batch * q.groups * q.cg * q.sz[0] * q.sz[1];
    const bool vec = q.sz[2] >= V16;
    const int64_t pieces = (q.sz[2] + (vec ? V16 : V) - 1) / (vec ? V16 : V), total = rows * pieces;
    if (total == 0) return hipSuccess;
    if (total >= 0x7fffffffLL) return hipErrorInvalidValue;
    const dim3 g((unsigned)((total + 255) / 256)), t(256);
    const FastDiv dp = make_fastdiv((uint32_t)pieces);
    if (vec) hipLaunchKernelGGL((phase_interleave_kernel<T, V16, true>), g, t, 0, s, (const T*)tmp, (T*)im, q, (uint32_t)total, dp, accumulate);
    else hipLaunchKernelGGL((phase_interleave_kernel<T, V, false>), g, t, 0, s, (const T*)tmp, (T*)im, q, (uint32_t)total, dp, accumulate);
    return hipGetLastError();
}
hipError_t launch_phase_interleave(int dtype, const void* tmp, void* im, const PhaseLayout& q, int accumulate, hipStream_t s) {
    switch (dtype) {
    case DT_F32: return launch_phase_interleave_t<float>(tmp, im, q, accumulate, s);
    case DT_F16: return launch_phase_interleave_t<_Float16>(tmp, im, q, accumulate, s);
    case DT_BF16: return launch_phase_interleave_t<__bf16>(tmp, im, q, accumulate, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace ntg
