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

// out[b][p][c] = in[b][c][p]: an image batch from channel planes to channels-last, 64 x 64 tiles through LDS so that
// both the loads (along p) and the stores (along c) are coalesced.
// Where pixel p of the source image goes in a copy that carries a border of zero pixels (on == 0: no border, Pp == P): every row
// skips the Wp - W border pixels beside it, every depth slice the Hp - H border rows
struct PixRemap { int64_t Pp; FastDiv div_w, div_hw; uint32_t on, row_skip, slice_skip, off0; };
__device__ __forceinline__ int64_t remap_pixel(const PixRemap& r, int64_t p) {
    if (!r.on) return p;
    uint32_t skip = fast_div((uint32_t)p, r.div_w) * r.row_skip + r.off0;      // (a padded image has fewer than 2^31 pixels)
    if (r.slice_skip) skip += fast_div((uint32_t)p, r.div_hw) * r.slice_skip;   // (uniform)
    return p + skip;
}
static PixRemap make_remap(const HaloMap* h, int64_t P) {
    PixRemap r;
    std::memset(&r, 0, sizeof r);
    r.Pp = P;
    if (h && h->Wp) {
        r.Pp = h->vol(); r.on = 1;
        r.div_w = make_fastdiv((uint32_t)h->W); r.div_hw = make_fastdiv((uint32_t)(h->H * h->W));
        r.row_skip = (uint32_t)(h->Wp - h->W); r.slice_skip = (uint32_t)((h->Hp - h->H) * h->Wp);
        r.off0 = (uint32_t)((h->front * h->Hp + h->top) * h->Wp + h->left);
    }
    return r;
}

// zeros the border pixels of a channels-last copy [B][Dp * Hp * Wp][C] (16-byte pieces; C * sizeof(T) a multiple of 16).
// Only the border is visited: its pixels are numbered front slices, back slices, then slice by slice the top rows, the bottom
// rows and the left and right pieces of the image's rows.
// (vectors first, first + step, ... of the per_image 16-byte vectors of one image's border)
__device__ __forceinline__ void zero_border_vectors(uint4* __restrict__ img, const uint32_t per_image, const uint32_t vec_per_pixel, const HaloMap& h,
                                                    const uint32_t first, const uint32_t step) {
    const uint32_t top_n = (uint32_t)(h.top * h.Wp), bot_n = (uint32_t)((h.Hp - h.top - h.H) * h.Wp), side = (uint32_t)(h.Wp - h.W);
    const uint32_t slice = (uint32_t)(h.Hp * h.Wp), slice_n = slice - (uint32_t)(h.H * h.W);
    const uint32_t front_n = (uint32_t)h.front * slice, back_n = (uint32_t)(h.Dp - h.front - h.D) * slice;
    for (uint32_t i = first; i < per_image; i += step) {
        uint32_t j = i / vec_per_pixel, pix, d0 = 0u;
        const uint32_t v = i - j * vec_per_pixel;
        if (h.Dp > 1) {                                               // (uniform)
            if (j < front_n + back_n) {
                pix = j < front_n ? j : j + (uint32_t)h.D * slice;
                img[(int64_t)pix * vec_per_pixel + v] = make_uint4(0u, 0u, 0u, 0u);
                continue;
            }
            j -= front_n + back_n;
            const uint32_t d = j / slice_n;
            j -= d * slice_n;
            d0 = ((uint32_t)h.front + d) * slice;
        }
        if (j < top_n) pix = j;
        else if (j < top_n + bot_n) pix = (uint32_t)((h.top + h.H) * h.Wp) + (j - top_n);
        else {
            j -= top_n + bot_n;
            const uint32_t row = j / side, c = j - row * side;
            pix = (uint32_t)((h.top + row) * h.Wp) + (c < (uint32_t)h.left ? c : (uint32_t)h.W + c);
        }
        img[(int64_t)(d0 + pix) * vec_per_pixel + v] = make_uint4(0u, 0u, 0u, 0u);
    }
}
__global__ void __launch_bounds__(256) halo_zero_kernel(uint4* __restrict__ out, const uint32_t per_image, const uint32_t vec_per_pixel, const HaloMap h) {
    zero_border_vectors(out + (int64_t)blockIdx.y * h.vol() * vec_per_pixel, per_image, vec_per_pixel, h, blockIdx.x * 256u + threadIdx.x, gridDim.x * 256u);
}
hipError_t launch_halo_zero(int64_t es, void* out, int64_t batch, int64_t C, const HaloMap& h, hipStream_t s) {
    if ((C * es) % 16 != 0 || (reinterpret_cast<uintptr_t>(out) & 15) != 0) return hipErrorInvalidValue;
    const int64_t vpp = C * es / 16, border = h.border(), per_image = border * vpp;
    if (batch <= 0 || per_image <= 0) return hipSuccess;
    if (per_image > 0x7fffffffLL || h.vol() > 0x7fffffffLL) return hipErrorInvalidValue;
    const int64_t gx = std::min<int64_t>((per_image + 255) / 256, 64);
    for (int64_t b0 = 0; b0 < batch; b0 += 65535) {
        const int64_t nb = std::min<int64_t>(batch - b0, 65535);
        hipLaunchKernelGGL(halo_zero_kernel, dim3((unsigned)gx, (unsigned)nb), dim3(256), 0, s,
                           (uint4*)out + b0 * h.vol() * vpp, (uint32_t)per_image, (uint32_t)vpp, h);
    }
    return hipGetLastError();
}

template <class T>
__global__ void __launch_bounds__(256) nchw_to_nhwc_kernel(const T* __restrict__ in, T* __restrict__ out, const int64_t C, const int64_t P, const PixRemap r) {
    __shared__ T tile[64][65];
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int64_t p0 = (int64_t)blockIdx.x * 64, c0 = (int64_t)blockIdx.y * 64, b = blockIdx.z;
    const T* src = in + b * C * P;
    T* dst = out + b * C * r.Pp;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int64_t c = c0 + ty + 4 * i, pp = p0 + tx;
        if (c < C && pp < P) tile[ty + 4 * i][tx] = src[c * P + pp];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int64_t pp = p0 + ty + 4 * i, c = c0 + tx;
        if (c < C && pp < P) dst[remap_pixel(r, pp) * C + c] = tile[tx][ty + 4 * i];
    }
}

// element idx of the two weight permutations (see weights_channels_last_kernel, flip_weights_channels_last_kernel)
template <class T>
__device__ __forceinline__ void weights_channels_last_elem(const T* __restrict__ w, T* __restrict__ wp, const int64_t idx, const int64_t cg, const int64_t cgp,
                                                           const int64_t taps, const int64_t chunk) {
    const int64_t c = idx % cgp;
    const int64_t t = (idx / cgp) % taps;
    const int64_t o = idx / (cgp * taps);
    // chunk != 0: the k order (run of `chunk` channels, tap, channel inside the run) instead of (tap, channel)
    const int64_t dst = chunk ? o * taps * cgp + ((c / chunk) * taps + t) * chunk + c % chunk : idx;
    wp[dst] = c < cg ? w[(o * cg + c) * taps + t] : (T)0;
}
template <class T>
__device__ __forceinline__ void flip_weights_channels_last_elem(const T* __restrict__ w, T* __restrict__ wt, const int64_t idx, const int64_t og, const int64_t ogp,
                                                                const int64_t cg, const int64_t taps, const int64_t chunk) {
    const int64_t oc = idx % ogp;
    int64_t r = idx / ogp;
    const int64_t t = r % taps;
    r /= taps;
    const int64_t c = r % cg;
    const int64_t g = r / cg;
    // chunk != 0: the k order (run of `chunk` out channels, tap, out channel inside the run) instead of (tap, out channel)
    const int64_t dst = chunk ? r * taps * ogp + ((oc / chunk) * taps + t) * chunk + oc % chunk : idx;
    wt[dst] = oc < og ? w[((g * og + oc) * cg + c) * taps + (taps - 1 - t)] : (T)0;
}
// what a channels-last copy takes along: the border of zero pixels of its own output and a weight permutation
struct CopyExtras { HaloMap h; uint32_t border_vecs, vpp; WeightsJob job; int64_t job_total; };

// The same copy with 16-byte accesses on both sides (C and P multiples of one 16-byte vector, aligned pointers): a
// thread loads VEC pixels of one channel, the tile goes through LDS as single elements (row pitch chosen so that the
// column-wise read-back spreads over the banks), and a thread stores VEC channels of one pixel.
template <class T>
__global__ void __launch_bounds__(256) nchw_to_nhwc_vec_kernel(const T* __restrict__ in, T* __restrict__ out, const int64_t C, const int64_t P, const PixRemap r,
                                                               const CopyExtras ex) {
    constexpr int VEC = 16 / (int)sizeof(T), VPR = 64 / VEC;            // elements per vector, vectors per tile row
    constexpr int PITCH = sizeof(T) == 2 ? 66 : 65;                     // elements: 33 / 65 words
    typedef T TV __attribute__((ext_vector_type(VEC)));
    __shared__ T tile[64 * PITCH];
    const int64_t p0 = (int64_t)blockIdx.x * 64, c0 = (int64_t)blockIdx.y * 64, b = blockIdx.z;
    const T* src = in + b * C * P;
    T* dst = out + b * C * r.Pp;
#pragma unroll
    for (int i = 0; i < 64 * VPR / 256; ++i) {
        const int v = threadIdx.x + 256 * i, c = v / VPR, pv = v % VPR;
        if (c0 + c < C && p0 + pv * VEC < P) {
            const TV x = *reinterpret_cast<const TV*>(src + (c0 + c) * P + p0 + pv * VEC);
#pragma unroll
            for (int e = 0; e < VEC; ++e) tile[c * PITCH + pv * VEC + e] = x[e];
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 64 * VPR / 256; ++i) {
        const int v = threadIdx.x + 256 * i, pp = v / VPR, cv = v % VPR;
        if (c0 + cv * VEC < C && p0 + pp < P) {
            TV x;
#pragma unroll
            for (int e = 0; e < VEC; ++e) x[e] = tile[(cv * VEC + e) * PITCH + pp];
            *reinterpret_cast<TV*>(dst + remap_pixel(r, p0 + pp) * C + c0 + cv * VEC) = x;
        }
    }
    // the blocks of an image share its border, all blocks of the launch the weight permutation (a few elements each)
    const uint32_t per_image = gridDim.x * gridDim.y, bid = blockIdx.y * gridDim.x + blockIdx.x;
    if (ex.border_vecs)
        zero_border_vectors(reinterpret_cast<uint4*>(dst), ex.border_vecs, ex.vpp, ex.h, bid * 256u + threadIdx.x, per_image * 256u);
    if (ex.job.kind) {
        const int64_t step = (int64_t)gridDim.z * per_image * 256;
        for (int64_t idx = ((int64_t)blockIdx.z * per_image + bid) * 256 + threadIdx.x; idx < ex.job_total; idx += step) {
            if (ex.job.kind == 1) weights_channels_last_elem<T>((const T*)ex.job.w, (T*)ex.job.wp, idx, ex.job.cg, ex.job.cgp, ex.job.taps, ex.job.chunk);
            else flip_weights_channels_last_elem<T>((const T*)ex.job.w, (T*)ex.job.wp, idx, ex.job.og, ex.job.ogp, ex.job.cg, ex.job.taps, ex.job.chunk);
        }
    }
}

hipError_t launch_nchw_to_nhwc(int64_t es, const void* in, void* out, int64_t batch, int64_t C, int64_t P, hipStream_t s, const HaloMap* halo,
                               const WeightsJob* job, bool* took_along) {
    if (took_along) *took_along = false;
    if (batch * C * P == 0) return hipSuccess;
    const PixRemap r = make_remap(halo, P);
    const int64_t gx = (P + 63) / 64, gy = (C + 63) / 64;
    if (gx > 0x7fffffffLL || gy > 65535) return hipErrorInvalidValue;
    const int64_t vec = 16 / es;
    const bool vec_ok = C % vec == 0 && P % vec == 0 && ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
    CopyExtras ex;
    std::memset(&ex, 0, sizeof ex);
    if (vec_ok && (es == 2 || es == 4) && took_along) {
        // (the caller acts on *took_along: without it the copy stays what it was)
        const int64_t vpp = C * es / 16, border = halo && halo->Wp ? halo->border() : 0;
        if (border * vpp <= 0x7fffffffLL && (!halo || halo->vol() <= 0x7fffffffLL)) {
            if (border > 0) { ex.h = *halo; ex.border_vecs = (uint32_t)(border * vpp); ex.vpp = (uint32_t)vpp; }
            if (job && job->kind) {
                ex.job = *job;
                ex.job_total = job->kind == 1 ? job->a * job->cgp * job->taps : job->a * job->ogp * job->cg * job->taps;
                // Small images have few blocks, and an element is a chain of divisions and a strided read, about 0.55 us: eight a thread
                // take as long as a launch, beyond that the permutation goes out on its own (Float32 1 x 512 x 4 x 4 x 4 -> 128
                // channels by 3 x 3 x 3, eight blocks: 864 elements a thread, image gradient 1960 us; on its own 84 us).
                if (ex.job_total > 8 * 256 * gx * gy * std::min<int64_t>(batch, 65535)) {
                    const WeightsJob& j = *job;
                    const hipError_t e = j.kind == 1 ? launch_weights_channels_last(es, j.w, j.wp, j.a, j.cg, j.cgp, j.taps, s, j.chunk)
                                                     : launch_flip_weights_channels_last(es, j.w, j.wp, j.a, j.og, j.ogp, j.cg, j.taps, s, j.chunk);
                    if (e != hipSuccess) return e;
                    ex.job.kind = 0;
                }
            }
            *took_along = true;
        }
    }
    for (int64_t b0 = 0; b0 < batch; b0 += 65535) {                    // (grid z limit)
        const int64_t nb = batch - b0 < 65535 ? batch - b0 : 65535;
        const dim3 g((unsigned)gx, (unsigned)gy, (unsigned)nb), t(256);
        const char* src = static_cast<const char*>(in) + b0 * C * P * es;
        char* dst = static_cast<char*>(out) + b0 * C * r.Pp * es;
        if (es == 2 && vec_ok) hipLaunchKernelGGL(nchw_to_nhwc_vec_kernel<uint16_t>, g, t, 0, s, (const uint16_t*)src, (uint16_t*)dst, C, P, r, ex);
        else if (es == 4 && vec_ok) hipLaunchKernelGGL(nchw_to_nhwc_vec_kernel<uint32_t>, g, t, 0, s, (const uint32_t*)src, (uint32_t*)dst, C, P, r, ex);
        else if (es == 2) hipLaunchKernelGGL(nchw_to_nhwc_kernel<uint16_t>, g, t, 0, s, (const uint16_t*)src, (uint16_t*)dst, C, P, r);
        else if (es == 4) hipLaunchKernelGGL(nchw_to_nhwc_kernel<uint32_t>, g, t, 0, s, (const uint32_t*)src, (uint32_t*)dst, C, P, r);
        else return hipErrorInvalidValue;
        ex.job.kind = 0;                                               // (the first launch has done the weights)
    }
    return hipGetLastError();
}

// wt[g][c][t][oc] = w[g*og + oc][c][taps-1-t]: the weights of the convolution that maps the output gradient back to the
// image (channel axes swapped inside each group, taps reversed), with the out channels of one tap consecutive and
// padded with zeros from og to ogp per tap.
template <class T>
__global__ void __launch_bounds__(256) flip_weights_channels_last_kernel(const T* __restrict__ w, T* __restrict__ wt, const int64_t groups,
                                                                         const int64_t og, const int64_t ogp, const int64_t cg, const int64_t taps,
                                                                         const int64_t chunk) {
    const int64_t total = groups * ogp * cg * taps;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += stride)
        flip_weights_channels_last_elem<T>(w, wt, idx, og, ogp, cg, taps, chunk);
}

hipError_t launch_flip_weights_channels_last(int64_t es, const void* w, void* wt, int64_t groups, int64_t og, int64_t ogp, int64_t cg, int64_t taps, hipStream_t s,
                                             int64_t chunk) {
    const int64_t total = groups * ogp * cg * taps;
    if (total == 0) return hipSuccess;
    const dim3 g(grid_for(total)), t(256);
    switch (es) {
    case 2: hipLaunchKernelGGL(flip_weights_channels_last_kernel<uint16_t>, g, t, 0, s, (const uint16_t*)w, (uint16_t*)wt, groups, og, ogp, cg, taps, chunk); break;
    case 4: hipLaunchKernelGGL(flip_weights_channels_last_kernel<uint32_t>, g, t, 0, s, (const uint32_t*)w, (uint32_t*)wt, groups, og, ogp, cg, taps, chunk); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// Weights of all phases of a strided convolution's image gradient, and the table of their products.  Phase e has the taps
// e + s (M - 1 - m) of w [g*og + oc][c][taps], reversed, as wt[g][c][(run, m0, m1, m2, oc in run)] with the out channels padded with
// zeros from og to ogp and in runs of `chunk` (see ConvGeom::tap_inner).  One thread per (group, image channel, tap, out channel):
// every tap belongs to one phase.  The table, one thread an item, is the work of the blocks behind those of the weights: an item is a
// walk over the phases and four 64-bit divisions, which behind a weight of its own was the kernel's whole length; index arithmetic in
// 32 bits (I) where the weights allow it, as a 64-bit division is some hundred instructions and a weight takes three
// (Float16 128 x 64 x 4 x 4 at stride 2: 9.5 -> 8.2 us, the rest the latency of its strided reads).
template <class T, class I>
__global__ void __launch_bounds__(256) phase_setup_kernel(const T* __restrict__ w, T* __restrict__ wt, RingItem* __restrict__ items, const PhaseLayout q,
                                                          const uint32_t weight_blocks) {
    const int taps = q.k[0] * q.k[1] * q.k[2];
    const int64_t total = (int64_t)q.groups * q.cg * taps * q.ogp;
    const int64_t stride = (int64_t)weight_blocks * 256;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; blockIdx.x < weight_blocks && i < total; i += stride) {
        const I idx = (I)i, row = idx / (I)q.ogp, gc = row / (I)taps;
        const int oc = (int)(idx - row * (I)q.ogp);
        int tap = (int)(row - gc * (I)taps);
        const int src_tap = tap;
        const int64_t r = (int64_t)gc;                                 // g * cg + c
        int e[3], m[3];
#pragma unroll
        for (int a = 2; a >= 0; --a) {
            const int i = tap % q.k[a];
            tap /= q.k[a];
            e[a] = i % q.s[a];
            m[a] = q.M[a][e[a]] - 1 - i / q.s[a];
        }
        const int ph = (e[0] * q.s[1] + e[1]) * q.s[2] + e[2];
        if (q.plane_off[ph] < 0) continue;
        const int ptaps = q.M[0][e[0]] * q.M[1][e[1]] * q.M[2][e[2]], t = (m[0] * q.M[1][e[1]] + m[1]) * q.M[2][e[2]] + m[2];
        const int64_t g = (int64_t)(gc / (I)q.cg), c = r - g * q.cg;
        wt[q.w_off[ph] + r * ptaps * q.ogp + ((int64_t)(oc / q.chunk) * ptaps + t) * q.chunk + oc % q.chunk] =
            oc < q.og ? w[((g * q.og + oc) * q.cg + c) * taps + src_tap] : (T)0;
    }
    // item (live phase, group)
    if (blockIdx.x < weight_blocks) return;
    const int64_t i = (int64_t)(blockIdx.x - weight_blocks) * 256 + threadIdx.x;
    if (i < (int64_t)q.phases * q.groups) {
        const int want = (int)(i / q.groups), g = (int)(i % q.groups);
        const int tiles_m = (q.cg + q.tile_rows - 1) / q.tile_rows;
        int64_t start = 0;
        int live = 0;
        for (int ph = 0; ph < q.s[0] * q.s[1] * q.s[2]; ++ph) {
            if (q.plane_off[ph] < 0) continue;
            const int e2 = ph % q.s[2], e1 = ph / q.s[2] % q.s[1], e0 = ph / (q.s[2] * q.s[1]);
            const int N = q.n[0][e0] * q.n[1][e1] * q.n[2][e2], tiles_n = (N + q.tile_cols - 1) / q.tile_cols;
            const int64_t per_group = (int64_t)tiles_m * tiles_n * q.batch;
            if (live++ < want) { start += per_group * q.groups; continue; }
            const int ptaps = q.M[0][e0] * q.M[1][e1] * q.M[2][e2], ochp = q.groups * q.ogp;
            RingItem it;
            it.K = ptaps * q.ogp; it.N = N; it.ldc = phase_plane(q, e0, e1, e2);
            it.a = q.w_off[ph] + (int64_t)g * q.cg * it.K;
            it.b = (((int64_t)q.org[0][e0] * q.yp[1] + q.org[1][e1]) * q.yp[2] + q.org[2][e2]) * ochp + (int64_t)g * q.ogp;
            it.c = q.plane_off[ph] + (int64_t)g * q.cg * it.ldc;
            it.k_d = q.M[0][e0]; it.k_r = q.M[1][e1]; it.k_c = q.M[2][e2];
            it.Wo = q.n[2][e2]; it.HoWo = q.n[1][e1] * q.n[2][e2];
            it.first = (int)(start + per_group * g); it.tiles_n = tiles_n;
            it.div_wo = make_fastdiv((uint32_t)it.Wo); it.div_howo = make_fastdiv((uint32_t)it.HoWo);
            items[i] = it;
            break;
        }
    }
}

hipError_t launch_phase_setup(int64_t es, const void* w, void* wt, RingItem* items, const PhaseLayout& q, hipStream_t s) {
    const int64_t total = (int64_t)q.groups * q.cg * q.k[0] * q.k[1] * q.k[2] * q.ogp;
    const uint32_t wb = (uint32_t)grid_for(total);
    const int64_t ib = ((int64_t)q.phases * q.groups + 255) / 256;
    if (ib > 0x3fffffffLL) return hipErrorInvalidValue;
    const dim3 g(wb + (uint32_t)ib), t(256);
    const bool narrow = total <= 0x7fffffffLL;
    switch (es) {
    case 2:
        if (narrow) hipLaunchKernelGGL((phase_setup_kernel<uint16_t, uint32_t>), g, t, 0, s, (const uint16_t*)w, (uint16_t*)wt, items, q, wb);
        else hipLaunchKernelGGL((phase_setup_kernel<uint16_t, int64_t>), g, t, 0, s, (const uint16_t*)w, (uint16_t*)wt, items, q, wb);
        break;
    case 4:
        if (narrow) hipLaunchKernelGGL((phase_setup_kernel<uint32_t, uint32_t>), g, t, 0, s, (const uint32_t*)w, (uint32_t*)wt, items, q, wb);
        else hipLaunchKernelGGL((phase_setup_kernel<uint32_t, int64_t>), g, t, 0, s, (const uint32_t*)w, (uint32_t*)wt, items, q, wb);
        break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// im[b][c][z][y][x] (+)= the element of the phase plane that holds it: phase e = (position + p) % s per axis stores the image
// positions s (a0 + a) + e - p as its positions a; phases without taps contribute zero.  A thread does V consecutive elements of
// an image row (16 bytes in one store where the rows allow it): the divisions are made once per row piece and the column phase
// advances by counting (Float16 32 x 64 x 56 x 56: one element per thread with all its divisions 19.8 us, this 12.9).  At a column
// stride of two, the one in common use, a piece is half a chunk of one phase's row and half a chunk of the other's: two loads at any element
// where the counting makes one of two bytes for each of its elements, 8.5 us (25.7 MB: 5.5 at the rate of a large copy).
template <class T, int V, bool STORE16>
__global__ void __launch_bounds__(256) phase_interleave_kernel(const T* __restrict__ tmp, T* __restrict__ im, const PhaseLayout q, const uint32_t total,
                                                               const FastDiv div_pieces, const int accumulate) {
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= total) return;
    const uint32_t pieces = (uint32_t)(q.sz[2] + V - 1) / V;
    const uint32_t row = fast_div(idx, div_pieces), x0 = (idx - row * pieces) * V;
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
        if (q.s[2] == 2) {                                             // (uniform)
            typedef T TV __attribute__((ext_vector_type(V)));
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
    if constexpr (STORE16) {
        typedef T TV __attribute__((ext_vector_type(V)));
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
    const bool vec = q.sz[2] % V16 == 0 && (reinterpret_cast<uintptr_t>(im) & 15) == 0;
    const int64_t pieces = vec ? q.sz[2] / V16 : (q.sz[2] + V - 1) / V, total = rows * pieces;
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

// wp[o][t][c] = w[o][c][t]: convolution weights with the channel index fastest (the k order of the channels-last gather),
// the channels of one tap padded with zeros from cg to cgp
template <class T>
__global__ void __launch_bounds__(256) weights_channels_last_kernel(const T* __restrict__ w, T* __restrict__ wp, const int64_t rows,
                                                                    const int64_t cg, const int64_t cgp, const int64_t taps, const int64_t chunk) {
    const int64_t total = rows * cgp * taps;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += stride)
        weights_channels_last_elem<T>(w, wp, idx, cg, cgp, taps, chunk);
}

hipError_t launch_weights_channels_last(int64_t es, const void* w, void* wp, int64_t rows, int64_t cg, int64_t cgp, int64_t taps, hipStream_t s, int64_t chunk) {
    const int64_t total = rows * cgp * taps;
    if (total == 0) return hipSuccess;
    const dim3 g(grid_for(total)), t(256);
    switch (es) {
    case 2: hipLaunchKernelGGL(weights_channels_last_kernel<uint16_t>, g, t, 0, s, (const uint16_t*)w, (uint16_t*)wp, rows, cg, cgp, taps, chunk); break;
    case 4: hipLaunchKernelGGL(weights_channels_last_kernel<uint32_t>, g, t, 0, s, (const uint32_t*)w, (uint32_t*)wp, rows, cg, cgp, taps, chunk); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// wp[o][r][q][c] = w[o][c][r][q] with every tap row padded with zeros from k_c to kq_pad taps and the channels from cg to cgp
template <class T>
__global__ void __launch_bounds__(256) weights_channels_last_rows_kernel(const T* __restrict__ w, T* __restrict__ wp, const int64_t rows, const int64_t cg,
                                                                         const int64_t cgp, const int64_t k_r, const int64_t k_c, const int64_t kq_pad) {
    const int64_t total = rows * k_r * kq_pad * cgp;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += stride) {
        const int64_t c = idx % cgp;
        int64_t t = idx / cgp;
        const int64_t q = t % kq_pad;
        t /= kq_pad;
        const int64_t r = t % k_r, o = t / k_r;
        wp[idx] = (c < cg && q < k_c) ? w[((o * cg + c) * k_r + r) * k_c + q] : (T)0;
    }
}

hipError_t launch_weights_channels_last_rows(int64_t es, const void* w, void* wp, int64_t rows, int64_t cg, int64_t cgp, int64_t k_r, int64_t k_c,
                                             int64_t kq_pad, hipStream_t s) {
    const int64_t total = rows * k_r * kq_pad * cgp;
    if (total == 0) return hipSuccess;
    const dim3 g(grid_for(total)), t(256);
    switch (es) {
    case 2: hipLaunchKernelGGL(weights_channels_last_rows_kernel<uint16_t>, g, t, 0, s, (const uint16_t*)w, (uint16_t*)wp, rows, cg, cgp, k_r, k_c, kq_pad); break;
    case 4: hipLaunchKernelGGL(weights_channels_last_rows_kernel<uint32_t>, g, t, 0, s, (const uint32_t*)w, (uint32_t*)wp, rows, cg, cgp, k_r, k_c, kq_pad); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// out[b][p][g*cgp + c] = in[b][g*cg + c][p] for c < cg, 0 for cg <= c < cgp: the channels-last copy with the channels of
// every group padded to cgp.  64 x 64 tiles of (channel inside the group, pixel) through LDS, like the plain copy.
template <class T>
__global__ void __launch_bounds__(256) nchw_to_nhwc_pad_kernel(const T* __restrict__ in, T* __restrict__ out, const int64_t groups,
                                                               const int64_t cg, const int64_t cgp, const int64_t P, const int cblocks, const PixRemap r) {
    __shared__ T tile[64][65];
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int64_t g = blockIdx.y / cblocks, c0 = (int64_t)(blockIdx.y % cblocks) * 64;
    const int64_t p0 = (int64_t)blockIdx.x * 64, b = blockIdx.z;
    const T* src = in + (b * groups + g) * cg * P;
    T* dst = out + b * r.Pp * groups * cgp + g * cgp;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int64_t c = c0 + ty + 4 * i, pp = p0 + tx;
        tile[ty + 4 * i][tx] = (c < cg && pp < P) ? src[c * P + pp] : (T)0;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int64_t pp = p0 + ty + 4 * i, c = c0 + tx;
        if (c < cgp && pp < P) dst[remap_pixel(r, pp) * groups * cgp + c] = tile[tx][ty + 4 * i];
    }
}

// The same for groups of at most 32 bytes of channels (padded to 16 or 32 bytes): one thread per pixel and group reads its
// cg channels (each a coalesced stream over the pixels) and stores the padded run with 16-byte stores.
template <class T, int CP>
__global__ void __launch_bounds__(256) nchw_to_nhwc_few_kernel(const T* __restrict__ in, T* __restrict__ out, const int64_t total, const int64_t groups,
                                                               const int64_t cg, const int64_t P, const PixRemap r) {
    constexpr int VEC = 16 / (int)sizeof(T);
    typedef T TV __attribute__((ext_vector_type(VEC)));
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    const int64_t pp = idx % P, bg = idx / P, b = bg / groups, g = bg - b * groups;
    const T* src = in + bg * cg * P + pp;
    TV* dst = reinterpret_cast<TV*>(out + ((b * r.Pp + remap_pixel(r, pp)) * groups + g) * CP);
#pragma unroll
    for (int v = 0; v < CP / VEC; ++v) {
        TV x;
#pragma unroll
        for (int e = 0; e < VEC; ++e) x[e] = (v * VEC + e) < cg ? src[(int64_t)(v * VEC + e) * P] : (T)0;
        dst[v] = x;
    }
}

hipError_t launch_nchw_to_nhwc_padded(int64_t es, const void* in, void* out, int64_t batch, int64_t groups, int64_t cg, int64_t cgp, int64_t P, hipStream_t s,
                                      const HaloMap* halo) {
    if (batch * groups * cgp * P == 0) return hipSuccess;
    const PixRemap r = make_remap(halo, P);
    if (cgp * es <= 32 && (cgp * es) % 16 == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0) {
        const int64_t total = batch * groups * P, blocks = (total + 255) / 256;
        if (blocks <= 0x7fffffffLL) {
            const dim3 g((unsigned)blocks), t(256);
            if (es == 2 && cgp == 8) hipLaunchKernelGGL((nchw_to_nhwc_few_kernel<uint16_t, 8>), g, t, 0, s, (const uint16_t*)in, (uint16_t*)out, total, groups, cg, P, r);
            else if (es == 2) hipLaunchKernelGGL((nchw_to_nhwc_few_kernel<uint16_t, 16>), g, t, 0, s, (const uint16_t*)in, (uint16_t*)out, total, groups, cg, P, r);
            else if (es == 4 && cgp == 4) hipLaunchKernelGGL((nchw_to_nhwc_few_kernel<uint32_t, 4>), g, t, 0, s, (const uint32_t*)in, (uint32_t*)out, total, groups, cg, P, r);
            else if (es == 4) hipLaunchKernelGGL((nchw_to_nhwc_few_kernel<uint32_t, 8>), g, t, 0, s, (const uint32_t*)in, (uint32_t*)out, total, groups, cg, P, r);
            else return hipErrorInvalidValue;
            return hipGetLastError();
        }
    }
    const int64_t cblocks = (cgp + 63) / 64, gx = (P + 63) / 64, gy = cblocks * groups;
    if (gx > 0x7fffffffLL || gy > 65535) return hipErrorInvalidValue;
    for (int64_t b0 = 0; b0 < batch; b0 += 65535) {                    // (grid z limit)
        const int64_t nb = batch - b0 < 65535 ? batch - b0 : 65535;
        const dim3 g((unsigned)gx, (unsigned)gy, (unsigned)nb), t(256);
        const char* src = static_cast<const char*>(in) + b0 * groups * cg * P * es;
        char* dst = static_cast<char*>(out) + b0 * groups * cgp * r.Pp * es;
        if (es == 2) hipLaunchKernelGGL(nchw_to_nhwc_pad_kernel<uint16_t>, g, t, 0, s, (const uint16_t*)src, (uint16_t*)dst, groups, cg, cgp, P, (int)cblocks, r);
        else if (es == 4) hipLaunchKernelGGL(nchw_to_nhwc_pad_kernel<uint32_t>, g, t, 0, s, (const uint32_t*)src, (uint32_t*)dst, groups, cg, cgp, P, (int)cblocks, r);
        else return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace ntg
