// What a channels-last convolution needs before its product, in one launch: copies of images (or gradients) from channel planes to [pixel][channel], the
// borders of zero pixels around them, the convolution's weights in the order of the product's k, and the table of a strided gradient's phases.
#include "ntg_common.h"

#include <algorithm>
#include <cstring>
#include <type_traits>

namespace ntg {

// A group of launches that each took 2.5 to 5 us for next to no data is what a small layer's time was (copy, border, weights and phases: four of nine launches;
// the copy's own blocks did up to eight weights a thread, a chain of divisions and strided reads each).  Here every part has blocks of its own, side by
// side, a thread makes 16 bytes of weights from eight reads in flight, and all divisions are by multiplication.
//   tile blocks     64 pixels x 64 channels through LDS: 16-byte loads along the pixels at any element (the last of a row piecewise), 16-byte stores along the
//                   channels; padded channels are rows of zeros.  Bound by HBM: 64 x 256 x 56 x 56 in BFloat16, 213 MB, 35 us
//   few blocks      up to 32 bytes of channels a pixel, where a tile would be mostly empty: a thread reads the channels of one pixel, 256 pixels a block
//                   (64 bytes: 60 x 32 x 32^3 in BFloat16 99 us so, 57 in tiles)
//   border blocks   1024 vectors of one image's border
// Training steps before | now, us: BFloat16 15 x 64 x 39 x 39 -> 48 by 3 x 3 (13 launches before, 6 now) 80 | 49, Float32 3 x 96 x 13 x 13 -> 256 by one tap 53 | 42.
struct ClCopy {
    const void* in;
    void* out;
    uint32_t first, border_blocks, border_per_image, tiles_p, tiles_c;      // first block; blocks of an image's border; tiles of an image
    uint32_t P, cg, cgp, C, Ctot, few, vpp, border_vecs;                    // pixels; channels of a group here and in the copy, and in all
    uint32_t on, row_skip, slice_skip, off0;                                // where pixels go in a copy with a border
    FastDiv div_tp, div_tc, div_bpi, div_cgp, div_w, div_hw;
    int64_t Pp;                                                             // pixels of an image of the copy
    HaloMap h;
};
// kind 1: wp[o][t][c] = w[o][c][t], the channels of a tap consecutive and padded with zeros from cg to cgp; chunk != 0: k order (run of `chunk`
//         channels, tap, channel inside the run)
//      2: wp[g][c][t][oc] = w[g og + oc][c][taps - 1 - t]: the weights of the convolution that maps the output gradient back to the image (channel axes
//         swapped inside each group, taps reversed), out channels padded from cg (= og here) to cgp; chunk as above
//      3: kind 1 with every tap row padded from k_c to kq_pad taps
struct ClWeights {
    const void* w;
    void* wp;
    uint32_t kind, blocks, weight_blocks;            // (phases: the blocks behind weight_blocks write the table)
    int64_t vecs;                                    // 16-byte vectors of wp
    uint32_t cgv, cgp, cg, taps, other, k_r, k_c, kq_pad, chunk;      // cgv = vectors of a tap; other: the image channels of a group (kind 2)
    FastDiv div_cgv, div_taps, div_other, div_kq, div_kr;
};
struct ClArgs { ClCopy copy[3]; uint32_t n; ClWeights w; };
struct ClPhases { PhaseLayout q; RingItem* items; };
struct ClNone {};

// vectors first, first + step, ... of the per_image 16-byte vectors of one image's border.  Only the border is visited: its pixels are numbered front
// slices, back slices, then slice by slice the top rows, the bottom rows and the left and right pieces of the image's rows.
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

__device__ __forceinline__ int64_t copied_pixel(const ClCopy& r, uint32_t p) {
    if (!r.on) return p;                                               // (uniform)
    uint32_t skip = fast_div(p, r.div_w) * r.row_skip + r.off0;        // (a padded image has fewer than 2^31 pixels)
    if (r.slice_skip) skip += fast_div(p, r.div_hw) * r.slice_skip;    // (uniform)
    return (int64_t)p + skip;
}

// 16 bytes of weights: vector i of wp
template <class T>
__device__ __forceinline__ void weight_vector(const ClWeights& j, const int64_t i) {
    constexpr int VEC = 16 / (int)sizeof(T);
    typedef T TV __attribute__((ext_vector_type(VEC)));
    const T* w = static_cast<const T*>(j.w);
    // (the rows of wp as 32-bit numbers: weights of 2^35 bytes and more have their leading part taken off first)
    int64_t row = 0;
    uint32_t cv;
    if (i < 0x7fffffffLL) {
        const uint32_t r = fast_div((uint32_t)i, j.div_cgv);
        cv = (uint32_t)i - r * j.cgv;
        row = r;
    } else {
        row = i / j.cgv;
        cv = (uint32_t)(i - row * j.cgv);
    }
    const uint32_t c0 = cv * VEC, rr = (uint32_t)row;                  // (rows: fewer than 2^31 -- a row is a tap of a channel or filter)
    TV x;
    int64_t dst = i * VEC;
    if (j.kind == 3u) {                                                // (uniform)
        const uint32_t t = fast_div(rr, j.div_kq), q = rr - t * j.kq_pad;
        const uint32_t o = fast_div(t, j.div_kr), r = t - o * j.k_r;
#pragma unroll
        for (int e = 0; e < VEC; ++e) x[e] = c0 + e < j.cg && q < j.k_c ? w[(((int64_t)o * j.cg + c0 + e) * j.k_r + r) * j.k_c + q] : (T)0;
    } else {
        const uint32_t o = fast_div(rr, j.div_taps), t = rr - o * j.taps;        // (kind 2: o = group * channels + channel)
        if (j.kind == 1u) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) x[e] = c0 + e < j.cg ? w[((int64_t)o * j.cg + c0 + e) * j.taps + t] : (T)0;
        } else {
            const uint32_t g = fast_div(o, j.div_other), c = o - g * j.other;
#pragma unroll
            for (int e = 0; e < VEC; ++e)
                x[e] = c0 + e < j.cg ? w[(((int64_t)g * j.cg + c0 + e) * j.other + c) * j.taps + (j.taps - 1 - t)] : (T)0;
        }
        if (j.chunk) dst = (int64_t)o * j.taps * j.cgp + (int64_t)(c0 / j.chunk * j.taps + t) * j.chunk + c0 % j.chunk;
    }
    *reinterpret_cast<TV*>(static_cast<T*>(j.wp) + dst) = x;
}

// Weights of all phases of a strided convolution's image gradient.  Phase e has the taps e + s (M - 1 - m) of w [g*og + oc][c][taps], reversed, as
// wt[g][c][(run, m0, m1, m2, oc in run)] with the out channels padded with zeros from og to ogp and in runs of `chunk` (see ConvGeom::tap_inner).  One
// vector per (group, image channel, tap, eight or four out channels): every tap belongs to one phase.
template <class T>
__device__ __forceinline__ void phase_weight_vector(const ClWeights& j, const PhaseLayout& q, const int64_t i) {
    constexpr int VEC = 16 / (int)sizeof(T);
    typedef T TV __attribute__((ext_vector_type(VEC)));
    const T* w = static_cast<const T*>(j.w);
    const int64_t row = i < 0x7fffffffLL ? (int64_t)fast_div((uint32_t)i, j.div_cgv) : i / j.cgv;
    const int oc = (int)(i - row * j.cgv) * VEC;
    const uint32_t gc = fast_div((uint32_t)row, j.div_taps);           // g * cg + c
    int tap = (int)((uint32_t)row - gc * j.taps);
    const int src_tap = tap;
    int e[3], m[3];
#pragma unroll
    for (int a = 2; a >= 0; --a) {
        const int k = tap % q.k[a];
        tap /= q.k[a];
        e[a] = k % q.s[a];
        m[a] = q.M[a][e[a]] - 1 - k / q.s[a];
    }
    const int ph = (e[0] * q.s[1] + e[1]) * q.s[2] + e[2];
    if (q.plane_off[ph] < 0) return;
    const int ptaps = q.M[0][e[0]] * q.M[1][e[1]] * q.M[2][e[2]], t = (m[0] * q.M[1][e[1]] + m[1]) * q.M[2][e[2]] + m[2];
    const uint32_t g = fast_div(gc, j.div_other), c = gc - g * j.other;
    TV x;
#pragma unroll
    for (int v = 0; v < VEC; ++v) x[v] = oc + v < q.og ? w[(((int64_t)g * q.og + oc + v) * q.cg + c) * j.taps + src_tap] : (T)0;
    *reinterpret_cast<TV*>(static_cast<T*>(j.wp) + q.w_off[ph] + (int64_t)gc * ptaps * q.ogp + ((int64_t)(oc / q.chunk) * ptaps + t) * q.chunk + oc % q.chunk) = x;
}
// ... and the table of their products: item i = (live phase, group)
__device__ __forceinline__ void phase_item(const PhaseLayout& q, RingItem* __restrict__ items, const int64_t i) {
    if (i >= (int64_t)q.phases * q.groups) return;
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

template <class T, class Phases>
__global__ void __launch_bounds__(256) channels_last_kernel(const ClArgs a, const Phases ph) {
    constexpr int VEC = 16 / (int)sizeof(T), VPR = 64 / VEC;           // elements per vector, vectors per tile row
    constexpr int PITCH = sizeof(T) == 2 ? 66 : 65;                    // elements: 33 / 65 words
    typedef T TV __attribute__((ext_vector_type(VEC)));
    typedef T TU __attribute__((ext_vector_type(VEC), aligned(sizeof(T))));
    __shared__ T tile[64 * PITCH];
    uint32_t id = blockIdx.x;
    if (id < a.w.blocks) {
        if constexpr (std::is_same<Phases, ClPhases>::value) {
            if (id >= a.w.weight_blocks) { phase_item(ph.q, ph.items, (int64_t)(id - a.w.weight_blocks) * 256 + threadIdx.x); return; }
        }
        const int64_t step = (int64_t)a.w.weight_blocks * 256;
        for (int64_t i = (int64_t)id * 256 + threadIdx.x; i < a.w.vecs; i += step) {
            if constexpr (std::is_same<Phases, ClPhases>::value) phase_weight_vector<T>(a.w, ph.q, i);
            else weight_vector<T>(a.w, i);
        }
        return;
    }
    const ClCopy& r = a.copy[a.n > 2 && id >= a.copy[2].first ? 2 : a.n > 1 && id >= a.copy[1].first ? 1 : 0];
    id -= r.first;
    if (id < r.border_blocks) {
        const uint32_t b = fast_div(id, r.div_bpi), part = id - b * r.border_per_image;
        zero_border_vectors(reinterpret_cast<uint4*>(static_cast<T*>(r.out) + (int64_t)b * r.Pp * r.Ctot), r.border_vecs, r.vpp, r.h, part * 256u + threadIdx.x,
                            r.border_per_image * 256u);
        return;
    }
    id -= r.border_blocks;
    const uint32_t t = fast_div(id, r.div_tp), pt = id - t * r.tiles_p;
    const uint32_t b = fast_div(t, r.div_tc), ct = t - b * r.tiles_c;
    const T* src = static_cast<const T*>(r.in) + (int64_t)b * r.C * r.P;
    T* dst = static_cast<T*>(r.out) + (int64_t)b * r.Pp * r.Ctot;
    if (r.few) {                                                       // (uniform)
        const uint32_t p = pt * 256u + threadIdx.x;
        if (p >= r.P) return;
        TV* d = reinterpret_cast<TV*>(dst + copied_pixel(r, p) * r.Ctot);
        for (uint32_t c0 = 0; c0 < r.Ctot; c0 += VEC) {
            const uint32_t g = fast_div(c0, r.div_cgp), c = c0 - g * r.cgp;      // (cgp is whole vectors)
            TV x;
#pragma unroll
            for (int e = 0; e < VEC; ++e) x[e] = c + e < r.cg ? src[(int64_t)(g * r.cg + c + e) * r.P + p] : (T)0;
            d[c0 / VEC] = x;
        }
        return;
    }
    const uint32_t p0 = pt * 64u, c0 = ct * 64u;
#pragma unroll
    for (int i = 0; i < 64 * VPR / 256; ++i) {
        const uint32_t v = threadIdx.x + 256u * i, c = v / VPR, p = p0 + v % VPR * VEC;
        const uint32_t ch = c0 + c, g = fast_div(ch, r.div_cgp), cc = ch - g * r.cgp;
        TV x = {};
        if (ch < r.Ctot && cc < r.cg && p < r.P) {
            const T* s = src + (int64_t)(g * r.cg + cc) * r.P + p;
            if (p + VEC <= r.P) x = *reinterpret_cast<const TU*>(s);
            else {
#pragma unroll
                for (int e = 0; e < VEC; ++e)
                    if (p + e < r.P) x[e] = s[e];
            }
        }
#pragma unroll
        for (int e = 0; e < VEC; ++e) tile[c * PITCH + v % VPR * VEC + e] = x[e];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 64 * VPR / 256; ++i) {
        const uint32_t v = threadIdx.x + 256u * i, pp = v / VPR, cv = v % VPR;
        if (c0 + cv * VEC < r.Ctot && p0 + pp < r.P) {
            TV x;
#pragma unroll
            for (int e = 0; e < VEC; ++e) x[e] = tile[(cv * VEC + e) * PITCH + pp];
            *reinterpret_cast<TV*>(dst + copied_pixel(r, p0 + pp) * r.Ctot + c0 + cv * VEC) = x;
        }
    }
}

hipError_t launch_channels_last(int64_t es, const ChannelsLast& job, hipStream_t s) {
    if (es != 2 && es != 4) return hipErrorInvalidValue;
    const int64_t vec = 16 / es;
    ClArgs a;
    std::memset(&a, 0, sizeof a);
    int64_t blocks = 0;
    const WeightsJob& w = job.weights;
    if (w.kind) {
        if (w.cgp % vec != 0 || (reinterpret_cast<uintptr_t>(w.wp) & 15) != 0) return hipErrorInvalidValue;
        const int64_t rows = w.kind == 3 ? w.rows * w.k_r * w.kq_pad : w.rows * w.taps;
        if (rows >= 0x7fffffffLL) return hipErrorInvalidValue;
        a.w.w = w.w; a.w.wp = w.wp; a.w.kind = (uint32_t)w.kind;
        a.w.vecs = rows * (w.cgp / vec);
        a.w.cgv = (uint32_t)(w.cgp / vec); a.w.cgp = (uint32_t)w.cgp; a.w.cg = (uint32_t)w.cg; a.w.taps = (uint32_t)w.taps; a.w.other = (uint32_t)w.other;
        a.w.k_r = (uint32_t)w.k_r; a.w.k_c = (uint32_t)w.k_c; a.w.kq_pad = (uint32_t)w.kq_pad; a.w.chunk = (uint32_t)w.chunk;
        a.w.div_cgv = make_fastdiv(a.w.cgv); a.w.div_taps = make_fastdiv(std::max(a.w.taps, 1u)); a.w.div_other = make_fastdiv(std::max(a.w.other, 1u));
        a.w.div_kq = make_fastdiv(std::max(a.w.kq_pad, 1u)); a.w.div_kr = make_fastdiv(std::max(a.w.k_r, 1u));
        blocks = std::min<int64_t>((a.w.vecs + 255) / 256, 4096);
        a.w.weight_blocks = (uint32_t)blocks;
        if (job.phases) {
            const int64_t ib = ((int64_t)job.phases->phases * job.phases->groups + 255) / 256;
            if (ib > 0x3fffffffLL) return hipErrorInvalidValue;
            blocks += ib;
        }
        a.w.blocks = (uint32_t)blocks;
    }
    for (int i = 0; i < job.n; ++i) {
        const ChannelsLastCopy& c = job.copy[i];
        const int64_t Ctot = c.groups * c.cgp;
        if (c.batch * Ctot * c.P == 0) continue;
        if (c.cgp % vec != 0 || c.P > 0x7fffffffLL - 256 || Ctot > 0x7fffffffLL || c.groups * c.cg > 0x7fffffffLL || (reinterpret_cast<uintptr_t>(c.out) & 15) != 0)
            return hipErrorInvalidValue;
        ClCopy& r = a.copy[a.n++];
        r.in = c.in; r.out = c.out;
        r.P = (uint32_t)c.P; r.cg = (uint32_t)c.cg; r.cgp = (uint32_t)c.cgp; r.C = (uint32_t)(c.groups * c.cg); r.Ctot = (uint32_t)Ctot;
        r.Pp = c.P;
        if (c.bordered) {
            const HaloMap& h = c.halo;
            r.h = h; r.Pp = h.vol(); r.on = 1;
            r.div_w = make_fastdiv((uint32_t)h.W); r.div_hw = make_fastdiv((uint32_t)(h.H * h.W));
            r.row_skip = (uint32_t)(h.Wp - h.W); r.slice_skip = (uint32_t)((h.Hp - h.H) * h.Wp);
            r.off0 = (uint32_t)((h.front * h.Hp + h.top) * h.Wp + h.left);
            r.vpp = (uint32_t)(Ctot / vec);
            const int64_t vecs = h.border() * r.vpp;
            if (vecs > 0x7fffffffLL || h.vol() > 0x7fffffffLL) return hipErrorInvalidValue;
            r.border_vecs = (uint32_t)vecs;
        }
        r.border_per_image = std::max(1u, (r.border_vecs + 1023u) / 1024u);
        const int64_t bb = r.border_vecs ? c.batch * r.border_per_image : 0;
        r.few = Ctot * es <= 32;
        r.tiles_p = (uint32_t)((c.P + (r.few ? 255 : 63)) / (r.few ? 256 : 64));
        r.tiles_c = r.few ? 1u : (uint32_t)((Ctot + 63) / 64);
        r.first = (uint32_t)blocks;
        const int64_t all = blocks + bb + (int64_t)r.tiles_p * r.tiles_c * c.batch;
        if (all > 0x7fffffffLL) return hipErrorInvalidValue;
        r.border_blocks = (uint32_t)bb;
        r.div_tp = make_fastdiv(r.tiles_p); r.div_tc = make_fastdiv(r.tiles_c); r.div_bpi = make_fastdiv(r.border_per_image); r.div_cgp = make_fastdiv(r.cgp);
        blocks = all;
    }
    if (blocks == 0) return hipSuccess;
    const dim3 g((unsigned)blocks), t(256);
    if (job.phases) {
        const ClPhases ph = {*job.phases, job.items};
        if (es == 2) hipLaunchKernelGGL((channels_last_kernel<uint16_t, ClPhases>), g, t, 0, s, a, ph);
        else hipLaunchKernelGGL((channels_last_kernel<uint32_t, ClPhases>), g, t, 0, s, a, ph);
    } else if (es == 2) hipLaunchKernelGGL((channels_last_kernel<uint16_t, ClNone>), g, t, 0, s, a, ClNone{});
    else hipLaunchKernelGGL((channels_last_kernel<uint32_t, ClNone>), g, t, 0, s, a, ClNone{});
    return hipGetLastError();
}

}  // namespace ntg
