// Int8 / UInt8 on the matrix pipe: v_mfma_i32_32x32x32_i8 in the DMA-fed LDS ring kernel.  The reference multiplies and
// adds 8-bit integers with wrap-around in the element type (nt/mp/simde_traits/simde_traits_avx2.h:668-670); the low 8 bits
// of the exact products' 32-bit sum are that result for either signedness, so the outputs are bit-identical.  Rows that are
// not 16-byte multiples run on gemm_any_impl.h, rows shorter than 16 bytes on the vector ALU.  16-, 32- and 64-bit integer products: gemm_int_impl.h.
#include "gemm_ring_impl.h"
namespace ntg {
hipError_t launch_gemm_mfma_i8(int dtype, bool ta, bool tb, const GemmParams& p, hipStream_t s) {
    if ((p.tailA || p.tailB) && !ring_eligible(p, ta, 1)) return hipErrorInvalidValue;     // (only the DMA-fed kernel reads copied tail rows)
    if (!ring_eligible(p, ta, 1)) {
        if (any_eligible(p, dtype, ta, tb)) return launch_gemm_any(dtype, ta, tb, p, s);
        return launch_gemm_valu(dtype, ta, tb, p, s);
    }
    // (an MN-major 192-row tile of bytes has 12 chunks per k-row, which the chunk swizzle of the transposing reads does not fit)
    const int rect = ta ? RECT_128 : RECT_128 | RECT_192;
    auto launch = [&](int te, const GemmParams& q) {
        if (te == 256) return launch_ring_wb<DT_I8, 4>(ta, tb, q, s);
        if (te == 224) return tb ? launch_ring_cfg<DT_I8, false, true, 3, 4>(q, s) : launch_ring_cfg<DT_I8, false, false, 3, 4>(q, s);
        if (te == 192) return launch_ring_wb<DT_I8, 2, 4, 2>(ta, tb, q, s);     // (128-byte K-steps, as for the 16-bit products)
        if (te == 64) return launch_ring_wb<DT_I8, 1>(ta, tb, q, s);
        // (k in 16-bit elements: the same number of K-steps)
        if (ring16_deep128(ring16_tiles(128, q.M, q.N, q.batch), q.K / 2)) return launch_ring_wb<DT_I8, 2, 0, 2>(ta, tb, q, s);
        return launch_ring_wb<DT_I8, 2>(ta, tb, q, s);
    };
    if (p.batch == 1) {
        // (the estimate of the 16-bit kernel: a K-step of 64 bytes per row is 64 k here, so the same tile takes half the steps)
        const Ring16Split sp = ring16_split(p.M, p.N, p.K, rect);
        if (sp.axis) {
            GemmParams head, tail;
            ring_split_params(p, ta, tb, 1, sp, head, tail);
            const hipError_t e = launch(sp.head_edge, head);
            if (e != hipSuccess) return e;
            return launch(sp.tail_edge, tail);
        }
    }
    return launch(ring16_tile_edge(p.M, p.N, p.K, p.batch, rect), p);
}
// the DMA-fed kernel or nothing (the gated pair of an unvouched pointer-table batch)
hipError_t launch_gemm_ring_only_i8(int dtype, bool ta, bool tb, const GemmParams& p, hipStream_t s, bool* taken) {
    *taken = ring_eligible(p, ta, 1);
    return *taken ? launch_gemm_mfma_i8(dtype, ta, tb, p, s) : hipSuccess;
}
}  // namespace ntg
