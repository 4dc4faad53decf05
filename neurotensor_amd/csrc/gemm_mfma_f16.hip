// Float16 instantiations of the MFMA GEMM (v_mfma_f32_32x32x16_f16, fp32 accumulate).
#include "gemm_ring_impl.h"
namespace ntg {
hipError_t launch_gemm_mfma_f16(bool ta, bool tb, const GemmParams& p, hipStream_t s) {
    if ((p.tailA || p.tailB) && !ring_eligible(p, ta)) return hipErrorInvalidValue;       // (only the DMA-fed kernel reads copied tail rows)
    if (ring_eligible(p, ta)) return launch_ring16<DT_F16>(ta, tb, p, s);   // DMA-fed LDS ring; the tile (256 x 256 .. 64 x 64, 192 x 256, 128 x 256) follows ring16_tile_edge
    if (any_eligible(p, DT_F16, ta, tb)) return launch_gemm_any(DT_F16, ta, tb, p, s);
    if (p.cmode == C_PARTIAL) return hipErrorInvalidValue;      // (this kernel would round the sums to 16 bits)
    // rows shorter than a 16-byte chunk, pitches from 8 MiB on: 128 x 128 x 64 (256 x 256: 8192 x 4 x 8192 127 us against 78, 4096 x 2048 x 4096 at such a pitch 98 / 100)
    return launch_trans<DT_F16, 2, 2, 64>(ta, tb, p, s);
}
hipError_t launch_gemm_ring_only_f16(bool ta, bool tb, const GemmParams& p, hipStream_t s, bool* taken) {
    *taken = ring_eligible(p, ta);
    return *taken ? launch_ring16<DT_F16>(ta, tb, p, s) : hipSuccess;
}
// convolution / conv_dkernel with op(B) gathered from the image (tb: col^T), nd = 2 or 3 spatial axes.  128 x 128 x 64 tiles,
// two workgroups per CU: the gather's registers do not fit beside a 256 x 256 accumulator.
hipError_t launch_conv_mfma_f16(bool tb, int nd, const GemmParams& p, hipStream_t s) {
    if (nd == 3) return tb ? launch_conv_cfg<DT_F16, true, 3, 2, 2, 64>(p, s) : launch_conv_cfg<DT_F16, false, 3, 2, 2, 64>(p, s);
    return tb ? launch_conv_cfg<DT_F16, true, 2, 2, 2, 64>(p, s) : launch_conv_cfg<DT_F16, false, 2, 2, 2, 64>(p, s);
}
hipError_t launch_conv_nhwc_f16(const GemmParams& p, hipStream_t s) {
    if (p.M <= 32) return ring16_flat_wide(p) ? launch_ring_nhwc_cfg<DT_F16, 2, true>(p, s) : launch_ring_nhwc_cfg<DT_F16, 1, true>(p, s);
    return launch_conv_nhwc16_planned(p, s, [&](int te, const GemmParams& q) {
        if (te == 256) return launch_ring_nhwc_cfg<DT_F16, 4>(q, s);
        if (te == 64) return launch_ring_nhwc_cfg<DT_F16, 1>(q, s);
        return launch_ring_nhwc_cfg<DT_F16, 2>(q, s);
    });
}
hipError_t launch_conv_nhwc_items_f16(int edge, const GemmParams& p, int64_t blocks, hipStream_t s) {
    if (edge == 256) return launch_ring_items_cfg<DT_F16, 4>(p, blocks, s);
    if (edge == 64) return launch_ring_items_cfg<DT_F16, 1>(p, blocks, s);
    if (edge == 32) return launch_ring_items_cfg<DT_F16, 1, true>(p, blocks, s);
    return launch_ring_items_cfg<DT_F16, 2>(p, blocks, s);
}
hipError_t launch_conv_nhwc_dw_f16(bool ta, const GemmParams& p, hipStream_t s) { return launch_ring_nhwc_dw<DT_F16>(ta, p, s); }
}  // namespace ntg
