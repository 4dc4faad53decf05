// Int16 / Int32 / Int64 (and unsigned) products on the 8-bit matrix pipe.
#include "gemm_int_impl.h"
namespace ntg {
hipError_t launch_gemm_int(int planes, bool ta, bool tb, const GemmParams& p, hipStream_t s) {
    // 128 x 64 tiles (three quarters of the LDS reads and digits per product) where they put two on every CU: Int32 2048^3 79 us against 90, 8 x 1024^3 84 against
    // 92, Int16 2048^3 38 against 43; Int32 1024^3 (128 tiles) 29 against 18.6
    const bool wide = p.M > 64 && (int64_t)((p.M + 127) / 128) * ((p.N + 63) / 64) * p.batch >= 512;
    if (planes == 2) return wide ? launch_int_wb<2, 2>(ta, tb, p, s) : launch_int_wb<2, 1>(ta, tb, p, s);
    if (planes == 4) return wide ? launch_int_wb<4, 2>(ta, tb, p, s) : launch_int_wb<4, 1>(ta, tb, p, s);
    if (planes == 8) return launch_int_wb<8, 1>(ta, tb, p, s);
    return hipErrorInvalidValue;
}
}  // namespace ntg
