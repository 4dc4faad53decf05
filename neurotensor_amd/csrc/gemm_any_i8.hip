// Int8 / UInt8 instantiations of the product on rows that start anywhere.
#include "gemm_any_impl.h"
namespace ntg {
hipError_t launch_gemm_any_i8(bool ta, bool tb, const GemmParams& p, hipStream_t s) { return launch_any<DT_I8>(ta, tb, p, s); }
}  // namespace ntg
