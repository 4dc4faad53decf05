// Float32 instantiations of the product on rows that start anywhere.
#include "gemm_any_impl.h"
namespace ntg {
hipError_t launch_gemm_any_f32(bool ta, bool tb, const GemmParams& p, hipStream_t s) { return launch_any<DT_F32>(ta, tb, p, s); }
}  // namespace ntg
