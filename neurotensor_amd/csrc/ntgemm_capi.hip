// C ABI of the gfx950 matmult backend (declared in include/ntgemm.h): argument checks,
// dtype dispatch, host<->device staging for the host-pointer entry points, and the
// conv2d lowering.  No entry point throws; failures are reported as ntg_status plus a
// thread-local message.
#include "../../include/ntgemm.h"
#include "ntg_common.h"
#include "host_stage.h"

#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace ntg {
hipError_t launch_gemm_mfma_f32(bool ta, bool tb, const GemmParams& p, hipStream_t s);
hipError_t launch_gemm_mfma_f64(bool ta, bool tb, const GemmParams& p, hipStream_t s);
hipError_t launch_gemm_mfma_f16(bool ta, bool tb, const GemmParams& p, hipStream_t s);
hipError_t launch_gemm_mfma_bf16(bool ta, bool tb, const GemmParams& p, hipStream_t s);
hipError_t launch_gemm_skinny(int dtype, bool ta, bool tb, const GemmParams& p, hipStream_t s, bool* handled);
hipError_t launch_gemm_ring_only_f32(bool ta, bool tb, const GemmParams& p, hipStream_t s, bool* taken);
hipError_t launch_gemm_ring_only_f16(bool ta, bool tb, const GemmParams& p, hipStream_t s, bool* taken);
hipError_t launch_gemm_ring_only_bf16(bool ta, bool tb, const GemmParams& p, hipStream_t s, bool* taken);
hipError_t launch_gemm_ring_only_i8(int dtype, bool ta, bool tb, const GemmParams& p, hipStream_t s, bool* taken);
hipError_t launch_gemm_ring_only_f64(bool ta, bool tb, const GemmParams& p, hipStream_t s, bool* taken);
hipError_t launch_gemm_ring_only(int dtype, bool ta, bool tb, const GemmParams& p, hipStream_t s, bool* taken) {
    *taken = false;
    switch (dtype) {
    case DT_I8: case DT_U8: return launch_gemm_ring_only_i8(dtype, ta, tb, p, s, taken);
    case DT_F32: return launch_gemm_ring_only_f32(ta, tb, p, s, taken);
    case DT_F64: return launch_gemm_ring_only_f64(ta, tb, p, s, taken);
    case DT_F16: return launch_gemm_ring_only_f16(ta, tb, p, s, taken);
    case DT_BF16: return launch_gemm_ring_only_bf16(ta, tb, p, s, taken);
    default: return hipSuccess;
    }
}
hipError_t launch_gemm_any_f32(bool ta, bool tb, const GemmParams& p, hipStream_t s);
hipError_t launch_gemm_any_f16(bool ta, bool tb, const GemmParams& p, hipStream_t s);
hipError_t launch_gemm_any_bf16(bool ta, bool tb, const GemmParams& p, hipStream_t s);
hipError_t launch_gemm_any_i8(bool ta, bool tb, const GemmParams& p, hipStream_t s);
hipError_t launch_gemm_any(int dtype, bool ta, bool tb, const GemmParams& p, hipStream_t s) {
    switch (dtype) {
    case DT_I8: case DT_U8: return launch_gemm_any_i8(ta, tb, p, s);
    case DT_F32: return launch_gemm_any_f32(ta, tb, p, s);
    case DT_F16: return launch_gemm_any_f16(ta, tb, p, s);
    case DT_BF16: return launch_gemm_any_bf16(ta, tb, p, s);
    default: return hipErrorInvalidValue;
    }
}
hipError_t launch_conv_mfma_f32(bool tb, int nd, const GemmParams& p, hipStream_t s);
hipError_t launch_conv_mfma_f64(bool tb, int nd, const GemmParams& p, hipStream_t s);
hipError_t launch_conv_mfma_f16(bool tb, int nd, const GemmParams& p, hipStream_t s);
hipError_t launch_conv_mfma_bf16(bool tb, int nd, const GemmParams& p, hipStream_t s);

hipError_t launch_conv_nhwc_f32(const GemmParams& p, hipStream_t s);
hipError_t launch_conv_nhwc_f16(const GemmParams& p, hipStream_t s);
hipError_t launch_conv_nhwc_bf16(const GemmParams& p, hipStream_t s);
hipError_t launch_conv_nhwc(int dtype, const GemmParams& p, hipStream_t s) {
    switch (dtype) {
    case DT_F32: return launch_conv_nhwc_f32(p, s);
    case DT_F16: return launch_conv_nhwc_f16(p, s);
    case DT_BF16: return launch_conv_nhwc_bf16(p, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_conv_nhwc_items_f32(int edge, const GemmParams& p, int64_t blocks, hipStream_t s);
hipError_t launch_conv_nhwc_items_f16(int edge, const GemmParams& p, int64_t blocks, hipStream_t s);
hipError_t launch_conv_nhwc_items_bf16(int edge, const GemmParams& p, int64_t blocks, hipStream_t s);
hipError_t launch_conv_nhwc_items(int dtype, int edge, const GemmParams& p, int64_t blocks, hipStream_t s) {
    switch (dtype) {
    case DT_F32: return launch_conv_nhwc_items_f32(edge, p, blocks, s);
    case DT_F16: return launch_conv_nhwc_items_f16(edge, p, blocks, s);
    case DT_BF16: return launch_conv_nhwc_items_bf16(edge, p, blocks, s);
    default: return hipErrorInvalidValue;
    }
}
hipError_t launch_conv_nhwc_dw_f32(bool ta, const GemmParams& p, hipStream_t s);
hipError_t launch_conv_nhwc_dw_f16(bool ta, const GemmParams& p, hipStream_t s);
hipError_t launch_conv_nhwc_dw_bf16(bool ta, const GemmParams& p, hipStream_t s);
hipError_t launch_conv_nhwc_dw(int dtype, bool ta, const GemmParams& p, hipStream_t s) {
    switch (dtype) {
    case DT_F32: return launch_conv_nhwc_dw_f32(ta, p, s);
    case DT_F16: return launch_conv_nhwc_dw_f16(ta, p, s);
    case DT_BF16: return launch_conv_nhwc_dw_bf16(ta, p, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_conv_mfma(int dtype, bool tb, int nd, const GemmParams& p, hipStream_t s) {
    switch (dtype) {
    case DT_F32: return launch_conv_mfma_f32(tb, nd, p, s);
    case DT_F64: return launch_conv_mfma_f64(tb, nd, p, s);
    case DT_F16: return launch_conv_mfma_f16(tb, nd, p, s);
    case DT_BF16: return launch_conv_mfma_bf16(tb, nd, p, s);
    default: return hipErrorInvalidValue;
    }
}
}  // namespace ntg

// Scratch memory of ntg_gemm_noalloc_dev: a fixed array in every GPU's copy of this code object, so that the entry point
// needs no allocator.  Host code never uses the array's name as an address: ntg::noalloc_scratch_of_current_device() asks the runtime
// for the address of the current device's copy once and keeps it.
static __device__ __align__(256) unsigned char scratch[NTG_NOALLOC_SCRATCH_BYTES];

// Flags of ntg_gemm_ptrs_dev's alignment check (one word per call, handed out round-robin), in the same kind of array and
// for the same reason: the device entry points allocate nothing.
#define NTG_GATE_SLOTS 1024
static __device__ __align__(256) int gate_flags[NTG_GATE_SLOTS];
namespace ntg {
// *flag = 1 when every entry of the three pointer tables is a multiple of 16 bytes, else 0
__global__ void __launch_bounds__(256) ptr_tables_aligned_kernel(const void* const* a, const void* const* b, void* const* c, const int batch, int* flag) {
    __shared__ unsigned bits;
    if (threadIdx.x == 0) bits = 0u;
    __syncthreads();
    unsigned mine = 0u;
    for (int i = threadIdx.x; i < batch; i += 256)
        mine |= (unsigned)(reinterpret_cast<uintptr_t>(a[i]) | reinterpret_cast<uintptr_t>(b[i]) | reinterpret_cast<uintptr_t>(c[i])) & 15u;
    if (mine) atomicOr(&bits, mine);
    __syncthreads();
    if (threadIdx.x == 0) *flag = bits == 0u ? 1 : 0;
}
}  // namespace ntg

namespace {

thread_local std::string g_last_error;

int fail(int status, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_last_error = buf;
    return status;
}

int hip_fail(hipError_t e, const char* what) {
    if (e == hipErrorOutOfMemory) return fail(NTG_ERR_OUT_OF_MEMORY, "%s: %s", what, hipGetErrorString(e));
    if (e == hipErrorNoDevice || e == hipErrorInvalidDevice) return fail(NTG_ERR_NO_DEVICE, "%s: %s", what, hipGetErrorString(e));
    return fail(NTG_ERR_DEVICE, "%s: %s", what, hipGetErrorString(e));
}

#define HIP_TRY(expr)                                   \
    do {                                                \
        hipError_t e__ = (expr);                        \
        if (e__ != hipSuccess) return hip_fail(e__, #expr); \
    } while (0)


inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

bool is_int_dtype(int dt) {
    switch (dt) {
    case ntg::DT_I8: case ntg::DT_I16: case ntg::DT_I32: case ntg::DT_I64:
    case ntg::DT_U8: case ntg::DT_U16: case ntg::DT_U32: case ntg::DT_U64: return true;
    default: return false;
    }
}

bool is_complex_dtype(int dt) { return dt == ntg::DT_C32 || dt == ntg::DT_C64 || dt == ntg::DT_C128; }
// integers and the complex types: computed lane by lane on the vector ALU, bit-exact; no matrix-pipe or gathering forms
bool is_valu_dtype(int dt) { return is_int_dtype(dt) || is_complex_dtype(dt); }

// 16-, 32- and 64-bit integers on the 8-bit matrix pipe (gemm_int_impl.h): bytes per element
static int int_planes_of(int dtype) {
    switch (dtype) {
    case ntg::DT_I16: case ntg::DT_U16: return 2;
    case ntg::DT_I32: case ntg::DT_U32: return 4;
    case ntg::DT_I64: case ntg::DT_U64: return 8;
    default: return 0;
    }
}
// Every contiguous extent holds the eight elements of a group, 32-bit lane offsets, 32-bit sums of a shift's products (P K 2^14 < 2^31).
// What misses this runs on the vector ALU, bit for bit the same; so does Int64 of up to 16 k, one pass of that kernel and half a K-step here, on more than
// 256 tiles (one wavefront a SIMD here): 4096 x 16 x 4096 64 us against 76, 2048 x 16 x 2048 20.3 / 21.8, 1500 x 8 x 1500 14.9 / 17.9, 1024 x (16 x 16 x 16)
// 13.5 / 16.8, but 1024 x 16 x 1024 10.2 / 7.4; from 17 k on the digits win on any number of tiles (4096 x 20 x 4096 87 / 76, 2048 x 20 x 2048 27 / 22).  Int16 and
// Int32 win everywhere (4096 x 8 x 4096 25 / 20 and 34 / 22.5, 4096 x (8 x 8 x 8) 19 / 12 and 23 / 20).
static bool int_pipe_eligible(const ntg::GemmParams& p, int dtype, bool ta, bool tb) {
    const int64_t P = int_planes_of(dtype);
    if (P == 8 && p.K <= 16 && (int64_t)((p.M + 63) / 64) * ((p.N + 63) / 64) * p.batch > 256) return false;
    return P != 0 && p.K > 0 && (ta ? p.M : p.K) >= 8 && (tb ? p.K : p.N) >= 8 && P * (int64_t)p.K < (1 << 17) && p.lda * P < (1 << 23) && p.ldb * P < (1 << 23);
}

// Fills the derived fields and launches the kernel family for the dtype.
int launch_gemm(ntg::GemmParams p, int dtype, bool ta, bool tb, hipStream_t s) {
    const int64_t es = ntg::elem_size(dtype);
    const int64_t ve = 16 / es;
    p.vecA_ok = (p.lda % ve == 0) && (p.Aptr || p.sA % ve == 0) && (p.krange_items == 0 || p.sAk % ve == 0);
    p.vecB_ok = (p.ldb % ve == 0) && (p.Bptr || p.sB % ve == 0) && (p.krange_items == 0 || p.sBk % ve == 0);
    hipError_t e;
    // relu_ on the result: inside the epilogue of the DMA-fed kernels, of those for rows as they lie and of the streaming ones for up to 32 rows,
    // else as a pass over C after whichever kernel runs
    const int act = p.act;
    p.act = ntg::ACT_NONE;
    if (act != ntg::ACT_NONE) {
        if (p.Cptr || !(dtype == ntg::DT_F32 || dtype == ntg::DT_F64 || dtype == ntg::DT_F16 || dtype == ntg::DT_BF16))
            return fail(NTG_ERR_INVALID_ARGUMENT, "the relu epilogue takes strided floating-point results");
        if (p.M > 32 && p.cmode != ntg::C_PARTIAL) {
            ntg::GemmParams q = p;
            q.act = act;
            bool taken = false;
            e = ntg::launch_gemm_ring_only(dtype, ta, tb, q, s, &taken);
            if (e != hipSuccess) return hip_fail(e, "gemm launch");
            if (taken) return NTG_OK;
            if (ntg::any_eligible(p, dtype, ta, tb)) {
                e = ntg::launch_gemm_any(dtype, ta, tb, q, s);
                return e == hipSuccess ? NTG_OK : hip_fail(e, "gemm launch");
            }
        }
    }
    const auto finish = [&]() -> int {
        if (act == ntg::ACT_NONE) return NTG_OK;
        const hipError_t ea = ntg::launch_relu_inplace(dtype, p.C, p.ldc, p.sC, p.M, p.N, p.batch, s);
        return ea == hipSuccess ? NTG_OK : hip_fail(ea, "relu launch");
    };
    if (dtype == ntg::DT_I8 || dtype == ntg::DT_U8) {
        e = ntg::launch_gemm_mfma_i8(dtype, ta, tb, p, s);
    } else if (int_pipe_eligible(p, dtype, ta, tb)) {
        e = ntg::launch_gemm_int(int_planes_of(dtype), ta, tb, p, s);
    } else if (is_int_dtype(dtype)) {
        e = ntg::launch_gemm_valu(dtype, ta, tb, p, s);
    } else if (is_complex_dtype(dtype)) {
        e = ntg::launch_gemm_complex(dtype, ta, tb, p, s);
    } else {
        bool handled = false;
        // (the streaming kernels for up to 32 rows split k over their wavefronts: not for a caller who wants the one chain.  Items in groups or k ranges go there
        //  in Float32, where the eight short chains are what a result errs by: 2 x 512 x 28 x 28 -> 32 by one tap in 2 groups 1.17e-7 against 2.87e-7; 16-bit
        //  results err by their rounding, and the tiles' kernels are faster)
        e = hipSuccess;
        if (dtype == ntg::DT_F32 ? !p.keep_k_order : p.krange_items == 0) {
            p.act = act;                                                   // (its epilogue clamps)
            e = ntg::launch_gemm_skinny(dtype, ta, tb, p, s, &handled);
            p.act = ntg::ACT_NONE;
        }
        if (e != hipSuccess) return hip_fail(e, "skinny gemm launch");
        if (handled) return NTG_OK;
        switch (dtype) {
        case ntg::DT_F32: e = ntg::launch_gemm_mfma_f32(ta, tb, p, s); break;
        case ntg::DT_F64: e = ntg::launch_gemm_mfma_f64(ta, tb, p, s); break;
        case ntg::DT_F16: e = ntg::launch_gemm_mfma_f16(ta, tb, p, s); break;
        case ntg::DT_BF16: e = ntg::launch_gemm_mfma_bf16(ta, tb, p, s); break;
        default: return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
        }
    }
    if (e != hipSuccess) return hip_fail(e, "gemm launch");
    return finish();
}

// Split-K.  A product whose output tiles cannot occupy the 256 CUs but whose K is deep (a Linear layer on a few
// hundred rows) is cut into `splits` equal k ranges, computed as one batched launch of the ordinary kernels into a
// workspace [splits][M][N] (fp32 sums for the 16-bit dtypes, so nothing is rounded early), and added up in ascending
// range order by a second kernel.  Deterministic; applied only when the caller supplies the workspace.
// The plan is a function of ONE item's M, N, K (and dtype, flags, alignment) only, never of the batch count: a split
// changes the order of summation over k, and an item must come out bit for bit the same alone and inside a batch
// (the reference's batched == per-item rule, tests/src/matmult_test.cpp:108-189).  A batch whose items are split runs one
// batched launch per k range into [splits][batch][M][N] and one reduction over all items.
struct SplitPlan { int splits; int64_t kc; int64_t bytes; };

// Padded copies.  The DMA-fed kernels need 16-byte rows (leading dimensions, batch strides, base pointers, and K, N -- M
// under transpose_a -- multiples of one 16-byte chunk); a product that misses this runs on rows as they lie (gemm_any_impl.h), Float64 on
// the register-staged kernel at 0.8 of the rate.  With a workspace the operands that need it
// are copied into rows padded with zeros to whole chunks (zero products add nothing: bit-identical integers, the same
// single rounding for the 16-bit floats), the product runs on the DMA-fed kernel, and a result whose own rows are not
// 16-byte multiples is computed into a padded copy and copied back.  Taken for products large enough to repay the copies.
struct PadPlan {
    bool ok, pays, padA, padB, padC;   // ok: it can be done; pays: nothing else is faster
    bool stripA, stripB;            // the operand stays where it is, only its last k-rows are copied (and continued with zeros)
    int strip_k0, strip_rows;
    int Mp, Kp, Np;
    int64_t lda2, ldb2, rowsA2, rowsB2, a_bytes, b_bytes, c_bytes;
    int64_t bytes() const { return a_bytes + b_bytes + c_bytes; }
};
SplitPlan plan_splitk(const ntg::GemmParams& p, int dtype, bool ta);
static PadPlan plan_pad(const ntg::GemmParams& p, int dtype, bool ta, bool tb) {
    PadPlan pl;
    std::memset(&pl, 0, sizeof pl);
    const bool half = dtype == ntg::DT_F16 || dtype == ntg::DT_BF16, byte = dtype == ntg::DT_I8 || dtype == ntg::DT_U8;
    const bool wide = dtype == ntg::DT_F32 || dtype == ntg::DT_F64;
    if ((!half && !byte && !wide) || p.Aptr || p.Bptr || p.Cptr || p.M <= 32) return pl;
    const int64_t es = ntg::elem_size(dtype), ve = 16 / es;
    // From where copies of an operand's last k-rows, as good as free, pay; Float64: from where whole copies pay against the register-staged kernel.
    // (Whole copies of the other types: see below.)
    const double macs = (double)p.M * p.N * p.K * p.batch;
    const double from = byte ? 268435456.0 : half ? 2147483648.0 : dtype == ntg::DT_F32 ? 4294967296.0 : 8589934592.0;
    if (macs < from) return pl;
    // (an item that alone is too small for copies, and is split along k instead, keeps that order of summation in a batch that is not: Float64)
    if (macs / p.batch < from && plan_splitk(p, dtype, ta).splits > 1) return pl;
    auto up = [&](int64_t v) { return (v + ve - 1) / ve * ve; };
    pl.Kp = (int)up(p.K); pl.Np = (int)up(p.N); pl.Mp = ta ? (int)up(p.M) : p.M;
    auto misaligned = [&](const void* ptr, int64_t ld, int64_t stride) {
        return ld % ve != 0 || (p.batch > 1 && stride % ve != 0) || (reinterpret_cast<uintptr_t>(ptr) & 15) != 0;
    };
    pl.padA = misaligned(p.A, p.lda, p.sA) || pl.Kp != p.K || pl.Mp != p.M;
    pl.padB = misaligned(p.B, p.ldb, p.sB) || pl.Kp != p.K || pl.Np != p.N;
    pl.padC = misaligned(p.C, p.ldc, p.sC) || pl.Np != p.N || pl.Mp != p.M;
    if (!pl.padA && !pl.padB && !pl.padC) return pl;                       // nothing that padding would fix
    // (the copies' rows start on 128-byte boundaries: a pitch that is only a multiple of 16 bytes splits the cache lines that the
    //  kernel fetches, which costs it 3 - 13 %)
    auto line_pitch = [&](int64_t elems) { return (elems * es + 127) / 128 * 128 / es; };
    pl.lda2 = line_pitch(ta ? pl.Mp : pl.Kp); pl.rowsA2 = ta ? pl.Kp : p.M;
    pl.ldb2 = line_pitch(tb ? pl.Kp : pl.Np); pl.rowsB2 = tb ? pl.Np : pl.Kp;
    const int64_t ldmax = (int64_t)(1 << 23) / es;                         // (the kernels' 32-bit lane offsets)
    if ((pl.padA ? pl.lda2 : p.lda) >= ldmax || (pl.padB ? pl.ldb2 : p.ldb) >= ldmax) return pl;
    // An operand stored [k][m] / [k][n] that only lacks k-rows up to a whole chunk: its rows keep the 16-byte rule, so the kernel
    // reads it in place and takes its last k-rows (from a multiple of 128, which every kernel's K-step divides) from a copy of at
    // most 128 rows that continues with rows of zeros, instead of a copy of everything.
    if (pl.Kp != p.K && p.K > 128) {
        pl.strip_k0 = (pl.Kp - 1) / 128 * 128;
        pl.strip_rows = pl.Kp - pl.strip_k0;
        pl.stripA = pl.padA && ta && !misaligned(p.A, p.lda, p.sA) && pl.Mp == p.M;
        pl.stripB = pl.padB && !tb && !misaligned(p.B, p.ldb, p.sB) && pl.Np == p.N;
        if (pl.stripA) { pl.padA = false; pl.a_bytes = (int64_t)align_up((size_t)((p.sA == 0 ? 1 : p.batch) * pl.strip_rows * p.lda * es), 256); }
        if (pl.stripB) { pl.padB = false; pl.b_bytes = (int64_t)align_up((size_t)((p.sB == 0 ? 1 : p.batch) * pl.strip_rows * p.ldb * es), 256); }
    }
    if (pl.padA) pl.a_bytes = (int64_t)align_up((size_t)((p.sA == 0 ? 1 : p.batch) * pl.rowsA2 * pl.lda2 * es), 256);
    if (pl.padB) pl.b_bytes = (int64_t)align_up((size_t)((p.sB == 0 ? 1 : p.batch) * pl.rowsB2 * pl.ldb2 * es), 256);
    if (pl.padC) pl.c_bytes = (int64_t)align_up((size_t)((int64_t)p.batch * pl.Mp * pl.Np * es), 256);
    pl.ok = true;
    // The kernel that takes rows as they lie (gemm_any_impl.h) makes whole copies pay later; where only the last k-rows are copied they are as good
    // as free.  Copies against no copies: Float16 1023 x 1537 x 2049 (3.2e9) 30.4 us against 26.7, 27 x 1704 x 229 x 960 (1.0e10) 64 against 56, 8 x 1201 x
    // 1301 x 903 (1.1e10) 57.2 against 53.7, 2049^3 (8.6e9) 50.4 against 49.7; BFloat16 2813 x 803 x 2240 (5.1e9) 28.0 against 23.3, 8192 x 999 x 999
    // A^T.B (8.2e9) 40.8 against 29.8, 3618 x 739 x 9392 (2.5e10) 73 against 84, 4095^3 145 against 192; Float32 2049^3 211 against 187, 1504 x 727 x
    // 8952 (9.8e9) 180 against 191; Int8 2049^3 36.7 against 33.3, 1002 x 257 x 2431 14.8 against 9.8.
    pl.pays = !(pl.padA || pl.padB || pl.padC) || !ntg::any_eligible(p, dtype, ta, tb) || macs >= (byte ? 1.7e10 : half ? 1.6e10 : dtype == ntg::DT_F32 ? 9.0e9 : 0.0);
    return pl;
}
static int run_padded(const ntg::GemmParams& p, const PadPlan& pl, int dtype, bool ta, bool tb, void* ws, hipStream_t s) {
    const int64_t es = ntg::elem_size(dtype);
    char* a2 = static_cast<char*>(ws);
    char* b2 = a2 + pl.a_bytes;
    char* c2 = b2 + pl.b_bytes;
    ntg::GemmParams q = p;
    q.M = pl.Mp; q.K = pl.Kp; q.N = pl.Np;
    hipError_t e;
    ntg::PadJobs jobs;
    std::memset(&jobs, 0, sizeof jobs);
    const int64_t itemsA = p.sA == 0 ? 1 : p.batch, itemsB = p.sB == 0 ? 1 : p.batch;
    auto copy = [&](const void* src, int64_t ld_src, int64_t s_src, void* dst, int64_t ld_dst, int64_t rows, int64_t cols, int64_t rows_dst, int64_t items) {
        ntg::PadJob& j = jobs.job[jobs.n++];
        j.src = src; j.ld_src = ld_src; j.s_src = s_src;
        j.dst = dst; j.ld_dst = ld_dst; j.s_dst = rows_dst * ld_dst;
        j.rows = rows; j.cols = cols; j.rows_dst = rows_dst; j.batch = items;
    };
    if (pl.padA) {
        copy(p.A, p.lda, p.sA, a2, pl.lda2, ta ? p.K : p.M, ta ? p.M : p.K, pl.rowsA2, itemsA);
        q.A = a2; q.lda = pl.lda2; q.sA = p.sA == 0 ? 0 : pl.rowsA2 * pl.lda2;
    } else if (pl.stripA) {
        copy(static_cast<const char*>(p.A) + (int64_t)pl.strip_k0 * p.lda * es, p.lda, p.sA, a2, p.lda, p.K - pl.strip_k0, p.M, pl.strip_rows, itemsA);
        q.tailA = a2; q.s_tailA = p.sA == 0 ? 0 : (int64_t)pl.strip_rows * p.lda; q.tail_k0 = pl.strip_k0;
    }
    if (pl.padB) {
        copy(p.B, p.ldb, p.sB, b2, pl.ldb2, tb ? p.N : p.K, tb ? p.K : p.N, pl.rowsB2, itemsB);
        q.B = b2; q.ldb = pl.ldb2; q.sB = p.sB == 0 ? 0 : pl.rowsB2 * pl.ldb2;
    } else if (pl.stripB) {
        copy(static_cast<const char*>(p.B) + (int64_t)pl.strip_k0 * p.ldb * es, p.ldb, p.sB, b2, p.ldb, p.K - pl.strip_k0, p.N, pl.strip_rows, itemsB);
        q.tailB = b2; q.s_tailB = p.sB == 0 ? 0 : (int64_t)pl.strip_rows * p.ldb; q.tail_k0 = pl.strip_k0;
    }
    if (pl.padC && p.cmode == ntg::C_ACCUMULATE) copy(p.C, p.ldc, p.sC, c2, pl.Np, p.M, p.N, pl.Mp, p.batch);
    if (jobs.n) {
        e = ntg::launch_pad_copies(es, jobs, s);
        if (e != hipSuccess) return hip_fail(e, "padded copies");
    }
    if (pl.padC) {
        const int64_t sc2 = (int64_t)pl.Mp * pl.Np;
        if (p.cmode == ntg::C_BIAS) {
            // the bias becomes the initial accumulator in the padded layout (reading it at padded indices would leave its array)
            e = ntg::launch_bias_fill(es, p.bias, p.bias_bs, p.bias_rs, p.bias_cs, c2, pl.Np, sc2, p.M, p.N, pl.Mp, p.batch, s);
            if (e != hipSuccess) return hip_fail(e, "bias fill");
            q.cmode = ntg::C_ACCUMULATE;
            q.bias = nullptr;
        }
        q.C = c2; q.ldc = pl.Np; q.sC = sc2;
    }
    const int rc = launch_gemm(q, dtype, ta, tb, s);
    if (rc) return rc;
    if (pl.padC) {
        e = ntg::launch_unpad_copy(es, c2, pl.Np, (int64_t)pl.Mp * pl.Np, p.C, p.ldc, p.sC, p.M, p.N, p.batch, s);
        if (e != hipSuccess) return hip_fail(e, "copy of the padded result");
    }
    return NTG_OK;
}

SplitPlan plan_splitk(const ntg::GemmParams& p, int dtype, bool ta) {
    SplitPlan none{1, p.K, 0};
    const int64_t es = ntg::elem_size(dtype);
    if (is_valu_dtype(dtype) || es == 0 || p.batch < 1 || p.batch > 65535 || p.Aptr || p.Bptr || p.Cptr || p.keep_k_order) return none;
    if (p.M <= 32 && dtype != ntg::DT_F64) return none;                       // the streaming kernels take these
    const bool half = dtype == ntg::DT_F16 || dtype == ntg::DT_BF16;
    if (half) {
        // only the DMA-fed kernel writes fp32 partial sums: 16-byte rows everywhere
        if (p.K % 8 || p.N % 8 || (ta && p.M % 8) || p.lda % 8 || p.ldb % 8 || p.lda >= (1 << 22) || p.ldb >= (1 << 22)) return none;
        if ((reinterpret_cast<uintptr_t>(p.A) & 15) || (reinterpret_cast<uintptr_t>(p.B) & 15)) return none;
        if (p.batch > 1 && (p.sA % 8 || p.sB % 8)) return none;
        // Both sides from the tile estimate of the 16-bit kernels (ring16_cost_us): the product as it is, against S batched
        // products over K / S (the tiles that the batched launch picks) plus the second pass, measured at about 4 us + the
        // fp32 partial sums written and read (8 S M N bytes) at 4 TB/s.  A split has to win by 5 %.  On a sweep of 23
        // shapes (64 .. 1024 rows, k 2048 .. 16384) the choice is the best measured S in 20 and within 5 % in two more
        // (1024 x 4096 x 1024: no split, 20.9 us against 24.5; 64 x 8192 x 8192: two ranges, 26.9 us against 38.3).
        const int rect = ntg::RECT_128 | ntg::RECT_192;
        const int edge1 = ntg::ring16_tile_edge(p.M, p.N, p.K, 1, rect);
        if (edge1 == 256) return none;                                // (larger problems fill the chip by themselves)
        const double whole_us = ntg::ring16_cost_us(edge1, ntg::ring16_tiles(edge1, p.M, p.N, 1), p.K);
        int64_t best = 1;
        double best_us = whole_us;
        for (int64_t sp = 2; sp <= 16; ++sp) {
            if (p.K % (sp * 32) != 0 || p.K / sp < 256) continue;
            const int edge = ntg::ring16_tile_edge(p.M, p.N, p.K / sp, sp, rect);
            const double us = ntg::ring16_cost_us(edge, ntg::ring16_tiles(edge, p.M, p.N, sp), p.K / sp) + 4.0 +
                              8.0 * (double)sp * (double)p.M * (double)p.N / 4.0e6;
            if (us < 0.95 * whole_us && us < best_us) { best = sp; best_us = us; }
        }
        if (best == 1) return none;
        return SplitPlan{(int)best, p.K / best, best * (int64_t)p.batch * p.M * p.N * 4};
    }
    // fp32 / fp64: their kernels go down to 64 x 64 tiles by themselves; a split pays only when those leave CUs without a
    // tile.  Same kind of estimate: a CU spends about 14.4 ns (fp32) / 28.8 ns (fp64) per k on each 64 x 64 tile it is
    // handed; the second pass costs about 5 us + the partial sums written and read at 4 TB/s.
    const int64_t tiles = ((p.M + 63) / 64) * ((p.N + 63) / 64);
    if (tiles > 255) return none;
    const double per_k = dtype == ntg::DT_F32 ? 0.0144 : 0.0288;
    auto estimate_us = [&](int64_t sp) {
        const double rounds = (double)((tiles * sp + 255) / 256);
        const double second_pass = sp == 1 ? 0.0 : 5.0 + 2.0 * (double)sp * (double)p.M * (double)p.N * (double)es / 4.0e6;
        return rounds * (double)(p.K / sp) * per_k + second_pass;
    };
    int64_t best = 1;
    double best_us = estimate_us(1);
    for (int64_t sp = 2; sp <= 16; ++sp) {
        if (p.K % (sp * 32) != 0 || p.K / sp < 64) continue;
        const double us = estimate_us(sp);
        if (us < 0.9 * best_us) { best = sp; best_us = us; }
    }
    if (best > 1) return SplitPlan{(int)best, p.K / best, best * (int64_t)p.batch * p.M * p.N * es};
    return none;
}

// k ranges of a product whose rows miss the 16-byte rule by their SIZES (gemm_any_impl.h serves it): for floats, as plan_splitk, a function of one
// item's sizes and pitches only.  kc is a whole number of K-steps, the last range is what is left.  Rows of the partial sums hold whole 16-byte chunks.
// The integers of more than a byte likewise (gemm_int_impl.h).
// inside: a workgroup runs all ranges of its tile (the sums of these are added in registers, in the order of the second pass: the same bits).  It needs
// no room; 256 bytes stand for the caller's leave to change the order of summation, which a workspace is.
struct AnySplitPlan { int splits; int64_t kc, ldp, bytes; bool inside; double us; };      // us: estimated, where splits > 1
constexpr int64_t INSIDE_BYTES = 256;
// microseconds of a K-step on a 64 x 64 tile: of a workgroup alone on its CU, of each of several (measured, see the planners)
struct KStepUs { double alone, shared; };
static KStepUs k_step_us(int dtype) {
    switch (int_planes_of(dtype)) {
    case 2: return {0.35, 0.17};
    case 4: return {0.48, 0.35};
    case 8: return {1.4, 1.3};
    default: return dtype == ntg::DT_F32 ? KStepUs{0.71, 0.45} : ntg::elem_size(dtype) == 2 ? KStepUs{0.28, 0.18} : KStepUs{0.43, 0.25};
    }
}
// ... with all k ranges of a float's tile in one workgroup
static double inside_us(int64_t es, int64_t tiles, int64_t steps) {
    const double rounds = (double)tiles / 256.0;
    return es == 2 ? 5.5 + (double)steps * std::max(0.33, 0.3 * rounds) : 2.5 + (double)steps * std::max(0.71, 0.3 + 0.62 * rounds);
}
// A workgroup alone on its CU spends 0.35 / 0.48 / 1.4 us (16 / 32 / 64 bits) on each K-step of 32, several 0.17 / 0.35 / 1.3 us each (Int32 200 x 3000 x 200
// whole 48 us, 8 / 16 ranges 12.4 / 10.8; Int16 709 x 3136 x 450, ranges 1 / 4 / 8 / 16: 36 / 16.9 / 15.8 / 19.4; Int64 576 x 3968 x 281, 1 / 4 / 8: 183 / 53 / 58).
// The sums wrap, so their order is nobody's concern: the batch counts among the tiles.  room: bytes of workspace there are.
AnySplitPlan plan_int_split(const ntg::GemmParams& p, int dtype, bool ta, bool tb, int64_t room) {
    AnySplitPlan pl{1, p.K, (p.N + 3) / 4 * 4, 0, false, 0.0};
    if (p.batch < 1 || p.batch > 65535 || p.Aptr || p.Bptr || p.Cptr || !int_pipe_eligible(p, dtype, ta, tb)) return pl;
    const int P = int_planes_of(dtype);
    const int64_t steps = (p.K + 31) / 32, tiles = ((p.M + 63) / 64) * ((p.N + 63) / 64) * (int64_t)p.batch;
    if (tiles > 255) return pl;
    const int64_t per_range = (int64_t)p.batch * p.M * pl.ldp * P;
    const double alone = k_step_us(dtype).alone, shared = k_step_us(dtype).shared;
    double best_us = 0.95 * (double)steps * alone;
    // (The second launch and its workspace take a host about 5 us, 8.3 -> 13.5 us a call through the Python face: what the GPU does meanwhile stays whole.
    //  64 x k x 64 through that face, whole / ranges: Int32 k = 384 9.0 / 13.9 us, 1000 17.7 / 13.6, 4096 59 / 13.6; Int16 k = 1000 10.3 / 13.5, 2048 17.0 / 13.7.)
    if (best_us < 13.0) return pl;
    for (int64_t sp = 2; sp <= 32 && sp <= steps / 2 && sp * per_range <= room; ++sp) {
        const int64_t per = (steps + sp - 1) / sp, ranges = (steps + per - 1) / per, wgs = tiles * ranges;
        const double us = (double)per * (wgs <= 256 ? alone : shared * (double)((wgs + 255) / 256)) + 4.0 + 2.0 * (double)ranges * (double)per_range / 4.0e6;
        if (us < best_us) { best_us = us; pl.splits = (int)ranges; pl.kc = per * 32; pl.bytes = ranges * per_range; pl.us = us; }
    }
    return pl;
}
AnySplitPlan plan_any_split(const ntg::GemmParams& p, int dtype, bool ta, bool tb) {
    AnySplitPlan none{1, p.K, 0, 0, false, 0.0};
    const bool byte = dtype == ntg::DT_I8 || dtype == ntg::DT_U8;
    if (p.batch < 1 || (byte && p.batch > 65535) || p.Aptr || p.Bptr || p.Cptr || p.keep_k_order || !ntg::any_eligible(p, dtype, ta, tb)) return none;
    if (p.M <= 32 && !byte) return none;                           // the streaming kernels take these
    const int64_t es = ntg::elem_size(dtype), ve = 16 / es, bk = 128 / es;
    if (p.K % ve == 0 && p.N % ve == 0 && (!ta || p.M % ve == 0) && p.lda % ve == 0 && p.ldb % ve == 0 && p.ldc % ve == 0) return none;
    // (the ranges of a float are one item's: an item comes out bit for bit the same alone and in a batch.  Bytes wrap: the batch counts among the tiles)
    const int64_t items = byte ? p.batch : 1;
    const int64_t tiles = ((p.M + 63) / 64) * ((p.N + 63) / 64) * items, steps = (p.K + bk - 1) / bk;
    if (tiles > 255) return none;
    // A workgroup alone on its CU spends 0.28 / 0.71 / 0.43 us (16-bit / Float32 / Int8) on each K-step, several on one CU 0.18 / 0.45 / 0.25 us
    // each; a launch costs about 2.5 us, the second pass 4 us + the partial sums written and read at 4 TB/s.  Of 2 .. 32 ranges the choice was the
    // best measured one or within 10 % of it on fourteen shapes (BFloat16 576 x 3797 x 448, ranges 1 / 2 / 4 / 8: 19.6 / 16.5 / 13.0 / 14.5 us;
    // 448 x 3704 x 166: 25.9 us whole, 10.4 in eight ranges; Float32 128 x 6463 x 720: 146 us whole, 24 in 21 ranges).
    const double alone = k_step_us(dtype).alone, shared = k_step_us(dtype).shared;
    auto estimate_us = [&](int64_t tls, int64_t its, int64_t sp, int64_t per) {
        const int64_t wgs = tls * sp;
        const double second_pass = sp == 1 ? 0.0 : 4.0 + 8.0 * (double)sp * (double)its * (double)p.M * (double)p.N / 4.0e6;
        return 2.5 + (double)per * (wgs <= 256 ? alone : shared * (double)((wgs + 255) / 256)) + second_pass;
    };
    const double whole_us = estimate_us(tiles, items, 1, steps);
    double best_us = 0.95 * whole_us;
    AnySplitPlan pl = none;
    for (int64_t sp = 2; sp <= 32 && sp <= steps / 2; ++sp) {
        const int64_t per = (steps + sp - 1) / sp, ranges = (steps + per - 1) / per;
        const double us = estimate_us(tiles, items, ranges, per);
        if (ranges * items * (int64_t)p.M * ((p.N + 3) / 4 * 4) * 4 > (int64_t)NTG_NOALLOC_SCRATCH_BYTES) break;      // (fits where nothing is allocated)
        if (us < best_us) { best_us = us; pl.splits = (int)ranges; pl.kc = per * bk; pl.us = us; }
    }
    if (pl.splits < 2) return none;
    pl.ldp = (p.N + 3) / 4 * 4;
    pl.bytes = (int64_t)pl.splits * p.batch * p.M * pl.ldp * 4;
    if (!byte && p.batch > 1) {
        // A batch: the items' ranges through memory, or inside a workgroup once the batch gives the CUs enough tiles (and where the sums would take more than
        // 64 MiB).  Measured in 2 .. 64 items of six shapes, the choice is the better one or within 10 % of it: Float16 128 x 6463 x 721 through memory / inside,
        // 6 items 30.7 / 37.0 us, 10 items 44.3 / 38.6, 32 items 148 / 113; Float32 200 x 1501 x 201, 6 items 25.9 / 36.7, 16 items 48.7 / 37.3, 64 items 175 /
        // 114; Float16 1000 x (70 x 2049 x 66) 237 / 135, Float32 64 x (128 x 6463 x 720) 892 / 740.  A K-step inside takes at least 0.33 / 0.71 us (16-bit / Float32).
        const int64_t all = tiles * p.batch;
        pl.inside = p.batch > 65535 || pl.bytes > (int64_t)NTG_NOALLOC_SCRATCH_BYTES || inside_us(es, all, steps) <= estimate_us(all, p.batch, pl.splits, pl.kc / bk);
        if (pl.inside) pl.bytes = INSIDE_BYTES;
    }
    return pl;
}

// the k ranges of a float's item inside one workgroup a tile: no workspace
static int run_ranges_inside(ntg::GemmParams p, const AnySplitPlan& ap, int dtype, bool ta, bool tb, hipStream_t s) {
    p.fold_steps = (int)(ap.kc * ntg::elem_size(dtype) / 128);
    const hipError_t e = ntg::launch_gemm_any(dtype, ta, tb, p, s);
    return e == hipSuccess ? NTG_OK : hip_fail(e, "gemm launch");
}

// A list of p.batch products behind pointer tables whose items are to have the bits that they have alone with their workspace (NTG_GEMM_PTRS_ITEM_ORDER).
// 0: one launch over the tables does that; else the workspace of one item, the list goes out item by item.  Integers have the same bits in any order; k ranges
// of odd rows run inside a workgroup; a split of 16-byte rows, and padded copies, are for single products only.  Where both ways are open the list's length
// decides: an item takes its own time and two launches, 9 us at least.  Item by item / one launch: BFloat16 448 x 3704 x 166 A^T.B, 2 items 22 / 21 us, 16 items 178 /
// 33, 64 items 774 / 80; Int32 200 x 3001 x 200, 2 items 23 / 50, 8 items 94 / 53; Int64 64 x 4096 x 64, 8 items 119 / 134, 16 items 237 / 134.
static int64_t table_item_bytes(const ntg::GemmParams& p, int dtype, bool ta, bool tb) {
    ntg::GemmParams one = p;
    one.batch = 1;
    const bool wide = int_planes_of(dtype) != 0;
    const AnySplitPlan ap = wide ? plan_int_split(one, dtype, ta, tb, NTG_NOALLOC_SCRATCH_BYTES) : plan_any_split(one, dtype, ta, tb);
    if (ap.splits > 1) {
        const int64_t bk = wide ? 32 : 128 / ntg::elem_size(dtype), steps = (p.K + bk - 1) / bk, tiles = (int64_t)((p.M + 63) / 64) * ((p.N + 63) / 64) * p.batch;
        const KStepUs c = k_step_us(dtype);
        const double table_us = is_int_dtype(dtype) ? 2.5 + (double)steps * (tiles <= 256 ? c.alone : c.shared * (double)((tiles + 255) / 256))
                                                    : inside_us(ntg::elem_size(dtype), tiles, steps);
        return table_us <= (double)p.batch * std::max(9.0, ap.us + 4.0) ? 0 : ap.bytes;
    }
    const PadPlan pp = plan_pad(one, dtype, ta, tb);
    return pp.ok && pp.pays ? pp.bytes() : plan_splitk(one, dtype, ta).bytes;
}

int run_gemm(ntg::GemmParams p, int dtype, bool ta, bool tb, hipStream_t s, void* workspace = nullptr, int64_t workspace_bytes = 0) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported by the gfx950 matmult backend", dtype);
    if (p.M == 0 || p.N == 0 || p.batch == 0) return NTG_OK;
    if (p.K == 0) {
        // empty sum: C keeps what it holds, or becomes the bias / zero.  The product kernels assume at least one k.
        if (p.cmode == ntg::C_ACCUMULATE && p.act == ntg::ACT_NONE) return NTG_OK;      // (with relu: C = relu_(C), below)
        if (p.Cptr) return fail(NTG_ERR_INVALID_ARGUMENT, "k = 0 with a C mode other than accumulate needs strided operands");
        hipError_t e = hipSuccess;
        if (is_int_dtype(dtype)) {
            e = ntg::launch_gemm_valu(dtype, ta, tb, p, s);                 // its k loop runs zero times
        } else if (is_complex_dtype(dtype)) {
            e = ntg::launch_gemm_complex(dtype, ta, tb, p, s);              // likewise
        } else {
            for (int b = 0; b < p.batch && e == hipSuccess; ++b) {
                ntg::GemmParams q = p;
                q.batch = 1;
                q.C = static_cast<char*>(p.C) + (int64_t)b * p.sC * es;
                if (p.bias) q.bias = static_cast<const char*>(p.bias) + (int64_t)b * p.bias_bs * es;
                e = ntg::launch_splitk_reduce(dtype, nullptr, 0, q, q.N, s);     // C0 plus no partial sums
            }
        }
        if (e != hipSuccess) return hip_fail(e, "empty-k launch");
        return NTG_OK;
    }
    {
        const AnySplitPlan ap = int_planes_of(dtype) ? plan_int_split(p, dtype, ta, tb, workspace ? workspace_bytes : 0) : plan_any_split(p, dtype, ta, tb);
        const bool offered = ap.splits > 1 && workspace && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0;
        if (offered && workspace_bytes >= INSIDE_BYTES && (ap.inside || workspace_bytes < ap.bytes) && !is_int_dtype(dtype))
            return run_ranges_inside(p, ap, dtype, ta, tb, s);
        if (offered && !ap.inside && workspace_bytes >= ap.bytes) {
            // launch index = range * batch + item
            ntg::GemmParams q = p;
            q.K = (int)ap.kc;
            q.k_total = p.K;
            q.C = workspace;
            q.ldc = ap.ldp;
            q.sC = (int64_t)p.M * ap.ldp;
            q.cmode = int_planes_of(dtype) ? ntg::C_OVERWRITE : ntg::C_PARTIAL;      // (sums in the element type: wrapping)
            q.bias = nullptr;
            q.act = ntg::ACT_NONE;
            q.batch = ap.splits * p.batch;
            q.krange_items = p.batch;
            q.sAk = ta ? ap.kc * p.lda : ap.kc;
            q.sBk = tb ? ap.kc : ap.kc * p.ldb;
            hipError_t e = int_planes_of(dtype) ? ntg::launch_gemm_int(int_planes_of(dtype), ta, tb, q, s) : ntg::launch_gemm_any(dtype, ta, tb, q, s);
            if (e != hipSuccess) return hip_fail(e, "gemm launch");
            e = ntg::launch_splitk_reduce(dtype, workspace, ap.splits, p, ap.ldp, s);
            if (e != hipSuccess) return hip_fail(e, "split-K reduction launch");
            return NTG_OK;
        }
    }
    {
        const PadPlan pp = plan_pad(p, dtype, ta, tb);
        if (pp.ok && pp.pays && workspace && workspace_bytes >= pp.bytes() && (reinterpret_cast<uintptr_t>(workspace) & 255) == 0)
            return run_padded(p, pp, dtype, ta, tb, workspace, s);
    }
    const SplitPlan plan = plan_splitk(p, dtype, ta);
    if (plan.splits > 1 && workspace && workspace_bytes >= plan.bytes && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0) {
        ntg::GemmParams q = p;
        q.K = (int)plan.kc;
        q.ldc = p.N;
        q.sC = (int64_t)p.M * p.N;
        q.cmode = (dtype == ntg::DT_F16 || dtype == ntg::DT_BF16) ? ntg::C_PARTIAL : ntg::C_OVERWRITE;
        q.bias = nullptr;
        q.act = ntg::ACT_NONE;                     // (the reduction applies it, after the last k range)
        const int64_t step_a = (ta ? plan.kc * p.lda : plan.kc), step_b = (tb ? plan.kc : plan.kc * p.ldb);   // elements from one k range to the next
        q.C = workspace;
        q.batch = plan.splits * p.batch;
        if (p.batch == 1) {
            // the k ranges are the items of one batched launch
            q.sA = step_a;
            q.sB = step_b;
        } else {
            // ... range r of item i is launch index r * batch + i
            q.krange_items = p.batch;
            q.sAk = step_a;
            q.sBk = step_b;
        }
        {
            int rc = launch_gemm(q, dtype, ta, tb, s);
            if (rc) return rc;
        }
        hipError_t e = ntg::launch_splitk_reduce(dtype, workspace, plan.splits, p, p.N, s);
        if (e != hipSuccess) return hip_fail(e, "split-K reduction launch");
        return NTG_OK;
    }
    return launch_gemm(p, dtype, ta, tb, s);
}

int check_sizes(int64_t m, int64_t k, int64_t n, int64_t batches) {
    if (m < 0 || k < 0 || n < 0 || batches < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "negative size (m=%lld k=%lld n=%lld batches=%lld)", (long long)m, (long long)k, (long long)n, (long long)batches);
    if (m > 0x7fffffffLL || k > 0x7fffffffLL || n > 0x7fffffffLL || batches > 0x7fffffffLL)
        return fail(NTG_ERR_INVALID_ARGUMENT, "a size exceeds 2^31-1");
    return NTG_OK;
}

int desc_to_params(const ntg_gemm_desc* d, ntg::GemmParams& p) {
    if (!d) return fail(NTG_ERR_INVALID_ARGUMENT, "null descriptor");
    if (ntg::elem_size(d->dtype) == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", d->dtype);
    int rc = check_sizes(d->m, d->k, d->n, d->batches);
    if (rc) return rc;
    if (d->c_mode < 0 || d->c_mode > 2) return fail(NTG_ERR_INVALID_ARGUMENT, "c_mode %d is not one of overwrite/accumulate/bias", d->c_mode);
    std::memset(&p, 0, sizeof p);
    p.M = (int)d->m; p.K = (int)d->k; p.N = (int)d->n; p.batch = (int)d->batches;
    p.lda = d->lda ? d->lda : (d->transpose_a ? d->m : d->k);
    p.ldb = d->ldb ? d->ldb : (d->transpose_b ? d->k : d->n);
    p.ldc = d->ldc ? d->ldc : d->n;
    if (p.lda < (d->transpose_a ? d->m : d->k) || p.ldb < (d->transpose_b ? d->k : d->n) || p.ldc < d->n)
        return fail(NTG_ERR_INVALID_ARGUMENT, "leading dimension smaller than the stored row length");
    p.sA = d->stride_a; p.sB = d->stride_b; p.sC = d->stride_c;
    p.cmode = d->c_mode;
    p.bias = d->bias;
    p.bias_bs = d->bias_batch_stride; p.bias_rs = d->bias_row_stride; p.bias_cs = d->bias_col_stride;
    if (p.cmode == NTG_C_BIAS && !p.bias) return fail(NTG_ERR_INVALID_ARGUMENT, "c_mode is bias but bias is null");
    p.keep_k_order = (d->flags & NTG_GEMM_KEEP_K_ORDER) != 0;
    return NTG_OK;
}

// The groups of a convolution are items of its one launch: item image * groups + group has its operands at group * (its own stride) +
// image * (the images' stride), its result at a uniform stride (rows of the groups follow each other in every layout used here).  A launch
// a group is `groups` times the 4-5 us that a launch costs the host and as many half-empty rounds: training steps in groups, us before | now:
// BFloat16 1 x 96 x 48 x 48 -> 16 by 3 x 3 in 4 groups 118 | 51, Float32 6 x 256 x 32 x 32 -> 96 by 5 x 5 at stride 2 in 4 groups 239 | 99,
// Float16 10 x 64 x 216 x 216 -> 192 by 3 x 3 in 4 groups 854 | 814.
struct GroupStrides { int64_t a_group, a_image, b_group, b_image, c_item; };      // elements
template <class Launch>
static hipError_t launch_groups(ntg::GemmParams p, int dtype, int64_t batch, int64_t groups, const GroupStrides& st, Launch&& launch) {
    const int64_t es = ntg::elem_size(dtype);
    // (a grid's 2^31 workgroups hold 32 x 32 tiles of any result that fits the memory, unless the groups are tiny and there are 2^31 of them)
    if ((double)((p.M + 31) / 32) * ((p.N + 31) / 32) * (double)batch * (double)groups < 2147483647.0) {
        p.batch = (int)(batch * groups);
        p.sC = st.c_item;
        p.sA = groups > 1 ? st.a_group : st.a_image;
        p.sB = groups > 1 ? st.b_group : st.b_image;
        if (groups > 1) { p.krange_items = (int)groups; p.sAk = st.a_image; p.sBk = st.b_image; }
        return launch(p);
    }
    for (int64_t g = 0; g < groups; ++g) {
        ntg::GemmParams q = p;
        q.batch = (int)batch;
        q.A = static_cast<const char*>(p.A) + g * st.a_group * es;
        q.B = static_cast<const char*>(p.B) + g * st.b_group * es;
        q.C = static_cast<char*>(p.C) + g * st.c_item * (p.cmode == ntg::C_PARTIAL ? 4 : es);
        q.sA = st.a_image; q.sB = st.b_image; q.sC = groups * st.c_item;
        const hipError_t e = launch(q);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace

// Device address of `scratch` on the current device (each GPU holds its own copy at its own address), looked up on the
// first call per device.  The function has external linkage on purpose: the compiler gives a file-scope static device
// variable a symbol the runtime can look up only when a host function with external linkage refers to it.
namespace ntg {
// One per GPU: the address of its copy of `scratch`, and what orders the users of that copy.  Calls that use the array are
// enqueued one at a time (the mutex spans a call's whole sequence of launches); a call on another stream than the previous
// user's first makes its stream wait for the event recorded behind that user's last kernel.  Streams under capture take no
// part in this (an event recorded inside a capture cannot be waited for from outside): their callers order such calls themselves.
struct NoallocState {
    std::mutex mutex;
    void* ptr = nullptr;
    hipEvent_t done = nullptr;
    hipStream_t last_stream = nullptr;
    bool used = false;
};
int noalloc_state_of_current_device(NoallocState** out) {
    constexpr int kMaxDevices = 64;
    static std::mutex setup_mutex;
    static NoallocState states[kMaxDevices];
    int dev = -1;
    HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(NTG_ERR_DEVICE, "device ordinal %d outside 0..%d", dev, kMaxDevices - 1);
    NoallocState& st = states[dev];
    std::lock_guard<std::mutex> lock(setup_mutex);
    if (!st.ptr) {
        void* ptr = nullptr;
        HIP_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        if (!ptr) return fail(NTG_ERR_DEVICE, "hipGetSymbolAddress returned a null address for the static scratch");
        HIP_TRY(hipEventCreateWithFlags(&st.done, hipEventDisableTiming));
        st.ptr = ptr;
    }
    *out = &st;
    return NTG_OK;
}
}  // namespace ntg

extern "C" {

const char* ntg_last_error(void) { return g_last_error.c_str(); }
int ntg_version(void) { return 100; }
int64_t ntg_dtype_size(int dtype) { return ntg::elem_size(dtype); }

int ntg_release_host_buffers(void) {
    ntg::HostSession::release_all();
    return NTG_OK;
}

int ntg_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

int ntg_gemm_dev(const ntg_gemm_desc* d, const void* dA, const void* dB, void* dC, void* stream) {
    ntg::GemmParams p;
    int rc = desc_to_params(d, p);
    if (rc) return rc;
    if (p.M == 0 || p.N == 0 || p.batch == 0) return NTG_OK;
    if (!dA || !dB || !dC) return fail(NTG_ERR_INVALID_ARGUMENT, "null matrix pointer");
    if (p.batch > 1 && p.sC == 0) return fail(NTG_ERR_INVALID_ARGUMENT, "stride_c must be non-zero for a batch (outputs may not alias)");
    p.A = dA; p.B = dB; p.C = dC;
    return run_gemm(p, d->dtype, d->transpose_a != 0, d->transpose_b != 0, static_cast<hipStream_t>(stream), d->workspace, d->workspace_bytes);
}

int ntg_gemm_relu_dev(const ntg_gemm_desc* d, const void* dA, const void* dB, void* dC, void* stream) {
    ntg::GemmParams p;
    int rc = desc_to_params(d, p);
    if (rc) return rc;
    if (!(d->dtype == ntg::DT_F32 || d->dtype == ntg::DT_F64 || d->dtype == ntg::DT_F16 || d->dtype == ntg::DT_BF16))
        return fail(NTG_ERR_UNSUPPORTED_DTYPE, "ntg_gemm_relu_dev takes Float16, BFloat16, Float32 and Float64 (dtype %d)", d->dtype);
    if (p.M == 0 || p.N == 0 || p.batch == 0) return NTG_OK;
    if (!dC || (p.K > 0 && (!dA || !dB))) return fail(NTG_ERR_INVALID_ARGUMENT, "null matrix pointer");      // (k = 0: C = relu_(C0), no operands)
    if (p.batch > 1 && p.sC == 0) return fail(NTG_ERR_INVALID_ARGUMENT, "stride_c must be non-zero for a batch (outputs may not alias)");
    p.A = dA; p.B = dB; p.C = dC;
    p.act = ntg::ACT_RELU;
    return run_gemm(p, d->dtype, d->transpose_a != 0, d->transpose_b != 0, static_cast<hipStream_t>(stream), d->workspace, d->workspace_bytes);
}

int64_t ntg_gemm_workspace_bytes(const ntg_gemm_desc* d) {
    ntg::GemmParams p;
    if (desc_to_params(d, p)) return -1;
    if (p.M == 0 || p.N == 0 || p.batch == 0) return 0;
    if (d->flags & NTG_GEMM_PTRS_ITEM_ORDER) return table_item_bytes(p, d->dtype, d->transpose_a != 0, d->transpose_b != 0);
    if (int_planes_of(d->dtype)) return plan_int_split(p, d->dtype, d->transpose_a != 0, d->transpose_b != 0, NTG_NOALLOC_SCRATCH_BYTES).bytes;
    {
        const AnySplitPlan ap = plan_any_split(p, d->dtype, d->transpose_a != 0, d->transpose_b != 0);
        if (ap.splits > 1) return ap.bytes;                        // (no padded copies beside k ranges)
        const PadPlan pp = plan_pad(p, d->dtype, d->transpose_a != 0, d->transpose_b != 0);      // pointers taken as 16-byte aligned
        if (pp.ok && pp.pays) return pp.bytes();
    }
    return plan_splitk(p, d->dtype, d->transpose_a != 0).bytes;      // pointers taken as 16-byte aligned
}

int ntg_gemm_noalloc_dev(const ntg_gemm_desc* d, const void* dA, const void* dB, void* dC, void* stream) {
    ntg::GemmParams p;
    int rc = desc_to_params(d, p);
    if (rc) return rc;
    if (p.M == 0 || p.N == 0 || p.batch == 0) return NTG_OK;
    if (!dA || !dB || !dC) return fail(NTG_ERR_INVALID_ARGUMENT, "null matrix pointer");
    if (p.batch > 1 && p.sC == 0) return fail(NTG_ERR_INVALID_ARGUMENT, "stride_c must be non-zero for a batch (outputs may not alias)");
    const int64_t need = ntg_gemm_workspace_bytes(d);
    if (need < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "bad descriptor");
    if (need > (int64_t)NTG_NOALLOC_SCRATCH_BYTES)
        return fail(NTG_ERR_INVALID_ARGUMENT, "this product's workspace form needs %lld bytes, the static scratch of ntg_gemm_noalloc_dev holds %lld: "
                    "call ntg_gemm_dev with a workspace of the caller's, or ntg_gemm_dev without a workspace (the plain kernels: they allocate "
                    "nothing either, but a split along k is then not taken and floating-point sums may differ in their last bits)",
                    (long long)need, (long long)NTG_NOALLOC_SCRATCH_BYTES);
    p.A = dA; p.B = dB; p.C = dC;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool ta = d->transpose_a != 0, tb = d->transpose_b != 0;
    if (need == 0) return run_gemm(p, d->dtype, ta, tb, s);      // the plain kernels: the array is not used
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &capture) != hipSuccess) {      // (e.g. the default stream while another stream captures)
        (void)hipGetLastError();
        capture = hipStreamCaptureStatusActive;
    }
    const bool ordered = capture == hipStreamCaptureStatusNone;
    // k ranges of rows that start anywhere, and of integers, have forms of the same bits that keep nothing in memory.  They are taken under capture, where
    // nothing orders the users of the array (an odd row must not decide whether a graph may run beside them), and where they are the faster ones anyway.
    const AnySplitPlan ap = plan_any_split(p, d->dtype, ta, tb);
    if (ap.splits > 1 && !is_int_dtype(d->dtype) && (ap.inside || !ordered)) return run_ranges_inside(p, ap, d->dtype, ta, tb, s);
    if (!ordered && (int_planes_of(d->dtype) || ap.splits > 1)) return run_gemm(p, d->dtype, ta, tb, s);
    ntg::NoallocState* st = nullptr;
    rc = ntg::noalloc_state_of_current_device(&st);
    if (rc) return rc;
    std::lock_guard<std::mutex> lock(st->mutex);
    if (ordered && st->used && st->last_stream != s) HIP_TRY(hipStreamWaitEvent(s, st->done, 0));     // the previous user of the array finishes first
    rc = run_gemm(p, d->dtype, ta, tb, s, st->ptr, need);
    if (ordered) {
        HIP_TRY(hipEventRecord(st->done, s));
        st->last_stream = s;
        st->used = true;
    }
    return rc;
}

// Address of the current device's copy of gate_flags (looked up once per device) and the next slot of it.
static int next_gate_slot(int** out) {
    constexpr int kMaxDevices = 64;
    static std::mutex mutex;
    static int* base[kMaxDevices];
    static unsigned next[kMaxDevices];
    int dev = -1;
    HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(NTG_ERR_DEVICE, "device ordinal %d outside 0..%d", dev, kMaxDevices - 1);
    std::lock_guard<std::mutex> lock(mutex);
    if (!base[dev]) {
        void* ptr = nullptr;
        HIP_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(gate_flags)));
        if (!ptr) return fail(NTG_ERR_DEVICE, "hipGetSymbolAddress returned a null address for the gate flags");
        base[dev] = static_cast<int*>(ptr);
    }
    *out = base[dev] + (next[dev]++ % NTG_GATE_SLOTS);
    return NTG_OK;
}

// Pointer tables without the caller's vouch: the entries' alignment is a fact of device memory, so it is found out there.  A
// one-workgroup kernel ORs the low bits of all entries into a flag; then the product is launched twice, on the DMA-fed
// kernel (which needs 16-byte entries) and on the one that takes rows as they lie (Float64: register-staged), each returning at
// once unless the flag names it.  The two kernels give the same bits, so nothing depends on which one runs.  Worth two extra
// launches (about 4 us) only where the DMA-fed kernel gains more; the types that have both kernels, more than 32 rows.
static bool gated_tables_pay(const ntg::GemmParams& p, int dtype) {
    const bool byte = dtype == ntg::DT_I8 || dtype == ntg::DT_U8;
    if (dtype != ntg::DT_F32 && dtype != ntg::DT_F64 && dtype != ntg::DT_F16 && dtype != ntg::DT_BF16 && !byte) return false;
    if (p.M <= 32 || p.K <= 0 || p.act != ntg::ACT_NONE) return false;
    const double flops = 2.0 * (double)p.M * (double)p.N * (double)p.K * (double)p.batch;
    // Checked / rows as they lie, aligned tables: Int8 8 x 512^3 12.3 us / 7.2, 128 x (256 x 2048 x 256) 36 / 27, 24 x 1024^3 42 / 41, 32 x 1024^3 49 / 53, 4 x 2048^3
    // 40 / 48; BFloat16 64 x (256 x 1024 x 256) 23.0 / 18.1, 8 x (1024 x 512 x 1024) 17.2 / 17.6, 6 x 1024^3 23.2 / 25.1, 32 x 1024^3 73 / 91; Float32 64 x 256^3 28.1 /
    // 24.7, 16 x 512^3 42 / 41, 4 x 1024^3 71.5 / 75.2, 16 x 1024^3 244 / 279.  (Float64 still weighs against the register-staged kernel.)
    return flops >= (byte ? 6.0e10 : dtype == ntg::DT_F32 ? 6.0e9 : dtype == ntg::DT_F64 ? 3.2e10 : 1.2e10);
}
static int launch_gemm_tables_gated(ntg::GemmParams p, int dtype, bool ta, bool tb, hipStream_t s) {
    int* flag = nullptr;
    int rc = next_gate_slot(&flag);
    if (rc) return rc;
    hipLaunchKernelGGL(ntg::ptr_tables_aligned_kernel, dim3(1), dim3(256), 0, s, p.Aptr, p.Bptr, p.Cptr, p.batch, flag);
    HIP_TRY(hipGetLastError());
    const int64_t ve = 16 / ntg::elem_size(dtype);
    ntg::GemmParams q = p;
    q.vecA_ok = p.lda % ve == 0;
    q.vecB_ok = p.ldb % ve == 0;
    q.ptrs_aligned = 1; q.gate = flag; q.gate_want = 1;
    bool taken = false;
    hipError_t e = ntg::launch_gemm_ring_only(dtype, ta, tb, q, s, &taken);
    if (e != hipSuccess) return hip_fail(e, "gemm launch");
    p.ptrs_aligned = 0;
    if (taken) { p.gate = flag; p.gate_want = 0; }        // (not taken: sizes or pitches rule the DMA-fed kernel out anyway)
    return launch_gemm(p, dtype, ta, tb, s);
}

// aligned: the caller vouches that every table entry is a multiple of 16 bytes (true for the host entry points' own arena)
static int gemm_ptrs(const ntg_gemm_desc* d, const void* const* dA, const void* const* dB, void* const* dC, void* stream, bool aligned) {
    ntg::GemmParams p;
    int rc = desc_to_params(d, p);
    if (rc) return rc;
    if (p.M == 0 || p.N == 0 || p.batch == 0) return NTG_OK;
    if (!dA || !dB || !dC) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer table");
    AnySplitPlan item{1, p.K, 0, 0, false, 0.0};
    if ((d->flags & NTG_GEMM_PTRS_ITEM_ORDER) && !is_int_dtype(d->dtype)) {
        ntg::GemmParams one = p;
        one.batch = 1;
        item = plan_any_split(one, d->dtype, d->transpose_a != 0, d->transpose_b != 0);
        if (item.splits == 1 && plan_splitk(one, d->dtype, d->transpose_a != 0).splits > 1)
            return fail(NTG_ERR_INVALID_ARGUMENT, "no launch over pointer tables sums these items in the order that each has alone: run them one by one (ntg_gemm_workspace_bytes says so)");
    }
    p.Aptr = dA; p.Bptr = dB; p.Cptr = dC;
    p.ptrs_aligned = aligned ? 1 : 0;
    if (item.splits > 1) return run_ranges_inside(p, item, d->dtype, d->transpose_a != 0, d->transpose_b != 0, static_cast<hipStream_t>(stream));
    if (!aligned && gated_tables_pay(p, d->dtype))
        return launch_gemm_tables_gated(p, d->dtype, d->transpose_a != 0, d->transpose_b != 0, static_cast<hipStream_t>(stream));
    return run_gemm(p, d->dtype, d->transpose_a != 0, d->transpose_b != 0, static_cast<hipStream_t>(stream));
}

int ntg_gemm_ptrs_dev(const ntg_gemm_desc* d, const void* const* dA, const void* const* dB, void* const* dC, void* stream) {
    // (the tables are in device memory: their entries' alignment is what the caller says it is)
    return gemm_ptrs(d, dA, dB, dC, stream, d && (d->flags & NTG_GEMM_PTRS_ALIGNED16) != 0);
}

// The host-pointer entry points are the reference's own seam (nt_matmult / nt_matmult_batch / cpu::linear on host memory): there a
// Float32 product keeps the reference's order of summation -- no split along k, whose gain the transfers would hide anyway.
static int64_t host_entry_flags(int dtype) { return dtype == ntg::DT_F32 ? NTG_GEMM_KEEP_K_ORDER : 0; }

int ntg_matmult_dev(int dtype, const void* dA, const void* dB, void* dC, int64_t m, int64_t k, int64_t n,
                    int transpose_a, int transpose_b, void* stream) {
    ntg_gemm_desc d;
    std::memset(&d, 0, sizeof d);
    d.dtype = dtype; d.transpose_a = transpose_a; d.transpose_b = transpose_b; d.c_mode = NTG_C_ACCUMULATE;
    d.m = m; d.k = k; d.n = n; d.batches = 1;
    return ntg_gemm_dev(&d, dA, dB, dC, stream);
}

int ntg_matmult(int dtype, const void* A, const void* B, void* C,
                int64_t a_rows, int64_t a_cols, int64_t b_rows, int64_t b_cols,
                int transpose_a, int transpose_b) {
    const void* As[1] = {A};
    const void* Bs[1] = {B};
    void* Cs[1] = {C};
    return ntg_matmult_batch(dtype, As, Bs, Cs, 1, a_rows, a_cols, b_rows, b_cols, transpose_a, transpose_b);
}

// The host-pointer seam, pipelined: large operands cross the link in panels so that uploads, products and downloads
// overlap (the link is full duplex and the kernel is short beside the transfers).
//   one product:  B first (and A whole when it is stored [k][m]), then panels of rows: A's rows and C's rows up, the
//                 panel's product on a second stream, its rows of C down on a third while the next panels go up;
//   a batch of distinct matrices (or one shared A or B): the same with groups of items as panels.
// A C that is all zeros in the caller's memory (what functional::matmult hands over: zeros, then accumulate,
// matmult_cpu.cpp:110, :707) is not uploaded; the products overwrite instead, which gives the same bits (the sums start
// from +0 either way).  Panels are products of their own, so this form is taken only where that cannot change a bit: no
// workspace form exists for the whole product (a split along k would depend on the panel's rows), more than 32 rows.
// Returns -1 when the call is not one for this form (nothing has been done then).
static int matmult_host_pipelined(int dtype, const void* const* A, const void* const* B, void* const* C, int64_t batches,
                                  int64_t m, int64_t k, int64_t n, int ta, int tb) {
    const int64_t es = ntg::elem_size(dtype);
    const size_t a_bytes = (size_t)(m * k * es), b_bytes = (size_t)(k * n * es), c_bytes = (size_t)(m * n * es);
    if ((a_bytes + b_bytes + c_bytes) * (size_t)batches < ((size_t)48 << 20)) return -1;
    ntg_gemm_desc d;
    std::memset(&d, 0, sizeof d);
    d.dtype = dtype; d.transpose_a = ta; d.transpose_b = tb;
    d.m = m; d.k = k; d.n = n; d.batches = 1;
    d.flags = host_entry_flags(dtype);
    const size_t a_slot = align_up(a_bytes, 256), b_slot = align_up(b_bytes, 256), c_slot = align_up(c_bytes, 256);
    std::vector<ntg::HostSession::Range> up;
    if (batches == 1) {
        if (m < 1024 || ntg_gemm_workspace_bytes(&d) != 0) return -1;
        // rows per panel: multiples of 256, about 16 MiB of A and C rows together, at least four panels
        int64_t rows = (int64_t)(((size_t)16 << 20) / (size_t)((k + n) * es)) / 256 * 256;
        rows = std::max<int64_t>(256, std::min<int64_t>(rows, (m / 4) / 256 * 256));
        // (the rows that are left over join the last panel: a panel of 32 rows or fewer would run on the streaming kernel,
        //  whose sums over k have another order)
        const int panels = (int)std::max<int64_t>(1, m / rows);
        auto panel_rows = [&](int p) { return p == panels - 1 ? m - (int64_t)p * rows : rows; };
        ntg::HostSession mem;
        HIP_TRY(mem.reserve(a_slot + b_slot + c_slot));

        const size_t oa = 0, ob = a_slot, oc = a_slot + b_slot;
        // B (and an A stored [k][m]: a panel of rows of op(A) is a column block of the stored matrix) go first; C is looked
        // at while the stagers are busy with them
        up.push_back({ob, B[0], b_bytes, 0});
        if (ta) up.push_back({oa, A[0], a_bytes, 0});
        HIP_TRY(mem.begin_uploads(up.data(), up.size(), 1));
        const bool zero = ntg::HostSession::all_zero(C[0], c_bytes);
        HIP_TRY(mem.end_uploads());
        up.clear();
        for (int p = 0; p < panels; ++p) {
            const int64_t m0 = p * rows, mr = panel_rows(p);
            if (!ta) up.push_back({oa + (size_t)(m0 * k * es), static_cast<const char*>(A[0]) + m0 * k * es, (size_t)(mr * k * es), p});
            if (!zero) up.push_back({oc + (size_t)(m0 * n * es), static_cast<const char*>(C[0]) + m0 * n * es, (size_t)(mr * n * es), p});
        }
        HIP_TRY(mem.begin_uploads(up.data(), up.size(), panels));
        d.lda = ta ? m : k;
        d.c_mode = zero ? NTG_C_OVERWRITE : NTG_C_ACCUMULATE;
        for (int p = 0; p < panels; ++p) {
            const int64_t m0 = p * rows, mr = panel_rows(p);
            const size_t c_off = (size_t)(m0 * n * es);
            HIP_TRY(mem.uploaded_through(p));
            d.m = mr;
            const int rc = ntg_gemm_dev(&d, mem.at(oa + (size_t)((ta ? m0 : m0 * k) * es)), mem.at(ob), mem.at(oc + c_off), mem.compute_stream());
            if (rc) return rc;
            HIP_TRY(mem.download_async(static_cast<char*>(C[0]) + c_off, oc + c_off, (size_t)(mr * n * es), mem.compute_stream()));
        }
        HIP_TRY(mem.end_uploads());
        HIP_TRY(mem.finish_downloads());
        return NTG_OK;
    }
    // a batch: distinct A, B, C per item, or one B (or one A) for all
    if (m <= 32) return -1;
    bool a_same = true, b_same = true;
    for (int64_t i = 1; i < batches; ++i) { a_same = a_same && A[i] == A[0]; b_same = b_same && B[i] == B[0]; }
    {
        std::map<const void*, int64_t> seen;
        for (int64_t i = 0; i < batches && !a_same; ++i)
            if (!seen.emplace(A[i], i).second) return -1;
        seen.clear();
        for (int64_t i = 0; i < batches && !b_same; ++i)
            if (!seen.emplace(B[i], i).second) return -1;
        seen.clear();
        for (int64_t i = 0; i < batches; ++i)
            if (!seen.emplace(C[i], i).second) return -1;          // (aliasing outputs: the general path reports it)
    }
    const size_t per_item = (a_same ? 0 : a_bytes) + (b_same ? 0 : b_bytes) + c_bytes;
    int64_t group = std::max<int64_t>(1, (int64_t)(((size_t)24 << 20) / per_item));
    group = std::min(group, std::max<int64_t>(1, batches / 4));
    const int panels = (int)((batches + group - 1) / group);
    d.batches = group;
    d.stride_a = a_same ? 0 : (int64_t)(a_slot / (size_t)es);
    d.stride_b = b_same ? 0 : (int64_t)(b_slot / (size_t)es);
    d.stride_c = (int64_t)(c_slot / (size_t)es);
    if (a_slot % (size_t)es || b_slot % (size_t)es || c_slot % (size_t)es) return -1;
    const int64_t ws_bytes = ntg_gemm_workspace_bytes(&d);          // (planned per item: the same form for any group size)
    if (ws_bytes < 0) return -1;
    const size_t na = a_same ? 1 : (size_t)batches, nb = b_same ? 1 : (size_t)batches;
    const size_t oa = 0, ob = na * a_slot, oc = ob + nb * b_slot, ow = oc + (size_t)batches * c_slot;
    ntg::HostSession mem;
    HIP_TRY(mem.reserve(ow + (size_t)ws_bytes));
    // the shared operand and the first group's A and B go first; the outputs are looked at while the stagers are busy with them
    if (a_same) up.push_back({oa, A[0], a_bytes, 0});
    if (b_same) up.push_back({ob, B[0], b_bytes, 0});
    for (int64_t i = 0; i < std::min(group, batches); ++i) {
        if (!a_same) up.push_back({oa + (size_t)i * a_slot, A[i], a_bytes, 0});
        if (!b_same) up.push_back({ob + (size_t)i * b_slot, B[i], b_bytes, 0});
    }
    HIP_TRY(mem.begin_uploads(up.data(), up.size(), 1));
    bool zero = true;
    for (int64_t i = 0; i < batches && zero; ++i) zero = ntg::HostSession::all_zero(C[i], c_bytes);
    HIP_TRY(mem.end_uploads());
    up.clear();
    for (int64_t i = 0; i < batches; ++i) {
        const int p = (int)(i / group);
        if (!a_same && p > 0) up.push_back({oa + (size_t)i * a_slot, A[i], a_bytes, p});
        if (!b_same && p > 0) up.push_back({ob + (size_t)i * b_slot, B[i], b_bytes, p});
        if (!zero) up.push_back({oc + (size_t)i * c_slot, C[i], c_bytes, p});
    }
    HIP_TRY(mem.begin_uploads(up.data(), up.size(), panels));
    if (ws_bytes > 0) { d.workspace = mem.at(ow); d.workspace_bytes = ws_bytes; }
    d.c_mode = zero ? NTG_C_OVERWRITE : NTG_C_ACCUMULATE;
    for (int p = 0; p < panels; ++p) {
        const int64_t i0 = p * group, cnt = std::min(group, batches - i0);
        HIP_TRY(mem.uploaded_through(p));
        d.batches = cnt;
        const int rc = ntg_gemm_dev(&d, mem.at(oa + (a_same ? 0 : (size_t)i0 * a_slot)), mem.at(ob + (b_same ? 0 : (size_t)i0 * b_slot)),
                                    mem.at(oc + (size_t)i0 * c_slot), mem.compute_stream());
        if (rc) return rc;
        for (int64_t i = i0; i < i0 + cnt; ++i) HIP_TRY(mem.download_async(C[i], oc + (size_t)i * c_slot, c_bytes, mem.compute_stream()));
    }
    HIP_TRY(mem.end_uploads());
    HIP_TRY(mem.finish_downloads());
    return NTG_OK;
}

int ntg_matmult_batch(int dtype, const void* const* A, const void* const* B, void* const* C,
                      int64_t batches, int64_t a_rows, int64_t a_cols, int64_t b_rows, int64_t b_cols,
                      int transpose_a, int transpose_b) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported by the gfx950 matmult backend", dtype);
    if (a_cols != b_rows) return fail(NTG_ERR_INVALID_ARGUMENT, "inner sizes differ: a_cols=%lld b_rows=%lld", (long long)a_cols, (long long)b_rows);
    const int64_t m = a_rows, k = a_cols, n = b_cols;
    int rc = check_sizes(m, k, n, batches);
    if (rc) return rc;
    if (batches == 0 || m == 0 || n == 0 || k == 0) return NTG_OK;   // C += empty sum
    if (!A || !B || !C) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer array");
    for (int64_t i = 0; i < batches; ++i)
        if (!A[i] || !B[i] || !C[i]) return fail(NTG_ERR_INVALID_ARGUMENT, "null matrix pointer in item %lld", (long long)i);
    rc = matmult_host_pipelined(dtype, A, B, C, batches, m, k, n, transpose_a, transpose_b);
    if (rc >= 0) return rc;
    rc = NTG_OK;

    const size_t a_bytes = (size_t)(m * k * es), b_bytes = (size_t)(k * n * es), c_bytes = (size_t)(m * n * es);
    // every distinct input matrix gets one slot in a single device arena
    std::map<const void*, size_t> slotA, slotB;
    size_t off = 0;
    for (int64_t i = 0; i < batches; ++i)
        if (slotA.emplace(A[i], off).second) off += align_up(a_bytes, 256);
    for (int64_t i = 0; i < batches; ++i)
        if (slotB.emplace(B[i], off).second) off += align_up(b_bytes, 256);
    const size_t c_off = off;
    off += align_up(c_bytes, 256) * (size_t)batches;
    const size_t tab_off = off;
    off += align_up(3 * sizeof(void*) * (size_t)batches, 256);
    ntg_gemm_desc d;
    std::memset(&d, 0, sizeof d);
    d.dtype = dtype; d.transpose_a = transpose_a; d.transpose_b = transpose_b; d.c_mode = NTG_C_ACCUMULATE;
    d.m = m; d.k = k; d.n = n; d.batches = batches;
    d.flags = host_entry_flags(dtype);
    // The arena is this function's own: when every item's A (and B) is a new matrix, or all items share one, the slots
    // lie at a constant stride and the strided kernels (and their workspace forms) serve the batch; any other pattern of
    // repeated pointers goes through the pointer tables.
    auto constant_stride = [&](const std::map<const void*, size_t>& slot, const void* const* P, size_t bytes, int64_t& stride) {
        const size_t step = slot.size() == 1 ? 0 : align_up(bytes, 256);
        for (int64_t i = 0; i < batches; ++i)
            if (slot.at(P[i]) != slot.at(P[0]) + (size_t)i * step) return false;
        stride = (int64_t)(step / (size_t)es);
        return true;
    };
    const bool strided = constant_stride(slotA, A, a_bytes, d.stride_a) && constant_stride(slotB, B, b_bytes, d.stride_b);
    if (strided) d.stride_c = (int64_t)(align_up(c_bytes, 256) / (size_t)es);
    else d.stride_a = d.stride_b = 0;
    const size_t ws_off = off;
    int64_t ws_bytes = strided ? ntg_gemm_workspace_bytes(&d) : 0;
    // A pattern of repeated pointers runs as ONE table batch.  Where an item on its own would be given a workspace form whose order of
    // summation over k the tables do not have (a split), the items go out one by one in that form instead, so that an item comes out
    // bit for bit the same alone and in any batch (tests/src/matmult_test.cpp:108-189).
    bool per_item = false;
    if (!strided) {
        d.flags |= NTG_GEMM_PTRS_ITEM_ORDER;
        const int64_t wb = ntg_gemm_workspace_bytes(&d);
        if (wb > 0) { per_item = true; ws_bytes = wb; }
    }
    if (ws_bytes > 0) off += (size_t)ws_bytes;

    ntg::HostSession mem;
    HIP_TRY(mem.reserve(off));
    for (auto& kv : slotA) HIP_TRY(mem.upload(kv.second, kv.first, a_bytes));
    for (auto& kv : slotB) HIP_TRY(mem.upload(kv.second, kv.first, b_bytes));
    std::vector<void*> tab(3 * (size_t)batches);
    std::map<const void*, int64_t> seenC;
    for (int64_t i = 0; i < batches; ++i) {
        const auto ins = seenC.emplace(C[i], i);
        if (!ins.second) return fail(NTG_ERR_INVALID_ARGUMENT, "output pointers of items %lld and %lld alias", (long long)ins.first->second, (long long)i);
        const size_t dc_off = c_off + (size_t)i * align_up(c_bytes, 256);
        HIP_TRY(mem.upload(dc_off, C[i], c_bytes));   // accumulate contract: C is an input too
        tab[(size_t)i] = mem.at(slotA[A[i]]);
        tab[(size_t)(batches + i)] = mem.at(slotB[B[i]]);
        tab[(size_t)(2 * batches + i)] = mem.at(dc_off);
    }
    void** dtab = reinterpret_cast<void**>(mem.at(tab_off));
    if (ws_bytes > 0) { d.workspace = mem.at(ws_off); d.workspace_bytes = ws_bytes; }
    if (strided) {
        rc = ntg_gemm_dev(&d, tab[0], tab[(size_t)batches], tab[(size_t)(2 * batches)], mem.stream());
    } else if (per_item) {
        d.batches = 1;
        for (int64_t i = 0; i < batches && rc == NTG_OK; ++i)
            rc = ntg_gemm_dev(&d, tab[(size_t)i], tab[(size_t)(batches + i)], tab[(size_t)(2 * batches + i)], mem.stream());
    } else {
        HIP_TRY(mem.upload(tab_off, tab.data(), tab.size() * sizeof(void*)));
        rc = gemm_ptrs(&d, dtab, dtab + batches, dtab + 2 * batches, mem.stream(), true);     // (every slot of the arena is 256-byte aligned)
    }
    if (rc) return rc;
    for (int64_t i = 0; i < batches; ++i)
        HIP_TRY(mem.download(C[i], c_off + (size_t)i * align_up(c_bytes, 256), c_bytes));
    return NTG_OK;
}

int ntg_linear(int dtype, const void* X, const void* W, const void* bias, void* Y,
               int64_t m, int64_t k, int64_t n, int transpose_x, int transpose_w,
               int64_t bias_rows, int64_t bias_cols) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported by the gfx950 matmult backend", dtype);
    int rc = check_sizes(m, k, n, 1);
    if (rc) return rc;
    if ((bias_rows != 1 && bias_rows != m) || (bias_cols != 1 && bias_cols != n))
        return fail(NTG_ERR_INVALID_ARGUMENT, "bias shape [%lld, %lld] does not broadcast to [%lld, %lld]",
                    (long long)bias_rows, (long long)bias_cols, (long long)m, (long long)n);
    if (m == 0 || n == 0) return NTG_OK;
    if (!X || !W || !bias || !Y) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer");
    const size_t x_bytes = (size_t)(m * k * es), w_bytes = (size_t)(k * n * es), y_bytes = (size_t)(m * n * es);
    const size_t bias_bytes = (size_t)(bias_rows * bias_cols * es);
    ntg::HostSession mem;
    const size_t ox = 0, ow = align_up(x_bytes, 256), ob = ow + align_up(w_bytes, 256), oy = ob + align_up(bias_bytes, 256);
    HIP_TRY(mem.reserve(oy + y_bytes));
    if (x_bytes) HIP_TRY(mem.upload(ox, X, x_bytes));
    if (w_bytes) HIP_TRY(mem.upload(ow, W, w_bytes));
    HIP_TRY(mem.upload(ob, bias, bias_bytes));
    ntg_gemm_desc d;
    std::memset(&d, 0, sizeof d);
    d.dtype = dtype; d.transpose_a = transpose_x; d.transpose_b = transpose_w; d.c_mode = NTG_C_BIAS;
    d.m = m; d.k = k; d.n = n; d.batches = 1;
    d.flags = host_entry_flags(dtype);
    d.bias = mem.at(ob);
    d.bias_row_stride = (bias_rows == 1) ? 0 : bias_cols;
    d.bias_col_stride = (bias_cols == 1) ? 0 : 1;
    rc = ntg_gemm_dev(&d, mem.at(ox), mem.at(ow), mem.at(oy), mem.stream());
    if (rc) return rc;
    HIP_TRY(mem.download(Y, oy, y_bytes));
    return NTG_OK;
}

static int unfold_out(int64_t height, int64_t width, int64_t k_r, int64_t k_c, int64_t s_r, int64_t s_c,
                      int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c, int64_t& Ho, int64_t& Wo) {
    if (k_r < 1 || k_c < 1 || s_r < 1 || s_c < 1 || d_r < 1 || d_c < 1 || p_r < 0 || p_c < 0)
        return fail(NTG_ERR_INVALID_ARGUMENT, "kernel/stride/dilation must be >= 1 and padding >= 0");
    Ho = (height + 2 * p_r - d_r * (k_r - 1) - 1) / s_r + 1;
    Wo = (width + 2 * p_c - d_c * (k_c - 1) - 1) / s_c + 1;
    if (height + 2 * p_r - d_r * (k_r - 1) - 1 < 0 || width + 2 * p_c - d_c * (k_c - 1) - 1 < 0 || Ho <= 0 || Wo <= 0)
        return fail(NTG_ERR_INVALID_ARGUMENT, "the array of sliding blocks would be empty (Ho=%lld, Wo=%lld)", (long long)Ho, (long long)Wo);
    return NTG_OK;
}

int ntg_unfold2d_dev(int dtype, const void* image, void* col,
                     int64_t batch, int64_t channels, int64_t height, int64_t width,
                     int64_t k_r, int64_t k_c, int64_t s_r, int64_t s_c,
                     int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c, void* stream) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    if (batch < 0 || channels < 0 || height < 0 || width < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "negative size");
    int64_t Ho, Wo;
    int rc = unfold_out(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo);
    if (rc) return rc;
    if (batch == 0 || channels == 0) return NTG_OK;
    if (!image || !col) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer");
    hipError_t e = ntg::launch_unfold2d(es, image, col, batch, channels, height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c,
                                        static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return hip_fail(e, "unfold2d launch");
    return NTG_OK;
}

int ntg_unfold2d(int dtype, const void* image, void* col,
                 int64_t batch, int64_t channels, int64_t height, int64_t width,
                 int64_t k_r, int64_t k_c, int64_t s_r, int64_t s_c,
                 int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    int64_t Ho, Wo;
    int rc = unfold_out(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo);
    if (rc) return rc;
    if (batch <= 0 || channels <= 0) return batch < 0 || channels < 0 ? fail(NTG_ERR_INVALID_ARGUMENT, "negative size") : NTG_OK;
    if (!image || !col) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer");
    const size_t im_bytes = (size_t)(batch * channels * height * width * es);
    const size_t col_bytes = (size_t)(batch * channels * k_r * k_c * Ho * Wo * es);
    ntg::HostSession mem;
    const size_t oc = align_up(im_bytes, 256);
    HIP_TRY(mem.reserve(oc + col_bytes));
    HIP_TRY(mem.upload(0, image, im_bytes));
    rc = ntg_unfold2d_dev(dtype, mem.at(0), mem.at(oc), batch, channels, height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, mem.stream());
    if (rc) return rc;
    HIP_TRY(mem.download(col, oc, col_bytes));
    return NTG_OK;
}

// Geometry of a convolution over two or three spatial axes; axis 0 is the depth (size 1, one tap for two axes).
struct Geo3 {
    int nd;
    int64_t sz[3], k[3], s[3], p[3], d[3], o[3];
    int64_t vol() const { return sz[0] * sz[1] * sz[2]; }
    int64_t taps() const { return k[0] * k[1] * k[2]; }
    int64_t L() const { return o[0] * o[1] * o[2]; }
};

static Geo3 geo2(int64_t height, int64_t width, int64_t k_r, int64_t k_c, int64_t s_r, int64_t s_c, int64_t p_r, int64_t p_c,
                 int64_t d_r, int64_t d_c, int64_t Ho, int64_t Wo) {
    return Geo3{2, {1, height, width}, {1, k_r, k_c}, {1, s_r, s_c}, {0, p_r, p_c}, {1, d_r, d_c}, {1, Ho, Wo}};
}

// The geometry of the convolution that maps the output gradient back to the image (all strides 1): its "image" is the
// gradient, its outputs are the image elements, its padding is d*(k-1) - p (negative = the image is cropped).
static Geo3 geo_dimage(const Geo3& g) {
    Geo3 t = g;
    for (int a = 0; a < 3; ++a) {
        t.sz[a] = g.o[a]; t.o[a] = g.sz[a]; t.s[a] = 1;
        t.p[a] = g.d[a] * (g.k[a] - 1) - g.p[a];
    }
    return t;
}

// The floating dtypes gather the im2col operand inside the GEMM (no col buffer) when every index the kernel forms fits
// 32 bits with room for its out-of-range sentinels and the kernel has at most 8 taps per axis (one byte of tap mask).
static bool conv_implicit_g(int dtype, int64_t channels, const Geo3& g) {
    if (is_valu_dtype(dtype)) return false;
    const int64_t lim = 1 << 24;
    for (int a = 0; a < 3; ++a) {
        if (g.k[a] > 8) return false;
        if (g.sz[a] >= lim || g.s[a] >= lim || g.p[a] >= lim || g.p[a] <= -lim) return false;
        if (g.k[a] * g.d[a] >= lim || g.o[a] * g.s[a] >= lim) return false;
    }
    if (channels >= lim || g.taps() >= lim) return false;
    // byte offsets inside one image are formed in 32 bits
    if (channels * g.vol() * ntg::elem_size(dtype) >= 0x7fffffffLL || channels * g.taps() >= 0x7fffffffLL || g.L() >= 0x7fffffffLL) return false;
    return channels * g.vol() > 0;
}

static bool conv_implicit(int dtype, int64_t channels, int64_t height, int64_t width, int64_t k_r, int64_t k_c,
                          int64_t s_r, int64_t s_c, int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c, int64_t Ho, int64_t Wo) {
    return conv_implicit_g(dtype, channels, geo2(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo));
}

static void fill_conv_geom(ntg::ConvGeom& c, int64_t slice_channels, const Geo3& g) {
    c.D = (int)g.sz[0]; c.H = (int)g.sz[1]; c.W = (int)g.sz[2]; c.chan = (int)g.vol();
    c.s_d = (int)g.s[0]; c.s_r = (int)g.s[1]; c.s_c = (int)g.s[2];
    c.p_d = (int)g.p[0]; c.p_r = (int)g.p[1]; c.p_c = (int)g.p[2];
    c.d_d = (int)g.d[0]; c.d_r = (int)g.d[1]; c.d_c = (int)g.d[2];
    c.k_d = (int)g.k[0]; c.k_r = (int)g.k[1]; c.k_c = (int)g.k[2];
    c.k_rc = (int)(g.k[1] * g.k[2]); c.k_drc = (int)g.taps();
    c.Wo = (int)g.o[2]; c.HoWo = (int)(g.o[1] * g.o[2]);
    c.last = (int)(slice_channels * g.vol() - 1);
    c.div_kdrc = ntg::make_fastdiv((uint32_t)c.k_drc);
    c.div_krc = ntg::make_fastdiv((uint32_t)c.k_rc);
    c.div_kc = ntg::make_fastdiv((uint32_t)c.k_c);
    c.div_wo = ntg::make_fastdiv((uint32_t)c.Wo);
    c.div_howo = ntg::make_fastdiv((uint32_t)c.HoWo);
}

// A plain product per (image, group), strides in elements; the floating types in one launch.  reference_order: NTG_GEMM_KEEP_K_ORDER (a convolution of one tap
// through the host entry points is unfold + matmult bit for bit).
static int gemm_per_group(int dtype, bool ta, bool tb, int cmode, int64_t m, int64_t k, int64_t n, int64_t lda, int64_t ldb, int64_t ldc, int64_t batch, int64_t groups,
                          const void* A, int64_t a_group, int64_t a_image, const void* B, int64_t b_group, int64_t b_image, void* C, void* stream, bool reference_order) {
    const int64_t es = ntg::elem_size(dtype), c_item = m * ldc;
    const bool streaming = dtype != ntg::DT_F32 || m > 32 || batch * groups <= NTG_SKINNY_MAX_ITEMS;      // (in Float32 the kernels for few rows decide the sums)
    if (groups > 1 && !is_valu_dtype(dtype) && streaming && m > 0 && n > 0 && k > 0 && batch > 0) {
        const int rc = check_sizes(m, k, n, batch);
        if (rc) return rc;
        ntg::GemmParams p;
        std::memset(&p, 0, sizeof p);
        p.M = (int)m; p.K = (int)k; p.N = (int)n;
        p.A = A; p.B = B; p.C = C;
        p.lda = lda; p.ldb = ldb; p.ldc = ldc;
        p.cmode = cmode;
        p.keep_k_order = reference_order;
        int status = NTG_OK;
        const hipError_t e = launch_groups(p, dtype, batch, groups, {a_group, a_image, b_group, b_image, c_item}, [&](const ntg::GemmParams& q) {
            status = launch_gemm(q, dtype, ta, tb, static_cast<hipStream_t>(stream));
            return status == NTG_OK ? hipSuccess : hipErrorUnknown;
        });
        return e == hipSuccess ? NTG_OK : status;
    }
    for (int64_t g = 0; g < groups; ++g) {
        ntg_gemm_desc d;
        std::memset(&d, 0, sizeof d);
        d.dtype = dtype; d.transpose_a = ta; d.transpose_b = tb; d.c_mode = cmode;
        d.m = m; d.k = k; d.n = n;
        d.lda = lda; d.ldb = ldb; d.ldc = ldc; d.batches = batch;
        d.stride_a = a_image; d.stride_b = b_image; d.stride_c = groups * c_item;
        d.flags = reference_order ? NTG_GEMM_KEEP_K_ORDER : 0;
        const int rc = ntg_gemm_dev(&d, static_cast<const char*>(A) + g * a_group * es, static_cast<const char*>(B) + g * b_group * es,
                                    static_cast<char*>(C) + g * c_item * es, stream);
        if (rc) return rc;
    }
    return NTG_OK;
}

// out_b[g*og:(g+1)*og, L] = W_g[og, add] . col_b[g*add:(g+1)*add, L] with col_b gathered from the image by the B loader.
// The reference forms (col_b^T . W_g^T) and swaps rows/columns afterwards (conv.cpp:94, :143); each output element is the
// same ascending-k sum of the same products.
static int conv_forward_gather(int dtype, const void* image, const void* kernel, void* out, int64_t batch, int64_t channels,
                               int64_t out_channels, const Geo3& g, int64_t groups, hipStream_t hs) {
    const int64_t es = ntg::elem_size(dtype), cg = channels / groups, og = out_channels / groups;
    const int64_t L = g.L(), add = cg * g.taps(), vol = g.vol();
    ntg::GemmParams p;
    std::memset(&p, 0, sizeof p);
    p.M = (int)og; p.K = (int)add; p.N = (int)L;
    p.A = kernel; p.B = image; p.C = out;
    p.lda = add; p.ldb = L; p.ldc = L;
    p.cmode = ntg::C_OVERWRITE;
    p.vecA_ok = (add * es) % 16 == 0;
    fill_conv_geom(p.conv, cg, g);
    const hipError_t e = launch_groups(p, dtype, batch, groups, {og * add, 0, cg * vol, channels * vol, og * L},
                                       [&](const ntg::GemmParams& q) { return ntg::launch_conv_mfma(dtype, false, g.nd, q, hs); });
    if (e != hipSuccess) return hip_fail(e, "implicit convolution launch");
    return NTG_OK;
}

// A 1x1 kernel with unit stride and no padding unfolds the image onto itself (col_b == x_b as a [C, H*W] matrix), so the
// convolution is the batched product W_g . x_b on the image where it lies.  Integer dtypes always take it; the floating
// ones when rows of the image and of W are 16-byte multiples (what the DMA-fed kernels need), else they gather.
static bool conv_pointwise(const Geo3& g) {
    for (int a = 0; a < 3; ++a)
        if (g.k[a] != 1 || g.s[a] != 1 || g.p[a] != 0) return false;
    return true;
}
static bool conv_pointwise_ok(int dtype, int64_t channels, int64_t groups, const Geo3& g) {
    if (!conv_pointwise(g)) return false;
    if (is_valu_dtype(dtype)) return true;
    const int64_t es = ntg::elem_size(dtype);
    return (g.L() * es) % 16 == 0 && (channels / groups * es) % 16 == 0;
}
static int conv_forward_pointwise(int dtype, const void* image, const void* kernel, void* out, int64_t batch, int64_t channels,
                                  int64_t out_channels, const Geo3& g, int64_t groups, void* stream, bool reference_order) {
    const int64_t cg = channels / groups, og = out_channels / groups, L = g.L();
    return gemm_per_group(dtype, false, false, NTG_C_OVERWRITE, og, cg, L, cg, L, L, batch, groups, kernel, og * cg, 0, image, cg * L, channels * L, out, stream,
                          reference_order);
}

// Channels-last form of the same convolution, for the floating dtypes up to 32 bits: the image is first copied to
// [B][pixel][C] and the weights to [O][(taps, c)] in the workspace; then one K-step of the product is 64 bytes of consecutive
// channels of one tap, and the kernel's DMA gathers the operand in 16-byte pieces instead of element by element.

// Byte offsets inside a channels-last image are formed in 32 bits from two terms (the pixel of the window origin, and the
// tap reach with the padding taken off): both must stay below 2^30.  The tap counters run to the first tap behind the window, so
// the reach is k d and not (k - 1) d; over two axes there is no depth to step through (counted as one whole slice it refused
// images within one window's reach of 2^30 bytes).
static bool conv_nhwc_offsets_fit(int64_t channels, int64_t es, const Geo3& g) {
    auto mag = [](int64_t v) { return v < 0 ? -v : v; };
    const int64_t pd = mag(g.p[0]), pr = mag(g.p[1]), pc = mag(g.p[2]);
    const int64_t slices = g.nd == 3 ? pd + g.k[0] * g.d[0] : 0;
    const int64_t reach = ((slices * g.sz[1] + pr + g.k[1] * g.d[1]) * g.sz[2] + pc + g.k[2] * g.d[2]) * channels * es;
    return channels * g.vol() * es < (1LL << 30) && reach < (1LL << 30);
}
// A K-step of the channels-last kernel is 64 bytes of channels of one tap, so the copy pads the channels of each group
// with zeros to the next multiple of 64 bytes (and the permuted weights likewise).  The padding is arithmetic spent on
// zeros: accepted up to 4x for the 16-bit types, whose element-wise gather is bound by the vector ALU (beyond that --
// RGB input layers -- the gathering kernels are the better choice); Float32 takes whole runs only: its element-wise
// DMA gather was measured faster than a padded copy (24 -> 32 channels: 48 against 60 us).  0: not accepted.
static int64_t nhwc_padded_channels(int64_t es, int64_t cg) {
    const int64_t step = 64 / es, cgp = (cg + step - 1) / step * step;
    return cg > 0 && cgp <= (es == 2 ? 4 : 1) * cg ? cgp : 0;
}
// The channels-last copy carries the convolution's padding as a border of zero pixels (non-negative padding):
// the padded image is as large as the windows reach, every tap of every window then exists, and the kernel's gather needs
// neither a validity test nor a per-lane address select -- its DMA is that of a stored operand.  gp describes the padded
// image with padding 0 (what the kernel is told); hm where the copy puts the pixels.
struct HaloPlan { bool on; ntg::HaloMap hm; Geo3 gp; int64_t vol; };
static HaloPlan conv_halo(const Geo3& g) {
    HaloPlan h;
    std::memset(&h.hm, 0, sizeof h.hm);
    h.on = false; h.gp = g; h.vol = g.vol();
    int64_t ext[3];                                                   // the padded image: as far as the windows reach, and the image itself
    for (int a = 0; a < 3; ++a) {
        if (g.p[a] < 0) return h;
        ext[a] = std::max((g.o[a] - 1) * g.s[a] + (g.k[a] - 1) * g.d[a] + 1, g.p[a] + g.sz[a]);
    }
    const int64_t vol = ext[0] * ext[1] * ext[2];
    // (a border larger than the image: not worth the copy on two axes, where the validity bits serve; three axes have no such form,
    //  and the element-wise gather they fall back to loses more than the copy of three times the image costs; small maps under wide windows,
    //  where the copy is next to nothing, need it for their channels to go out in ranges: a step of Float16 4 x 1 x 8 x 8 -> 256 by 7 x 7 130 -> 36 us, BFloat16
    //  2 x 256 x 8 x 8 -> 192 by 7 x 7 in 2 groups 113 -> 59)
    if (vol > (g.nd == 3 || vol <= 1024 ? 4 : 2) * g.vol() + 64) return h;
    h.hm.W = g.sz[2]; h.hm.H = g.sz[1]; h.hm.D = g.sz[0];
    h.hm.Wp = ext[2]; h.hm.Hp = ext[1]; h.hm.Dp = ext[0];
    h.hm.left = g.p[2]; h.hm.top = g.p[1]; h.hm.front = g.p[0];
    for (int a = 0; a < 3; ++a) { h.gp.sz[a] = ext[a]; h.gp.p[a] = 0; }
    h.vol = vol;
    h.on = true;
    return h;
}

// How the copy holds the channels of a group (cgp 0: not at all): whole 64-byte runs, or behind a border in whole 16-byte slots (slot_v of them) where
// that is less; the kernel's K-steps are then four slots of whatever taps.  us of the forward product and what it needs, as whole runs, merged taps or
// element-wise gathers | in slots: BFloat16 16 x 24 x 56 x 56 -> 24 by 3 x 3 21 | 12, 16 x 48 x 47 x 47 -> 16 by 5 x 5 in 2 groups 43 | 18, 14 x 1 x 40^3 -> 32 by
// 3 x 3 x 3 365 | 83, Float32 32 x 3 x 224 x 224 -> 64 by 7 x 7 at stride 2 144 | 126, 16 x 24 x 56 x 56 -> 24 29 | 19, 16 x 48 x 47 x 47 -> 16 in 2 groups 104 | 46,
// 4 x 24 x 20^3 -> 40 47 | 33; equal on one or two tiles (Float32 1 x 24 x 12 x 12 -> 24 12 | 12).  Up to 128 output pixels the other forms stay for the
// workspaces that callers know (tests/test_abi.py holds some), not for speed: steps of n x 24 x 8 x 8 -> 24 take 21.0 us so | 20.2 in slots with one image in BFloat16,
// 21.7 | 20.9 with four, Float32 35.0 | 28.9 and 35.5 | 29.6, 72 -> 72 63 | 46.
// In 16 bits wide groups lose little to whole runs, whose taps meet a pixel's line while it is in L2: there slots are taken where they save a quarter of k, or on few
// pixels.  Steps in BFloat16, whole runs | slots: 72 channels (9 slots of 12) 32 x 56 x 56 by 3 x 3 131 | 125, 16 x 28 x 28 46 | 41; 104 (13 of 16) 168 | 178 and 53 | 51,
// 20^3 104 | 111; 168 (21 of 24) 343 | 347 and 77 | 90, 161 | 185; 232 (29 of 32) 476 | 486 and 98 | 107, 224 | 259; 4 x 28 x 28 of 104, 168, 232 37.7 | 35.1, 51 | 47, 64 | 60.
struct NhwcForm { int64_t cgp, slot_v; };
static NhwcForm nhwc_form(int64_t es, int64_t cg, int64_t taps, int nd, bool bordered, int64_t pixels) {
    const int64_t vel = 16 / es, slots = (cg + vel - 1) / vel, in_runs = (slots + 3) / 4 * 4;
    const bool fewer = es == 4 ? slots < in_runs : 4 * slots <= 3 * in_runs || (slots < in_runs && pixels < (in_runs <= 16 && nd < 3 ? 32768 : 8192));
    if (bordered && cg > 0 && pixels > 128 && fewer && taps * slots <= NTG_SLOT_TABLE) return {slots * vel, slots};
    return {nhwc_padded_channels(es, cg), 0};
}

// Few channels per group (up to 32 bytes of them): a pixel of the copy holds 16 or 32 bytes and a K-step covers 4 or 2
// consecutive taps of a tap row, the row padded to a multiple of that with zero weights -- an RGB 7 x 7 input layer in
// BFloat16 runs on K = 7 * 8 * 8 instead of 49 * 32.  Forward only.
struct MergedTaps { int64_t cgp, T, kq_pad; };
static bool conv_nhwc_merged(int dtype, int64_t batch, int64_t channels, int64_t out_channels, int64_t groups, const Geo3& g, MergedTaps& mt) {
    if (dtype != ntg::DT_F32 && dtype != ntg::DT_F16 && dtype != ntg::DT_BF16) return false;
    if (g.nd != 2 || !conv_implicit_g(dtype, channels, g) || out_channels <= 0) return false;
    const int64_t es = ntg::elem_size(dtype), cg = channels / groups;
    if (cg <= 0 || cg * es > 32 || nhwc_form(es, cg, g.taps(), g.nd, conv_halo(g).on, batch * g.L()).slot_v) return false;
    const int64_t cb = cg * es <= 16 ? 16 : 32;
    mt.cgp = cb / es; mt.T = 64 / cb; mt.kq_pad = (g.k[2] + mt.T - 1) / mt.T * mt.T;
    if (mt.kq_pad > 8 || mt.kq_pad * mt.cgp > 4 * g.k[2] * cg || out_channels * g.k[1] * mt.kq_pad >= 0x7fffffffLL) return false;          // (padding: at most 4x the arithmetic)
    return conv_nhwc_offsets_fit(groups * mt.cgp, es, g);
}
static int64_t conv_nhwc_merged_workspace(int dtype, int64_t batch, int64_t out_channels, int64_t groups, const Geo3& g, const MergedTaps& mt) {
    const int64_t es = ntg::elem_size(dtype);
    return (int64_t)align_up((size_t)(batch * groups * mt.cgp * g.vol() * es), 256) + out_channels * g.k[1] * mt.kq_pad * mt.cgp * es;
}
static bool conv_nhwc_ok(int dtype, int64_t batch, int64_t channels, int64_t out_channels, int64_t groups, const Geo3& g) {
    if (dtype != ntg::DT_F32 && dtype != ntg::DT_F16 && dtype != ntg::DT_BF16) return false;
    if (!conv_implicit_g(dtype, channels, g)) return false;
    const HaloPlan halo = conv_halo(g);
    if (g.nd == 3 && !halo.on) return false;                          // (three axes: the bordered copy is the only form)
    const int64_t es = ntg::elem_size(dtype), cgp = nhwc_form(es, channels / groups, g.taps(), g.nd, halo.on, batch * g.L()).cgp;
    return cgp > 0 && out_channels > 0 && out_channels * g.taps() < 0x7fffffffLL && conv_nhwc_offsets_fit(groups * cgp, es, g) &&
           conv_nhwc_offsets_fit(groups * cgp, es, halo.gp);
}
// Few output tiles and a deep k (a handful of small maps with many channels): the 64-byte runs of channels in `ranges` equal ranges, Float32 sums of
// each, added up in order by a second pass.  A workgroup alone on its CU takes 0.32 us a K-step in Float32 and 0.2 in 16 bits whatever the others do (2 x 256 x
// 13 x 13 -> 256 by 3 x 3: 24 tiles of 144 and 72 K-steps); shared by w workgroups a CU takes 0.25 w and 0.07 w.  The second pass costs 4.5 us and the traffic of
// the sums.  Measured: that layer 47 -> 11 + 3 us and 18 -> 8 + 3; 192 x 17 x 17 -> 32 by 7 x 7, 3 tiles of 588, 169 -> 33 + 4 us.  Under 64 K-steps there is too little
// to win.  Layers in groups alike (Float32 256 x 11^3 -> 128 by 3 x 3 x 3 at stride 2 in 4 groups, a step, 85 -> 62 us, 4 x 96 x 8 x 8 -> 16 by 5 x 5 at stride 2 in 2
// 56 -> 44).  Whether there are ranges, and how many, follows from one image, so up to 128 tiles in all an image's result is the same bits alone and among
// others (in whole runs: nhwc_form looks at all images' pixels).  That is ahead all the way: BFloat16 n x 256 x 13 x 13 -> 256 by
// 3 x 3, a step, without | with ranges in the products: 10 images 64.0 | 55.6 us; 256 x 16 x 16 -> 256, 8 images 62.8 | 58.9.
static int64_t conv_k_ranges(int64_t es, int64_t batch, int64_t rows, int64_t pixels, int64_t groups, const NhwcForm& form, int64_t taps) {
    const int64_t bk = 64 / es, runs = form.cgp / bk, steps = runs * taps, tiles = ((rows / groups + 63) / 64) * ((pixels + 63) / 64) * groups;
    if (form.slot_v || tiles * batch > 128 || steps < 64) return 1;
    int64_t r = 8;
    while (r > 1 && (runs % r != 0 || steps / r < 16)) --r;
    const double shared = (double)((tiles * r + 255) / 256), step_us = es == 4 ? 0.32 : 0.2, shared_us = std::max(step_us, (es == 4 ? 0.25 : 0.07) * shared);
    const double sums_us = 4.5 + 8.0 * (double)(r * rows * pixels) / 4.0e6;
    return (double)(steps / r) * shared_us + sums_us < 0.8 * (double)steps * step_us ? r : 1;
}
static int64_t conv_k_ranges_bytes(int64_t ranges, int64_t batch, int64_t rows, int64_t pixels) { return ranges > 1 ? ranges * batch * rows * ((pixels + 7) / 8 * 8) * 4 : 0; }
// the product p (weights by image, p.M rows a group; strides as in launch_groups) in ranges: partial sums at `part`, results at p.C in p.cmode
static hipError_t launch_conv_k_ranges(ntg::GemmParams p, int dtype, int64_t batch, int64_t groups, int64_t ranges, int64_t taps, const GroupStrides& st, char* part, hipStream_t hs) {
    const int64_t ldp = (p.N + 7) / 8 * 8, K = p.K;
    ntg::GemmParams q = p;
    // launch index = (range * images + image) * groups + group
    q.K = (int)(K / ranges);
    q.C = part;
    q.ldc = ldp; q.sC = p.M * ldp;
    q.cmode = ntg::C_PARTIAL;
    q.batch = (int)(batch * groups * ranges);
    q.krange_items = (int)(batch * groups);
    q.sA = groups > 1 ? st.a_group : 0; q.sAk = q.K;
    q.sB = groups > 1 ? st.b_group : st.b_image; q.sBk = q.K / taps;
    q.conv.range_groups = (int)groups;
    q.conv.range_image = st.b_image;
    hipError_t e = ntg::launch_conv_nhwc(dtype, q, hs);
    if (e != hipSuccess) return e;
    p.batch = (int)(batch * groups);
    p.sC = st.c_item;
    return ntg::launch_splitk_reduce(dtype, part, (int)ranges, p, ldp, hs);
}
static int64_t conv_nhwc_workspace(int dtype, int64_t batch, int64_t channels, int64_t out_channels, int64_t groups, const Geo3& g) {
    const HaloPlan halo = conv_halo(g);
    const int64_t es = ntg::elem_size(dtype);
    const NhwcForm form = nhwc_form(es, channels / groups, g.taps(), g.nd, halo.on, batch * g.L());
    const int64_t cgp = form.cgp, weights = out_channels * cgp * g.taps() * es;
    const int64_t sums = halo.on ? conv_k_ranges_bytes(conv_k_ranges(es, batch, out_channels, g.L(), groups, form, g.taps()), batch, out_channels, g.L()) : 0;
    return (int64_t)align_up((size_t)(batch * groups * cgp * halo.vol * es), 256) + (sums ? (int64_t)align_up((size_t)weights, 256) + sums : weights);
}
static void set_slots(ntg::ConvGeom& c, const NhwcForm& form) {
    c.slot_v = (int)form.slot_v;
    c.div_slot = ntg::make_fastdiv((uint32_t)std::max<int64_t>(form.slot_v, 1));
}
static void add_copy(ntg::ChannelsLast& cl, const void* in, void* out, int64_t batch, int64_t groups, int64_t cg, int64_t cgp, int64_t pixels, const HaloPlan& halo) {
    cl.copy[cl.n++] = {in, out, batch, groups, cg, cgp, pixels, halo.on, halo.hm};
}
static int conv_forward_nhwc(int dtype, const void* image, const void* kernel, void* out, void* ws, int64_t batch, int64_t channels,
                             int64_t out_channels, const Geo3& g, int64_t groups, hipStream_t hs, const MergedTaps* mt = nullptr) {
    const int64_t es = ntg::elem_size(dtype), cg = channels / groups, og = out_channels / groups;
    HaloPlan halo = conv_halo(g);
    const NhwcForm form = nhwc_form(es, cg, g.taps(), g.nd, halo.on, batch * g.L());
    const int64_t cgp = mt ? mt->cgp : form.cgp, chp = groups * cgp;      // channels per group / per pixel in the copy
    const int64_t L = g.L(), taps = g.taps(), vol = g.vol(), K = mt ? g.k[1] * mt->kq_pad * cgp : taps * cgp;
    if (mt) { halo.on = false; halo.vol = vol; halo.gp = g; }                    // (the merged-tap form keeps its validity bits)
    const int64_t volp = halo.vol;                                               // pixels per image of the copy
    const int64_t ranges = halo.on ? conv_k_ranges(es, batch, out_channels, L, groups, form, taps) : 1;
    // (neighbouring taps share pixels only at unit strides; ranges are of whole runs with all their taps)
    const bool tap_inner = halo.on && !form.slot_v && ((g.s[0] == 1 && g.s[1] == 1 && g.s[2] == 1) || ranges > 1);
    char* ws_img = static_cast<char*>(ws);
    char* ws_w = ws_img + align_up((size_t)(batch * chp * volp * es), 256);
    const int64_t wchunk = tap_inner ? 64 / es : 0;                              // (taps inside a 64-byte run of channels)
    ntg::ChannelsLast cl;
    std::memset(&cl, 0, sizeof cl);
    add_copy(cl, image, ws_img, batch, groups, cg, cgp, vol, halo);
    cl.weights = {mt ? 3 : 1, kernel, ws_w, out_channels, cg, cgp, taps, 0, g.k[1], g.k[2], mt ? mt->kq_pad : 0, wchunk};
    hipError_t e = ntg::launch_channels_last(es, cl, hs);
    if (e != hipSuccess) return hip_fail(e, "channels-last copy launch");
    ntg::GemmParams p;
    std::memset(&p, 0, sizeof p);
    p.M = (int)og; p.K = (int)K; p.N = (int)L;
    p.A = ws_w; p.B = ws_img; p.C = out;
    p.lda = K; p.ldb = chp; p.ldc = L;
    p.cmode = ntg::C_OVERWRITE;
    p.vecA_ok = 1; p.vecB_ok = 1;
    fill_conv_geom(p.conv, cgp, halo.gp);
    p.conv.chan = (int)chp;                        // elements from one pixel to the next
    p.conv.halo = halo.on ? 1 : 0;
    p.conv.tap_inner = tap_inner ? 1 : 0;
    if (mt) { p.conv.tap_step = (int)mt->T; p.conv.kq_pad = (int)mt->kq_pad; }
    else set_slots(p.conv, form);
    const GroupStrides st = {og * K, 0, cgp, chp * volp, og * L};
    if (ranges > 1) e = launch_conv_k_ranges(p, dtype, batch, groups, ranges, taps, st, ws_w + align_up((size_t)(out_channels * K * es), 256), hs);
    else e = launch_groups(p, dtype, batch, groups, st, [&](const ntg::GemmParams& q) { return ntg::launch_conv_nhwc(dtype, q, hs); });
    if (e != hipSuccess) return hip_fail(e, "channels-last convolution launch");
    return NTG_OK;
}

// dW: one batched GEMM  P_{b,g} [og, add] = dY_{b,g} [og, L] . col_{b,g}^T  with col gathered from the image, into
// ws [B][O][add]; then the per-image results are summed in batch order (the same additions, in the same order, as
// accumulating one GEMM per image into dW, conv.cpp:466-469).
static int conv_dkernel_gather(int dtype, const void* image, const void* grad_out, void* d_kernel, void* ws, int64_t batch,
                               int64_t channels, int64_t out_channels, const Geo3& g, int64_t groups, int accumulate, hipStream_t hs) {
    const int64_t es = ntg::elem_size(dtype), cg = channels / groups, og = out_channels / groups;
    const int64_t L = g.L(), add = cg * g.taps(), vol = g.vol();
    ntg::GemmParams p;
    std::memset(&p, 0, sizeof p);
    p.M = (int)og; p.K = (int)L; p.N = (int)add;
    p.A = grad_out; p.B = image; p.C = ws;
    p.lda = L; p.ldb = L; p.ldc = add;
    p.cmode = ntg::C_OVERWRITE;
    p.vecA_ok = (L * es) % 16 == 0 && (out_channels * L * es) % 16 == 0;
    fill_conv_geom(p.conv, cg, g);
    hipError_t e = launch_groups(p, dtype, batch, groups, {og * L, out_channels * L, cg * vol, channels * vol, og * add},
                                 [&](const ntg::GemmParams& q) { return ntg::launch_conv_mfma(dtype, true, g.nd, q, hs); });
    if (e != hipSuccess) return hip_fail(e, "implicit conv_dkernel launch");
    e = ntg::launch_reduce_batch(dtype, ws, d_kernel, batch, out_channels * add, accumulate, hs);
    if (e != hipSuccess) return hip_fail(e, "weight gradient reduction launch");
    return NTG_OK;
}

// dX (all strides 1): the convolution of dY with the channel-swapped, tap-reversed kernel (written to ws) and padding
// d*(k-1) - p, again as an implicit GEMM; one sum over (oc, taps) per element instead of the reference's GEMM over oc
// followed by col2im over the taps -- same terms, different rounding order, inside the stated tolerance.
static int conv_dimage_gather(int dtype, const void* kernel, const void* grad_out, void* d_image, void* ws, int64_t batch,
                              int64_t channels, int64_t out_channels, const Geo3& g, int64_t groups, int accumulate, hipStream_t hs) {
    const int64_t es = ntg::elem_size(dtype), cg = channels / groups, og = out_channels / groups;
    const int64_t L = g.L(), taps = g.taps(), vol = g.vol();
    hipError_t e = ntg::launch_flip_weights(es, kernel, ws, groups, og, cg, taps, hs);
    if (e != hipSuccess) return hip_fail(e, "weight flip launch");
    const Geo3 t = geo_dimage(g);
    ntg::GemmParams p;
    std::memset(&p, 0, sizeof p);
    p.M = (int)cg; p.K = (int)(og * taps); p.N = (int)vol;
    p.A = ws; p.B = grad_out; p.C = d_image;
    p.lda = og * taps; p.ldb = vol; p.ldc = vol;
    p.cmode = accumulate ? ntg::C_ACCUMULATE : ntg::C_OVERWRITE;
    p.vecA_ok = (og * taps * es) % 16 == 0;
    fill_conv_geom(p.conv, og, t);
    e = launch_groups(p, dtype, batch, groups, {cg * og * taps, 0, og * L, out_channels * L, cg * vol},
                      [&](const ntg::GemmParams& q) { return ntg::launch_conv_mfma(dtype, false, g.nd, q, hs); });
    if (e != hipSuccess) return hip_fail(e, "implicit conv_dimage launch");
    return NTG_OK;
}

// The same gradient through the channels-last kernel: dY is copied to [B][pixel][O] and the flipped weights to
// [C][(taps, oc)] in the workspace (out channels of a group in whole 64-byte runs, padded like the forward copy).
static bool conv_dimage_nhwc_ok(int dtype, int64_t batch, int64_t channels, int64_t out_channels, int64_t groups, const Geo3& g) {
    return conv_nhwc_ok(dtype, batch, out_channels, channels, groups, geo_dimage(g));
}
static int64_t conv_dimage_nhwc_workspace(int dtype, int64_t batch, int64_t channels, int64_t out_channels, int64_t groups, const Geo3& g) {
    return conv_nhwc_workspace(dtype, batch, out_channels, channels, groups, geo_dimage(g));
}
// (the image gradients and the channels-last weight gradient come in two parts, so that a call can make the copies of both in one launch:
//  with `cl` they only add theirs to it, without it they run on copies that have been made)
static int conv_dimage_nhwc(int dtype, const void* kernel, const void* grad_out, void* d_image, void* ws, int64_t batch,
                            int64_t channels, int64_t out_channels, const Geo3& g, int64_t groups, int accumulate, hipStream_t hs, ntg::ChannelsLast* cl) {
    const int64_t es = ntg::elem_size(dtype), cg = channels / groups, og = out_channels / groups;
    const Geo3 t = geo_dimage(g);
    const HaloPlan halo = conv_halo(t);                                         // (the "image" of this convolution is dY)
    const NhwcForm form = nhwc_form(es, og, g.taps(), g.nd, halo.on, batch * t.L());
    const int64_t ogp = form.cgp, ochp = groups * ogp;                          // out channels per group / per pixel in the copy
    const int64_t L = g.L(), taps = g.taps(), vol = g.vol(), K = taps * ogp;
    const int64_t Lp = halo.vol;
    const bool tap_inner = halo.on && !form.slot_v;                             // (all strides are 1)
    char* ws_gy = static_cast<char*>(ws);
    char* ws_w = ws_gy + align_up((size_t)(batch * ochp * Lp * es), 256);
    if (cl) {
        add_copy(*cl, grad_out, ws_gy, batch, groups, og, ogp, L, halo);
        cl->weights = {2, kernel, ws_w, channels, og, ogp, taps, cg, 0, 0, 0, tap_inner ? 64 / es : 0};
        return NTG_OK;
    }
    ntg::GemmParams p;
    std::memset(&p, 0, sizeof p);
    p.M = (int)cg; p.K = (int)K; p.N = (int)vol;
    p.A = ws_w; p.B = ws_gy; p.C = d_image;
    p.lda = K; p.ldb = ochp; p.ldc = vol;
    p.cmode = accumulate ? ntg::C_ACCUMULATE : ntg::C_OVERWRITE;
    p.vecA_ok = 1; p.vecB_ok = 1;
    fill_conv_geom(p.conv, ogp, halo.gp);
    p.conv.chan = (int)ochp;
    p.conv.halo = halo.on ? 1 : 0;
    p.conv.tap_inner = tap_inner ? 1 : 0;
    set_slots(p.conv, form);
    const int64_t ranges = halo.on ? conv_k_ranges(es, batch, channels, vol, groups, form, taps) : 1;
    const GroupStrides st = {cg * K, 0, ogp, ochp * Lp, cg * vol};
    const hipError_t e = ranges > 1 ? launch_conv_k_ranges(p, dtype, batch, groups, ranges, taps, st, ws_w + align_up((size_t)(channels * K * es), 256), hs)
                                    : launch_groups(p, dtype, batch, groups, st, [&](const ntg::GemmParams& q) { return ntg::launch_conv_nhwc(dtype, q, hs); });
    if (e != hipSuccess) return hip_fail(e, "channels-last conv_dimage launch");
    return NTG_OK;
}

// Float32: K-steps (16 multiply-adds) of one chain in a gathered product that stands for shorter ones of `n` multiply-adds each, added
// up: the largest power of two within n, from one K-step to sixteen (256 multiply-adds; longer chains gain no time), to eight in the weight
// gradients of layers in groups, which share the ranges that fill the CUs: theirs are fewer and longer.  Relative error with ranges for each group |
// shared ones in chains of 256 | of 128: 4 x 24 x 64 x 64 -> 32 by 5 x 5 in 4 groups 2.26e-7 | 3.01e-7 | 2.23e-7, 192 x 29^3 -> 48 by 3 x 3 x 3 at stride 2
// in 4 groups 2.14e-7 | 2.59e-7 | 1.95e-7.  Without groups 128 costs 0.6 % of a step (4 x 32 x 32^3 -> 64 by 3 x 3 x 3 395.3 | 397.7 us).
static int chain_steps(int64_t n, int most = 16) {
    int steps = 1;
    while (steps < most && 32 * steps <= n) steps *= 2;
    return steps;
}

// dX of a convolution with strides > 1 (dilation 1), without the col matrix: the image positions y with (y + p) mod s = e
// form one phase; they receive only the taps i = e + s m (m = 0 .. M_e - 1), and, with a = (y + p) / s,
//   dX[y] = sum_m dY[a - m] W[e + s m],
// a stride-1 convolution of dY with the M_e reversed taps.  So every phase (one per residue of each axis) is one channels-last
// convolution of the shared bordered copy of dY with its own small kernel, written to a plane of the phase's positions in the
// workspace; a last pass interleaves the planes into dX.  Exactly the products of the reference's GEMM + col2im, none wasted on
// the zeros a dilated gradient would hold.  All phases (and groups) are items of ONE launch: a phase alone is a small product
// (32 x 64 x 56 x 56 by 4 x 4 at stride 2: 416 tiles of k = 512), and four launches with a weight permutation each took 58 us
// where the one takes 25 and the set-up of all phases' weights 8.
struct PhasePlan {
    bool ok;
    int edge;
    NhwcForm form;
    int64_t gy_bytes, w_bytes, item_bytes, tmp_bytes, blocks;
    ntg::HaloMap hm;
    ntg::PhaseLayout lay;
    int64_t bytes() const { return gy_bytes + w_bytes + item_bytes + tmp_bytes; }
};
// Out channels of a group as the phases hold them, in whole 64-byte runs (0: not taken).  The alternative is the col matrix, which is ahead wherever
// Float32 would have to pad (16 x 64 x 56 x 56 -> 24 by 3 x 3 at stride 2, a step: 83 us against 93 by phases; 4 x 32 x 24^3 -> 24 by 3 x 3 x 3 84 / 101)
// except over three axes on images from 32 MiB on, the passes over col and image being the larger part there (9 x 256 x 29^3 -> 48 by one
// tap in 2 groups 621 / 406, 42 x 256 x 24^3 -> 96 by 3 x 3 x 3 in 4 groups 3291 / 2571).
static NhwcForm phase_form(int64_t es, int64_t og, int64_t batch, int64_t channels, const Geo3& g) {
    int64_t taps = 1;                                                             // of the largest phase
    for (int a = 0; a < 3; ++a) taps *= (g.k[a] + g.s[a] - 1) / g.s[a];
    const NhwcForm f = nhwc_form(es, og, taps, g.nd, true, batch * g.vol());
    // (a chain ends with a K-step at the earliest: in slots it would run through several taps of fewer than 16 channels)
    if (es == 4 && og < 16 && f.slot_v) return {16, 0};
    if (f.slot_v) return f;
    const int64_t step = 64 / es, ogp = (og + step - 1) / step * step;
    const int64_t most = es == 2 ? 4 : g.nd == 3 && batch * channels * g.vol() * es >= (1LL << 25) ? 2 : 1;
    return {og > 0 && ogp <= most * og ? ogp : 0, 0};
}
static PhasePlan plan_dimage_phases(int dtype, int64_t batch, int64_t channels, int64_t out_channels, int64_t groups, const Geo3& g) {
    PhasePlan pp;
    std::memset(&pp, 0, sizeof pp);
    if (dtype != ntg::DT_F32 && dtype != ntg::DT_F16 && dtype != ntg::DT_BF16) return pp;
    if (g.s[0] == 1 && g.s[1] == 1 && g.s[2] == 1) return pp;
    for (int a = 0; a < 3; ++a)
        if (g.d[a] != 1 || g.s[a] > 4 || g.p[a] < 0 || g.sz[a] >= (1 << 24) || g.k[a] >= (1 << 16)) return pp;
    const int64_t es = ntg::elem_size(dtype), vel = 16 / es, og = out_channels / groups, cg = channels / groups;
    const NhwcForm form = phase_form(es, og, batch, channels, g);
    const int64_t ogp = form.cgp, ochp = groups * ogp;
    // (the interleaving pass counts image elements in 32 bits; one image's planes, whose pitches are 16-byte multiples, are indexed in 32 bits)
    if (ogp == 0 || batch * channels * g.vol() >= 0x7fffffffLL || channels * (g.vol() + 64 * vel) >= 0x7fffffffLL) return pp;
    // the image channels of a group are the rows of these products: with a handful of them (an RGB input layer) a 64-row
    // tile is mostly padding, and the GEMM over (channel, tap) rows followed by col2im is the better form
    if (cg < 16) return pp;
    ntg::PhaseLayout& q = pp.lay;
    int64_t front[3];
    for (int ax = 0; ax < 3; ++ax) {
        q.sz[ax] = (int)g.sz[ax]; q.k[ax] = (int)g.k[ax]; q.s[ax] = (int)g.s[ax]; q.p[ax] = (int)g.p[ax];
        q.div_s[ax] = ntg::make_fastdiv((uint32_t)g.s[ax]);
        q.div_rows[ax] = ntg::make_fastdiv((uint32_t)g.sz[ax]);
        front[ax] = 0;
        for (int64_t e = 0; e < g.s[ax]; ++e) {
            q.M[ax][e] = (int)(e < g.k[ax] ? (g.k[ax] - e + g.s[ax] - 1) / g.s[ax] : 0);
            // image positions y = s a + e - p in [0, size): a from a0
            q.a0[ax][e] = (int)(g.p[ax] > e ? (g.p[ax] - e + g.s[ax] - 1) / g.s[ax] : 0);
            const int64_t last = g.sz[ax] - 1 + g.p[ax] - e;                      // largest s a
            q.n[ax][e] = (int)(last >= 0 && last / g.s[ax] >= q.a0[ax][e] ? last / g.s[ax] - q.a0[ax][e] + 1 : 0);
            // the window of the phase's first position begins (M - 1) - a0 before dY (behind it if negative)
            if (q.M[ax][e] && q.n[ax][e]) front[ax] = std::max<int64_t>(front[ax], q.M[ax][e] - 1 - q.a0[ax][e]);
        }
        int64_t ext = front[ax] + g.o[ax];
        for (int64_t e = 0; e < g.s[ax]; ++e) {
            q.org[ax][e] = (int)(front[ax] - (q.M[ax][e] - 1 - q.a0[ax][e]));
            if (q.M[ax][e] && q.n[ax][e]) ext = std::max<int64_t>(ext, q.org[ax][e] + q.n[ax][e] - 1 + q.M[ax][e]);
        }
        q.yp[ax] = (int)ext;
    }
    const int64_t volp = (int64_t)q.yp[0] * q.yp[1] * q.yp[2];
    const Geo3 reach = {g.nd, {q.yp[0], q.yp[1], q.yp[2]}, {g.k[0], g.k[1], g.k[2]}, {1, 1, 1}, {0, 0, 0}, {1, 1, 1}, {1, 1, 1}};
    // A border of many times dY: in Float32 the col matrix is the faster form (32 x 128 x 8 x 256 from 8 x 8 at stride 2, one row of 125
    // outputs, 256 out channels: 231 us against 541 by phases).  In 16 bits it is slower (247 against 128 us; a small one, 4 x 32 x 8 x 64,
    // 18 against 27) and rounds every entry of the col matrix besides the sum (2.4e-3 from the exact gradient against 1.7e-3), so the
    // phases keep what they served over two axes with windows of up to 8 taps, whose border is at most 7 positions on each side.
    const bool keep = es == 2 && g.nd == 2 && g.k[1] <= 8 && g.k[2] <= 8;
    if ((!keep && volp > 4 * g.L() + 64) || !conv_nhwc_offsets_fit(ochp, es, reach) || ogp * g.taps() >= 0x7fffffffLL) return pp;
    pp.hm.W = g.o[2]; pp.hm.H = g.o[1]; pp.hm.D = g.o[0];
    pp.hm.Wp = q.yp[2]; pp.hm.Hp = q.yp[1]; pp.hm.Dp = q.yp[0];
    pp.hm.left = front[2]; pp.hm.top = front[1]; pp.hm.front = front[0];
    q.groups = (int)groups; q.og = (int)og; q.ogp = (int)ogp; q.cg = (int)cg; q.batch = (int)batch;
    q.chunk = (int)(form.slot_v ? ogp : 64 / es); q.vel = (int)vel;
    int64_t w_elems = 0, tmp_elems = 0, n_max = 0, k_max = 0;
    for (int ph = 0; ph < NTG_MAX_PHASES; ++ph) q.plane_off[ph] = -1;
    for (int e0 = 0; e0 < q.s[0]; ++e0)
        for (int e1 = 0; e1 < q.s[1]; ++e1)
            for (int e2 = 0; e2 < q.s[2]; ++e2) {
                const int64_t taps = (int64_t)q.M[0][e0] * q.M[1][e1] * q.M[2][e2], n = (int64_t)q.n[0][e0] * q.n[1][e1] * q.n[2][e2];
                if (taps == 0 || n == 0) continue;
                const int ph = (e0 * q.s[1] + e1) * q.s[2] + e2;
                q.w_off[ph] = w_elems;
                q.plane_off[ph] = tmp_elems;
                w_elems += channels * taps * ogp;                                 // (ogp is a multiple of 64 bytes)
                tmp_elems += batch * channels * ntg::phase_plane(q, e0, e1, e2);
                n_max = std::max(n_max, n); k_max = std::max(k_max, taps * ogp);
                ++q.phases;
            }
    if (q.phases == 0) return pp;
    // one tile for all items, as if they were equal
    const int64_t items = (int64_t)q.phases * groups;
    if (es == 4) pp.edge = ntg::ring_f32_conv_edge(cg, n_max, batch * items);
    else pp.edge = cg <= 32 ? 32 : ntg::ring16_tile_edge(cg, n_max, k_max, batch * items);      // (32: flat tiles)
    q.tile_rows = pp.edge;
    q.tile_cols = pp.edge == 32 ? 128 : pp.edge;
    const int64_t tiles_m = (cg + pp.edge - 1) / pp.edge;
    for (int e0 = 0; e0 < q.s[0]; ++e0)
        for (int e1 = 0; e1 < q.s[1]; ++e1)
            for (int e2 = 0; e2 < q.s[2]; ++e2) {
                if (q.plane_off[(e0 * q.s[1] + e1) * q.s[2] + e2] < 0) continue;
                const int64_t n = (int64_t)q.n[0][e0] * q.n[1][e1] * q.n[2][e2];
                pp.blocks += tiles_m * ((n + q.tile_cols - 1) / q.tile_cols) * batch * groups;
            }
    if (pp.blocks > 0x7fffffffLL || channels * g.taps() >= 0x7fffffffLL) return pp;
    pp.form = form;
    pp.gy_bytes = (int64_t)align_up((size_t)(batch * ochp * volp * es), 256);
    pp.w_bytes = (int64_t)align_up((size_t)(w_elems * es), 256);
    pp.item_bytes = (int64_t)align_up((size_t)items * sizeof(ntg::RingItem), 256);
    pp.tmp_bytes = (int64_t)align_up((size_t)(tmp_elems * es), 256);
    pp.ok = true;
    return pp;
}
static int conv_dimage_phases(int dtype, const PhasePlan& pp, const void* kernel, const void* grad_out, void* d_image, void* ws, int64_t batch,
                              int64_t channels, const Geo3& g, int64_t groups, int accumulate, hipStream_t hs, ntg::ChannelsLast* cl) {
    const ntg::PhaseLayout& q = pp.lay;
    const int64_t og = q.og, ogp = q.ogp, ochp = groups * ogp;
    char* ws_gy = static_cast<char*>(ws);
    char* ws_w = ws_gy + pp.gy_bytes;
    ntg::RingItem* items = reinterpret_cast<ntg::RingItem*>(ws_w + pp.w_bytes);
    char* ws_tmp = ws_w + pp.w_bytes + pp.item_bytes;
    if (cl) {
        cl->copy[cl->n++] = {grad_out, ws_gy, batch, groups, og, ogp, g.L(), true, pp.hm};
        cl->weights = {4, kernel, ws_w, channels, og, ogp, g.taps(), q.cg, 0, 0, 0, 0};
        cl->phases = &pp.lay;
        cl->items = items;
        return NTG_OK;
    }
    ntg::GemmParams p;
    std::memset(&p, 0, sizeof p);
    p.M = q.cg; p.batch = (int)batch;
    p.A = ws_w; p.B = ws_gy; p.C = ws_tmp;
    p.ldb = ochp; p.sB = ochp * pp.hm.vol(); p.sC = channels;
    p.cmode = ntg::C_OVERWRITE;
    p.vecA_ok = 1; p.vecB_ok = 1;
    p.conv.D = q.yp[0]; p.conv.H = q.yp[1]; p.conv.W = q.yp[2]; p.conv.chan = (int)ochp;
    p.conv.s_d = p.conv.s_r = p.conv.s_c = 1;
    p.conv.d_d = p.conv.d_r = p.conv.d_c = 1;
    p.conv.k_drc = 1;                                      // (the items set their own taps; k runs taps-inner, which does not use it)
    p.conv.halo = 1; p.conv.tap_inner = 1;
    set_slots(p.conv, pp.form);
    p.conv.items = items; p.conv.n_items = q.phases * (int)groups;
    // (what the phases in slots and over three axes took over from the col matrix adds up one product per tap: no chain may be longer.  Float32 8 x 32 x 56 x 56
    //  -> 24 at stride 2 by 3 x 3 | 5 x 5 | 7 x 7, relative error: the col matrix 0.95e-7 | 1.03e-7 | 1.13e-7, one chain through all taps 1.44e-7 | 2.24e-7 | 3.06e-7)
    if (g.nd == 3 || pp.form.slot_v || og < 16) p.conv.k_segment = chain_steps(og);
    hipError_t e = ntg::launch_conv_nhwc_items(dtype, pp.edge, p, pp.blocks, hs);
    if (e != hipSuccess) return hip_fail(e, "phase convolution launch");
    e = ntg::launch_phase_interleave(dtype, ws_tmp, d_image, q, accumulate, hs);
    if (e != hipSuccess) return hip_fail(e, "phase interleave launch");
    return NTG_OK;
}

// dW through the channels-last kernel: the image is copied to [B][pixel][C]; the output pixels of ALL images counted through are
// cut into k ranges, and per range and group  P [og][(taps, c)] = dY [og, pixels] . col^T  gathered 16 bytes of channels at a
// time; the ranges' partial sums are added in order into the kernel's [O][c][taps] layout.  The copy pads the channels of a group to
// whole 16-byte runs and carries the convolution's padding as pixels of zeros.
static int64_t dkernel_padded_channels(int64_t es, int64_t cg) { const int64_t v = 16 / es; return (cg + v - 1) / v * v; }
static HaloPlan dkernel_halo(int64_t es, int64_t cg, int64_t groups, const Geo3& g) {
    HaloPlan h = conv_halo(g);
    const int64_t cgp = dkernel_padded_channels(es, cg);
    // (a copy that pads the channels grows by its border as well: on one and two axes that is kept to a quarter of the image, as it is from 17 x 17 pixels on for a
    //  3 x 3 window, for the workspace alone.  Steps with validity tests | with the border, us: BFloat16 64 x 3 x 16 x 16 -> 64 by 3 x 3 26.1 | 25.8, 256 x 3 x 32 x 32 ->
    //  64 by 5 x 5 132 | 128, Float32 39.5 | 39.0, 331 | 324, 256 x 6 x 16 x 16 -> 96 100 | 94, 64 x 102 x 14 x 14 -> 128 134 | 129; equal on 8 x 8)
    const bool wide_border = g.nd < 3 && cgp != cg && 4 * h.vol > 5 * g.vol();
    if (h.on && (wide_border || !conv_nhwc_offsets_fit(groups * cgp, es, h.gp))) {
        h.on = false; h.gp = g; h.vol = g.vol();
    }
    return h;
}
// What a launch of the gathering kernel takes: microseconds for `tiles` tiles of rows x cols with K output pixels each, by how many workgroups share a
// CU; the writes of the partial sums are the caller's.  Nanoseconds a pixel and tile, alone on its CU and for each of several:
//   Float32  64 x 64 25, 18.5 (the matrix pipe takes 13.3)   64 x 128 40, 33   32 x 128 26, 19.5   128 x 128 72, 60
//   16-bit   64 x 64 7.5, 3.5                                64 x 128 8.5, 5.5   32 x 128 7.5, 4.6   larger ones by their share of a CU's MFMA peak
// Wide tiles read the output gradient and wait at the barrier half as often, flat ones do half the work where a group has up to 32 out channels.  us of the
// gradient on 64 x 64 | 64 x 128 | 32 x 128: Float32 4 x 32 x 32^3 -> 64 by 3 x 3 x 3 158 | 144 | 171, 32 x 3 x 224 x 224 -> 64 by 7 x 7 at stride 2 142 | 134 |
// 151, 20 x 256 x 193 x 193 -> 16 by 3 x 3 in 4 groups 2216 | 2227 | 1433, 32 x 32 x 64 x 64 -> 32 by 5 x 5 139 | 143 | 95; Float16 8 x 64 x 32^3 -> 64 by 3 x 3 x 3
// 130 | 110 | 146, 13 x 48 x 128 x 128 -> 48 by 5 x 5 in 2 groups 82 | 64 | 57.  (32 x 256 was never the fastest.)
static double dkernel_cost_us(int64_t es, int rows, int cols, int64_t tiles, int64_t K) {
    const double w = (double)((tiles + 255) / 256), k = (double)K;
    if (es == 4) {
        const double alone = rows == 128 ? 0.072 : rows == 32 ? 0.026 : cols == 128 ? 0.040 : 0.025;
        const double each = rows == 128 ? 0.060 : rows == 32 ? 0.0195 : cols == 128 ? 0.033 : 0.0185;
        return 8.0 + k * std::max(alone, each * w);
    }
    const double cu_flops_per_us = 9.77e6, area = (double)rows * cols;
    if (rows == 256) return w * (2.0 * area * k / (cu_flops_per_us * 0.45) + 6.0);
    if (rows == 128) {
        if (tiles <= 256) return 2.0 * area * k / (cu_flops_per_us * 0.27) + 3.0;
        return (double)((tiles + 511) / 512) * (4.0 * area * k / (cu_flops_per_us * 0.41) + 3.0);
    }
    const double alone = cols == 64 || rows == 32 ? 0.0075 : 0.0085, each = cols == 64 ? 0.0035 : rows == 32 ? 0.0046 : 0.0055;
    return 3.0 + k * std::max(alone, each * w);
}
// How dW is cut up: `ranges` k ranges of `kr` output pixels (0: one product per image), tiles of rows x cols, dY read where it
// lies (its rows 16-byte multiples, an image a whole number of K-steps) or through a channels-last copy of its own (any range then), with
// the out channels of a group padded to 16 bytes: rows of zeros that the last pass skips.  Without that padding a layer with odd planes and odd
// channels ran on the element-wise gather, one chain an image: BFloat16 5 x 192 x 125 x 125 -> 48 by one tap in 4 groups, a step 2033 us before, 153 with
// it, Float32 2 x 24 x 63 x 63 transposed to 96 by 4 x 4 in 4 groups 773 | 100, BFloat16 1 x 223 x 223 -> 16 by 5 x 5 1518 | 60.  The partial sums are Float32 whatever the type, so that a 16-bit gradient
// is rounded once (rounded to 16 bits each, they left sqrt(2) of one rounding's error in the sum: BFloat16 2 x 256 x 32 x 32 -> 1024
// channels by 3 x 3 2.45e-3 against 1.66e-3).
// One product per image left a small layer on a handful of workgroups, each with the whole image as its k (3 x 3 x 3 x 32 -> 64
// channels on 4 volumes of 32^3 in Float32: 56 workgroups of 32768 pixels, 1285 us), and a 7 x 7 map of 64 images with 64
// times the partial sums it needs; the ranges are chosen so that tiles x ranges fill whole rounds over the CUs, against the
// cost of writing and reading the partial sums (4 TB/s) and of the copy of dY.
struct DkernelPlan { bool ok, copy_dy; int64_t ranges, kr, items; int rows, cols; };      // rows x cols: the tile
static DkernelPlan plan_dkernel(int dtype, int64_t batch, int64_t channels, int64_t out_channels, int64_t groups, const Geo3& g) {
    DkernelPlan pl;
    std::memset(&pl, 0, sizeof pl);
    if (dtype != ntg::DT_F32 && dtype != ntg::DT_F16 && dtype != ntg::DT_BF16) return pl;
    if (!conv_implicit_g(dtype, channels, g) || out_channels <= 0 || batch <= 0) return pl;
    const int64_t es = ntg::elem_size(dtype), bk = 64 / es, cg = channels / groups, og = out_channels / groups, L = g.L();
    if (g.k[1] * g.d[1] >= 32768 || g.k[2] * g.d[2] >= 32768) return pl;         // tap reach packed in 16 bits
    const int64_t cgp = dkernel_padded_channels(es, cg), N = cgp * g.taps();
    if (cgp > (es == 2 ? 8 : 4) * cg || N >= 0x7fffffffLL || !conv_nhwc_offsets_fit(groups * cgp, es, g)) return pl;
    if (g.nd == 3 && !dkernel_halo(es, cg, groups, g).on) return pl;             // (three axes: the bordered copy is the only form)
    const bool rows_16 = (L * es) % 16 == 0;
    const int64_t ogp = dkernel_padded_channels(es, og);                         // (rows of a copied dY)
    const int64_t total = batch * L, steps = (total + bk - 1) / bk;
    const bool countable = total < (1LL << 30);
    const bool lies = rows_16 && L % bk == 0 && countable, copied = countable;
    if (!rows_16 && !copied) return pl;
    const int64_t volp = dkernel_halo(es, cg, groups, g).vol;
    pl.ok = true;
    // measurement and test knob: NTG_DW_RANGES=r forces r ranges of dY where it lies where r is admissible, 0 one product per image
    const char* env = rows_16 ? std::getenv("NTG_DW_RANGES") : nullptr;
    const int64_t forced = env ? std::atoll(env) : 0;
    if (lies && forced > 0 && steps % forced == 0) {
        pl.ranges = pl.items = forced;
        pl.kr = total / forced;
        pl.rows = pl.cols = es == 2 ? ntg::ring16_tile_edge(og, N, pl.kr, forced) : 64;
    } else {
        // A range has the pixels of an image at least, where those are two to eight K-steps: over small maps ranges of eight are too few (a step of 58 x 64 x 17 -> 64
        // by 5 in 8 groups, in ranges from an image's pixels | from eight K-steps on: BFloat16 23.7 | 25.0 us, Float32 27.4 | 30.4; without groups 24.8 | 26.1, 36.4 |
        // 38.7), while shorter ones gain nothing and ask for a larger workspace than one gradient per image.
        const int64_t shortest = std::min<int64_t>(8, std::max<int64_t>(2, (L + bk - 1) / bk));
        double best = 0.0;
        const auto consider = [&](bool copy, int64_t ranges, int64_t items, int64_t kr, int rows, int cols) {
            const int64_t tiles = ((og + rows - 1) / rows) * ((N + cols - 1) / cols) * items * groups;
            const double us = (copy ? 4.0 + (double)(total * (out_channels + groups * ogp) * es) / 4.5e6 : 0.0) + dkernel_cost_us(es, rows, cols, tiles, kr) + 4.0 +
                              2.0 * (double)(items * groups * (copy ? ogp : og) * N * 4) / 4.0e6;
            if (pl.rows && us >= best) return;
            if ((kr / L + 2) * groups * cgp * volp * es >= (1LL << 36)) return;  // (window origins in 16 bytes from the range's first image: 32 bits)
            best = us;
            pl.copy_dy = copy; pl.ranges = ranges; pl.items = items; pl.kr = kr; pl.rows = rows; pl.cols = cols;
        };
        struct { int rows, cols; } const shapes[] = {{256, 256}, {128, 128}, {64, 64}, {64, 128}, {32, 128}};
        for (const auto [rows, cols] : shapes) {
            if (es == 4 && rows == 256) continue;
            if (rows_16) consider(false, 0, batch, L, rows, cols);
            if (env) continue;
            const int64_t tiles = ((og + rows - 1) / rows) * ((N + cols - 1) / cols) * groups;
            for (int64_t target : {256, 512, 768, 1024, 1536, 2048}) {
                const int64_t want = std::min(std::max<int64_t>(target / tiles, 1), std::max<int64_t>(steps / shortest, 1));
                const int64_t per = (steps + want - 1) / want, r = (steps + per - 1) / per;
                if (lies) consider(false, r, r, per * bk, rows, cols);
                if (copied) consider(true, r, r, per * bk, rows, cols);
            }
        }
        pl.ok = pl.rows != 0;
    }
    return pl;
}
static int64_t conv_dkernel_nhwc_workspace(int dtype, const DkernelPlan& pl, int64_t batch, int64_t channels, int64_t out_channels, int64_t groups, const Geo3& g) {
    const int64_t es = ntg::elem_size(dtype);
    const int64_t rows = pl.copy_dy ? groups * dkernel_padded_channels(es, out_channels / groups) : out_channels;
    const int64_t gy = pl.copy_dy ? (int64_t)align_up((size_t)(batch * rows * g.L() * es), 256) : 0;
    const int64_t cgp = dkernel_padded_channels(es, channels / groups);
    return (int64_t)align_up((size_t)(batch * groups * cgp * dkernel_halo(es, channels / groups, groups, g).vol * es), 256) + gy +
           pl.items * rows * cgp * g.taps() * 4;
}
static int conv_dkernel_nhwc(int dtype, const DkernelPlan& pl, const void* image, const void* grad_out, void* d_kernel, void* ws, int64_t batch,
                             int64_t channels, int64_t out_channels, const Geo3& g, int64_t groups, int accumulate, hipStream_t hs, ntg::ChannelsLast* cl) {
    const int64_t es = ntg::elem_size(dtype), bk = 64 / es, cg = channels / groups, og = out_channels / groups;
    const int64_t cgp = dkernel_padded_channels(es, cg), chp = groups * cgp;      // channels per group / per pixel in the copy
    const int64_t ogr = pl.copy_dy ? dkernel_padded_channels(es, og) : og, rows = groups * ogr;     // rows of a group and in all: a copied dY's are whole 16 bytes
    const int64_t L = g.L(), taps = g.taps(), vol = g.vol(), N = taps * cgp;
    const HaloPlan halo = dkernel_halo(es, cg, groups, g);
    const int64_t volp = halo.vol;                                                         // pixels per image of the copy
    char* ws_img = static_cast<char*>(ws);
    char* ws_gy = ws_img + align_up((size_t)(batch * chp * volp * es), 256);
    char* ws_part = ws_gy + (pl.copy_dy ? align_up((size_t)(batch * rows * L * es), 256) : 0);
    if (cl) {
        add_copy(*cl, image, ws_img, batch, groups, cg, cgp, vol, halo);
        if (pl.copy_dy) cl->copy[cl->n++] = {grad_out, ws_gy, batch, groups, og, ogr, L, false, {}};
        return NTG_OK;
    }
    ntg::GemmParams p;
    std::memset(&p, 0, sizeof p);
    p.M = (int)ogr; p.K = (int)(pl.ranges ? pl.kr : L); p.N = (int)N;
    p.A = pl.copy_dy ? static_cast<const void*>(ws_gy) : grad_out;
    p.lda = pl.copy_dy ? rows : L;
    p.B = ws_img; p.C = ws_part;
    p.ldb = chp; p.ldc = N;
    const int64_t a_item = pl.copy_dy ? pl.kr * rows : pl.ranges ? 0 : out_channels * L;     // (a range: or an image)
    p.cmode = ntg::C_PARTIAL;
    p.vecA_ok = 1; p.vecB_ok = 1;
    fill_conv_geom(p.conv, cgp, halo.gp);
    p.conv.chan = (int)chp;                        // elements from one pixel to the next
    p.conv.halo = halo.on ? 1 : 0;
    p.conv.tile_rows = pl.rows; p.conv.tile_cols = pl.cols;
    p.conv.k_segment = chain_steps(L, groups > 1 ? 8 : 16);
    if (pl.ranges) {
        p.conv.k_ranges = 1;
        p.conv.k_total = (int)(batch * L);
        p.conv.fold_L = (int)L;
        p.conv.div_fold = ntg::make_fastdiv((uint32_t)L);
        p.conv.fold_stride = chp * volp;
        if (!pl.copy_dy) {
            p.conv.a_steps = (int)(L / bk);
            p.conv.div_a_steps = ntg::make_fastdiv((uint32_t)(L / bk));
            p.conv.a_image_stride = out_channels * L;
        }
    }
    hipError_t e = launch_groups(p, dtype, pl.items, groups, {pl.copy_dy ? ogr : og * L, a_item, cgp, pl.ranges ? 0 : chp * volp, ogr * N},
                      [&](const ntg::GemmParams& q) { return ntg::launch_conv_nhwc_dw(dtype, pl.copy_dy, q, hs); });
    if (e != hipSuccess) return hip_fail(e, "channels-last conv_dkernel launch");
    // (groups are consecutive row blocks of both layouts, so one pass covers them all)
    e = ntg::launch_reduce_batch_taps_last(dtype, ws_part, d_kernel, pl.items, rows, og, ogr, cg, cgp, taps, accumulate, hs);
    if (e != hipSuccess) return hip_fail(e, "weight gradient reduction launch");
    return NTG_OK;
}

// The weight gradient from a stored col matrix (integers, complex types, four spatial axes): per group g
//   dW_g [og, add] (+)= sum over the images b of dY_{b,g} [og, L] . col_{b,g}^T   (col_{b,g} stored [add, L]).
// Integers: one accumulating product per (group, image) straight into dW (exact in any order).  Complex types: the
// reference's order, which the results are checked against bit for bit -- every image's product on its own from zero, the
// products added up in batch order in the element type, that sum added to dW last (conv.cpp:444-471: matmult(grad, image,
// false, true).sum(0), then d_kernel +=); the per-image products [B][O][add] lie behind the col matrix in the workspace.
static int64_t complex_dkernel_extra(int dtype, int64_t batch, int64_t out_channels, int64_t add, int64_t col_bytes) {
    if (!is_complex_dtype(dtype)) return 0;
    return (int64_t)(align_up((size_t)col_bytes, 256) - (size_t)col_bytes) + batch * out_channels * add * ntg::elem_size(dtype);
}
static int conv_dkernel_from_col(int dtype, const char* gy, char* col, void* d_kernel, int64_t batch, int64_t out_channels, int64_t ccol,
                                 int64_t groups, int64_t L, int accumulate, void* stream) {
    const int64_t es = ntg::elem_size(dtype), add = ccol / groups, og = out_channels / groups;
    ntg_gemm_desc d;
    int rc = NTG_OK;
    if (is_complex_dtype(dtype)) {
        char* per = col + align_up((size_t)(batch * ccol * L * es), 256);
        for (int64_t g = 0; g < groups && rc == NTG_OK; ++g) {
            std::memset(&d, 0, sizeof d);
            d.dtype = dtype; d.transpose_b = 1; d.c_mode = NTG_C_OVERWRITE;
            d.m = og; d.k = L; d.n = add;
            d.lda = L; d.ldb = L; d.ldc = add; d.batches = batch;
            d.stride_a = out_channels * L; d.stride_b = ccol * L; d.stride_c = out_channels * add;
            rc = ntg_gemm_dev(&d, gy + g * og * L * es, col + g * add * L * es, per + g * og * add * es, stream);
        }
        if (rc) return rc;
        hipError_t e = ntg::launch_reduce_batch(dtype, per, d_kernel, batch, out_channels * add, accumulate, static_cast<hipStream_t>(stream));
        if (e != hipSuccess) return hip_fail(e, "weight gradient reduction launch");
        return NTG_OK;
    }
    for (int64_t g = 0; g < groups; ++g)
        for (int64_t b = 0; b < batch; ++b) {
            std::memset(&d, 0, sizeof d);
            d.dtype = dtype; d.transpose_b = 1;
            d.c_mode = (b == 0 && !accumulate) ? NTG_C_OVERWRITE : NTG_C_ACCUMULATE;
            d.m = og; d.k = L; d.n = add;
            d.lda = L; d.ldb = L; d.ldc = add; d.batches = 1;
            rc = ntg_gemm_dev(&d, gy + ((b * out_channels + g * og) * L) * es, col + ((b * ccol + g * add) * L) * es,
                              static_cast<char*>(d_kernel) + g * og * add * es, stream);
            if (rc) return rc;
        }
    return NTG_OK;
}

// dW of one tap on rows of 16-byte multiples: dY_b . X_b^T per image on the operands where they lie, every image's pixels in `splits` equal ranges of
// whole K-steps so that tiles x images x groups x ranges fill the CUs, the Float32 sums of all of them added up in one pass.  With one range an
// image a few large images were a few workgroups, each a chain of all its pixels (Float16 4 x 128 x 192 x 192 -> 96, a step: 231 us, 56 with
// ranges; Float32 6 x 64 x 5992 -> 32 in 4 groups 299 | 139, 1 x 192 x 112 x 112 -> 48 104 | 37), and 16-bit gradients were rounded once an image.
struct PointwiseDwPlan { int64_t splits, bytes; };                               // splits 0: one product an image in the element type
static PointwiseDwPlan plan_pointwise_dw(int dtype, int64_t batch, int64_t channels, int64_t out_channels, int64_t groups, const Geo3& g) {
    PointwiseDwPlan pl = {0, 0};
    if (dtype != ntg::DT_F32 && dtype != ntg::DT_F16 && dtype != ntg::DT_BF16) return pl;
    const int64_t es = ntg::elem_size(dtype), bk = 64 / es, cg = channels / groups, og = out_channels / groups, L = g.L();
    if (!conv_pointwise_ok(dtype, channels, groups, g) || (og * es) % 16 != 0 || batch <= 0 || og <= 0) return pl;
    const int64_t tiles = ((og + 63) / 64) * ((cg + 63) / 64) * batch * groups;
    if (tiles >= 0x7fffffffLL || L >= 0x7fffffffLL) return pl;
    if (es == 2 && L >= (1 << 23) / es) return pl;       // (the rows are the operands' pitch, and no kernel for pitches from 8 MiB on writes Float32 sums of 16-bit operands)
    if (es == 4 && og <= 32 && batch * groups > NTG_SKINNY_MAX_ITEMS) return pl;
    const uint32_t steps = L % bk == 0 ? (uint32_t)(L / bk) : 1u;
    double best = 0.0;
    const auto consider = [&](uint32_t s) {
        if (s > 1 && tiles * s > 2048) return;           // (eight tiles a CU: more only makes more partial sums)
        const int64_t items = batch * groups * s, K = L / s;
        double us;
        if (es == 2) {
            const int te = ntg::ring16_tile_edge(og, cg, K, items);
            us = ntg::ring16_cost_us(te, ntg::ring16_tiles(te, og, cg, items), K);
        } else {
            us = std::min(ntg::ring_f32_cost(128, og, cg, items), ntg::ring_f32_cost(64, og, cg, items)) * ((double)K * 0.062 + 3.0);
        }
        us += 2.0 * (double)(items * og * cg * 4) / 4.0e6;
        if (pl.splits == 0 || us < best || (us == best && s < pl.splits)) { best = us; pl.splits = s; }
    };
    // (the divisors of steps in pairs: trying every number up to 2048 took 6 us of the host, in the query and in the call)
    for (uint32_t s = 1; (uint64_t)s * s <= steps; ++s) {
        if (steps % s != 0) continue;
        consider(s);
        if (steps / s != s) consider(steps / s);
    }
    pl.bytes = pl.splits * batch * out_channels * cg * 4;
    return pl;
}
static int conv_dkernel_pointwise(int dtype, const PointwiseDwPlan& pl, const void* image, const void* grad_out, void* d_kernel, void* ws, int64_t batch,
                                  int64_t channels, int64_t out_channels, const Geo3& g, int64_t groups, int accumulate, hipStream_t hs) {
    const int64_t cg = channels / groups, og = out_channels / groups, L = g.L();
    ntg::GemmParams p;
    std::memset(&p, 0, sizeof p);
    p.M = (int)og; p.K = (int)(L / pl.splits); p.N = (int)cg;
    p.A = grad_out; p.B = image; p.C = ws;
    p.lda = L; p.ldb = L; p.ldc = cg;
    // launch index = range * (images * groups) + image * groups + group
    p.batch = (int)(batch * groups * pl.splits);
    p.krange_items = (int)(batch * groups);
    p.sA = og * L; p.sB = cg * L; p.sAk = p.sBk = p.K; p.sC = og * cg;
    p.cmode = dtype == ntg::DT_F32 ? ntg::C_OVERWRITE : ntg::C_PARTIAL;
    const int rc = launch_gemm(p, dtype, false, true, hs);
    if (rc) return rc;
    hipError_t e = ntg::launch_reduce_batch_taps_last(dtype, ws, d_kernel, pl.splits * batch, out_channels, og, og, cg, cg, 1, accumulate, hs);
    if (e != hipSuccess) return hip_fail(e, "weight gradient reduction launch");
    return NTG_OK;
}

// Which backward gradients run as implicit GEMMs, and the workspace the call needs.
struct ConvBackwardPlan { bool gather_dw, gather_dx, nhwc_dx, nhwc_dw, phase_dx; int64_t need, need_both, need_nhwc_dx, need_nhwc_dw, need_phase_dx, need_wt_dx, wt_offset; PointwiseDwPlan pointwise; PhasePlan phases; DkernelPlan dkernel; };
// reference_order (Float32 through the host entry points): the forms whose sums are the reference's own, bit for bit -- the
// image gradient as W^T . dY into the col matrix + col2im (conv.cpp:318-346; the implicit forms run one chain over out
// channels and taps where the reference rounds in between), the weight gradient per image with k = the output pixels +
// the sum over the batch (conv.cpp:444-471; not the channels-last kernels, whose partial sums may span images).
static ConvBackwardPlan plan_conv_backward_g(int dtype, bool want_dx, bool want_dw, int64_t batch, int64_t channels, int64_t out_channels,
                                             const Geo3& g, int64_t groups, bool reference_order = false, bool in_place = false) {
    const int64_t es = ntg::elem_size(dtype);
    const int64_t cg = channels / groups, taps = g.taps();
    ConvBackwardPlan pl;
    std::memset(&pl, 0, sizeof pl);
    pl.gather_dw = want_dw && conv_implicit_g(dtype, channels, g);
    pl.gather_dx = want_dx && !reference_order && g.s[0] == 1 && g.s[1] == 1 && g.s[2] == 1 && conv_implicit_g(dtype, out_channels, geo_dimage(g));
    const int64_t col = batch * channels * taps * g.L() * es;
    int64_t need = 0;
    if (want_dw) need = std::max(need, pl.gather_dw ? batch * out_channels * cg * taps * es : col + complex_dkernel_extra(dtype, batch, out_channels, cg * taps, col));
    if (want_dx) need = std::max(need, pl.gather_dx ? out_channels * cg * taps * es : col);
    pl.need = need;
    pl.pointwise = want_dw && !reference_order ? plan_pointwise_dw(dtype, batch, channels, out_channels, groups, g) : PointwiseDwPlan{0, 0};
    if (in_place) return pl;                       // (one tap on operands where they lie: the call takes none of the forms below)
    // the channels-last form of dX is taken when the caller's workspace also holds the copy of dY
    pl.nhwc_dx = pl.gather_dx && conv_dimage_nhwc_ok(dtype, batch, channels, out_channels, groups, g);
    pl.need_nhwc_dx = pl.nhwc_dx ? conv_dimage_nhwc_workspace(dtype, batch, channels, out_channels, groups, g) : 0;
    if (pl.gather_dw && !reference_order) pl.dkernel = plan_dkernel(dtype, batch, channels, out_channels, groups, g);
    pl.nhwc_dw = pl.dkernel.ok;
    pl.need_nhwc_dw = pl.nhwc_dw ? conv_dkernel_nhwc_workspace(dtype, pl.dkernel, batch, channels, out_channels, groups, g) : 0;
    // strides > 1: dX phase by phase instead of GEMM + col2im, again when the workspace allows
    if (want_dx && !pl.gather_dx && !reference_order)
        pl.phases = plan_dimage_phases(dtype, batch, channels, out_channels, groups, g);
    pl.phase_dx = pl.phases.ok;
    pl.need_phase_dx = pl.phase_dx ? pl.phases.bytes() : 0;
    // both channels-last gradients with their copies side by side, made in one launch, as long as that is not much memory (the launch it saves is
    // 1 % of a step from there on)
    const int64_t both = (int64_t)align_up((size_t)pl.need_nhwc_dw, 256) + std::max(pl.need_nhwc_dx, pl.need_phase_dx);
    pl.need_both = pl.nhwc_dw && (pl.nhwc_dx || pl.phase_dx) && both <= (1LL << 26) ? both : 0;
    // strides > 1 on few channels: W^T . dY + col2im.  W_g is stored [og][channels of the group * taps]; where those rows miss the
    // 16-byte rule (3 channels by 7 x 7: 147) the product would run on rows as they lie, so W is copied to [..][og] behind the col matrix
    // and dY and col, whose rows keep the rule, stay where they are.  From 2^30 multiply-adds on, where every layer timed gains; us per backward
    // call as stored | transposed, at n * 2^30 multiply-adds: Float32 3 x 224 x 224 -> 64 by 7 x 7 at stride 2 n = 0.22 57 | 57, 0.44 80 | 73,
    // 1.76 214 | 181, 3.52 405 | 352; 3 x 256 x 256 -> 32 by 5 x 5 0.29 76 | 78, 1.17 237 | 230; BFloat16 0.22 49 | 48, 1.76 213 | 128, 3.52 362 | 209.
    // (The two meet near 0.25: between that and 2^30 the copy would gain up to a third.)
    pl.wt_offset = (int64_t)align_up((size_t)col, 256);
    const int64_t og = out_channels / groups, add = cg * taps;
    const bool wt = want_dx && !pl.gather_dx && !pl.phase_dx && !reference_order && g.nd <= 2 &&
                    (dtype == ntg::DT_F32 || dtype == ntg::DT_F16 || dtype == ntg::DT_BF16) && add > 32 && (add * es) % 16 != 0 && (og * es) % 16 == 0 &&
                    (g.L() * es) % 16 == 0 && (double)batch * (double)(og * add) * (double)g.L() >= 1073741824.0;
    pl.need_wt_dx = wt ? pl.wt_offset + groups * og * add * es : 0;
    return pl;
}

// The gradients that need no col matrix; d_image / d_kernel are set to null when done.  fast: the channels-last forms may be taken.
static int conv_gradients_implicit(int dtype, const ConvBackwardPlan& plan, const void* image, const void* kernel, const void* grad_out, void*& d_image, void*& d_kernel,
                                   char* ws, int64_t ws_bytes, int64_t batch, int64_t channels, int64_t out_channels, const Geo3& g, int64_t groups, int accumulate,
                                   hipStream_t hs, bool fast) {
    fast = fast && (reinterpret_cast<uintptr_t>(ws) & 15) == 0;
    const bool dw = d_kernel && fast && plan.nhwc_dw && ws_bytes >= plan.need_nhwc_dw && (reinterpret_cast<uintptr_t>(grad_out) & 15) == 0;
    const bool dx = d_image && fast && plan.nhwc_dx && ws_bytes >= plan.need_nhwc_dx, dx_phases = d_image && fast && plan.phase_dx && ws_bytes >= plan.need_phase_dx;
    const bool together = dw && (dx || dx_phases) && plan.need_both > 0 && ws_bytes >= plan.need_both;
    char* ws_dx = together ? ws + align_up((size_t)plan.need_nhwc_dw, 256) : ws;
    ntg::ChannelsLast cl;
    std::memset(&cl, 0, sizeof cl);
    const auto dw_part = [&](ntg::ChannelsLast* c) {
        return conv_dkernel_nhwc(dtype, plan.dkernel, image, grad_out, d_kernel, ws, batch, channels, out_channels, g, groups, accumulate, hs, c);
    };
    const auto dx_part = [&](ntg::ChannelsLast* c) {
        return dx ? conv_dimage_nhwc(dtype, kernel, grad_out, d_image, ws_dx, batch, channels, out_channels, g, groups, accumulate, hs, c)
                  : conv_dimage_phases(dtype, plan.phases, kernel, grad_out, d_image, ws_dx, batch, channels, g, groups, accumulate, hs, c);
    };
    const auto copies = [&]() -> int {
        const hipError_t e = ntg::launch_channels_last(ntg::elem_size(dtype), cl, hs);
        return e == hipSuccess ? NTG_OK : hip_fail(e, "channels-last copy launch");
    };
    int rc = NTG_OK;
    if (dw) {
        dw_part(&cl);
        if (together) dx_part(&cl);
        if ((rc = copies()) || (rc = dw_part(nullptr))) return rc;
    } else if (d_kernel && plan.gather_dw) {
        rc = conv_dkernel_gather(dtype, image, grad_out, d_kernel, ws, batch, channels, out_channels, g, groups, accumulate, hs);
        if (rc) return rc;
    }
    if (plan.gather_dw) d_kernel = nullptr;
    if (dx || dx_phases) {
        if (!together) {
            std::memset(&cl, 0, sizeof cl);
            dx_part(&cl);
            if ((rc = copies())) return rc;
        }
        rc = dx_part(nullptr);
        d_image = nullptr;
    } else if (d_image && plan.gather_dx) {
        rc = conv_dimage_gather(dtype, kernel, grad_out, d_image, ws, batch, channels, out_channels, g, groups, accumulate, hs);
        d_image = nullptr;
    }
    return rc;
}

int64_t ntg_conv2d_fast_workspace_bytes(int dtype, int64_t batch, int64_t channels, int64_t height, int64_t width,
                                        int64_t out_channels, int64_t k_r, int64_t k_c, int64_t s_r, int64_t s_c,
                                        int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c, int64_t groups) {
    const int64_t es = ntg::elem_size(dtype);
    int64_t Ho, Wo;
    if (es == 0 || unfold_out(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo)) return -1;
    const Geo3 g = geo2(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo);
    const bool groups_ok = groups >= 1 && channels % groups == 0 && out_channels % groups == 0;      // (the call itself reports bad groups)
    if (groups_ok && conv_pointwise_ok(dtype, channels, groups, g)) return 0;
    MergedTaps mt;
    if (groups_ok && conv_nhwc_merged(dtype, batch, channels, out_channels, groups, g, mt)) return conv_nhwc_merged_workspace(dtype, batch, out_channels, groups, g, mt);
    if (groups_ok && conv_nhwc_ok(dtype, batch, channels, out_channels, groups, g)) return conv_nhwc_workspace(dtype, batch, channels, out_channels, groups, g);
    return ntg_conv2d_forward_workspace_bytes(dtype, batch, channels, height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c);
}

int64_t ntg_conv2d_forward_workspace_bytes(int dtype, int64_t batch, int64_t channels, int64_t height, int64_t width,
                                           int64_t k_r, int64_t k_c, int64_t s_r, int64_t s_c,
                                           int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c) {
    const int64_t es = ntg::elem_size(dtype);
    int64_t Ho, Wo;
    if (es == 0 || unfold_out(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo)) return -1;
    if (conv_implicit(dtype, channels, height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo)) return 0;
    if (conv_pointwise(geo2(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo))) return 0;
    return batch * channels * k_r * k_c * Ho * Wo * es;
}

int64_t ntg_conv2d_workspace_bytes(int dtype, int64_t batch, int64_t channels, int64_t height, int64_t width,
                                   int64_t k_r, int64_t k_c, int64_t s_r, int64_t s_c,
                                   int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c) {
    const int64_t es = ntg::elem_size(dtype);
    int64_t Ho, Wo;
    if (es == 0 || unfold_out(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo)) return -1;
    return batch * channels * k_r * k_c * Ho * Wo * es;
}

static int conv2d_dev_impl(int dtype, const void* image, const void* kernel, void* out,
                   void* workspace, int64_t workspace_bytes,
                   int64_t batch, int64_t channels, int64_t height, int64_t width,
                   int64_t out_channels, int64_t k_r, int64_t k_c,
                   int64_t s_r, int64_t s_c, int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c,
                   int64_t groups, void* stream, bool reference_order) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    if (batch < 0 || channels < 0 || out_channels < 0 || height < 0 || width < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "negative size");
    if (groups < 1) return fail(NTG_ERR_INVALID_ARGUMENT, "groups must be >= 1");
    // conv.cpp:97-98
    if (channels % groups != 0) return fail(NTG_ERR_INVALID_ARGUMENT, "image channels (%lld) not divisible by groups (%lld)", (long long)channels, (long long)groups);
    if (out_channels % groups != 0) return fail(NTG_ERR_INVALID_ARGUMENT, "out channels (%lld) not divisible by groups (%lld)", (long long)out_channels, (long long)groups);
    int64_t Ho, Wo;
    int rc = unfold_out(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo);
    if (rc) return rc;
    if (batch == 0 || out_channels == 0) return NTG_OK;
    if (!image || !kernel || !out) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer");
    const int64_t L = Ho * Wo, ckk = channels * k_r * k_c;
    const int64_t add = (channels / groups) * k_r * k_c, og = out_channels / groups;
    {
        const Geo3 g = geo2(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo);
        if (conv_pointwise_ok(dtype, channels, groups, g) &&
            (is_valu_dtype(dtype) || ((reinterpret_cast<uintptr_t>(image) | reinterpret_cast<uintptr_t>(kernel) | reinterpret_cast<uintptr_t>(out)) & 15) == 0))
            return conv_forward_pointwise(dtype, image, kernel, out, batch, channels, out_channels, g, groups, stream, reference_order);
        // with the workspace of ntg_conv2d_fast_workspace_bytes: channels-last copy of the image, 16-byte gathers
        MergedTaps mt;
        if (conv_nhwc_merged(dtype, batch, channels, out_channels, groups, g, mt) && workspace && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0 &&
            workspace_bytes >= conv_nhwc_merged_workspace(dtype, batch, out_channels, groups, g, mt))
            return conv_forward_nhwc(dtype, image, kernel, out, workspace, batch, channels, out_channels, g, groups, static_cast<hipStream_t>(stream), &mt);
        if (conv_nhwc_ok(dtype, batch, channels, out_channels, groups, g) && workspace && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0 &&
            workspace_bytes >= conv_nhwc_workspace(dtype, batch, channels, out_channels, groups, g))
            return conv_forward_nhwc(dtype, image, kernel, out, workspace, batch, channels, out_channels, g, groups, static_cast<hipStream_t>(stream));
        if (conv_implicit_g(dtype, channels, g))      // col_b is never stored: the GEMM's B loader gathers it from the image
            return conv_forward_gather(dtype, image, kernel, out, batch, channels, out_channels, g, groups, static_cast<hipStream_t>(stream));
    }
    const int64_t need = batch * channels * k_r * k_c * Ho * Wo * es;
    if (need > 0 && (!workspace || workspace_bytes < need))
        return fail(NTG_ERR_INVALID_ARGUMENT, "workspace of %lld bytes needed, %lld given", (long long)need, (long long)workspace_bytes);
    rc = ntg_unfold2d_dev(dtype, image, workspace, batch, channels, height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, stream);
    if (rc) return rc;
    for (int64_t g = 0; g < groups; ++g) {
        ntg_gemm_desc d;
        std::memset(&d, 0, sizeof d);
        d.dtype = dtype; d.c_mode = NTG_C_OVERWRITE;
        d.m = og; d.k = add; d.n = L;
        d.lda = add; d.ldb = L; d.ldc = L;
        d.batches = batch;
        d.stride_a = 0; d.stride_b = ckk * L; d.stride_c = out_channels * L;
        rc = ntg_gemm_dev(&d, static_cast<const char*>(kernel) + g * og * add * es,
                          static_cast<const char*>(workspace) + g * add * L * es,
                          static_cast<char*>(out) + g * og * L * es, stream);
        if (rc) return rc;
    }
    return NTG_OK;
}

int ntg_conv2d_dev(int dtype, const void* image, const void* kernel, void* out,
                   void* workspace, int64_t workspace_bytes,
                   int64_t batch, int64_t channels, int64_t height, int64_t width,
                   int64_t out_channels, int64_t k_r, int64_t k_c,
                   int64_t s_r, int64_t s_c, int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c,
                   int64_t groups, void* stream) {
    return conv2d_dev_impl(dtype, image, kernel, out, workspace, workspace_bytes, batch, channels, height, width, out_channels, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c,
                           groups, stream, false);
}

int ntg_conv2d(int dtype, const void* image, const void* kernel, void* out,
               int64_t batch, int64_t channels, int64_t height, int64_t width,
               int64_t out_channels, int64_t k_r, int64_t k_c,
               int64_t s_r, int64_t s_c, int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c,
               int64_t groups) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    if (batch < 0 || channels < 0 || out_channels < 0 || height < 0 || width < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "negative size");
    if (groups < 1 || channels % groups != 0 || out_channels % groups != 0)
        return fail(NTG_ERR_INVALID_ARGUMENT, "channels (%lld) and out channels (%lld) must be divisible by groups (%lld)",
                    (long long)channels, (long long)out_channels, (long long)groups);
    int64_t Ho, Wo;
    int rc = unfold_out(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo);
    if (rc) return rc;
    if (batch == 0 || out_channels == 0) return NTG_OK;
    if (!image || !kernel || !out) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer");
    const size_t im_bytes = (size_t)(batch * channels * height * width * es);
    const size_t k_bytes = (size_t)(out_channels * (channels / groups) * k_r * k_c * es);
    const size_t o_bytes = (size_t)(batch * out_channels * Ho * Wo * es);
    // Float32 at the reference's seam: the gathering kernels (no workspace), whose k axis is im2col's own -- the result is
    // unfold + matmult bit for bit (conv.cpp:86-95); the channels-last kernels sum the same products taps-outermost, and what
    // they would gain is small beside the transfers of this call.  The other dtypes take the faster form.
    const int64_t ws = dtype == ntg::DT_F32
        ? ntg_conv2d_forward_workspace_bytes(dtype, batch, channels, height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c)
        : ntg_conv2d_fast_workspace_bytes(dtype, batch, channels, height, width, out_channels, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, groups);
    if (ws < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "the array of sliding blocks would be empty");
    ntg::HostSession mem;
    const size_t ok_ = align_up(im_bytes, 256), oo = ok_ + align_up(k_bytes, 256), ow = oo + align_up(o_bytes, 256);
    HIP_TRY(mem.reserve(ow + (size_t)ws));
    if (im_bytes) HIP_TRY(mem.upload(0, image, im_bytes));
    if (k_bytes) HIP_TRY(mem.upload(ok_, kernel, k_bytes));
    rc = conv2d_dev_impl(dtype, mem.at(0), mem.at(ok_), mem.at(oo), mem.at(ow), ws, batch, channels, height, width,
                         out_channels, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, groups, mem.stream(), dtype == ntg::DT_F32);
    if (rc) return rc;
    HIP_TRY(mem.download(out, oo, o_bytes));
    return NTG_OK;
}

int ntg_unfold2d_backward_dev(int dtype, const void* col, void* image,
                              int64_t batch, int64_t channels, int64_t height, int64_t width,
                              int64_t k_r, int64_t k_c, int64_t s_r, int64_t s_c,
                              int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c, int accumulate, void* stream) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    if (batch < 0 || channels < 0 || height < 0 || width < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "negative size");
    int64_t Ho, Wo;
    int rc = unfold_out(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo);
    if (rc) return rc;
    if (batch == 0 || channels == 0) return NTG_OK;
    if (!col || !image) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer");
    hipError_t e = ntg::launch_col2im(dtype, col, image, batch, channels, height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c,
                                      accumulate, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return hip_fail(e, "col2im launch");
    return NTG_OK;
}

int ntg_unfold2d_backward(int dtype, const void* col, void* image,
                          int64_t batch, int64_t channels, int64_t height, int64_t width,
                          int64_t k_r, int64_t k_c, int64_t s_r, int64_t s_c,
                          int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c, int accumulate) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    if (batch < 0 || channels < 0 || height < 0 || width < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "negative size");
    int64_t Ho, Wo;
    int rc = unfold_out(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo);
    if (rc) return rc;
    if (batch == 0 || channels == 0) return NTG_OK;
    if (!col || !image) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer");
    const size_t im_bytes = (size_t)(batch * channels * height * width * es);
    const size_t col_bytes = (size_t)(batch * channels * k_r * k_c * Ho * Wo * es);
    ntg::HostSession mem;
    const size_t oc = align_up(im_bytes, 256);
    HIP_TRY(mem.reserve(oc + col_bytes));
    if (accumulate) HIP_TRY(mem.upload(0, image, im_bytes));
    HIP_TRY(mem.upload(oc, col, col_bytes));
    rc = ntg_unfold2d_backward_dev(dtype, mem.at(oc), mem.at(0), batch, channels, height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c,
                                   accumulate, mem.stream());
    if (rc) return rc;
    HIP_TRY(mem.download(image, 0, im_bytes));
    return NTG_OK;
}

static ConvBackwardPlan plan_conv_backward(int dtype, bool want_dx, bool want_dw, int64_t batch, int64_t channels, int64_t height, int64_t width,
                                           int64_t out_channels, int64_t k_r, int64_t k_c, int64_t s_r, int64_t s_c, int64_t p_r, int64_t p_c,
                                           int64_t d_r, int64_t d_c, int64_t groups, int64_t Ho, int64_t Wo, bool reference_order = false, bool in_place = false) {
    return plan_conv_backward_g(dtype, want_dx, want_dw, batch, channels, out_channels,
                                geo2(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo), groups, reference_order, in_place);
}

int64_t ntg_conv2d_backward_workspace_bytes(int dtype, int64_t batch, int64_t channels, int64_t height, int64_t width,
                                            int64_t out_channels, int64_t k_r, int64_t k_c, int64_t s_r, int64_t s_c,
                                            int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c, int64_t groups) {
    int64_t Ho, Wo;
    if (ntg::elem_size(dtype) == 0 || groups < 1 || channels % groups != 0 || out_channels % groups != 0 ||
        unfold_out(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo)) return -1;
    // the larger of what the call needs at least and what lets dX take its channels-last form (copy of dY + flipped weights)
    const ConvBackwardPlan pl = plan_conv_backward(dtype, true, true, batch, channels, height, width, out_channels, k_r, k_c, s_r, s_c, p_r, p_c,
                                                   d_r, d_c, groups, Ho, Wo);
    return std::max({pl.need, pl.need_phase_dx, pl.need_wt_dx, pl.need_nhwc_dx, pl.need_nhwc_dw, pl.need_both, pl.pointwise.bytes});
}

static int conv2d_backward_dev_impl(int dtype, const void* image, const void* kernel, const void* grad_out,
                                    void* d_image, void* d_kernel, void* workspace, int64_t workspace_bytes,
                                    int64_t batch, int64_t channels, int64_t height, int64_t width,
                                    int64_t out_channels, int64_t k_r, int64_t k_c,
                                    int64_t s_r, int64_t s_c, int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c,
                                    int64_t groups, int accumulate, void* stream, bool reference_order) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    if (batch < 0 || channels < 0 || out_channels < 0 || height < 0 || width < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "negative size");
    if (groups < 1 || channels % groups != 0 || out_channels % groups != 0)
        return fail(NTG_ERR_INVALID_ARGUMENT, "channels (%lld) and out channels (%lld) must be divisible by groups (%lld)",
                    (long long)channels, (long long)out_channels, (long long)groups);
    int64_t Ho, Wo;
    int rc = unfold_out(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo);
    if (rc) return rc;
    if (batch == 0 || out_channels == 0 || channels == 0) return NTG_OK;
    if (!kernel || !grad_out || (d_kernel && !image)) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer");
    const int64_t L = Ho * Wo, ckk = channels * k_r * k_c;
    const int64_t add = (channels / groups) * k_r * k_c, og = out_channels / groups;
    const Geo3 geo = geo2(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo);
    // 1x1 kernel, unit stride, no padding (floating dtypes, 16-byte rows): col is the image itself, so both gradients are
    // products on the tensors where they lie: dX_b = W_g^T . dY_b, and dW_g = sum_b dY_b . X_b^T through per-image results
    // in the workspace (the amount the gathering form needs), summed in batch order, or through those of ranges of the images' pixels.
    const bool in_place = !is_valu_dtype(dtype) && !(reference_order && accumulate) && conv_pointwise_ok(dtype, channels, groups, geo) && (og * es) % 16 == 0 &&
                          ((reinterpret_cast<uintptr_t>(image) | reinterpret_cast<uintptr_t>(kernel) | reinterpret_cast<uintptr_t>(grad_out) |
                            reinterpret_cast<uintptr_t>(d_image) | reinterpret_cast<uintptr_t>(d_kernel) | reinterpret_cast<uintptr_t>(workspace)) & 15) == 0;
    const ConvBackwardPlan plan = plan_conv_backward(dtype, d_image != nullptr, d_kernel != nullptr, batch, channels, height, width,
                                                     out_channels, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, groups, Ho, Wo, reference_order, in_place);
    if (plan.need > 0 && (!workspace || workspace_bytes < plan.need))
        return fail(NTG_ERR_INVALID_ARGUMENT, "workspace of %lld bytes needed, %lld given", (long long)plan.need, (long long)workspace_bytes);
    const char* kern = static_cast<const char*>(kernel);
    const char* gy = static_cast<const char*>(grad_out);
    char* ws = static_cast<char*>(workspace);
    hipStream_t hs = static_cast<hipStream_t>(stream);
    ntg_gemm_desc d;
    if (in_place) {
        const int64_t cg = channels / groups;
        if (d_image) {
            rc = gemm_per_group(dtype, true, false, accumulate ? NTG_C_ACCUMULATE : NTG_C_OVERWRITE, cg, og, L, cg, L, L, batch, groups, kern, og * cg, 0,
                                gy, og * L, out_channels * L, d_image, stream, reference_order);
            if (rc) return rc;
        }
        if (d_kernel && plan.pointwise.splits > 0 && workspace_bytes >= plan.pointwise.bytes)
            return conv_dkernel_pointwise(dtype, plan.pointwise, image, grad_out, d_kernel, ws, batch, channels, out_channels, geo, groups, accumulate, hs);
        if (d_kernel) {
            rc = gemm_per_group(dtype, false, true, NTG_C_OVERWRITE, og, L, cg, L, L, cg, batch, groups, gy, og * L, out_channels * L,
                                image, cg * L, channels * L, ws, stream, reference_order);
            if (rc) return rc;
        }
        if (d_kernel) {
            hipError_t e = ntg::launch_reduce_batch(dtype, ws, d_kernel, batch, out_channels * cg, accumulate, hs);
            if (e != hipSuccess) return hip_fail(e, "weight gradient reduction launch");
        }
        return NTG_OK;
    }
    rc = conv_gradients_implicit(dtype, plan, image, kernel, grad_out, d_image, d_kernel, ws, workspace_bytes, batch, channels, out_channels, geo, groups, accumulate, hs, true);
    if (rc) return rc;
    if (d_kernel) {
        // col = im2col(image); per group g:  dW_g [og, add] (+)= sum_b dY_{b,g} [og, L] . col_{b,g}^T  (col_{b,g} stored [add, L])
        rc = ntg_unfold2d_dev(dtype, image, ws, batch, channels, height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, stream);
        if (rc) return rc;
        rc = conv_dkernel_from_col(dtype, gy, ws, d_kernel, batch, out_channels, ckk, groups, L, accumulate, stream);
        if (rc) return rc;
    }
    if (d_image) {
        // d_col_{b,g} [add, L] = W_g^T . dY_{b,g}   (W_g stored [og, add] -> transpose_a, or its copy [add, og]), then col2im
        const bool wt = plan.need_wt_dx > 0 && workspace_bytes >= plan.need_wt_dx &&
                        ((reinterpret_cast<uintptr_t>(ws) | reinterpret_cast<uintptr_t>(grad_out)) & 15) == 0;
        if (wt) {
            ntg::ChannelsLast cl;
            std::memset(&cl, 0, sizeof cl);
            cl.copy[cl.n++] = {kern, ws + plan.wt_offset, groups, 1, og, og, add, false, {}};
            const hipError_t e = ntg::launch_channels_last(es, cl, hs);
            if (e != hipSuccess) return hip_fail(e, "transposed weights launch");
        }
        rc = gemm_per_group(dtype, !wt, false, NTG_C_OVERWRITE, add, og, L, wt ? og : add, L, L, batch, groups, wt ? ws + plan.wt_offset : kern, og * add, 0,
                            gy, og * L, out_channels * L, ws, stream, reference_order);
        if (rc) return rc;
        rc = ntg_unfold2d_backward_dev(dtype, ws, d_image, batch, channels, height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c,
                                       accumulate, stream);
        if (rc) return rc;
    }
    return NTG_OK;
}

int ntg_conv2d_backward_dev(int dtype, const void* image, const void* kernel, const void* grad_out,
                            void* d_image, void* d_kernel, void* workspace, int64_t workspace_bytes,
                            int64_t batch, int64_t channels, int64_t height, int64_t width,
                            int64_t out_channels, int64_t k_r, int64_t k_c,
                            int64_t s_r, int64_t s_c, int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c,
                            int64_t groups, int accumulate, void* stream) {
    return conv2d_backward_dev_impl(dtype, image, kernel, grad_out, d_image, d_kernel, workspace, workspace_bytes, batch, channels, height, width,
                                    out_channels, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, groups, accumulate, stream, false);
}

// conv_transpose2d = the image gradient of the convolution whose output is `input`: per group
// out_g [cog, Rout*Cout] = flipped, channel-swapped kernel . unfold(zero-dilated input), which is what
// the reference forms explicitly (conv.cpp:614-676: dilate by stride, pad by output_padding, unfold2d
// with padding d*(k-1) - p and stride 1, matmult with w.transpose(0,1).flip).  Here it is the
// conv_dimage path of ntg_conv2d_backward_dev with the roles renamed; kernel is [in_channels,
// out_channels/groups, k_r, k_c] as in the reference.
static int conv_transpose_out(int64_t in_h, int64_t in_w, int64_t k_r, int64_t k_c, int64_t s_r, int64_t s_c, int64_t p_r, int64_t p_c,
                              int64_t d_r, int64_t d_c, int64_t op_r, int64_t op_c, int64_t& out_h, int64_t& out_w) {
    if (k_r < 1 || k_c < 1) return fail(NTG_ERR_INVALID_ARGUMENT, "kernel size must be >= 1");
    if (s_r < 1 || s_c < 1) return fail(NTG_ERR_INVALID_ARGUMENT, "Conv2d Transpose stride cannot be less than 1 but got (%lld, %lld)", (long long)s_r, (long long)s_c);
    if (d_r < 1 || d_c < 1) return fail(NTG_ERR_INVALID_ARGUMENT, "Conv2d Transpose dilation cannot be less than 1 but got (%lld, %lld)", (long long)d_r, (long long)d_c);
    if (p_r < 0 || p_c < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "Conv2d Transpose padding cannot be less than 0 but got (%lld, %lld)", (long long)p_r, (long long)p_c);
    if (op_r < 0 || op_c < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "Conv2d Transpose output_padding cannot be less than 0 but got (%lld, %lld)", (long long)op_r, (long long)op_c);
    // the reference accepts any output_padding; rows past the reach of the kernel would be zero.  This backend needs the
    // forward convolution of the result to reproduce the input size, which holds for output_padding < stride.
    if (op_r >= s_r || op_c >= s_c) return fail(NTG_ERR_INVALID_ARGUMENT, "output_padding (%lld, %lld) must be smaller than stride (%lld, %lld)",
                                                (long long)op_r, (long long)op_c, (long long)s_r, (long long)s_c);
    if (in_h < 1 || in_w < 1) return fail(NTG_ERR_INVALID_ARGUMENT, "empty input");
    out_h = (in_h - 1) * s_r - 2 * p_r + d_r * (k_r - 1) + 1 + op_r;
    out_w = (in_w - 1) * s_c - 2 * p_c + d_c * (k_c - 1) + 1 + op_c;
    if (out_h < 1 || out_w < 1) return fail(NTG_ERR_INVALID_ARGUMENT, "the output of the transposed convolution would be empty");
    // a padding wider than the kernel reach would make the matching convolution read fewer input rows than exist
    if ((out_h + 2 * p_r - d_r * (k_r - 1) - 1) / s_r + 1 != in_h || (out_w + 2 * p_c - d_c * (k_c - 1) - 1) / s_c + 1 != in_w)
        return fail(NTG_ERR_INVALID_ARGUMENT, "geometry is not the transpose of a convolution");
    return NTG_OK;
}

int64_t ntg_conv_transpose2d_workspace_bytes(int dtype, int64_t batch, int64_t in_channels, int64_t in_h, int64_t in_w,
                                             int64_t out_channels, int64_t k_r, int64_t k_c, int64_t s_r, int64_t s_c,
                                             int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c, int64_t op_r, int64_t op_c, int64_t groups) {
    int64_t oh, ow, Ho, Wo;
    if (ntg::elem_size(dtype) == 0 || groups < 1 || in_channels % groups != 0 || out_channels % groups != 0 ||
        conv_transpose_out(in_h, in_w, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, op_r, op_c, oh, ow) ||
        unfold_out(oh, ow, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo)) return -1;
    const ConvBackwardPlan pl = plan_conv_backward(dtype, true, false, batch, out_channels, oh, ow, in_channels, k_r, k_c, s_r, s_c, p_r, p_c,
                                                   d_r, d_c, groups, Ho, Wo);
    return std::max(pl.need, std::max(pl.need_nhwc_dx, pl.need_phase_dx));      // (the larger amount lets it run channels-last)
}

int ntg_conv_transpose2d_dev(int dtype, const void* input, const void* kernel, void* out, void* workspace, int64_t workspace_bytes,
                             int64_t batch, int64_t in_channels, int64_t in_h, int64_t in_w, int64_t out_channels,
                             int64_t k_r, int64_t k_c, int64_t s_r, int64_t s_c, int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c,
                             int64_t op_r, int64_t op_c, int64_t groups, void* stream) {
    if (ntg::elem_size(dtype) == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    if (batch < 0 || in_channels < 0 || out_channels < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "negative size");
    if (groups < 1) return fail(NTG_ERR_INVALID_ARGUMENT, "groups must be >= 1");
    if (in_channels % groups != 0)
        return fail(NTG_ERR_INVALID_ARGUMENT, "Expected image channels to be divisible by groups in Conv2d Transpose but got %lld %% %lld != 0",
                    (long long)in_channels, (long long)groups);
    if (out_channels % groups != 0) return fail(NTG_ERR_INVALID_ARGUMENT, "out channels (%lld) not divisible by groups (%lld)", (long long)out_channels, (long long)groups);
    int64_t oh, ow;
    int rc = conv_transpose_out(in_h, in_w, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, op_r, op_c, oh, ow);
    if (rc) return rc;
    if (batch == 0 || out_channels == 0) return NTG_OK;
    if (in_channels == 0) {
        hipError_t e = ntg::launch_col2im(dtype, nullptr, out, batch, out_channels, oh, ow, 0, 0, 1, 1, 0, 0, 1, 1, 0, static_cast<hipStream_t>(stream));
        if (e != hipSuccess) return hip_fail(e, "zero fill");
        return NTG_OK;
    }
    return ntg_conv2d_backward_dev(dtype, nullptr, kernel, input, out, nullptr, workspace, workspace_bytes, batch, out_channels, oh, ow,
                                   in_channels, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, groups, 0, stream);
}

int ntg_conv_transpose2d(int dtype, const void* input, const void* kernel, void* out,
                         int64_t batch, int64_t in_channels, int64_t in_h, int64_t in_w, int64_t out_channels,
                         int64_t k_r, int64_t k_c, int64_t s_r, int64_t s_c, int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c,
                         int64_t op_r, int64_t op_c, int64_t groups) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    if (batch < 0 || in_channels < 0 || out_channels < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "negative size");
    if (groups < 1 || in_channels % groups != 0 || out_channels % groups != 0)
        return fail(NTG_ERR_INVALID_ARGUMENT, "channels (%lld) and out channels (%lld) must be divisible by groups (%lld)",
                    (long long)in_channels, (long long)out_channels, (long long)groups);
    int64_t oh, ow;
    int rc = conv_transpose_out(in_h, in_w, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, op_r, op_c, oh, ow);
    if (rc) return rc;
    if (batch == 0 || out_channels == 0) return NTG_OK;
    if (!input || !kernel || !out) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer");
    const size_t in_bytes = (size_t)(batch * in_channels * in_h * in_w * es);
    const size_t k_bytes = (size_t)(in_channels * (out_channels / groups) * k_r * k_c * es);
    const size_t o_bytes = (size_t)(batch * out_channels * oh * ow * es);
    const int64_t wsb = ntg_conv_transpose2d_workspace_bytes(dtype, batch, in_channels, in_h, in_w, out_channels, k_r, k_c, s_r, s_c,
                                                             p_r, p_c, d_r, d_c, op_r, op_c, groups);
    if (wsb < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "invalid geometry");
    ntg::HostSession mem;
    const size_t o_k = align_up(in_bytes, 256), o_o = o_k + align_up(k_bytes, 256), o_ws = o_o + align_up(o_bytes, 256);
    HIP_TRY(mem.reserve(o_ws + (size_t)wsb));
    if (in_bytes) HIP_TRY(mem.upload(0, input, in_bytes));
    if (k_bytes) HIP_TRY(mem.upload(o_k, kernel, k_bytes));
    rc = ntg_conv_transpose2d_dev(dtype, mem.at(0), mem.at(o_k), mem.at(o_o), mem.at(o_ws), wsb, batch, in_channels, in_h, in_w, out_channels,
                                  k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, op_r, op_c, groups, mem.stream());
    if (rc) return rc;
    HIP_TRY(mem.download(out, o_o, o_bytes));
    return NTG_OK;
}

int ntg_conv2d_backward(int dtype, const void* image, const void* kernel, const void* grad_out,
                        void* d_image, void* d_kernel,
                        int64_t batch, int64_t channels, int64_t height, int64_t width,
                        int64_t out_channels, int64_t k_r, int64_t k_c,
                        int64_t s_r, int64_t s_c, int64_t p_r, int64_t p_c, int64_t d_r, int64_t d_c,
                        int64_t groups, int accumulate) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    if (batch < 0 || channels < 0 || out_channels < 0 || height < 0 || width < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "negative size");
    if (groups < 1 || channels % groups != 0 || out_channels % groups != 0)
        return fail(NTG_ERR_INVALID_ARGUMENT, "channels (%lld) and out channels (%lld) must be divisible by groups (%lld)",
                    (long long)channels, (long long)out_channels, (long long)groups);
    int64_t Ho, Wo;
    int rc = unfold_out(height, width, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, Ho, Wo);
    if (rc) return rc;
    if (batch == 0 || out_channels == 0 || channels == 0) return NTG_OK;
    if (!image || !kernel || !grad_out) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer");
    const size_t im_bytes = (size_t)(batch * channels * height * width * es);
    const size_t k_bytes = (size_t)(out_channels * (channels / groups) * k_r * k_c * es);
    const size_t g_bytes = (size_t)(batch * out_channels * Ho * Wo * es);
    // Float32 at the reference's seam: its own two algorithms (see plan_conv_backward_g), whose results are conv_dimage's and
    // conv_dkernel's bit for bit; what the faster forms would gain is small beside the transfers of this call
    const bool reference_order = dtype == ntg::DT_F32;
    const int64_t wsb = reference_order
        ? plan_conv_backward(dtype, d_image != nullptr, d_kernel != nullptr, batch, channels, height, width, out_channels, k_r, k_c, s_r, s_c,
                             p_r, p_c, d_r, d_c, groups, Ho, Wo, true).need
        : ntg_conv2d_backward_workspace_bytes(dtype, batch, channels, height, width, out_channels, k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, groups);
    ntg::HostSession mem;
    const size_t o_k = align_up(im_bytes, 256), o_g = o_k + align_up(k_bytes, 256), o_di = o_g + align_up(g_bytes, 256);
    const size_t o_dk = o_di + align_up(im_bytes, 256), o_ws = o_dk + align_up(k_bytes, 256);
    HIP_TRY(mem.reserve(o_ws + (size_t)wsb));
    HIP_TRY(mem.upload(0, image, im_bytes));
    HIP_TRY(mem.upload(o_k, kernel, k_bytes));
    HIP_TRY(mem.upload(o_g, grad_out, g_bytes));
    if (accumulate && d_image) HIP_TRY(mem.upload(o_di, d_image, im_bytes));
    if (accumulate && d_kernel) HIP_TRY(mem.upload(o_dk, d_kernel, k_bytes));
    rc = conv2d_backward_dev_impl(dtype, mem.at(0), mem.at(o_k), mem.at(o_g), d_image ? mem.at(o_di) : nullptr,
                                  d_kernel ? mem.at(o_dk) : nullptr, mem.at(o_ws), wsb, batch, channels, height, width, out_channels,
                                  k_r, k_c, s_r, s_c, p_r, p_c, d_r, d_c, groups, accumulate, mem.stream(), reference_order);
    if (rc) return rc;
    if (d_image) HIP_TRY(mem.download(d_image, o_di, im_bytes));
    if (d_kernel) HIP_TRY(mem.download(d_kernel, o_dk, k_bytes));
    return NTG_OK;
}

// ---------------------------------------------------------------------------------------------------
// Convolutions over 1..4 spatial axes (conv3d conv.cpp:122-175, convnd :177-316, their gradients :347, :472 and
// conv_transpose3d / conv_transposend :678-905): unfold -> matmult like the reference.  One and two axes go to
// the 2-d entry points above (implicit GEMM); three and four axes store the unfolded matrix.
// Geometry arrays hold `ndim` entries, slowest axis first (depth, rows, columns).
static int fill_nd(ntg::UnfoldNdParams& u, int64_t batch, int64_t channels, int ndim, const int64_t* size, const int64_t* k,
                   const int64_t* s, const int64_t* p, const int64_t* d) {
    if (ndim < 1 || ndim > NTG_MAX_SPATIAL) return fail(NTG_ERR_INVALID_ARGUMENT, "ndim must be 1..%d but got %d", NTG_MAX_SPATIAL, ndim);
    if (!size || !k || !s || !p || !d) return fail(NTG_ERR_INVALID_ARGUMENT, "null geometry array");
    if (batch < 0 || channels < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "negative size");
    std::memset(&u, 0, sizeof u);
    u.nd = ndim; u.batch = batch; u.channels = channels;
    u.taps = 1; u.L = 1; u.vol = 1;
    for (int a = 0; a < ndim; ++a) {
        if (size[a] < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "negative size");
        if (k[a] < 1 || s[a] < 1 || d[a] < 1 || p[a] < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "kernel/stride/dilation must be >= 1 and padding >= 0");
        const int64_t span = size[a] + 2 * p[a] - d[a] * (k[a] - 1) - 1;
        const int64_t o = span / s[a] + 1;
        if (span < 0 || o <= 0) return fail(NTG_ERR_INVALID_ARGUMENT, "the array of sliding blocks would be empty (axis %d)", a);
        u.size[a] = size[a]; u.k[a] = k[a]; u.s[a] = s[a]; u.p[a] = p[a]; u.d[a] = d[a]; u.out[a] = o;
        u.taps *= k[a]; u.L *= o; u.vol *= size[a];
    }
    u.ccol = channels * u.taps;
    u.total = batch * u.ccol * u.L;
    return NTG_OK;
}

// trailing two axes of a 1- or 2-axis geometry as (rows, columns) for the 2-d entry points
struct Geo2 { int64_t h, w, kr, kc, sr, sc, pr, pc, dr, dc; };
static Geo2 as_2d(int ndim, const int64_t* size, const int64_t* k, const int64_t* s, const int64_t* p, const int64_t* d) {
    if (ndim == 1) return {1, size[0], 1, k[0], 1, s[0], 0, p[0], 1, d[0]};
    return {size[0], size[1], k[0], k[1], s[0], s[1], p[0], p[1], d[0], d[1]};
}

static Geo3 geo_from(const ntg::UnfoldNdParams& u) {
    Geo3 g{3, {1, 1, 1}, {1, 1, 1}, {1, 1, 1}, {0, 0, 0}, {1, 1, 1}, {1, 1, 1}};
    for (int a = 0; a < 3; ++a) { g.sz[a] = u.size[a]; g.k[a] = u.k[a]; g.s[a] = u.s[a]; g.p[a] = u.p[a]; g.d[a] = u.d[a]; g.o[a] = u.out[a]; }
    return g;
}

int ntg_unfoldnd_dev(int dtype, const void* image, void* col, int64_t batch, int64_t channels, int ndim, const int64_t* size,
                     const int64_t* kernel_size, const int64_t* stride, const int64_t* padding, const int64_t* dilation, void* stream) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    ntg::UnfoldNdParams u;
    int rc = fill_nd(u, batch, channels, ndim, size, kernel_size, stride, padding, dilation);
    if (rc) return rc;
    if (u.total == 0) return NTG_OK;
    if (!image || !col) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer");
    hipError_t e = ntg::launch_unfoldnd(es, image, col, u, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return hip_fail(e, "unfoldnd launch");
    return NTG_OK;
}

int ntg_unfoldnd_backward_dev(int dtype, const void* col, void* image, int64_t batch, int64_t channels, int ndim, const int64_t* size,
                              const int64_t* kernel_size, const int64_t* stride, const int64_t* padding, const int64_t* dilation,
                              int accumulate, void* stream) {
    if (ntg::elem_size(dtype) == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    ntg::UnfoldNdParams u;
    int rc = fill_nd(u, batch, channels, ndim, size, kernel_size, stride, padding, dilation);
    if (rc) return rc;
    if (batch * channels * u.vol == 0) return NTG_OK;
    if (!image || !col) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer");
    hipError_t e = ntg::launch_col2imnd(dtype, col, image, u, accumulate, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return hip_fail(e, "col2imnd launch");
    return NTG_OK;
}

static int check_groups(int64_t channels, int64_t out_channels, int64_t groups) {
    if (channels < 0 || out_channels < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "negative size");
    if (groups < 1) return fail(NTG_ERR_INVALID_ARGUMENT, "groups must be >= 1");
    if (channels % groups != 0) return fail(NTG_ERR_INVALID_ARGUMENT, "image channels (%lld) not divisible by groups (%lld)", (long long)channels, (long long)groups);
    if (out_channels % groups != 0) return fail(NTG_ERR_INVALID_ARGUMENT, "out channels (%lld) not divisible by groups (%lld)", (long long)out_channels, (long long)groups);
    return NTG_OK;
}

int64_t ntg_convnd_workspace_bytes(int dtype, int64_t batch, int64_t channels, int64_t out_channels, int ndim, const int64_t* size,
                                   const int64_t* kernel_size, const int64_t* stride, const int64_t* padding, const int64_t* dilation,
                                   int64_t groups, int backward) {
    const int64_t es = ntg::elem_size(dtype);
    ntg::UnfoldNdParams u;
    if (es == 0 || check_groups(channels, out_channels, groups) || fill_nd(u, batch, channels, ndim, size, kernel_size, stride, padding, dilation)) return -1;
    if (ndim <= 2) {
        const Geo2 g = as_2d(ndim, size, kernel_size, stride, padding, dilation);
        return backward ? ntg_conv2d_backward_workspace_bytes(dtype, batch, channels, g.h, g.w, out_channels, g.kr, g.kc, g.sr, g.sc, g.pr, g.pc, g.dr, g.dc, groups)
                        : ntg_conv2d_forward_workspace_bytes(dtype, batch, channels, g.h, g.w, g.kr, g.kc, g.sr, g.sc, g.pr, g.pc, g.dr, g.dc);
    }
    if (ndim == 3) {
        const Geo3 g = geo_from(u);
        if (backward) return plan_conv_backward_g(dtype, true, true, batch, channels, out_channels, g, groups).need;
        if (conv_implicit_g(dtype, channels, g)) return 0;
    }
    return u.total * es + (backward ? complex_dkernel_extra(dtype, batch, out_channels, (channels / groups) * u.taps, u.total * es) : 0);
}

int64_t ntg_convnd_fast_workspace_bytes(int dtype, int64_t batch, int64_t channels, int64_t out_channels, int ndim, const int64_t* size,
                                        const int64_t* kernel_size, const int64_t* stride, const int64_t* padding, const int64_t* dilation,
                                        int64_t groups, int backward) {
    const int64_t least = ntg_convnd_workspace_bytes(dtype, batch, channels, out_channels, ndim, size, kernel_size, stride, padding, dilation, groups, backward);
    if (least < 0) return least;
    if (ndim <= 2) {
        const Geo2 g = as_2d(ndim, size, kernel_size, stride, padding, dilation);
        return backward ? least : ntg_conv2d_fast_workspace_bytes(dtype, batch, channels, g.h, g.w, out_channels, g.kr, g.kc, g.sr, g.sc, g.pr, g.pc, g.dr, g.dc, groups);
    }
    if (ndim != 3) return least;
    ntg::UnfoldNdParams u;
    if (fill_nd(u, batch, channels, ndim, size, kernel_size, stride, padding, dilation)) return -1;
    const Geo3 g = geo_from(u);
    if (backward) {
        const ConvBackwardPlan pl = plan_conv_backward_g(dtype, true, true, batch, channels, out_channels, g, groups);
        const int64_t fast = std::max({pl.need_phase_dx, pl.need_nhwc_dx, pl.need_nhwc_dw, pl.need_both});
        return fast > 0 ? std::max(fast, least + 256) : least;        // (more than `least` is what asks for the fast forms)
    }
    return conv_nhwc_ok(dtype, batch, channels, out_channels, groups, g) ? conv_nhwc_workspace(dtype, batch, channels, out_channels, groups, g) : least;
}

int ntg_convnd_dev(int dtype, const void* image, const void* kernel, void* out, void* workspace, int64_t workspace_bytes,
                   int64_t batch, int64_t channels, int64_t out_channels, int ndim, const int64_t* size, const int64_t* kernel_size,
                   const int64_t* stride, const int64_t* padding, const int64_t* dilation, int64_t groups, void* stream) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    int rc = check_groups(channels, out_channels, groups);
    if (rc) return rc;
    ntg::UnfoldNdParams u;
    rc = fill_nd(u, batch, channels, ndim, size, kernel_size, stride, padding, dilation);
    if (rc) return rc;
    if (ndim <= 2) {
        const Geo2 g = as_2d(ndim, size, kernel_size, stride, padding, dilation);
        return ntg_conv2d_dev(dtype, image, kernel, out, workspace, workspace_bytes, batch, channels, g.h, g.w, out_channels, g.kr, g.kc,
                              g.sr, g.sc, g.pr, g.pc, g.dr, g.dc, groups, stream);
    }
    if (batch == 0 || out_channels == 0) return NTG_OK;
    if (!image || !kernel || !out) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer");
    if (ndim == 3) {
        const Geo3 g = geo_from(u);
        if (conv_nhwc_ok(dtype, batch, channels, out_channels, groups, g) && workspace && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0 &&
            workspace_bytes >= conv_nhwc_workspace(dtype, batch, channels, out_channels, groups, g))
            return conv_forward_nhwc(dtype, image, kernel, out, workspace, batch, channels, out_channels, g, groups, static_cast<hipStream_t>(stream));
        if (conv_implicit_g(dtype, channels, g))      // three axes, floating dtype: gathered inside the GEMM, no col buffer
            return conv_forward_gather(dtype, image, kernel, out, batch, channels, out_channels, g, groups, static_cast<hipStream_t>(stream));
    }
    const int64_t need = u.total * es;
    if (need > 0 && (!workspace || workspace_bytes < need))
        return fail(NTG_ERR_INVALID_ARGUMENT, "workspace of %lld bytes needed, %lld given", (long long)need, (long long)workspace_bytes);
    hipError_t e = ntg::launch_unfoldnd(es, image, workspace, u, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return hip_fail(e, "unfoldnd launch");
    // out_b[g*og:(g+1)*og, L] = W_g[og, add] . col_b[g*add:(g+1)*add, L]   (the reference's (col^T . W^T)^T, conv.cpp:143, :171)
    const int64_t add = (channels / groups) * u.taps, og = out_channels / groups;
    for (int64_t g = 0; g < groups; ++g) {
        ntg_gemm_desc d;
        std::memset(&d, 0, sizeof d);
        d.dtype = dtype; d.c_mode = NTG_C_OVERWRITE;
        d.m = og; d.k = add; d.n = u.L;
        d.lda = add; d.ldb = u.L; d.ldc = u.L;
        d.batches = batch;
        d.stride_a = 0; d.stride_b = u.ccol * u.L; d.stride_c = out_channels * u.L;
        rc = ntg_gemm_dev(&d, static_cast<const char*>(kernel) + g * og * add * es, static_cast<const char*>(workspace) + g * add * u.L * es,
                          static_cast<char*>(out) + g * og * u.L * es, stream);
        if (rc) return rc;
    }
    return NTG_OK;
}

// channels_last = false (Float32 through the host entry point): the element-wise gathering forms, whose weight gradient sums the
// output pixels of each image in ascending order like the reference
static int convnd_backward_dev_impl(int dtype, const void* image, const void* kernel, const void* grad_out, void* d_image, void* d_kernel,
                                    void* workspace, int64_t workspace_bytes, int64_t batch, int64_t channels, int64_t out_channels, int ndim,
                                    const int64_t* size, const int64_t* kernel_size, const int64_t* stride, const int64_t* padding,
                                    const int64_t* dilation, int64_t groups, int accumulate, void* stream, bool channels_last) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    int rc = check_groups(channels, out_channels, groups);
    if (rc) return rc;
    ntg::UnfoldNdParams u;
    rc = fill_nd(u, batch, channels, ndim, size, kernel_size, stride, padding, dilation);
    if (rc) return rc;
    if (ndim <= 2) {
        const Geo2 g = as_2d(ndim, size, kernel_size, stride, padding, dilation);
        return ntg_conv2d_backward_dev(dtype, image, kernel, grad_out, d_image, d_kernel, workspace, workspace_bytes, batch, channels, g.h, g.w,
                                       out_channels, g.kr, g.kc, g.sr, g.sc, g.pr, g.pc, g.dr, g.dc, groups, accumulate, stream);
    }
    if (batch == 0 || out_channels == 0 || channels == 0) return NTG_OK;
    if (!kernel || !grad_out || (d_kernel && !image)) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer");
    int64_t need = u.total * es + (d_kernel ? complex_dkernel_extra(dtype, batch, out_channels, (channels / groups) * u.taps, u.total * es) : 0);
    bool reference_order = !channels_last && dtype == ntg::DT_F32;
    if (ndim == 3) {
        const Geo3 g = geo_from(u);
        const ConvBackwardPlan plan = plan_conv_backward_g(dtype, d_image != nullptr, d_kernel != nullptr, batch, channels, out_channels, g, groups);
        need = plan.need;
        if (need > 0 && (!workspace || workspace_bytes < need))
            return fail(NTG_ERR_INVALID_ARGUMENT, "workspace of %lld bytes needed, %lld given", (long long)need, (long long)workspace_bytes);
        // a workspace of ntg_convnd_workspace_bytes asks for the reference's order, even where a fast form would fit into it
        const bool fast = channels_last && workspace_bytes > ntg_convnd_workspace_bytes(dtype, batch, channels, out_channels, ndim, size, kernel_size, stride,
                                                                                        padding, dilation, groups, 1);
        reference_order = !fast && dtype == ntg::DT_F32;
        rc = conv_gradients_implicit(dtype, plan, image, kernel, grad_out, d_image, d_kernel, static_cast<char*>(workspace), workspace_bytes, batch, channels,
                                     out_channels, g, groups, accumulate, static_cast<hipStream_t>(stream), fast);
        if (rc) return rc;
        if (!d_kernel && !d_image) return NTG_OK;
    }
    if (!workspace || workspace_bytes < need)
        return fail(NTG_ERR_INVALID_ARGUMENT, "workspace of %lld bytes needed, %lld given", (long long)need, (long long)workspace_bytes);
    const int64_t L = u.L, add = (channels / groups) * u.taps, og = out_channels / groups;
    const char* kern = static_cast<const char*>(kernel);
    const char* gy = static_cast<const char*>(grad_out);
    char* ws = static_cast<char*>(workspace);
    ntg_gemm_desc d;
    if (d_kernel) {
        hipError_t e = ntg::launch_unfoldnd(es, image, ws, u, static_cast<hipStream_t>(stream));
        if (e != hipSuccess) return hip_fail(e, "unfoldnd launch");
        rc = conv_dkernel_from_col(dtype, gy, ws, d_kernel, batch, out_channels, u.ccol, groups, L, accumulate, stream);
        if (rc) return rc;
    }
    if (d_image) {
        rc = gemm_per_group(dtype, true, false, NTG_C_OVERWRITE, add, og, L, add, L, L, batch, groups, kern, og * add, 0, gy, og * L, out_channels * L, ws, stream,
                            reference_order);
        if (rc) return rc;
        hipError_t e = ntg::launch_col2imnd(dtype, ws, d_image, u, accumulate, static_cast<hipStream_t>(stream));
        if (e != hipSuccess) return hip_fail(e, "col2imnd launch");
    }
    return NTG_OK;
}

int ntg_convnd_backward_dev(int dtype, const void* image, const void* kernel, const void* grad_out, void* d_image, void* d_kernel,
                            void* workspace, int64_t workspace_bytes, int64_t batch, int64_t channels, int64_t out_channels, int ndim,
                            const int64_t* size, const int64_t* kernel_size, const int64_t* stride, const int64_t* padding,
                            const int64_t* dilation, int64_t groups, int accumulate, void* stream) {
    return convnd_backward_dev_impl(dtype, image, kernel, grad_out, d_image, d_kernel, workspace, workspace_bytes, batch, channels, out_channels, ndim,
                                    size, kernel_size, stride, padding, dilation, groups, accumulate, stream, true);
}

// output size of the transposed convolution per axis; the geometry of the convolution it is the adjoint of
static int transpose_nd_out(int ndim, const int64_t* in_size, const int64_t* k, const int64_t* s, const int64_t* p, const int64_t* d,
                            const int64_t* op, int64_t* out_size) {
    if (ndim < 1 || ndim > NTG_MAX_SPATIAL) return fail(NTG_ERR_INVALID_ARGUMENT, "ndim must be 1..%d but got %d", NTG_MAX_SPATIAL, ndim);
    if (!in_size || !k || !s || !p || !d || !op) return fail(NTG_ERR_INVALID_ARGUMENT, "null geometry array");
    for (int a = 0; a < ndim; ++a) {
        if (k[a] < 1 || s[a] < 1 || d[a] < 1 || p[a] < 0 || op[a] < 0)
            return fail(NTG_ERR_INVALID_ARGUMENT, "kernel/stride/dilation must be >= 1 and padding/output_padding >= 0");
        if (op[a] >= s[a]) return fail(NTG_ERR_INVALID_ARGUMENT, "output_padding (%lld) must be smaller than stride (%lld)", (long long)op[a], (long long)s[a]);
        if (in_size[a] < 1) return fail(NTG_ERR_INVALID_ARGUMENT, "empty input");
        out_size[a] = (in_size[a] - 1) * s[a] - 2 * p[a] + d[a] * (k[a] - 1) + 1 + op[a];
        if (out_size[a] < 1) return fail(NTG_ERR_INVALID_ARGUMENT, "the output of the transposed convolution would be empty");
    }
    return NTG_OK;
}

int64_t ntg_conv_transposend_workspace_bytes(int dtype, int64_t batch, int64_t in_channels, int64_t out_channels, int ndim,
                                             const int64_t* in_size, const int64_t* kernel_size, const int64_t* stride,
                                             const int64_t* padding, const int64_t* dilation, const int64_t* output_padding, int64_t groups) {
    int64_t os[NTG_MAX_SPATIAL];
    if (ntg::elem_size(dtype) == 0 || check_groups(in_channels, out_channels, groups) ||
        transpose_nd_out(ndim, in_size, kernel_size, stride, padding, dilation, output_padding, os)) return -1;
    if (ndim <= 2) {
        const Geo2 g = as_2d(ndim, in_size, kernel_size, stride, padding, dilation);
        return ntg_conv_transpose2d_workspace_bytes(dtype, batch, in_channels, g.h, g.w, out_channels, g.kr, g.kc, g.sr, g.sc, g.pr, g.pc, g.dr, g.dc,
                                                    ndim == 1 ? 0 : output_padding[0], output_padding[ndim - 1], groups);
    }
    return ntg_convnd_fast_workspace_bytes(dtype, batch, out_channels, in_channels, ndim, os, kernel_size, stride, padding, dilation, groups, 1);
}

int ntg_conv_transposend_dev(int dtype, const void* input, const void* kernel, void* out, void* workspace, int64_t workspace_bytes,
                             int64_t batch, int64_t in_channels, int64_t out_channels, int ndim, const int64_t* in_size,
                             const int64_t* kernel_size, const int64_t* stride, const int64_t* padding, const int64_t* dilation,
                             const int64_t* output_padding, int64_t groups, void* stream) {
    if (ntg::elem_size(dtype) == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    int rc = check_groups(in_channels, out_channels, groups);
    if (rc) return rc;
    int64_t os[NTG_MAX_SPATIAL];
    rc = transpose_nd_out(ndim, in_size, kernel_size, stride, padding, dilation, output_padding, os);
    if (rc) return rc;
    if (ndim <= 2) {
        const Geo2 g = as_2d(ndim, in_size, kernel_size, stride, padding, dilation);
        return ntg_conv_transpose2d_dev(dtype, input, kernel, out, workspace, workspace_bytes, batch, in_channels, g.h, g.w, out_channels, g.kr, g.kc,
                                        g.sr, g.sc, g.pr, g.pc, g.dr, g.dc, ndim == 1 ? 0 : output_padding[0], output_padding[ndim - 1], groups, stream);
    }
    if (batch == 0 || out_channels == 0) return NTG_OK;
    if (in_channels == 0) return fail(NTG_ERR_INVALID_ARGUMENT, "empty input");
    // the image gradient of the convolution [out_channels -> in_channels] over an image of the output's size
    return ntg_convnd_backward_dev(dtype, nullptr, kernel, input, out, nullptr, workspace, workspace_bytes, batch, out_channels, in_channels, ndim,
                                   os, kernel_size, stride, padding, dilation, groups, 0, stream);
}

// host-pointer forms (synchronous)
int ntg_convnd(int dtype, const void* image, const void* kernel, void* out, int64_t batch, int64_t channels, int64_t out_channels, int ndim,
               const int64_t* size, const int64_t* kernel_size, const int64_t* stride, const int64_t* padding, const int64_t* dilation, int64_t groups) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    int rc = check_groups(channels, out_channels, groups);
    if (rc) return rc;
    ntg::UnfoldNdParams u;
    rc = fill_nd(u, batch, channels, ndim, size, kernel_size, stride, padding, dilation);
    if (rc) return rc;
    if (batch == 0 || out_channels == 0) return NTG_OK;
    if (!image || !kernel || !out) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer");
    const size_t im_bytes = (size_t)(batch * channels * u.vol * es), k_bytes = (size_t)(out_channels * (channels / groups) * u.taps * es);
    const size_t o_bytes = (size_t)(batch * out_channels * u.L * es);
    // (Float32 at the reference's seam keeps the gathering kernels and with them im2col's order of k, see ntg_conv2d; so do one and two axes)
    const int64_t wsb = (dtype == ntg::DT_F32 || ndim != 3 ? ntg_convnd_workspace_bytes : ntg_convnd_fast_workspace_bytes)(
        dtype, batch, channels, out_channels, ndim, size, kernel_size, stride, padding, dilation, groups, 0);
    ntg::HostSession mem;
    const size_t o_k = align_up(im_bytes, 256), o_o = o_k + align_up(k_bytes, 256), o_ws = o_o + align_up(o_bytes, 256);
    HIP_TRY(mem.reserve(o_ws + (size_t)wsb));
    if (im_bytes) HIP_TRY(mem.upload(0, image, im_bytes));
    if (k_bytes) HIP_TRY(mem.upload(o_k, kernel, k_bytes));
    if (ndim <= 2) {
        const Geo2 g = as_2d(ndim, size, kernel_size, stride, padding, dilation);
        rc = conv2d_dev_impl(dtype, mem.at(0), mem.at(o_k), mem.at(o_o), mem.at(o_ws), wsb, batch, channels, g.h, g.w, out_channels, g.kr, g.kc,
                             g.sr, g.sc, g.pr, g.pc, g.dr, g.dc, groups, mem.stream(), dtype == ntg::DT_F32);
    } else {
        rc = ntg_convnd_dev(dtype, mem.at(0), mem.at(o_k), mem.at(o_o), mem.at(o_ws), wsb, batch, channels, out_channels, ndim, size, kernel_size,
                            stride, padding, dilation, groups, mem.stream());
    }
    if (rc) return rc;
    HIP_TRY(mem.download(out, o_o, o_bytes));
    return NTG_OK;
}

int ntg_convnd_backward(int dtype, const void* image, const void* kernel, const void* grad_out, void* d_image, void* d_kernel,
                        int64_t batch, int64_t channels, int64_t out_channels, int ndim, const int64_t* size, const int64_t* kernel_size,
                        const int64_t* stride, const int64_t* padding, const int64_t* dilation, int64_t groups, int accumulate) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    int rc = check_groups(channels, out_channels, groups);
    if (rc) return rc;
    ntg::UnfoldNdParams u;
    rc = fill_nd(u, batch, channels, ndim, size, kernel_size, stride, padding, dilation);
    if (rc) return rc;
    if (batch == 0 || out_channels == 0 || channels == 0) return NTG_OK;
    if (!image || !kernel || !grad_out) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer");
    if (ndim <= 2) {        // (the two-axis host entry point: it keeps the reference's order of summation for Float32)
        const Geo2 g = as_2d(ndim, size, kernel_size, stride, padding, dilation);
        return ntg_conv2d_backward(dtype, image, kernel, grad_out, d_image, d_kernel, batch, channels, g.h, g.w, out_channels, g.kr, g.kc,
                                   g.sr, g.sc, g.pr, g.pc, g.dr, g.dc, groups, accumulate);
    }
    const size_t im_bytes = (size_t)(batch * channels * u.vol * es), k_bytes = (size_t)(out_channels * (channels / groups) * u.taps * es);
    const size_t g_bytes = (size_t)(batch * out_channels * u.L * es);
    // (Float32 takes the forms that follow the reference's order and reserves no more than those use)
    const int64_t wsb = (dtype == ntg::DT_F32 ? ntg_convnd_workspace_bytes : ntg_convnd_fast_workspace_bytes)(
        dtype, batch, channels, out_channels, ndim, size, kernel_size, stride, padding, dilation, groups, 1);
    ntg::HostSession mem;
    const size_t o_k = align_up(im_bytes, 256), o_g = o_k + align_up(k_bytes, 256), o_di = o_g + align_up(g_bytes, 256);
    const size_t o_dk = o_di + align_up(im_bytes, 256), o_ws = o_dk + align_up(k_bytes, 256);
    HIP_TRY(mem.reserve(o_ws + (size_t)wsb));
    HIP_TRY(mem.upload(0, image, im_bytes));
    HIP_TRY(mem.upload(o_k, kernel, k_bytes));
    HIP_TRY(mem.upload(o_g, grad_out, g_bytes));
    if (accumulate && d_image) HIP_TRY(mem.upload(o_di, d_image, im_bytes));
    if (accumulate && d_kernel) HIP_TRY(mem.upload(o_dk, d_kernel, k_bytes));
    rc = convnd_backward_dev_impl(dtype, mem.at(0), mem.at(o_k), mem.at(o_g), d_image ? mem.at(o_di) : nullptr, d_kernel ? mem.at(o_dk) : nullptr,
                                  mem.at(o_ws), wsb, batch, channels, out_channels, ndim, size, kernel_size, stride, padding, dilation, groups,
                                  accumulate, mem.stream(), dtype != ntg::DT_F32);
    if (rc) return rc;
    if (d_image) HIP_TRY(mem.download(d_image, o_di, im_bytes));
    if (d_kernel) HIP_TRY(mem.download(d_kernel, o_dk, k_bytes));
    return NTG_OK;
}

int ntg_conv_transposend(int dtype, const void* input, const void* kernel, void* out, int64_t batch, int64_t in_channels, int64_t out_channels,
                         int ndim, const int64_t* in_size, const int64_t* kernel_size, const int64_t* stride, const int64_t* padding,
                         const int64_t* dilation, const int64_t* output_padding, int64_t groups) {
    const int64_t es = ntg::elem_size(dtype);
    if (es == 0) return fail(NTG_ERR_UNSUPPORTED_DTYPE, "dtype %d is not supported", dtype);
    int rc = check_groups(in_channels, out_channels, groups);
    if (rc) return rc;
    int64_t os[NTG_MAX_SPATIAL];
    rc = transpose_nd_out(ndim, in_size, kernel_size, stride, padding, dilation, output_padding, os);
    if (rc) return rc;
    if (batch == 0 || out_channels == 0) return NTG_OK;
    if (!input || !kernel || !out) return fail(NTG_ERR_INVALID_ARGUMENT, "null pointer");
    int64_t in_vol = 1, out_vol = 1, taps = 1;
    for (int a = 0; a < ndim; ++a) { in_vol *= in_size[a]; out_vol *= os[a]; taps *= kernel_size[a]; }
    const size_t in_bytes = (size_t)(batch * in_channels * in_vol * es), k_bytes = (size_t)(in_channels * (out_channels / groups) * taps * es);
    const size_t o_bytes = (size_t)(batch * out_channels * out_vol * es);
    const int64_t wsb = ntg_conv_transposend_workspace_bytes(dtype, batch, in_channels, out_channels, ndim, in_size, kernel_size, stride, padding,
                                                             dilation, output_padding, groups);
    if (wsb < 0) return fail(NTG_ERR_INVALID_ARGUMENT, "invalid geometry");
    ntg::HostSession mem;
    const size_t o_k = align_up(in_bytes, 256), o_o = o_k + align_up(k_bytes, 256), o_ws = o_o + align_up(o_bytes, 256);
    HIP_TRY(mem.reserve(o_ws + (size_t)wsb));
    if (in_bytes) HIP_TRY(mem.upload(0, input, in_bytes));
    if (k_bytes) HIP_TRY(mem.upload(o_k, kernel, k_bytes));
    rc = ntg_conv_transposend_dev(dtype, mem.at(0), mem.at(o_k), mem.at(o_o), mem.at(o_ws), wsb, batch, in_channels, out_channels, ndim, in_size,
                                  kernel_size, stride, padding, dilation, output_padding, groups, mem.stream());
    if (rc) return rc;
    HIP_TRY(mem.download(out, o_o, o_bytes));
    return NTG_OK;
}

}  // extern "C"
