// c_api.hip -- the extern "C" boundary declared in include/iq4xs_mi355x.h.
// Argument checks mirror the reference launchers (hipErrorInvalidValue for
// null pointers and bad shapes, real_stock_dp4a_comparator.hip:487,513;
// impl_gemv_dp4a_gfx1100.hip:299-300) and run before anything is launched.
#include <stdlib.h>

#include <mutex>
#include <vector>

#include "iq4xs_device.h"
#include "iq4xs_internal.h"
#include "iq4xs_mi355x.h"

using namespace iq4xs;

// The static device scratch of iq4xs_mul_mat_noalloc (its host-side lookup is
// noalloc_scratch below).
static __device__ __align__(256) uint8_t scratch[(size_t)IQ4XS_NOALLOC_SCRATCH_BYTES];

namespace {

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

bool valid_k(int64_t K) { return K > 0 && K % QK_K == 0; }

// Largest tensor the int32/int64 index arithmetic of the kernels is sized for.
constexpr int64_t MAX_DIM = (int64_t)1 << 31;

bool valid_mat(const void* W, const void* X, const void* Y, int64_t K, int64_t N, int64_t M) {
    return W && X && Y && valid_k(K) && N > 0 && M > 0 && K < MAX_DIM && N < MAX_DIM && M < MAX_DIM;
}

// Per-call Q8_1 scratch of the reference-named entry points comes from a
// stream-ordered pool that this library creates for each device and owns.
// The pool keeps freed blocks instead of returning them to the driver, so a
// repeated call is a pool hit.  The device's default pool, which the rest of
// the process (a host application, PyTorch) may use, is left untouched.
constexpr int MAX_DEVICES = 64;
std::once_flag g_pool_once[MAX_DEVICES];
hipMemPool_t g_pool[MAX_DEVICES];
hipError_t g_pool_err[MAX_DEVICES];

hipError_t pool_alloc(void** p, size_t bytes, hipStream_t stream) {
    int dev = 0;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return err;
    if (dev < 0 || dev >= MAX_DEVICES) return hipErrorInvalidDevice;
    std::call_once(g_pool_once[dev], [dev]() {
        hipMemPoolProps props{};
        props.allocType = hipMemAllocationTypePinned;
        props.handleTypes = hipMemHandleTypeNone;
        props.location.type = hipMemLocationTypeDevice;
        props.location.id = dev;
        hipError_t e = hipMemPoolCreate(&g_pool[dev], &props);
        if (e == hipSuccess) {
            uint64_t keep = UINT64_MAX;
            e = hipMemPoolSetAttribute(g_pool[dev], hipMemPoolAttrReleaseThreshold, &keep);
        }
        g_pool_err[dev] = e;
    });
    if (g_pool_err[dev] != hipSuccess) return g_pool_err[dev];
    return hipMallocFromPoolAsync(p, bytes, g_pool[dev], stream);
}

// Q8_1 workspace of iq4xs_mul_mat_noalloc: a file-scope device array of a fixed
// size.  Every GPU the library runs on holds its own copy until the process
// ends.  In host code `scratch` names a host-side stand-in, not device memory:
// its device address is looked up once per device (hipGetSymbolAddress, with
// that device current) and only that address is ever passed to a kernel.
constexpr size_t NOALLOC_SCRATCH_BYTES = (size_t)IQ4XS_NOALLOC_SCRATCH_BYTES;

std::once_flag g_scratch_once[MAX_DEVICES];
void* g_scratch_ptr[MAX_DEVICES];
hipError_t g_scratch_err[MAX_DEVICES];

// The current device's copy of `scratch` (looked up on the first call on that device).
hipError_t noalloc_scratch(void** ptr) {
    int dev = 0;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return err;
    if (dev < 0 || dev >= MAX_DEVICES) return hipErrorInvalidDevice;
    std::call_once(g_scratch_once[dev], [dev]() {
        void* p = nullptr;
        g_scratch_err[dev] = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        g_scratch_ptr[dev] = g_scratch_err[dev] == hipSuccess ? p : nullptr;
    });
    if (g_scratch_err[dev] != hipSuccess) return g_scratch_err[dev];
    if (g_scratch_ptr[dev] == nullptr) return hipErrorInvalidSymbol;
    *ptr = g_scratch_ptr[dev];
    return hipSuccess;
}

struct Planar {
    int8_t* qs;
    uint32_t* ds;
    uint32_t* hq;
};

Planar planar_view(const void* ws, int64_t K, int64_t M) {
    uint8_t* base = static_cast<uint8_t*>(const_cast<void*>(ws));
    return {reinterpret_cast<int8_t*>(base), reinterpret_cast<uint32_t*>(base + planar_ds_offset(K, M)),
            reinterpret_cast<uint32_t*>(base + planar_hq_offset(K, M))};
}

hipError_t mul_mat_planar(const uint8_t* W, const void* ws, float* Y, int64_t K, int64_t N, int64_t M, int layout,
                          int path, int32_t* dbg, hipStream_t stream) {
    const Planar p = planar_view(ws, K, M);
    const int64_t ldy_m = (layout == LAYOUT_MK) ? N : 1;
    const int64_t ldy_n = (layout == LAYOUT_MK) ? 1 : M;
    if (path == IQ4XS_PATH_AUTO) path = (M <= GEMV_MAX_COLS) ? IQ4XS_PATH_GEMV : IQ4XS_PATH_GEMM;
    if (path == IQ4XS_PATH_GEMV) {
        if (M > GEMV_MAX_COLS) return hipErrorInvalidValue;
        return launch_gemv(W, p.qs, p.ds, Y, K, N, M, ldy_m, ldy_n, dbg, stream);
    }
    if (path == IQ4XS_PATH_GEMM) return launch_gemm(W, p.qs, p.ds, p.hq, Y, K, N, M, ldy_m, ldy_n, dbg, stream);
    return hipErrorInvalidValue;
}

// Single-column calls with K up to these bounds run the GEMV with the Q8_1
// quantisation in its prologue (one launch, no workspace).  Every workgroup
// quantises the whole column, so the prologue grows with K.  A 16-byte
// aligned column is loaded as vectors and quantised in up to five rounds: it
// fuses up to K = 20480 (measured on the decode set: down_proj, K = 17408,
// 0.6 us per layer faster fused).  Other columns take per-element loads in at
// most two rounds: up to K = 8192 (measured: 8192 ahead of 6144 and of 17408).
// Past the bound (and for M > 1) a separate quantiser launch is cheaper.
constexpr int64_t FUSED_MAX_K = 8192;

int64_t fused_max_k_override() {
    static const int64_t v = []() -> int64_t {
        const char* e = getenv("IQ4XS_FUSED_MAX_K");  // tuning override of both bounds
        return e ? atoll(e) : -1;
    }();
    return v;
}

bool prefer_fused(int64_t K, int64_t M, const float* X) {
    const int64_t o = fused_max_k_override();
    const int64_t bound = o >= 0 ? o : (reinterpret_cast<uintptr_t>(X) % 16 == 0 ? GEMV_FUSED_VEC_MAX_K : FUSED_MAX_K);
    return M == 1 && K <= bound;
}

hipError_t mul_mat_fused(const uint8_t* W, const float* X, float* Y, int64_t K, int64_t N, int64_t M, int layout,
                         int32_t* dbg, hipStream_t stream) {
    const int64_t ldy_m = (layout == LAYOUT_MK) ? N : 1;
    const int64_t ldy_n = (layout == LAYOUT_MK) ? 1 : M;
    const int64_t sc = (layout == LAYOUT_MK) ? K : 1;
    const int64_t sk = (layout == LAYOUT_MK) ? 1 : M;
    return launch_gemv_fused(W, X, sc, sk, Y, K, N, M, ldy_m, ldy_n, dbg, stream);
}

// quantise + multiply with scratch from the stream-ordered pool
hipError_t mul_mat_pooled(const void* W, const float* X, float* Y, int64_t K, int64_t N, int64_t M, int layout,
                          hipStream_t stream) {
    if (!valid_mat(W, X, Y, K, N, M)) return hipErrorInvalidValue;
    if (prefer_fused(K, M, X)) {
        const hipError_t e = mul_mat_fused(static_cast<const uint8_t*>(W), X, Y, K, N, M, layout, nullptr, stream);
        if (e != hipErrorNotSupported) return e;
    }
    void* ws = nullptr;
    hipError_t err = pool_alloc(&ws, planar_bytes(K, M), stream);
    if (err != hipSuccess) return err;
    const Planar p = planar_view(ws, K, M);
    err = launch_quantize(X, K, M, layout, p.qs, p.ds, p.hq, nullptr, stream);
    if (err == hipSuccess)
        err = mul_mat_planar(static_cast<const uint8_t*>(W), ws, Y, K, N, M, layout, IQ4XS_PATH_AUTO, nullptr,
                             stream);
    const hipError_t ferr = hipFreeAsync(ws, stream);
    return err != hipSuccess ? err : ferr;
}

}  // namespace

extern "C" {

int quantize_row_q8_1_gpu(const float* x, void* y, int64_t K, void* stream) {
    if (!x || !y || K <= 0 || K % QK8_1 != 0 || K >= MAX_DIM) return hipErrorInvalidValue;
    return launch_quantize(x, K, 1, LAYOUT_MK, nullptr, nullptr, nullptr, static_cast<block_q8_1*>(y),
                           as_stream(stream));
}

int quantize_row_q8_1_batched_gpu(const float* X, void* Y, int64_t K, int64_t M, void* stream) {
    if (!X || !Y || K <= 0 || K % QK8_1 != 0 || M <= 0 || K >= MAX_DIM || M >= MAX_DIM) return hipErrorInvalidValue;
    return launch_quantize(X, K, M, LAYOUT_KM, nullptr, nullptr, nullptr, static_cast<block_q8_1*>(Y),
                           as_stream(stream));
}

int gemv_iq4xs_stock_dp4a_gpu(const void* W, const float* x, float* y, int64_t K, int64_t N, void* stream) {
    return mul_mat_pooled(W, x, y, K, N, 1, LAYOUT_MK, as_stream(stream));
}

int gemv_iq4xs_dp4a_coop_gpu(const void* W, const float* x, float* y, int64_t K, int64_t N, void* stream) {
    return mul_mat_pooled(W, x, y, K, N, 1, LAYOUT_MK, as_stream(stream));
}

int gemv_iq4xs_dp4a_gfx1100_gpu(const void* W, const float* x, float* y, int64_t K, int64_t N, void* stream) {
    return mul_mat_pooled(W, x, y, K, N, 1, LAYOUT_MK, as_stream(stream));
}

int gemv_iq4xs_dp4a_gfx1100_prequantized_gpu(const void* W, const void* AQ, float* y, int64_t K, int64_t N,
                                             void* stream) {
    if (!valid_mat(W, AQ, y, K, N, 1) || reinterpret_cast<uintptr_t>(AQ) % 16 != 0) return hipErrorInvalidValue;
    hipStream_t s = as_stream(stream);
    void* ws = nullptr;
    hipError_t err = pool_alloc(&ws, planar_bytes(K, 1), s);
    if (err != hipSuccess) return err;
    const Planar p = planar_view(ws, K, 1);
    err = launch_coop_to_planar(static_cast<const uint8_t*>(AQ), K / QK8_1, p.qs, p.ds, p.hq, s);
    if (err == hipSuccess)
        err = mul_mat_planar(static_cast<const uint8_t*>(W), ws, y, K, N, 1, LAYOUT_MK, IQ4XS_PATH_AUTO, nullptr, s);
    const hipError_t ferr = hipFreeAsync(ws, s);
    return err != hipSuccess ? err : ferr;
}

int gemv_iq4xs_gfx1100_gpu(const void* W, const float* x, float* y, int64_t K, int64_t N, void* stream) {
    if (!valid_mat(W, x, y, K, N, 1)) return hipErrorInvalidValue;
    return launch_gfx1100_fp64(static_cast<const uint8_t*>(W), x, y, K, N, as_stream(stream));
}

int gemv_iq4xs_stock_gpu(const void* W, const float* x, float* y, int64_t K, int64_t N, void* stream) {
    if (!valid_mat(W, x, y, K, N, 1)) return hipErrorInvalidValue;
    return launch_stock_fp64(static_cast<const uint8_t*>(W), x, y, K, N, 1, as_stream(stream));
}

int gemm_iq4xs_stock_gpu(const void* W, const float* X, float* Y, int64_t K, int64_t N, int64_t M, void* stream) {
    if (!valid_mat(W, X, Y, K, N, M)) return hipErrorInvalidValue;
    return launch_stock_fp64(static_cast<const uint8_t*>(W), X, Y, K, N, M, as_stream(stream));
}

// The reference's fp16-WMMA GEMM family and its tiled fallbacks share one
// signature (X [K][M], Y [N][M]); here they all run the matrix-core GEMM on
// Q8_1 activations, the same kernel as gemm_iq4xs_stock_dp4a_gpu.
int gemm_iq4xs_wmma_stream_gpu(const void* W, const float* X, float* Y, int64_t K, int64_t N, int64_t M,
                               void* stream) {
    return mul_mat_pooled(W, X, Y, K, N, M, LAYOUT_KM, as_stream(stream));
}
int gemm_iq4xs_wmma_p4_xor_gpu(const void* W, const float* X, float* Y, int64_t K, int64_t N, int64_t M,
                               void* stream) {
    return mul_mat_pooled(W, X, Y, K, N, M, LAYOUT_KM, as_stream(stream));
}
int gemm_iq4xs_wmma_64x64_gpu(const void* W, const float* X, float* Y, int64_t K, int64_t N, int64_t M,
                              void* stream) {
    return mul_mat_pooled(W, X, Y, K, N, M, LAYOUT_KM, as_stream(stream));
}
int gemm_iq4xs_stream_tiled_gpu(const void* W, const float* X, float* Y, int64_t K, int64_t N, int64_t M,
                                void* stream) {
    return mul_mat_pooled(W, X, Y, K, N, M, LAYOUT_KM, as_stream(stream));
}
int gemm_iq4xs_wmma_gpu(const void* W, const float* X, float* Y, int64_t K, int64_t N, int64_t M, void* stream) {
    return mul_mat_pooled(W, X, Y, K, N, M, LAYOUT_KM, as_stream(stream));
}
int gemm_iq4xs_tiled_gpu(const void* W, const float* X, float* Y, int64_t K, int64_t N, int64_t M, void* stream) {
    return mul_mat_pooled(W, X, Y, K, N, M, LAYOUT_KM, as_stream(stream));
}

int gemm_iq4xs_lut_gpu(const void* W, const void* LUT, const float* X, float* Y, int64_t K, int64_t N, int64_t M,
                       void* stream) {
    (void)LUT;  // the IQ4_NL codebook is fixed by the format; the kernels carry it
    if (!W || !X || !Y || K % QK_K != 0) return hipErrorInvalidValue;
    // the reference's shape gate, kept so that callers relying on its fallback behave the same
    const bool gate = M % 16 == 0 && N % 16 == 0 && K % 16 == 0 && M >= 512 && N >= 32 && K >= 32;
    if (!gate) return hipErrorInvalidConfiguration;
    return mul_mat_pooled(W, X, Y, K, N, M, LAYOUT_KM, as_stream(stream));
}

int gemm_iq4xs_stock_dp4a_gpu(const void* W, const float* X, float* Y, int64_t K, int64_t N, int64_t M,
                              void* stream) {
    return mul_mat_pooled(W, X, Y, K, N, M, LAYOUT_KM, as_stream(stream));
}

int dequant_iq4xs_gpu(const void* src, float* dst, int64_t n_blocks, int warp_size, void* stream) {
    if (n_blocks < 0 || n_blocks >= MAX_DIM || (warp_size != 32 && warp_size != 64)) return hipErrorInvalidValue;
    if (n_blocks == 0) return hipSuccess;  // the reference launches a grid that writes nothing
    if (!src || !dst) return hipErrorInvalidValue;
    return launch_dequant(static_cast<const uint8_t*>(src), dst, n_blocks, as_stream(stream));
}

// The dispatch below computes one column (it has no M argument), so the gate
// accepts exactly M == 1, as the reference's does (patch:274-277); small
// batches reach the GEMV through custom_gemm_iq4xs_dispatch and the explicit
// API.
bool custom_gemv_iq4xs_can_handle(int64_t K, int64_t N, int64_t M, int type) {
    return type == IQ4XS_GGML_TYPE_IQ4_XS && M == 1 && valid_k(K) && K < MAX_DIM && N > 0 && N < MAX_DIM;
}

int custom_gemv_iq4xs_dispatch(const void* W, const float* x, float* y, int64_t K, int64_t N, void* stream) {
    return mul_mat_pooled(W, x, y, K, N, 1, LAYOUT_MK, as_stream(stream));
}

bool custom_gemm_iq4xs_can_handle(int64_t K, int64_t N, int64_t M, int type) {
    return type == IQ4XS_GGML_TYPE_IQ4_XS && M >= 1 && M < MAX_DIM && valid_k(K) && K < MAX_DIM && N > 0 &&
           N < MAX_DIM;
}

int custom_gemm_iq4xs_dispatch(const void* W, const float* X, float* Y, int64_t K, int64_t N, int64_t M,
                               void* stream) {
    return mul_mat_pooled(W, X, Y, K, N, M, LAYOUT_MK, as_stream(stream));
}

size_t iq4xs_workspace_bytes(int64_t K, int64_t M) {
    if (K <= 0 || K % QK8_1 != 0 || M <= 0 || K >= MAX_DIM || M >= MAX_DIM) return 0;
    return planar_bytes(K, M);
}

int iq4xs_quantize_q8_1(const float* X, int64_t K, int64_t M, int layout, void* ws, size_t ws_bytes,
                        void* stream) {
    if (!X || !ws || K <= 0 || K % QK8_1 != 0 || M <= 0 || K >= MAX_DIM || M >= MAX_DIM) return hipErrorInvalidValue;
    if ((layout != LAYOUT_KM && layout != LAYOUT_MK) || ws_bytes < planar_bytes(K, M)) return hipErrorInvalidValue;
    if (reinterpret_cast<uintptr_t>(ws) % 256 != 0) return hipErrorInvalidValue;
    const Planar p = planar_view(ws, K, M);
    return launch_quantize(X, K, M, layout, p.qs, p.ds, p.hq, nullptr, as_stream(stream));
}

int iq4xs_mul_mat_q8_1(const void* W, const void* ws, float* Y, int64_t K, int64_t N, int64_t M, int layout,
                       int path, void* stream) {
    if (!valid_mat(W, ws, Y, K, N, M) || (layout != LAYOUT_KM && layout != LAYOUT_MK)) return hipErrorInvalidValue;
    if (reinterpret_cast<uintptr_t>(ws) % 256 != 0) return hipErrorInvalidValue;
    return mul_mat_planar(static_cast<const uint8_t*>(W), ws, Y, K, N, M, layout, path, nullptr, as_stream(stream));
}

int iq4xs_mul_mat_q8_1_group(int count, const void* const* W, float* const* Y, const int64_t* N, const void* ws,
                             int64_t K, int64_t M, int layout, void* stream) {
    if (count < 1 || count > GEMV_GROUP_MAX || !W || !Y || !N) return hipErrorInvalidValue;
    if (layout != LAYOUT_KM && layout != LAYOUT_MK) return hipErrorInvalidValue;
    if (reinterpret_cast<uintptr_t>(ws) % 256 != 0) return hipErrorInvalidValue;
    for (int i = 0; i < count; ++i)
        if (!valid_mat(W[i], ws, Y[i], K, N[i], M)) return hipErrorInvalidValue;
    const Planar p = planar_view(ws, K, M);
    const uint8_t* Wb[GEMV_GROUP_MAX];
    for (int i = 0; i < count; ++i) Wb[i] = static_cast<const uint8_t*>(W[i]);
    if (M > GEMV_MAX_COLS)
        return launch_gemm_group(count, Wb, Y, N, p.qs, p.ds, p.hq, K, M, layout == LAYOUT_MK, as_stream(stream));
    return launch_gemv_group(count, Wb, Y, N, p.qs, p.ds, K, M, layout == LAYOUT_MK, as_stream(stream));
}

int iq4xs_mul_mat(const void* W, const float* X, float* Y, int64_t K, int64_t N, int64_t M, int layout, void* ws,
                  size_t ws_bytes, void* stream) {
    if (!valid_mat(W, X, Y, K, N, M) || !ws) return hipErrorInvalidValue;
    if ((layout != LAYOUT_KM && layout != LAYOUT_MK) || ws_bytes < planar_bytes(K, M)) return hipErrorInvalidValue;
    if (reinterpret_cast<uintptr_t>(ws) % 256 != 0) return hipErrorInvalidValue;
    if (prefer_fused(K, M, X)) {
        const hipError_t e =
            mul_mat_fused(static_cast<const uint8_t*>(W), X, Y, K, N, M, layout, nullptr, as_stream(stream));
        if (e != hipErrorNotSupported) return e;
    }
    const int err = iq4xs_quantize_q8_1(X, K, M, layout, ws, ws_bytes, stream);
    if (err != hipSuccess) return err;
    return mul_mat_planar(static_cast<const uint8_t*>(W), ws, Y, K, N, M, layout, IQ4XS_PATH_AUTO, nullptr,
                          as_stream(stream));
}

// iq4xs_mul_mat with the Q8_1 workspace in the library's static device scratch:
// no allocation of any kind.  Calls that overlap on one GPU share the scratch
// and race; the quantiser rewrites every byte a multiply reads, so nothing is
// cleared between calls.
int iq4xs_mul_mat_noalloc(const void* W, const float* X, float* Y, int64_t K, int64_t N, int64_t M, int layout,
                          void* stream) {
    if (!valid_mat(W, X, Y, K, N, M) || (layout != LAYOUT_KM && layout != LAYOUT_MK)) return hipErrorInvalidValue;
    if (planar_bytes(K, M) > NOALLOC_SCRATCH_BYTES) return hipErrorInvalidValue;  // beyond the static scratch
    void* ws = nullptr;
    hipError_t err = noalloc_scratch(&ws);
    if (err != hipSuccess) return err;
    hipStream_t s = as_stream(stream);
    if (prefer_fused(K, M, X)) {
        const hipError_t e = mul_mat_fused(static_cast<const uint8_t*>(W), X, Y, K, N, M, layout, nullptr, s);
        if (e != hipErrorNotSupported) return e;
    }
    const Planar p = planar_view(ws, K, M);
    err = launch_quantize(X, K, M, layout, p.qs, p.ds, p.hq, nullptr, s);
    if (err != hipSuccess) return err;
    return mul_mat_planar(static_cast<const uint8_t*>(W), ws, Y, K, N, M, layout, IQ4XS_PATH_AUTO, nullptr, s);
}

int iq4xs_mul_mat_fused(const void* W, const float* X, float* Y, int64_t K, int64_t N, int64_t M, int layout,
                        int32_t* S, void* stream) {
    if (!valid_mat(W, X, Y, K, N, M) || (layout != LAYOUT_KM && layout != LAYOUT_MK)) return hipErrorInvalidValue;
    if (M > GEMV_MAX_COLS) return hipErrorNotSupported;
    return mul_mat_fused(static_cast<const uint8_t*>(W), X, Y, K, N, M, layout, S, as_stream(stream));
}

namespace {
// [a, a + a_bytes) and [b, b + b_bytes) share a byte (null never overlaps).
bool overlaps(const void* a, size_t a_bytes, const void* b, size_t b_bytes) {
    const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
    return a && b && x < y + b_bytes && y < x + a_bytes;
}
bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }
}  // namespace

int iq4xs_rms_norm_q8_1(const float* X, const float* R, float* H, const float* gamma, float eps, int64_t K,
                        int64_t M, void* ws, size_t ws_bytes, void* stream) {
    if (!X || !ws || K <= 0 || K % QK8_1 != 0 || M <= 0 || K >= MAX_DIM || M >= MAX_DIM) return hipErrorInvalidValue;
    if (!(eps >= 0.0f) || ws_bytes < planar_bytes(K, M) || reinterpret_cast<uintptr_t>(ws) % 256 != 0)
        return hipErrorInvalidValue;
    if (!aligned16(X) || !aligned16(R) || !aligned16(H)) return hipErrorInvalidValue;
    // H is either its own buffer or exactly X or R (an in-place residual add)
    const size_t bytes = (size_t)K * (size_t)M * sizeof(float), wsb = planar_bytes(K, M);
    if ((H != X && overlaps(H, bytes, X, bytes)) || (H != R && overlaps(H, bytes, R, bytes)))
        return hipErrorInvalidValue;
    if (overlaps(ws, wsb, X, bytes) || overlaps(ws, wsb, R, bytes) || overlaps(ws, wsb, H, bytes))
        return hipErrorInvalidValue;
    const Planar p = planar_view(ws, K, M);
    return launch_rms_norm_q8_1(X, R, H, gamma, eps, K, M, p.qs, p.ds, p.hq, as_stream(stream));
}

int iq4xs_swiglu_q8_1(const float* G, const float* U, int64_t K, int64_t M, void* ws, size_t ws_bytes,
                      void* stream) {
    if (!G || !U || !ws || K <= 0 || K % QK8_1 != 0 || M <= 0 || K >= MAX_DIM || M >= MAX_DIM)
        return hipErrorInvalidValue;
    if (ws_bytes < planar_bytes(K, M) || reinterpret_cast<uintptr_t>(ws) % 256 != 0) return hipErrorInvalidValue;
    const Planar p = planar_view(ws, K, M);
    return launch_swiglu_q8_1(G, U, K, M, p.qs, p.ds, p.hq, as_stream(stream));
}

int iq4xs_rms_norm_mul_mat_group(int count, const void* const* W, float* const* Y, const int64_t* N, const float* X,
                                 const float* R, float* H, const float* gamma, float eps, int64_t K, void* stream) {
    if (count < 1 || count > GEMV_GROUP_MAX || !W || !Y || !N || !X || !valid_k(K) || K >= MAX_DIM)
        return hipErrorInvalidValue;
    if (!(eps >= 0.0f) || !aligned16(X) || !aligned16(R) || !aligned16(H) || !aligned16(gamma))
        return hipErrorInvalidValue;
    // workgroup 0 writes H while the others still read X and R: no aliasing
    const size_t bytes = (size_t)K * sizeof(float);
    if (overlaps(H, bytes, X, bytes) || overlaps(H, bytes, R, bytes)) return hipErrorInvalidValue;
    for (int i = 0; i < count; ++i) {
        if (!W[i] || !Y[i] || N[i] <= 0 || N[i] >= MAX_DIM) return hipErrorInvalidValue;
        const size_t yb = (size_t)N[i] * sizeof(float);
        if (overlaps(Y[i], yb, X, bytes) || overlaps(Y[i], yb, R, bytes) || overlaps(Y[i], yb, H, bytes))
            return hipErrorInvalidValue;
    }
    const uint8_t* Wb[GEMV_GROUP_MAX];
    for (int i = 0; i < count; ++i) Wb[i] = static_cast<const uint8_t*>(W[i]);
    return launch_gemv_rms_group(count, Wb, Y, N, X, R, H, gamma, eps, K, as_stream(stream));
}

int iq4xs_rms_norm_mul_mat_swiglu(const void* W_gate, const void* W_up, int64_t N, const float* X, const float* R,
                                  float* H, const float* gamma, float eps, int64_t K, float* Y_gate, float* Y_up,
                                  float* S, void* stream) {
    if (!W_gate || !W_up || !X || !S || !valid_k(K) || K >= MAX_DIM || N <= 0 || N >= MAX_DIM)
        return hipErrorInvalidValue;
    if (!(eps >= 0.0f) || !aligned16(X) || !aligned16(R) || !aligned16(H) || !aligned16(gamma))
        return hipErrorInvalidValue;
    const size_t bytes = (size_t)K * sizeof(float), yb = (size_t)N * sizeof(float);
    if (overlaps(H, bytes, X, bytes) || overlaps(H, bytes, R, bytes)) return hipErrorInvalidValue;
    float* const outs[3] = {Y_gate, Y_up, S};
    for (int i = 0; i < 3; ++i) {
        if (overlaps(outs[i], yb, X, bytes) || overlaps(outs[i], yb, R, bytes) || overlaps(outs[i], yb, H, bytes))
            return hipErrorInvalidValue;
        for (int j = 0; j < i; ++j)
            if (overlaps(outs[i], yb, outs[j], yb)) return hipErrorInvalidValue;
    }
    return launch_gemv_rms_swiglu(static_cast<const uint8_t*>(W_gate), static_cast<const uint8_t*>(W_up), Y_gate,
                                  Y_up, S, N, X, R, H, gamma, eps, K, as_stream(stream));
}

int iq4xs_q8_1_to_blocks(const void* ws, void* blocks, int64_t K, int64_t M, void* stream) {
    if (!ws || !blocks || K <= 0 || K % QK8_1 != 0 || M <= 0 || K >= MAX_DIM || M >= MAX_DIM) return hipErrorInvalidValue;
    const Planar p = planar_view(ws, K, M);
    return launch_planar_to_blocks(p.qs, p.ds, K, M, static_cast<block_q8_1*>(blocks), as_stream(stream));
}

int iq4xs_subblock_sums(const void* W, const void* ws, int32_t* S, float* Y, int64_t K, int64_t N, int64_t M,
                        int path, void* stream) {
    if (!valid_mat(W, ws, Y, K, N, M) || !S) return hipErrorInvalidValue;
    if (path != IQ4XS_PATH_GEMV && path != IQ4XS_PATH_GEMM) return hipErrorInvalidValue;
    return mul_mat_planar(static_cast<const uint8_t*>(W), ws, Y, K, N, M, LAYOUT_MK, path, S, as_stream(stream));
}

int iq4xs_probe_mfma_i8(const int8_t* A, const int8_t* B, int32_t* C, void* stream) {
    if (!A || !B || !C) return hipErrorInvalidValue;
    return launch_probe_mfma(A, B, C, as_stream(stream));
}

int iq4xs_fill_synthetic_weights(void* W, int64_t n_blocks, uint64_t seed, int64_t first_block, void* stream) {
    if (!W || n_blocks <= 0 || first_block < 0) return hipErrorInvalidValue;
    return launch_fill_weights(static_cast<uint8_t*>(W), n_blocks, seed, first_block, as_stream(stream));
}

int iq4xs_fill_synthetic_activations(float* x, int64_t n, uint64_t seed, int outliers, void* stream) {
    if (!x || n <= 0) return hipErrorInvalidValue;
    return launch_fill_activations(x, n, seed, outliers, as_stream(stream));
}

const char* iq4xs_version(void) { return "iq4xs_mi355x 0.1.0 gfx950"; }

}  // extern "C"
