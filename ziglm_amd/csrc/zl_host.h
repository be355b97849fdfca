// Host-side helpers shared by the hip_bridge translation units: error recording, launch
// checks, grid sizing. Not part of the C-ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "../../include/hip_bridge.h"

namespace zl {

// Record an op error for hip_bridge_last_error() (thread-local, first error wins until read).
void set_error(int code);

// After a launch: record hipGetLastError() if the launch failed.
inline void check_launch() {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) set_error((int)e);
}

inline hipStream_t stream_of(HipStream_t s) { return reinterpret_cast<hipStream_t>(s); }

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Compute units of the current device, looked up once (the persistent kernels size their
// grids by it); 256 if the query fails.
inline int device_cus() {
    static std::atomic<int> cus{0};
    int c = cus.load(std::memory_order_relaxed);
    if (c == 0) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || c <= 0) {
            (void)hipGetLastError();  // the failed query's error is not an op's
            c = 256;
        }
        cus.store(c, std::memory_order_relaxed);
    }
    return c;
}

// Matrix-core GEMM (gemm.hip) for batches of at least gemm_mfma_min_batch(qtype, rows, cols) tokens:
// launches and returns true when the type, shape (cols % 32 == 0, K-quants % 256) and
// alignment suit it, else launches nothing and returns false (the caller takes the vector
// path).
// Products at least this deep count as deep: K in two halves at more tiles, and their own crossovers
// (gemm.hip).
constexpr int kSplitMinCols = 4096;
// Rows from which 32-row tiles alone fill the chip's CUs, and most of them.
constexpr int kWideRows = 8192, kMidRows = 5120;
// y[0, n) = 0 (a kernel, not hipMemsetAsync, so that graph captures of the products that
// add into y replay correctly)
void launch_zero_f32(float* y, int64_t n, hipStream_t s);
// The batch from which the matrix-core GEMM (k_gemm_mfma; F16, F32: k_gemm_dense) is faster than
// the kernels for smaller ones, where k_gemm_skinny does not take the call. Wide products (us,
// 10240 x 2560, GEMM / k_gemm_skinny / k_gemv_mb): Q4_0 24 tokens 23.5 / 19.4 / 39.3, 40 tokens
// 25.7 / 32.4 / 40.4; Q4_K 45 33.0 / 38.7 / 30.9, 63 34.8 / 40.4 / 43.4; Q6_K 40 34.2 / 43.8 / 72.0; Q8_0
// 24 24.5 / 26.0 / 39.8; BF16 24 22.0 / 26.3 / 29.3. 6144 x 1536 Q4_K: 45 tokens 16.9 / 16.3 / 20.7, 80
// 23.3 / 29.1 / 21.3, 96 24.5 / 30.1 / 40.8. Narrower ones keep the crossovers of the GEMM against
// k_gemv_mb and the vector kernels: from 64 tokens where deep, else 128 (K-quants 96).
inline int gemm_mfma_min_batch(int qtype, int rows, int cols) {
    const bool deep = cols >= kSplitMinCols, q4k = qtype == HIP_BRIDGE_Q4_K;
    if (qtype == HIP_BRIDGE_F16 || qtype == HIP_BRIDGE_F32) return rows >= kWideRows ? 96 : deep ? 64 : 128;
    const bool single = qtype == HIP_BRIDGE_Q8_0 || qtype == HIP_BRIDGE_BF16;
    if (rows >= kWideRows) return single ? 17 : q4k && cols <= 5120 ? 49 : 33;  // (k_gemv_mb's longest rows)
    if (rows >= kMidRows && !deep) return single ? 33 : q4k ? 96 : 65;
    return q4k || qtype == HIP_BRIDGE_Q6_K ? 96 : deep ? 64 : 128;
}
bool launch_gemm_mfma(int qtype, const void* w, int64_t row_bytes, const float* x, float* y, int rows, int cols,
                      int batch, hipStream_t s);
bool launch_gemm_skinny(int qtype, const void* w, int64_t row_bytes, int x_dtype, const void* x, float* y, int rows,
                        int cols, int batch, hipStream_t s);
// The same for any batch with f32 or bf16 activations and output and an optional up matrix
// (y = gelu(W x) * (U x)); returns 0 when launched, else a HIP_BRIDGE_* code (nothing launched).
int launch_gemm_mfma_ex(int qtype, const void* w, const void* wu, int64_t row_bytes, int x_dtype, const void* x,
                        int y_dtype, void* y, int rows, int cols, int batch, hipStream_t s);

}  // namespace zl
