// kh_rows.h -- int8 rows at any alignment: 16-byte loads that stay inside the
// operand, and rows copied to an aligned stride.  Internal header.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace kh {
namespace rows {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef i32x4 i32x4_any __attribute__((aligned(1)));

// The 16 bytes v of an operand chunk, of which the first `sh` belong to the
// bytes before it (the load was pulled back by sh) and only `n` are wanted.
__device__ __forceinline__ i32x4 tail_bytes(i32x4 v, int sh, int n) {
    typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
    u64x2 w = __builtin_bit_cast(u64x2, v);
    unsigned long long lo = w.x, hi = w.y;
    if (sh >= 8) {
        lo = hi;
        hi = 0;
        sh -= 8;
    }
    if (sh >= 8) lo = 0;
    else if (sh > 0) {
        lo = (lo >> (8 * sh)) | (hi << (64 - 8 * sh));
        hi >>= 8 * sh;
    }
    if (n <= 0) lo = 0;
    else if (n < 8) lo &= (1ull << (8 * n)) - 1;
    if (n <= 8) hi = 0;
    else if (n < 16) hi &= (1ull << (8 * (n - 8))) - 1;
    w.x = lo;
    w.y = hi;
    return __builtin_bit_cast(i32x4, w);
}

// The rows of A [M, K] and then of B [N, K] copied to a stride of Kp bytes (a
// multiple of 16, zeros past K), 16 bytes a thread.  M K and N K >= 16 (an
// operand without rows is not read).
static __global__ __launch_bounds__(256) void pad_rows_kernel(const int8_t* __restrict__ A,
                                                              const int8_t* __restrict__ B, int M, int N, int K,
                                                              int Kp, int8_t* __restrict__ out) {
    const int chunks = Kp / 16;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t row = idx / chunks;
    if (row >= (int64_t)M + N) return;
    const int k = (int)(idx - row * chunks) * 16;
    const int8_t* const base = row < M ? A : B;
    const int64_t off = (row < M ? row : row - M) * K + k, last = (int64_t)(row < M ? M : N) * K - 16;
    const int64_t at = min(off, last);
    i32x4 v = *reinterpret_cast<const i32x4_any*>(base + at);
    if (k + 16 > K) v = tail_bytes(v, (int)(off - at), K - k);
    *reinterpret_cast<i32x4*>(out + idx * 16) = v;
}

}  // namespace rows
}  // namespace kh
