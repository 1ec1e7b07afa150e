// kh_quant.hip -- symmetric int8 quantize / dequantize kernels for gfx950.
//
// Semantics are the reference's, bit for bit (python/kansai/quantize.py:66-70
// and :76):
//   m = max|v|;  s = m / 127.0 in binary64 (1.0 when m == 0);
//   q = clamp(round_half_even(fl64(v / s)), -127, 127);
//   dequantized = (float)((double)q * s).
//
// Exact division without paying a binary64 divide per element: with
// rf = (float)(1.0 / s), the binary32 FMA a = fl32(v * rf + 1.5*2^23) rounds
// the EXACT product v * rf to the nearest integer k (ties to even) and
// d = fl32(v * rf - k) is its distance to k.  |v * rf - v / s| <= 7.6e-6 for
// |v| <= m (rf carries one binary64 and one binary32 rounding, relative
// 6e-8, on a quotient of magnitude <= 127.0000001), and fl64(v / s) is within
// 1.5e-14 of v / s, so when |d| <= 0.5 - kTieEps (kTieEps = 2^-15, four
// times that bound) k is the reference's round(fl64(v / s)).  Elements that
// fail the test take the exact path: a correctly rounded binary64 divide and
// rint (ties to even).  Rows whose max is below 2^-64 (where 127/m could
// overflow binary32) take the exact path throughout.  The fast path cannot
// leave [-127, 127] (|v * rf| <= 127 * (1 + 2^-23)), so only the exact path
// clamps.
//
// Memory layout: x, q row-major contiguous; per-row kernels keep the whole
// row in registers between the absmax and the quantize step, so each fp32
// value crosses HBM once (5 bytes moved per element: 4 read + 1 written).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "kh_common.h"

#pragma clang fp contract(off)

#include "kh_quant_math.h"

using namespace kh::quant;

namespace {

// ---------------------------------------------------------------------------
// Per-row quantize, row held in registers.  ROW_THREADS = 64 * WAVES_PER_ROW
// threads own one row; a 256-thread block owns 256 / ROW_THREADS rows.
// Requires cols % 4 == 0, x 16-byte and q 4-byte aligned, cols <= ROW_THREADS * 4 * VPT.
// ---------------------------------------------------------------------------
// Buffer resources (V#) over one row: loads beyond num_records return 0 and
// stores beyond it are dropped, so the row edge needs no per-access test,
// and each access needs one VGPR offset (the per-step offset is an SGPR).
constexpr int kBufferFlags = 0x00020000;  // dword 3 of a raw gfx9 buffer resource (32-bit data)
constexpr int kCacheNontemporal = 2;      // buffer instruction cache-policy operand: nt

__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_rsrc(const void* base, int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, kBufferFlags);
}

template <int WAVES_PER_ROW, int VPT>
__global__ __launch_bounds__(256) void quant_rows_reg_kernel(const float* __restrict__ x, int8_t* __restrict__ q,
                                                             double* __restrict__ scales, int64_t rows,
                                                             int64_t cols, unsigned* __restrict__ fault) {
    constexpr int ROW_THREADS = 64 * WAVES_PER_ROW;
    constexpr int ROWS_PER_BLOCK = 256 / ROW_THREADS;
    __shared__ unsigned red[4];
    const int lt = threadIdx.x % ROW_THREADS;
    // A wave lies within one row's threads: the row, and so each row's
    // buffer resource, is wave-uniform.  Said explicitly, the resources live
    // in scalar registers; derived from threadIdx.x they were vector values,
    // and every store became a loop over the lanes' distinct resources.
    const int sub = __builtin_amdgcn_readfirstlane((int)threadIdx.x / ROW_THREADS);
    const int64_t row = (int64_t)blockIdx.x * ROWS_PER_BLOCK + sub;
    const bool active = row < rows;
    // An inactive slot (past the last row) gets an empty resource: loads read 0.
    const __amdgpu_buffer_rsrc_t xr = row_rsrc(x + (active ? row : 0) * cols, active ? cols * 4 : 0);

    // Each value is read once: nontemporal loads (the row is not read again
    // unless a group takes the exact path); the codes are stored normally.
    f32x4 v[VPT];
    AbsMax am;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        v[i] = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, lt * 16, i * ROW_THREADS * 16, kCacheNontemporal));
        am.add4(v[i]);
    }
    unsigned mb = wave_max(am.bits());
    if (WAVES_PER_ROW > 1) {
        const int w = threadIdx.x / 64;
        if ((threadIdx.x & 63) == 0) red[w] = mb;
        __syncthreads();
        const int w0 = sub * WAVES_PER_ROW;
        mb = red[w0];
#pragma unroll
        for (int i = 1; i < WAVES_PER_ROW; ++i) mb = max(mb, red[w0 + i]);
    }
    if (!active) return;
    const Scale sc = make_scale(mb);
    if (lt == 0) {
        scales[row] = sc.s;
        if (sc.bad) flag_nonfinite(fault);
    }
    // Fast path for every element, stored as it is produced; the registers
    // holding the row die group by group.  A group of four holding an
    // undecided element (|d| within kTieEps of a half; about one per 30k
    // elements) is then redone from memory by the exact path and stored again.
    const __amdgpu_buffer_rsrc_t qr = row_rsrc(q + row * cols, cols);
    unsigned redo = sc.fast ? 0u : (VPT >= 32 ? ~0u : ((1u << VPT) - 1u));
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        bool ok = true;
        const unsigned w = pack4_fast(v[i], sc.rf, ok);
        if (!ok) redo |= 1u << i;
        __builtin_amdgcn_raw_buffer_store_b32(w, qr, lt * 4, i * ROW_THREADS * 4, 0);
    }
    while (redo) {
        const int i = __builtin_ctz(redo);
        redo &= redo - 1;
        const f32x4 vv =
            __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, lt * 16, i * ROW_THREADS * 16, 0));
        __builtin_amdgcn_raw_buffer_store_b32(pack4(vv, sc), qr, lt * 4, i * ROW_THREADS * 4, 0);
    }
}

// The same for rows of any length >= 4 at any float address and any code
// address: 16-byte loads of x at 4-byte alignment and dword stores at byte
// alignment (both plain global accesses).  A chunk past the row's end is pulled
// back to its last four values, so the last two chunks may overlap and store the
// same codes; chunks wholly past it store nothing.  16384 x 4099: 144 us with one
// value at a time, read twice; now 60.
typedef f32x4 f32x4_any __attribute__((aligned(4)));
typedef unsigned u32_any __attribute__((aligned(1)));

template <int WAVES_PER_ROW, int VPT>
__global__ __launch_bounds__(256) void quant_rows_any_kernel(const float* __restrict__ x, int8_t* __restrict__ q,
                                                             double* __restrict__ scales, int64_t rows, int cols,
                                                             unsigned* __restrict__ fault) {
    constexpr int ROW_THREADS = 64 * WAVES_PER_ROW;
    constexpr int ROWS_PER_BLOCK = 256 / ROW_THREADS;
    __shared__ unsigned red[4];
    const int lt = threadIdx.x % ROW_THREADS;
    const int sub = __builtin_amdgcn_readfirstlane((int)threadIdx.x / ROW_THREADS);
    const int64_t row = (int64_t)blockIdx.x * ROWS_PER_BLOCK + sub;
    const bool active = row < rows;
    const float* const xr = x + (active ? row : rows - 1) * cols;
    int8_t* const qr = q + (active ? row : rows - 1) * cols;
    f32x4 v[VPT];
    AbsMax am;
#pragma unroll
    for (int i = 0; i < VPT; ++i)
        v[i] = *reinterpret_cast<const f32x4_any*>(xr + min((lt + i * ROW_THREADS) * 4, cols - 4));
#pragma unroll
    for (int i = 0; i < VPT; ++i) am.add4(v[i]);
    unsigned mb = wave_max(am.bits());
    if (WAVES_PER_ROW > 1) {
        const int w = threadIdx.x / 64;
        if ((threadIdx.x & 63) == 0) red[w] = mb;
        __syncthreads();
        const int w0 = sub * WAVES_PER_ROW;
        mb = red[w0];
#pragma unroll
        for (int i = 1; i < WAVES_PER_ROW; ++i) mb = max(mb, red[w0 + i]);
    }
    if (!active) return;
    const Scale sc = make_scale(mb);
    if (lt == 0) {
        scales[row] = sc.s;
        if (sc.bad) flag_nonfinite(fault);
    }
    unsigned redo = sc.fast ? 0u : (VPT >= 32 ? ~0u : ((1u << VPT) - 1u));
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int c = (lt + i * ROW_THREADS) * 4;
        bool ok = true;
        const unsigned w = pack4_fast(v[i], sc.rf, ok);
        if (!ok) redo |= 1u << i;
        if (c < cols) *reinterpret_cast<u32_any*>(qr + min(c, cols - 4)) = w;
    }
    while (redo) {
        const int i = __builtin_ctz(redo);
        redo &= redo - 1;
        const int c = (lt + i * ROW_THREADS) * 4, at = min(c, cols - 4);
        if (c < cols) *reinterpret_cast<u32_any*>(qr + at) = pack4(*reinterpret_cast<const f32x4_any*>(xr + at), sc);
    }
}

// Per-row quantize for any shape/alignment: one block per row, two passes
// (the second pass re-reads the row, normally from L2).
__global__ __launch_bounds__(256) void quant_rows_generic_kernel(const float* __restrict__ x, int8_t* __restrict__ q,
                                                                 double* __restrict__ scales, int64_t cols,
                                                                 unsigned* __restrict__ fault) {
    __shared__ unsigned red[4];
    const int64_t row = blockIdx.x;
    const float* xr = x + row * cols;
    AbsMax am;
    for (int64_t c = threadIdx.x; c < cols; c += 256) am.add1(xr[c]);
    unsigned mb = wave_max(am.bits());
    if ((threadIdx.x & 63) == 0) red[threadIdx.x / 64] = mb;
    __syncthreads();
    mb = max(max(red[0], red[1]), max(red[2], red[3]));
    const Scale sc = make_scale(mb);
    if (threadIdx.x == 0) {
        scales[row] = sc.s;
        if (sc.bad) flag_nonfinite(fault);
    }
    int8_t* qr = q + row * cols;
    for (int64_t c = threadIdx.x; c < cols; c += 256) qr[c] = (int8_t)quant_one(xr[c], sc);
}

// ---------------------------------------------------------------------------
// Per-tensor quantize: pass 1 writes one absmax (as bits) per block into
// `partials`; pass 2 reduces the partials in every block, then quantizes.
// VEC: x 16-byte aligned and q 4-byte aligned (float4 body, scalar tail).
// ---------------------------------------------------------------------------
template <bool VEC>
__global__ __launch_bounds__(256) void absmax_partials_kernel(const float* __restrict__ x, int64_t n,
                                                              unsigned* __restrict__ partials) {
    __shared__ unsigned red[4];
    AbsMax am;
    const int64_t stride = (int64_t)gridDim.x * 256;
    if (VEC) {
        const int64_t n4 = n >> 2;
        const f32x4* x4 = reinterpret_cast<const f32x4*>(x);
        for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += stride) am.add4(x4[i]);
        if (blockIdx.x == 0)
            for (int64_t i = n4 * 4 + threadIdx.x; i < n; i += 256) am.add1(x[i]);
    } else {
        for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) am.add1(x[i]);
    }
    unsigned mb = wave_max(am.bits());
    if ((threadIdx.x & 63) == 0) red[threadIdx.x / 64] = mb;
    __syncthreads();
    if (threadIdx.x == 0) partials[blockIdx.x] = max(max(red[0], red[1]), max(red[2], red[3]));
}

constexpr int kTensorUnroll = 4;

template <bool VEC>
__global__ __launch_bounds__(256) void quant_tensor_kernel(const float* __restrict__ x, int64_t n,
                                                           int8_t* __restrict__ q, double* __restrict__ scale,
                                                           const unsigned* __restrict__ partials, int nparts,
                                                           unsigned* __restrict__ fault) {
    __shared__ unsigned red[4];
    const int64_t stride = (int64_t)gridDim.x * 256;
    const int64_t n4 = n >> 2;
    const f32x4* x4 = reinterpret_cast<const f32x4*>(x);
    // kTensorUnroll float4 per thread in flight before the first code is
    // stored (one load at a time per wave left HBM idle between them).  The
    // first batch is requested before the partials, so the workgroup waits
    // for one memory round trip before its first store, not two.
    constexpr int U = kTensorUnroll;
    const int64_t first = (int64_t)blockIdx.x * 256 * U + threadIdx.x;
    f32x4 v[U];
    auto load = [&](int64_t i0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t i = i0 + (int64_t)u * 256;
            v[u] = i < n4 ? x4[i] : f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };
    if (VEC) load(first);
    const unsigned mb = block_reduce_partials(partials, nparts, red);
    const Scale sc = make_scale(mb);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        scale[0] = sc.s;
        if (sc.bad) flag_nonfinite(fault);
    }
    if (VEC) {
        unsigned* q4 = reinterpret_cast<unsigned*>(q);
        for (int64_t i0 = first; i0 < n4; i0 += stride * U) {
            if (i0 != first) load(i0);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t i = i0 + (int64_t)u * 256;
                if (i < n4) q4[i] = pack4(v[u], sc);
            }
        }
        if (blockIdx.x == 0)
            for (int64_t i = n4 * 4 + threadIdx.x; i < n; i += 256) q[i] = (int8_t)quant_one(x[i], sc);
    } else {
        for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) q[i] = (int8_t)quant_one(x[i], sc);
    }
}

// Per-tensor quantize of a small tensor (n <= kSmallPer * 4 * 1024, x 16-byte
// and q 4-byte aligned) in one launch: one 1024-thread workgroup holds the
// values in registers, reduces the absmax, and stores the codes -- the same
// arithmetic as the two-pass path, without the second launch (latency-bound
// sizes such as a Linear's activations).
constexpr int kSmallThreads = 1024;
constexpr int kSmallPer = 16;  // float4 per thread
constexpr int64_t kSmallTensor = (int64_t)kSmallPer * 4 * kSmallThreads;

__global__ __launch_bounds__(kSmallThreads) void quant_tensor_small_kernel(const float* __restrict__ x, int64_t n,
                                                                           int8_t* __restrict__ q,
                                                                           double* __restrict__ scale,
                                                                           unsigned* __restrict__ fault) {
    __shared__ unsigned red[kSmallThreads / 64];
    const int tid = threadIdx.x;
    const int n4 = (int)(n >> 2), tail = (int)(n - 4 * (int64_t)n4);
    const f32x4* x4 = reinterpret_cast<const f32x4*>(x);
    f32x4 v[kSmallPer];
    AbsMax am;
#pragma unroll
    for (int i = 0; i < kSmallPer; ++i) {
        const int idx = tid + i * kSmallThreads;
        v[i] = idx < n4 ? x4[idx] : f32x4{0.f, 0.f, 0.f, 0.f};
        if (idx < n4) am.add4(v[i]);
    }
    const float xt = tid < tail ? x[4 * (int64_t)n4 + tid] : 0.0f;
    if (tid < tail) am.add1(xt);
    unsigned mb = wave_max(am.bits());
    if ((tid & 63) == 0) red[tid >> 6] = mb;
    __syncthreads();
    mb = red[0];
#pragma unroll
    for (int w = 1; w < kSmallThreads / 64; ++w) mb = max(mb, red[w]);
    const Scale sc = make_scale(mb);
    if (tid == 0) {
        scale[0] = sc.s;
        if (sc.bad) flag_nonfinite(fault);
    }
    unsigned* q4 = reinterpret_cast<unsigned*>(q);
#pragma unroll
    for (int i = 0; i < kSmallPer; ++i) {
        const int idx = tid + i * kSmallThreads;
        if (idx < n4) q4[idx] = pack4(v[i], sc);
    }
    if (tid < tail) q[4 * (int64_t)n4 + tid] = (int8_t)quant_one(xt, sc);
}

// ---------------------------------------------------------------------------
// Per-column (per output channel) absmax of a [k, n] weight, and the
// transpose-quantize that packs codes K-contiguous ([n, k]).
// ---------------------------------------------------------------------------
__global__ void fill_u32_kernel(unsigned* __restrict__ p, int64_t count, unsigned value) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) p[i] = value;
}

// Rows of w per absmax workgroup.  Each workgroup writes its columns' maxima as
// one row of partials, which the packing kernel reduces: no atomics and no
// clearing launch.  At least kColRows rows a workgroup, and no more partials than
// the scratch area's initial 1 MiB holds (one a column for the widest), so that a
// weight quantized under graph capture does not make it grow.
constexpr int64_t kColRows = 128, kColPartBytes = 1 << 20;

// VEC (n % 4 == 0, w 16-byte aligned): a thread takes four columns, the
// workgroup 256 of them and four rows at a time, eight rows' loads in flight per
// thread (one at a time, each waiting for the last, 4096 x 11008 took 43 us,
// now 27, 6.7 TB/s).  Otherwise a thread takes one column.
template <bool VEC>
__global__ __launch_bounds__(256) void col_absmax_kernel(const float* __restrict__ w, int64_t k, int64_t n,
                                                         int rows_per, unsigned* __restrict__ partials) {
    constexpr int U = 8;
    const int64_t i0 = (int64_t)blockIdx.y * rows_per, last = min(k, i0 + rows_per) - 1;
    if (VEC) {
        __shared__ unsigned red[4][256];
        const int c = threadIdx.x & 63, r = threadIdx.x >> 6;
        // Columns and rows past the end read the last one again.
        const int64_t j = min((int64_t)blockIdx.x * 256 + c * 4, n - 4);
        unsigned m[4] = {0, 0, 0, 0};
        for (int64_t i = i0 + r; i <= last; i += 4 * U) {
            f32x4 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = *reinterpret_cast<const f32x4*>(w + min(i + 4 * u, last) * n + j);
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int e = 0; e < 4; ++e) m[e] = max(m[e], abs_bits(v[u][e]));
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) red[r][c * 4 + e] = m[e];
        __syncthreads();
        const int64_t jo = (int64_t)blockIdx.x * 256 + threadIdx.x;
        const int t = threadIdx.x;
        if (jo < n) partials[blockIdx.y * n + jo] = max(max(red[0][t], red[1][t]), max(red[2][t], red[3][t]));
    } else {
        const int64_t jo = (int64_t)blockIdx.x * 256 + threadIdx.x, j = min(jo, n - 1);
        unsigned m = 0;
        for (int64_t i = i0; i <= last; i += U) {
            float v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = w[min(i + u, last) * n + j];
#pragma unroll
            for (int u = 0; u < U; ++u) m = max(m, abs_bits(v[u]));
        }
        if (jo < n) partials[blockIdx.y * n + jo] = m;
    }
}

// Quantizes a tile of 128 k x 64 columns and writes it K-contiguous (q_packed[j
// * k + i]) with the scales.  PER_COL: `maxbits` holds nparts rows of n partial
// maxima; otherwise nparts maxima of the whole weight.
//
// A thread takes four columns of eight rows, two runs of four consecutive k, so
// that four codes of one column make a dword of the LDS tile (33 dwords a
// column: the 64 lanes' writes fall on distinct banks).  A column's 128 codes
// then leave as one 128-byte run.  A workgroup walks the tiles blockIdx.y,
// blockIdx.y + gridDim.y, ... of its columns, so the scales (two binary64 divides
// behind the partials' loads) are made once, under the first tile's loads, and
// the next tile's loads are in flight while one is written.  4096 x 11008: 36.6
// us traced, against 50 for 64 x 64 tiles of byte writes and 43.5 with one tile a workgroup.
constexpr int kPackK = 128, kPackN = 64, kPackRow = kPackK / 4 + 1;

template <bool PER_COL, bool VEC>
__global__ __launch_bounds__(256) void pack_quant_kernel(const float* __restrict__ w, int64_t k, int64_t n,
                                                         const unsigned* __restrict__ maxbits, int nparts,
                                                         int8_t* __restrict__ qp, double* __restrict__ scales,
                                                         unsigned* __restrict__ fault) {
    __shared__ unsigned tile[kPackN * kPackRow];
    __shared__ double s_col[kPackN];
    __shared__ float rf_col[kPackN];
    __shared__ unsigned flags_col[kPackN];  // bit 0 fast, bit 1 bad
    __shared__ unsigned red[4];
    const int64_t j0 = (int64_t)blockIdx.x * kPackN;
    const int t = threadIdx.x, cg = t & 15, rg = t >> 4;

    // v[p][e]: row 64 p + 4 rg + e, columns 4 cg .. 4 cg + 3; past the end, the
    // last one again (never stored).
    f32x4 v[2][4];
    auto load = [&](int64_t i0) {
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float* const row = w + min(i0 + 64 * p + 4 * rg + e, k - 1) * n;
                if (VEC) {
                    v[p][e] = *reinterpret_cast<const f32x4*>(row + min(j0 + 4 * cg, n - 4));
                } else {
#pragma unroll
                    for (int c = 0; c < 4; ++c) v[p][e][c] = row[min(j0 + 4 * cg + c, n - 1)];
                }
            }
    };
    load((int64_t)blockIdx.y * kPackK);
    __builtin_amdgcn_sched_barrier(0);
    if (PER_COL) {
        if (t < kPackN) {
            const int64_t j = j0 + t, jc = min(j, n - 1);
            unsigned mb = 0;
#pragma unroll 8
            for (int q = 0; q < nparts; ++q) mb = max(mb, maxbits[q * n + jc]);
            const Scale sc = make_scale(mb);
            s_col[t] = sc.s;
            rf_col[t] = sc.rf;
            flags_col[t] = (sc.fast ? 1u : 0u) | (sc.bad ? 2u : 0u);
            if (blockIdx.y == 0 && j < n) {
                scales[j] = sc.s;
                if (sc.bad) flag_nonfinite(fault);
            }
        }
    } else {
        const Scale sc = make_scale(block_reduce_partials(maxbits, nparts, red));
        if (t < kPackN) {
            s_col[t] = sc.s;
            rf_col[t] = sc.rf;
            flags_col[t] = (sc.fast ? 1u : 0u) | (sc.bad ? 2u : 0u);
        }
        if (blockIdx.x == 0 && blockIdx.y == 0 && t == 0) {
            scales[0] = sc.s;
            if (sc.bad) flag_nonfinite(fault);
        }
    }
    __syncthreads();
    Scale sc[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        sc[c].s = s_col[4 * cg + c];
        sc[c].rf = rf_col[4 * cg + c];
        sc[c].fast = flags_col[4 * cg + c] & 1u;
        sc[c].bad = flags_col[4 * cg + c] & 2u;
    }
    for (int64_t i0 = (int64_t)blockIdx.y * kPackK; i0 < k; i0 += (int64_t)gridDim.y * kPackK) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int p = 0; p < 2; ++p)
                tile[(4 * cg + c) * kPackRow + 16 * p + rg] =
                    pack4(f32x4{v[p][0][c], v[p][1][c], v[p][2][c], v[p][3][c]}, sc[c]);
        const int64_t next = i0 + (int64_t)gridDim.y * kPackK;
        if (next < k) load(next);
        __syncthreads();
        // Thread t writes 16 codes of columns t / 8 and 32 + t / 8.
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int col = 32 * h + (t >> 3), part = t & 7;
            const int64_t jo = j0 + col, io = i0 + part * 16;
            if (jo >= n || io >= k) continue;
            const unsigned* const src = tile + col * kPackRow + part * 4;
            int8_t* const dst = qp + jo * k + io;
            if (io + 16 <= k && kh::aligned(dst, 16)) {
                *reinterpret_cast<uint4*>(dst) = uint4{src[0], src[1], src[2], src[3]};
            } else {
                for (int e = 0; e < 16 && io + e < k; ++e) dst[e] = (int8_t)(src[e >> 2] >> (8 * (e & 3)));
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Dequantize (quantize.py:76): out = (float)((double)q * s).
// ---------------------------------------------------------------------------
__device__ __forceinline__ float deq_one(int8_t q, double s) { return (float)((double)q * s); }

__device__ __forceinline__ f32x4 deq4(unsigned w, double s) {
    return f32x4{deq_one((int8_t)(w & 0xFF), s), deq_one((int8_t)((w >> 8) & 0xFF), s),
                 deq_one((int8_t)((w >> 16) & 0xFF), s), deq_one((int8_t)(w >> 24), s)};
}

// Vector dequantize.  Block (bx, row) covers kDeqPerBlock consecutive codes of
// one row (per-row scale uniform over the block; per-tensor: rows == 1).
// Each lane reads 4 codes (one u32) and writes one 16-byte float4 per step,
// so every load and store instruction covers a contiguous span of the wave.
// Codes load through the cache normally; the fp32 output is written with
// nontemporal stores (measured fastest of the four load/store policy pairs).
// Requires cols % 4 == 0, q 4-byte and out 16-byte aligned.
// STEPS of 1024 codes per block: 4 for rows of more than 3072 codes, fewer
// for shorter rows, so that a block issues no steps past its row's end.
constexpr int kDeqSteps = 4;
typedef int i32x4raw __attribute__((ext_vector_type(4)));  // a 16-byte buffer store's data
constexpr int kDeqPerBlock = 256 * 4 * kDeqSteps;

template <int STEPS>
__global__ __launch_bounds__(256) void dequant_vec_kernel(const int8_t* __restrict__ q, int64_t cols,
                                                          const double* __restrict__ scales, int per_row,
                                                          float* __restrict__ out) {
    const int64_t row = blockIdx.y;
    const double s = scales[per_row ? row : 0];
    // The block's span of the row, as buffer resources: every step's load is
    // issued before the first conversion (loads past the row's end read 0,
    // stores past it are dropped).  With a bounds test around each step the
    // compiler waited for each load before issuing the next.
    constexpr int kPerBlock = 1024 * STEPS;
    const int64_t c0 = (int64_t)blockIdx.x * kPerBlock;
    const int span = (int)min((int64_t)kPerBlock, cols - c0);
    const __amdgpu_buffer_rsrc_t rq = row_rsrc(q + row * cols + c0, span);
    const __amdgpu_buffer_rsrc_t ro = row_rsrc(out + row * cols + c0, (int64_t)span * 4);
    unsigned w[STEPS];
#pragma unroll
    for (int step = 0; step < STEPS; ++step)
        w[step] = __builtin_amdgcn_raw_buffer_load_b32(rq, threadIdx.x * 4, step * 1024, 0);
#pragma unroll
    for (int step = 0; step < STEPS; ++step)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(i32x4raw, deq4(w[step], s)), ro, threadIdx.x * 16,
                                               step * 4096, kCacheNontemporal);
}

// The same for rows of any length >= 7 at any code and float address: the row's
// values from its first 16-byte boundary on are stored as 16-byte runs (their
// codes loaded as dwords at any address), the up to three before and behind them
// one by one.  16384 x 4099: 136 us one value at a time, 106 with unaligned 16-byte
// stores; now 60.
template <int STEPS>
__global__ __launch_bounds__(256) void dequant_any_kernel(const int8_t* __restrict__ q, int64_t cols,
                                                          const double* __restrict__ scales, int per_row,
                                                          float* __restrict__ out) {
    const int64_t row = blockIdx.y;
    const double s = scales[per_row ? row : 0];
    const int8_t* const qr = q + row * cols;
    float* const orow = out + row * cols;
    const int head = (int)(-(reinterpret_cast<uintptr_t>(orow) >> 2) & 3);
    const int64_t end = head + (cols - head) / 4 * 4;  // of the 16-byte runs (at least one)
    const int64_t c0 = head + (int64_t)blockIdx.x * 1024 * STEPS + threadIdx.x * 4;
    unsigned w[STEPS];
#pragma unroll
    for (int step = 0; step < STEPS; ++step)
        w[step] = *reinterpret_cast<const u32_any*>(qr + min(c0 + step * 1024, end - 4));
#pragma unroll
    for (int step = 0; step < STEPS; ++step)
        if (c0 + step * 1024 < end)
            __builtin_nontemporal_store(deq4(w[step], s), reinterpret_cast<f32x4*>(orow + c0 + step * 1024));
    if (blockIdx.x == 0 && threadIdx.x < 8) {
        const int t = threadIdx.x & 3;
        const int64_t c = threadIdx.x < 4 ? t : end + t;
        if (threadIdx.x < 4 ? t < head : c < cols) orow[c] = deq_one(qr[c], s);
    }
}

// Any shape / alignment.
__global__ __launch_bounds__(256) void dequant_generic_kernel(const int8_t* __restrict__ q, int64_t n, int64_t cols,
                                                              const double* __restrict__ scales, int per_row,
                                                              float* __restrict__ out) {
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride)
        out[i] = deq_one(q[i], scales[per_row ? i / cols : 0]);
}

// out[i, j] = (float)((double)qp[j * k + i] * s_j), back to the [k, n] layout.
constexpr int kTile = 64;

__global__ __launch_bounds__(256) void dequant_packed_kernel(const int8_t* __restrict__ qp, int64_t k, int64_t n,
                                                             const double* __restrict__ scales, int64_t scales_n,
                                                             float* __restrict__ out) {
    __shared__ __attribute__((aligned(16))) int8_t tile[kTile][kTile + 4];
    const int64_t i0 = (int64_t)blockIdx.y * kTile;
    const int64_t j0 = (int64_t)blockIdx.x * kTile;
    const int t = threadIdx.x;
    // Read codes: thread (jj = t / 4) reads 16 k of column j0 + jj.
    {
        const int jj = t >> 2;
        const int ii = (t & 3) * 16;
        for (int e = 0; e < 16; ++e) {
            const int64_t i = i0 + ii + e, j = j0 + jj;
            tile[jj][ii + e] = (i < k && j < n) ? qp[j * k + i] : (int8_t)0;
        }
    }
    __syncthreads();
    const int c = t & 63;
    const int64_t j = j0 + c;
    if (j >= n) return;
    const double s = scales[scales_n == 1 ? 0 : j];
    for (int r = t >> 6; r < kTile; r += 4) {
        const int64_t i = i0 + r;
        if (i < k) out[i * n + j] = deq_one(tile[c][r], s);
    }
}

int grid_for(int64_t work_items, int per_thread, int cap) {
    int64_t g = (work_items + 256LL * per_thread - 1) / (256LL * per_thread);
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return (int)g;
}

constexpr int kMaxPartials = 1024;

}  // namespace


namespace {

__global__ void fill_f64_kernel(double* __restrict__ p, int64_t count, double value) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) p[i] = value;
}

// Empty slices: max() defaults to 0.0, so the scale is 1.0 (quantize.py:67-68).
int fill_scales_one(kh::Device* d, double* scales, int64_t count) {
    fill_f64_kernel<<<(unsigned)((count + 255) / 256), 256, 0, d->stream>>>(scales, count, 1.0);
    return kh::launch_status("fill_f64");
}

// Pass 1 of a per-tensor quantize: per-block absmax bits into library scratch.
int tensor_absmax(kh::Device* d, const float* x, int64_t n, bool vec, unsigned** partials, int* nparts) {
    const int g = grid_for(vec ? (n >> 2) : n, 8, kMaxPartials);
    unsigned* p = static_cast<unsigned*>(kh::scratch_area(d, kMaxPartials * sizeof(unsigned)));
    if (!p) return KH_ERR_OOM;
    if (vec)
        absmax_partials_kernel<true><<<g, 256, 0, d->stream>>>(x, n, p);
    else
        absmax_partials_kernel<false><<<g, 256, 0, d->stream>>>(x, n, p);
    *partials = p;
    *nparts = g;
    return kh::launch_status("absmax_partials");
}

}  // namespace

extern "C" {

int kh_quantize_tensor(const float* x, int64_t n, int8_t* q, double* scale) {
    KH_REQUIRE(n >= 0, "kh_quantize_tensor: negative size");
    KH_REQUIRE(scale, "kh_quantize_tensor: null scale");
    KH_REQUIRE(n == 0 || (x && q), "kh_quantize_tensor: null pointer");
    KH_DEVICE_OR_RETURN(d);
    if (n == 0) return fill_scales_one(d, scale, 1);
    const bool vec = kh::aligned(x, 16) && kh::aligned(q, 4);
    if (vec && n <= kSmallTensor) {
        quant_tensor_small_kernel<<<1, kSmallThreads, 0, d->stream>>>(x, n, q, scale, d->fault);
        return kh::launch_status("quant_tensor_small");
    }
    unsigned* partials = nullptr;
    int nparts = 0;
    int rc = tensor_absmax(d, x, n, vec, &partials, &nparts);
    if (rc) return rc;
    const int g = grid_for(vec ? (n >> 2) : n, 8, 8192);
    if (vec)
        quant_tensor_kernel<true><<<g, 256, 0, d->stream>>>(x, n, q, scale, partials, nparts, d->fault);
    else
        quant_tensor_kernel<false><<<g, 256, 0, d->stream>>>(x, n, q, scale, partials, nparts, d->fault);
    return kh::launch_status("quant_tensor");
}

int kh_absmax_parts(const float* x, int64_t n, unsigned* parts, int max_parts, int* nparts) {
    KH_REQUIRE(n >= 0 && max_parts > 0 && parts && nparts, "kh_absmax_parts: bad arguments");
    KH_REQUIRE(n == 0 || x, "kh_absmax_parts: null pointer");
    KH_DEVICE_OR_RETURN(d);
    if (n == 0) {
        fill_u32_kernel<<<1, 256, 0, d->stream>>>(parts, 1, 0u);
        *nparts = 1;
        return kh::launch_status("fill_u32");
    }
    const bool vec = kh::aligned(x, 16);
    const int g = grid_for(vec ? (n >> 2) : n, 8, std::min(max_parts, kMaxPartials));
    if (vec)
        absmax_partials_kernel<true><<<g, 256, 0, d->stream>>>(x, n, parts);
    else
        absmax_partials_kernel<false><<<g, 256, 0, d->stream>>>(x, n, parts);
    *nparts = g;
    return kh::launch_status("absmax_partials");
}

int kh_quantize_tensor_parts(const float* x, int64_t n, const unsigned* parts, int nparts, int8_t* q, double* scale) {
    KH_REQUIRE(n >= 0, "kh_quantize_tensor_parts: negative size");
    KH_REQUIRE(scale && parts && nparts > 0, "kh_quantize_tensor_parts: bad partials or scale");
    KH_REQUIRE(n == 0 || (x && q), "kh_quantize_tensor_parts: null pointer");
    KH_DEVICE_OR_RETURN(d);
    if (n == 0) return fill_scales_one(d, scale, 1);
    const bool vec = kh::aligned(x, 16) && kh::aligned(q, 4);
    const int g = grid_for(vec ? (n >> 2) : n, 8, 8192);
    if (vec)
        quant_tensor_kernel<true><<<g, 256, 0, d->stream>>>(x, n, q, scale, parts, nparts, d->fault);
    else
        quant_tensor_kernel<false><<<g, 256, 0, d->stream>>>(x, n, q, scale, parts, nparts, d->fault);
    return kh::launch_status("quant_tensor");
}

int kh_quantize_rows(const float* x, int64_t rows, int64_t cols, int8_t* q, double* scales) {
    KH_REQUIRE(rows >= 0 && cols >= 0, "kh_quantize_rows: negative shape");
    if (rows == 0) return KH_OK;
    KH_REQUIRE(scales, "kh_quantize_rows: null scales");
    KH_REQUIRE(cols == 0 || (x && q), "kh_quantize_rows: null pointer");
    KH_REQUIRE(rows <= 0x7FFFFFFFLL, "kh_quantize_rows: too many rows");
    KH_DEVICE_OR_RETURN(d);
    if (cols == 0) return fill_scales_one(d, scales, rows);
    const bool vec = (cols % 4 == 0) && kh::aligned(x, 16) && kh::aligned(q, 4);
    const bool any = !vec && cols >= 4 && kh::aligned(x, 4);
    // The smallest row slot (threads x float4 per thread) that holds the row:
    // slots past the row's end still cost their loads' issue.
    auto go = [&](auto waves, auto vpt) {
        constexpr int W = decltype(waves)::value, V = decltype(vpt)::value;
        const unsigned blocks = (unsigned)((rows * W + 3) / 4);
        if (vec) quant_rows_reg_kernel<W, V><<<blocks, 256, 0, d->stream>>>(x, q, scales, rows, cols, d->fault);
        else quant_rows_any_kernel<W, V><<<blocks, 256, 0, d->stream>>>(x, q, scales, rows, (int)cols, d->fault);
    };
    using std::integral_constant;
    using W1 = integral_constant<int, 1>;
    using W2 = integral_constant<int, 2>;
    using W4 = integral_constant<int, 4>;
    if (!(vec || any) || cols > 32768)
        quant_rows_generic_kernel<<<(unsigned)rows, 256, 0, d->stream>>>(x, q, scales, cols, d->fault);
    else if (cols <= 256) go(W1(), integral_constant<int, 1>());
    else if (cols <= 512) go(W1(), integral_constant<int, 2>());
    else if (cols <= 1024) go(W1(), integral_constant<int, 4>());
    else if (cols <= 1536) go(W2(), integral_constant<int, 3>());
    else if (cols <= 2048) go(W2(), integral_constant<int, 4>());
    else if (cols <= 4096) go(W4(), integral_constant<int, 4>());
    else if (cols <= 6144) go(W4(), integral_constant<int, 6>());
    else if (cols <= 8192) go(W4(), integral_constant<int, 8>());
    else if (cols <= 12288) go(W4(), integral_constant<int, 12>());
    else if (cols <= 16384) go(W4(), integral_constant<int, 16>());
    else go(W4(), integral_constant<int, 32>());
    return kh::launch_status("quant_rows");
}

static int quantize_packed(const float* w, int64_t k, int64_t n, int8_t* qp, double* scales, bool per_col) {
    KH_DEVICE_OR_RETURN(d);
    // As many workgroups as are resident at once (five to a CU).
    const int64_t tiles_n = (n + kPackN - 1) / kPackN, tiles_k = (k + kPackK - 1) / kPackK;
    const dim3 tiles((unsigned)tiles_n,
                     (unsigned)std::min(tiles_k, std::max<int64_t>(1, 5 * (int64_t)d->cus / tiles_n)));
    const bool vec = n % 4 == 0 && kh::aligned(w, 16);
    unsigned* partials = nullptr;
    int nparts = 0;
    if (per_col) {
        const int64_t most = std::max<int64_t>(1, kColPartBytes / (n * (int64_t)sizeof(unsigned)));
        const int64_t rows_per = std::max<int64_t>(kColRows, (k + most - 1) / most);
        nparts = (int)((k + rows_per - 1) / rows_per);
        partials = static_cast<unsigned*>(kh::scratch_area(d, (size_t)nparts * (size_t)n * sizeof(unsigned)));
        if (!partials) return KH_ERR_OOM;
        const dim3 g((unsigned)((n + 255) / 256), (unsigned)nparts);
        if (vec) col_absmax_kernel<true><<<g, 256, 0, d->stream>>>(w, k, n, (int)rows_per, partials);
        else col_absmax_kernel<false><<<g, 256, 0, d->stream>>>(w, k, n, (int)rows_per, partials);
        if (vec)
            pack_quant_kernel<true, true><<<tiles, 256, 0, d->stream>>>(w, k, n, partials, nparts, qp, scales, d->fault);
        else
            pack_quant_kernel<true, false><<<tiles, 256, 0, d->stream>>>(w, k, n, partials, nparts, qp, scales, d->fault);
    } else {
        int rc = tensor_absmax(d, w, k * n, kh::aligned(w, 16), &partials, &nparts);
        if (rc) return rc;
        if (vec)
            pack_quant_kernel<false, true><<<tiles, 256, 0, d->stream>>>(w, k, n, partials, nparts, qp, scales, d->fault);
        else
            pack_quant_kernel<false, false><<<tiles, 256, 0, d->stream>>>(w, k, n, partials, nparts, qp, scales, d->fault);
    }
    return kh::launch_status("pack_quant");
}

int kh_quantize_cols_packed(const float* w, int64_t k, int64_t n, int8_t* q_packed, double* scales) {
    KH_REQUIRE(k >= 0 && n >= 0, "kh_quantize_cols_packed: negative shape");
    if (n == 0) return KH_OK;
    KH_REQUIRE(scales, "kh_quantize_cols_packed: null scales");
    if (k == 0) {
        KH_DEVICE_OR_RETURN(d);
        return fill_scales_one(d, scales, n);
    }
    KH_REQUIRE(w && q_packed, "kh_quantize_cols_packed: null pointer");
    KH_REQUIRE(n <= 0x7FFFFFFFLL * 64 && k <= 0xFFFFLL * 64, "kh_quantize_cols_packed: shape too large");
    return quantize_packed(w, k, n, q_packed, scales, true);
}

int kh_quantize_tensor_packed(const float* w, int64_t k, int64_t n, int8_t* q_packed, double* scale) {
    KH_REQUIRE(k >= 0 && n >= 0, "kh_quantize_tensor_packed: negative shape");
    KH_REQUIRE(scale, "kh_quantize_tensor_packed: null scale");
    if (k == 0 || n == 0) {
        KH_DEVICE_OR_RETURN(d);
        return fill_scales_one(d, scale, 1);
    }
    KH_REQUIRE(w && q_packed, "kh_quantize_tensor_packed: null pointer");
    KH_REQUIRE(n <= 0x7FFFFFFFLL * 64 && k <= 0xFFFFLL * 64, "kh_quantize_tensor_packed: shape too large");
    return quantize_packed(w, k, n, q_packed, scale, false);
}

static int dequant(const int8_t* q, int64_t rows, int64_t cols, const double* scales, float* out, bool per_row) {
    KH_DEVICE_OR_RETURN(d);
    const bool vec = (cols % 4 == 0) && kh::aligned(q, 4) && kh::aligned(out, 16);
    const bool any = !vec && cols >= 7 && kh::aligned(out, 4);
    if ((vec || any) && rows <= 0x7FFFFFFFLL && (cols + kDeqPerBlock - 1) / kDeqPerBlock <= 0x7FFFFFFFLL) {
        // As few workgroups of up to 4 steps as the row needs, evenly filled.
        const int64_t per = (cols + kDeqPerBlock - 1) / kDeqPerBlock;
        const int steps = (int)((cols + 1024 * per - 1) / (1024 * per));
        const unsigned gx = (unsigned)((cols + 1024 * steps - 1) / (1024 * steps));
        // grid.y is limited to 65535: walk the rows in slabs.
        for (int64_t r0 = 0; r0 < rows; r0 += 65535) {
            const dim3 g(gx, (unsigned)min((int64_t)65535, rows - r0));
            const int8_t* const qq = q + r0 * cols;
            const double* const ss = scales + (per_row ? r0 : 0);
            float* const oo = out + r0 * cols;
            auto go = [&](auto st) {
                constexpr int S = decltype(st)::value;
                if (vec) dequant_vec_kernel<S><<<g, 256, 0, d->stream>>>(qq, cols, ss, per_row ? 1 : 0, oo);
                else dequant_any_kernel<S><<<g, 256, 0, d->stream>>>(qq, cols, ss, per_row ? 1 : 0, oo);
            };
            if (steps == 4) go(std::integral_constant<int, 4>());
            else if (steps == 3) go(std::integral_constant<int, 3>());
            else if (steps == 2) go(std::integral_constant<int, 2>());
            else go(std::integral_constant<int, 1>());
        }
    } else {
        const int64_t n = rows * cols;
        const int g = grid_for(n, 16, 16384);
        dequant_generic_kernel<<<g, 256, 0, d->stream>>>(q, n, cols, scales, per_row ? 1 : 0, out);
    }
    return kh::launch_status("dequant");
}

int kh_dequantize_tensor(const int8_t* q, int64_t n, const double* scale, float* out) {
    KH_REQUIRE(n >= 0, "kh_dequantize_tensor: negative size");
    if (n == 0) return KH_OK;
    KH_REQUIRE(q && scale && out, "kh_dequantize_tensor: null pointer");
    return dequant(q, 1, n, scale, out, false);
}

int kh_dequantize_rows(const int8_t* q, int64_t rows, int64_t cols, const double* scales, float* out) {
    KH_REQUIRE(rows >= 0 && cols >= 0, "kh_dequantize_rows: negative shape");
    if (rows == 0 || cols == 0) return KH_OK;
    KH_REQUIRE(q && scales && out, "kh_dequantize_rows: null pointer");
    return dequant(q, rows, cols, scales, out, true);
}

int kh_dequantize_packed(const int8_t* q_packed, int64_t k, int64_t n, const double* scales, int64_t scales_n,
                         float* out) {
    KH_REQUIRE(k >= 0 && n >= 0, "kh_dequantize_packed: negative shape");
    if (k == 0 || n == 0) return KH_OK;
    KH_REQUIRE(q_packed && scales && out, "kh_dequantize_packed: null pointer");
    KH_REQUIRE(scales_n == 1 || scales_n == n, "kh_dequantize_packed: scales_n must be 1 or n");
    KH_REQUIRE(n <= 0x7FFFFFFFLL * 64 && k <= 0xFFFFLL * 64, "kh_dequantize_packed: shape too large");
    KH_DEVICE_OR_RETURN(d);
    dim3 g((unsigned)((n + kTile - 1) / kTile), (unsigned)((k + kTile - 1) / kTile));
    dequant_packed_kernel<<<g, 256, 0, d->stream>>>(q_packed, k, n, scales, scales_n, out);
    return kh::launch_status("dequant_packed");
}

}  // extern "C"
