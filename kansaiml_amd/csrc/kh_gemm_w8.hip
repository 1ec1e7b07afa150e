// kh_gemm_w8.hip -- fp32 activations times an int8 weight: the reference's
// weight-only Linear, x.matmul(dequantize(W)).add(bias)
// (python/kansai/quantize.py:115-122), without the fp32 weight being written.
//
//   out[i, j] = (float)((double)(sum_k x[i, k] q[j, k]) * s_j) + bias[j]
//
// The reference rounds each weight q s to binary32 and sums in binary32; here
// the scale multiplies the sum, so the weights are exact, and the products run
// on the bf16 matrix cores, which are 16 times the fp32 ones: a code needs 8
// bits, which bf16 holds, and x = h + m + l exactly as three bf16 values of 8
// significand bits each (round to nearest, each of what the ones before left), so
// three products x code per value are exact and only their binary32 sums round.
// Error against binary64 at 64 x 4096 x 4096: 6.3e-7 of the result's norm
// unsplit, 2.2e-7 with K split in eight; the dequantize + fp32 matmul it replaces
// 1.1e-6.  Time there (one MI355X): 389 -> 22 us; 4096^3 1055 -> 410, 300 x 487 x
// 1728 227 -> 16.
//
// Range: every row of x is first scaled by a power of two that brings its
// largest finite magnitude to [2^100, 2^101), undone in binary64 in the epilogue:
// the sums stay below 2^127 (K <= 2^19), and values down to 2^-203 of the largest
// keep all three parts above binary32's smallest normal.  A row that spans more
// (it must hold values both above 2^73 and below 2^-73) has its outputs computed
// by the plain binary32 loop in the epilogue.  A NaN or infinity is its own first
// part, with zeros behind it.
//
// Two launches: split_rows_kernel (x -> planes h, m, l [3, rows, Kp] and the row
// factors) and gemm_w8_kernel, plus a sum of partials where K is split.
//
// gemm_w8_kernel: workgroup tile BM x BN, 4 waves as 2 x 2, 32x32 blocks of
// v_mfma_f32_32x32x16_bf16, K in steps of 64 through a ring of NS LDS stages
// (three planes of BM x 128 bytes, BN x 64 bytes of codes) filled by LDS-DMA; the
// ring and the fragments' double buffering are gemm_i8_tile_kernel's.  In
// product (t, u) of a step lane half h covers k = 16 (2 t + h) + 8 u .. + 7: bytes
// 8 u .. 8 u + 7 of the lane's 16-byte chunk of codes, turned into bf16 in
// registers, and 16 bytes of each plane.  Bound: for a few rows the
// weight's bytes; for many the matrix cores (three products a value), with the
// LDS reads of the planes close behind, which is why the tile is as wide as the
// grid allows.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "kh_common.h"
#include "kh_lanes.h"
#include "kh_pipeline.h"
#include "kh_rows.h"

#pragma clang fp contract(off)

namespace {

using namespace kh::pipe;
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kTargetExp = 100, kSpan = 200;
constexpr int64_t kMaxK = 1 << 19;

// One row of x per workgroup: its factor (the inverse of its power of two, or
// NaN for a row that spans too much), then its three planes, zeros from K to Kp.
// Up to 4096 values stay in registers between the two; VEC: 16-byte loads.
constexpr int kSplitRegs = 4;

template <bool VEC>
__global__ __launch_bounds__(256) void split_rows_kernel(const float* __restrict__ x, int64_t rows, int K, int Kp,
                                                         __bf16* __restrict__ planes, double* __restrict__ factors) {
    __shared__ unsigned red[2][4];
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    const int64_t row = blockIdx.x;
    const float* const xr = x + row * K;
    // Four values from k, zeros past K (the address is held inside the row
    // instead of a test, behind which the compiler would wait for each load).
    auto load = [&](int k) {
        f32x4 v;
        if (VEC) {
            v = *reinterpret_cast<const f32x4*>(xr + min(k, K - 4));
            if (k >= K) v = f32x4{0.f, 0.f, 0.f, 0.f};
        } else {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float w = xr[min(k + u, K - 1)];
                v[u] = k + u < K ? w : 0.0f;
            }
        }
        return v;
    };
    unsigned hi = 0, lo = 0;  // the largest bits, and the complement of (the smallest nonzero bits - 1)
    auto look = [&](f32x4 v) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const unsigned b = __float_as_uint(v[u]) & 0x7FFFFFFFu;
            hi = max(hi, b < KH_NONFINITE_BITS ? b : 0u);
            lo = max(lo, ~(b - 1u));
        }
    };
    f32x4 kept[kSplitRegs];
#pragma unroll
    for (int i = 0; i < kSplitRegs; ++i) kept[i] = load(threadIdx.x * 4 + i * 1024);
#pragma unroll
    for (int i = 0; i < kSplitRegs; ++i) look(kept[i]);
    for (int k = threadIdx.x * 4 + kSplitRegs * 1024; k < K; k += 1024) look(load(k));
    hi = kh::lanes::wave_max(hi);
    lo = kh::lanes::wave_max(lo);
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = hi;
        red[1][threadIdx.x >> 6] = lo;
    }
    __syncthreads();
    hi = max(max(red[0][0], red[0][1]), max(red[0][2], red[0][3]));
    lo = ~max(max(red[1][0], red[1][1]), max(red[1][2], red[1][3])) + 1u;
    const int e = hi ? ilogbf(__uint_as_float(hi)) : kTargetExp;  // 2^e <= the largest finite |x| < 2^(e + 1)
    if (threadIdx.x == 0) {
        const bool wide = hi && e - ilogbf(__uint_as_float(lo)) > kSpan;
        factors[row] = wide ? __longlong_as_double(0x7FF8000000000000LL) : ldexp(1.0, e - kTargetExp);
    }
    __bf16* const out = planes + row * Kp;
    const int64_t plane = rows * Kp;
    auto emit = [&](int k, f32x4 v) {
        bf16x4 p[3];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const float w = ldexpf(v[u], kTargetExp - e);
            const bool finite = (__float_as_uint(w) & 0x7FFFFFFFu) < KH_NONFINITE_BITS;
            const __bf16 h = (__bf16)w;
            const float r = finite ? w - (float)h : 0.0f;
            const __bf16 m = (__bf16)r;
            p[0][u] = h;
            p[1][u] = m;
            p[2][u] = (__bf16)(r - (float)m);
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x4*>(out + i * plane + k) = p[i];
    };
#pragma unroll
    for (int i = 0; i < kSplitRegs; ++i)
        if (threadIdx.x * 4 + i * 1024 < Kp) emit(threadIdx.x * 4 + i * 1024, kept[i]);
    for (int k = threadIdx.x * 4 + kSplitRegs * 1024; k < Kp; k += 1024) emit(k, load(k));
}

// Eight codes (two dwords, byte order = k order) as bf16.
__device__ __forceinline__ bf16x8 codes_bf16(int lo, int hi) {
    unsigned w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int d = i < 2 ? lo : hi;
        const int s = (i & 1) * 16;
        const float f0 = (float)(int8_t)(d >> s), f1 = (float)(int8_t)(d >> (s + 8));
        // The high halves: a code's binary32 form has nothing below.
        w[i] = __builtin_amdgcn_perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
    }
    return __builtin_bit_cast(bf16x8, i32x4{(int)w[0], (int)w[1], (int)w[2], (int)w[3]});
}

struct W8Out {
    const double* factors;  // [M]: the rows' powers of two
    const double* scales;   // 1 or N
    int per_col;
    const float* bias;
    float* out;      // [M, N]; or
    float* partial;  // [splits, M, N]: sums only
    // The operands as given, for the rows split_rows_kernel leaves.
    const float* x;
    const int8_t* q;
    int64_t K;
};

// quantize.py:115-122 for one output of a wide row.
__device__ __attribute__((noinline)) float w8_plain(const W8Out& o, int64_t i, int64_t j) {
    const double s = o.scales[o.per_col ? j : 0];
    float sum = 0.0f;
    for (int64_t k = 0; k < o.K; ++k) sum += o.x[i * o.K + k] * (float)((double)o.q[j * o.K + k] * s);
    return sum;
}

__device__ __forceinline__ float w8_value(const W8Out& o, float acc, int64_t i, int64_t j) {
    const double f = o.factors[i];
    float y = (float)((double)acc * (o.scales[o.per_col ? j : 0] * f));
    if (f != f) y = w8_plain(o, i, j);
    return o.bias ? y + o.bias[j] : y;
}

template <int BM, int BN, int NS>
__global__ __launch_bounds__(256, 1) void gemm_w8_kernel(const __bf16* __restrict__ X, const int8_t* __restrict__ Q,
                                                         int M, int N, int K, int Kp, int kper, W8Out o) {
    constexpr int BK = 64, kTM = BM / 64, kTN = BN / 64;
    constexpr int kPlane = BM * 128, kLdsB = 3 * kPlane, kStage = kLdsB + BN * BK;
    constexpr int kAInst = BM / 32, kBInst = BN / 64;  // LDS-DMA instructions per wave: per plane, and of codes
    constexpr int kLoads = 3 * kAInst + kBInst;
    static_assert(NS == 2 || NS == 4, "a turn of the ring below");
    __shared__ __attribute__((aligned(1024))) int8_t lds[NS * kStage];

    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    int tm, tn;
    tile_of(blockIdx.x, tiles_m, tiles_n, 8, tm, tn);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int rows_a = min(BM, M - tm * BM), rows_b = min(BN, N - tn * BN);
    auto swz_a = [](int r) { return (r >> 1) & 7; };  // 128-byte rows, 16 of them per conflict-free read
    auto swz_b = [](int r) { return (r >> 2) & 3; };  // 64-byte rows
    const int k_steps = Kp / BK;
    const int kt0 = blockIdx.y * kper, kt1 = min(k_steps, kt0 + kper);

    const int fr = lane & 31, fh = lane >> 5;
    int a_off[2][2][kTM], b_off[2][kTN];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int a = 0; a < kTM; ++a) {
                const int r = wm * (BM / 2) + a * 32 + fr;
                a_off[t][u][a] = r * 128 + (((2 * (2 * t + fh) + u) ^ swz_a(r)) << 4);
            }
#pragma unroll
        for (int b = 0; b < kTN; ++b) {
            const int r = wn * (BN / 2) + b * 32 + fr;
            b_off[t][b] = kLdsB + r * BK + (((2 * t + fh) ^ swz_b(r)) << 4);
        }
    }
    f32x16 acc[kTM][kTN];
#pragma unroll
    for (int a = 0; a < kTM; ++a)
#pragma unroll
        for (int b = 0; b < kTN; ++b) acc[a][b] = f32x16{0};

    struct Frags {
        bf16x8 a[3][2][2][kTM];
        i32x4 b[2][kTN];
    };
    Frags f0, f1;
    auto read = [&](const int8_t* base, Frags& f) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
            for (int b = 0; b < kTN; ++b) f.b[t][b] = *reinterpret_cast<const i32x4*>(base + b_off[t][b]);
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int a = 0; a < kTM; ++a)
#pragma unroll
                    for (int p = 0; p < 3; ++p)
                        f.a[p][t][u][a] = *reinterpret_cast<const bf16x8*>(base + p * kPlane + a_off[t][u][a]);
        }
    };
    auto multiply = [&](const Frags& f) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                bf16x8 q[kTN];
#pragma unroll
                for (int b = 0; b < kTN; ++b) q[b] = codes_bf16(f.b[t][b][2 * u], f.b[t][b][2 * u + 1]);
                // The smallest parts first.
#pragma unroll
                for (int p = 2; p >= 0; --p)
#pragma unroll
                    for (int a = 0; a < kTM; ++a)
#pragma unroll
                        for (int b = 0; b < kTN; ++b)
                            acc[a][b] =
                                __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[p][t][u][a], q[b], acc[a][b], 0, 0, 0);
            }
    };
    auto meet = [&]() {
        __builtin_amdgcn_s_waitcnt(wait_imm(63, 0));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };

    // Rows past M (N) lie outside the resources: their loads return zeros, as do
    // codes at k >= K (K % 16 == 0, so a chunk is whole or past).
    const int64_t plane = (int64_t)M * Kp;
    __amdgpu_buffer_rsrc_t ra[3];
#pragma unroll
    for (int p = 0; p < 3; ++p)
        ra[p] = make_rsrc(X + p * plane + (int64_t)tm * BM * Kp, (uint32_t)rows_a * (uint32_t)Kp * 2u);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(Q + (int64_t)tn * BN * K, (uint32_t)rows_b * (uint32_t)K);
    constexpr int kPast = 0x7FFF0000;
    int a_voff[kAInst], b_voff[kBInst], b_k[kBInst];
#pragma unroll
    for (int i = 0; i < kAInst; ++i) {
        const int r = (wave * kAInst + i) * 8 + (lane >> 3);
        a_voff[i] = r * Kp * 2 + (((lane & 7) ^ swz_a(r)) << 4);
    }
#pragma unroll
    for (int i = 0; i < kBInst; ++i) {
        const int r = (wave * kBInst + i) * 16 + (lane >> 2);
        b_k[i] = ((lane & 3) ^ swz_b(r)) << 4;
        b_voff[i] = r * K + b_k[i];
    }
    auto issue = [&](int kt, int slot) {
        int8_t* base = lds + slot * kStage;
        const int k0 = kt * BK;
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int i = 0; i < kAInst; ++i)
                lds_dma16(ra[p], base + p * kPlane + (wave * kAInst + i) * 1024, a_voff[i], k0 * 2);
        if (k0 + BK <= K) {
#pragma unroll
            for (int i = 0; i < kBInst; ++i)
                lds_dma16(rb, base + kLdsB + (wave * kBInst + i) * 1024, b_voff[i], k0);
        } else {
#pragma unroll
            for (int i = 0; i < kBInst; ++i)
                lds_dma16(rb, base + kLdsB + (wave * kBInst + i) * 1024, k0 + b_k[i] >= K ? kPast : b_voff[i], k0);
        }
    };
#pragma unroll
    for (int s = 0; s < NS; ++s)
        if (kt0 + s < kt1) issue(kt0 + s, s);
    wait_loads_beyond<kLoads>(min(NS - 1, kt1 - 1 - kt0));
    meet();
    read(lds, f0);
    // Step j of a turn of the ring (kt = kt0 + j mod NS).  Steady: every stage it
    // touches exists, so nothing is tested.
    auto step = [&](int kt, auto jc, auto steady, const Frags& cur, Frags& next) {
        constexpr int j = decltype(jc)::value;
        if constexpr (decltype(steady)::value)
            __builtin_amdgcn_s_waitcnt(wait_imm((NS - 2) * kLoads, 15));
        else
            wait_loads_beyond<kLoads>(max(0, min(NS - 2, kt1 - 2 - kt)));
        meet();  // stage kt + 1 landed, stage kt read
        if (decltype(steady)::value || kt + NS < kt1) issue(kt + NS, j);
        if (decltype(steady)::value || kt + 1 < kt1) read(lds + (j + 1) % NS * kStage, next);
        __builtin_amdgcn_sched_barrier(0);
        multiply(cur);
        __builtin_amdgcn_sched_barrier(0);
    };
    using std::integral_constant;
    int kt = kt0;
    for (; kt + 2 * NS <= kt1; kt += NS) {
        step(kt, integral_constant<int, 0>(), std::true_type(), f0, f1);
        step(kt + 1, integral_constant<int, 1>(), std::true_type(), f1, f0);
        if constexpr (NS == 4) {
            step(kt + 2, integral_constant<int, 2>(), std::true_type(), f0, f1);
            step(kt + 3, integral_constant<int, 3>(), std::true_type(), f1, f0);
        }
    }
    for (; kt < kt1; kt += NS) {
        step(kt, integral_constant<int, 0>(), std::false_type(), f0, f1);
        if (kt + 1 < kt1) step(kt + 1, integral_constant<int, 1>(), std::false_type(), f1, f0);
        if constexpr (NS == 4) {
            if (kt + 2 < kt1) step(kt + 2, integral_constant<int, 2>(), std::false_type(), f0, f1);
            if (kt + 3 < kt1) step(kt + 3, integral_constant<int, 3>(), std::false_type(), f1, f0);
        }
    }

    // 32x32 result layout: register r of lane l holds row 8 (r / 4) + 4 (l / 32)
    // + r % 4, column l % 32.
#pragma unroll
    for (int a = 0; a < kTM; ++a)
#pragma unroll
        for (int b = 0; b < kTN; ++b) {
            const int64_t j = (int64_t)tn * BN + wn * (BN / 2) + b * 32 + fr;
            if (j >= N) continue;
            const int64_t i0 = (int64_t)tm * BM + wm * (BM / 2) + a * 32 + 4 * fh;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t i = i0 + 8 * (r >> 2) + (r & 3);
                if (i >= M) continue;
                if (o.partial) o.partial[((int64_t)blockIdx.y * M + i) * N + j] = acc[a][b][r];
                else o.out[i * N + j] = w8_value(o, acc[a][b][r], i, j);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
}

// The K splits' sums, in order, and the epilogue.  Every split's load is issued
// before the first is used; a thread takes V = 4 columns where N % 4 == 0.
template <int S, int V>
__global__ __launch_bounds__(256) void w8_sum_kernel(int M, int N, W8Out o) {
    typedef float fv __attribute__((ext_vector_type(V == 4 ? 4 : 2)));
    const int64_t mn = (int64_t)M * N, idx = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
    if (idx >= mn) return;
    fv p[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if constexpr (V == 4) p[s] = *reinterpret_cast<const fv*>(o.partial + s * mn + idx);
        else p[s].x = o.partial[s * mn + idx];
    }
    const int64_t i = idx / N, j = idx - i * N;
#pragma unroll
    for (int u = 0; u < V; ++u) {
        float sum = p[0][u];
#pragma unroll
        for (int s = 1; s < S; ++s) sum += p[s][u];
        o.out[idx + u] = w8_value(o, sum, i, j + u);
    }
}

template <int S>
int launch_w8_sum(kh::Device* d, int64_t M, int64_t N, const W8Out& o) {
    if (N % 4 == 0)
        w8_sum_kernel<S, 4><<<(unsigned)((M * N / 4 + 255) / 256), 256, 0, d->stream>>>((int)M, (int)N, o);
    else
        w8_sum_kernel<S, 1><<<(unsigned)((M * N + 255) / 256), 256, 0, d->stream>>>((int)M, (int)N, o);
    return kh::launch_status("w8_sum");
}

template <int BM, int BN, int NS>
int launch_w8(kh::Device* d, const __bf16* X, const int8_t* Q, int64_t M, int64_t N, int64_t K, int64_t Kp, int S,
              const W8Out& o) {
    const unsigned tiles = (unsigned)(((M + BM - 1) / BM) * ((N + BN - 1) / BN));
    const int kper = (int)((Kp / 64 + S - 1) / S);
    gemm_w8_kernel<BM, BN, NS>
        <<<dim3(tiles, (unsigned)S), 256, 0, d->stream>>>(X, Q, (int)M, (int)N, (int)K, (int)Kp, kper, o);
    return kh::launch_status("gemm_w8");
}

}  // namespace

extern "C" int kh_linear_w8(const float* x, int64_t M, int64_t K, const int8_t* q_packed, int64_t N,
                            const double* scales, int64_t scales_n, const float* bias, float* out) {
    KH_REQUIRE(M >= 0 && N >= 0 && K >= 0, "kh_linear_w8: negative shape");
    if (M == 0 || N == 0) return KH_OK;
    KH_REQUIRE(out, "kh_linear_w8: null out");
    KH_REQUIRE(K == 0 || (x && q_packed && scales), "kh_linear_w8: null operand");
    KH_REQUIRE(scales_n == 1 || scales_n == N, "kh_linear_w8: scales_n must be 1 or N");
    KH_REQUIRE(M <= 0xFFFFLL * 128 && N <= 0x7FFFFFFFLL, "kh_linear_w8: shape too large");
    KH_DEVICE_OR_RETURN(d);
    const int64_t cus = d->cus;
    if (N * K < 16 || K > kMaxK) {
        // Weights of less than 16 bytes (the kernels load 16 at a time), and
        // sums that could pass binary32's range: the weight in fp32.
        void* w = nullptr;
        int rc = kh_alloc((size_t)(K * N) * sizeof(float), &w);
        if (rc) return rc;
        rc = kh_dequantize_packed(q_packed, K, N, scales, scales_n, static_cast<float*>(w));
        if (!rc) rc = kh_matmul_f32(x, static_cast<const float*>(w), out, M, K, N, bias);
        kh_free(w);  // stream-ordered: reused only by work queued after the product
        return rc;
    }
    const int64_t Kp = (K + 63) / 64 * 64;
    const bool pad = K % 16 != 0 || !kh::aligned(q_packed, 16);
    // The planes of at most 256 MiB of rows at a time, so that they stay in the
    // last-level cache and a long x needs no more.
    const int64_t slab = min(M, max((int64_t)128, (int64_t)(256 << 20) / (6 * Kp) / 128 * 128));
    // 64 x 128 tiles where they fill the chip, 64 x 64 otherwise (both two
    // workgroups to a CU): 4096^3 446 -> 377 us, 2048 x 4096 x 1024 73 -> 64;
    // 300 x 487 x 1728 20 against 29.  K is split until the tiles come to two a
    // CU, each split keeping four steps: 64 x 4096 x 4096 36.6 -> 17.2 us.
    const bool wide = ((slab + 63) / 64) * ((N + 127) / 128) >= cus;
    const int64_t tiles = ((slab + 63) / 64) * ((N + (wide ? 127 : 63)) / (wide ? 128 : 64)), steps = Kp / 64;
    KH_REQUIRE(tiles <= 0x7FFFFFFF && N * (Kp / 16) / 256 < 0x7FFFFFFF, "kh_linear_w8: shape too large");
    int S = 1;
    while (!wide && S < 8 && tiles * S * 2 <= 2 * cus && steps >= 8 * S) S *= 2;
    const size_t planes_bytes = (size_t)(3 * slab * Kp) * sizeof(__bf16);
    const size_t factors_at = planes_bytes, codes_at = factors_at + (size_t)(slab + 1) / 2 * 2 * sizeof(double);
    const size_t sums_at = codes_at + (pad ? (size_t)(N * Kp) : 0);  // (a multiple of 16)
    void* work = nullptr;
    int rc = kh_alloc(sums_at + (S > 1 ? (size_t)S * (size_t)(slab * N) * sizeof(float) : 0), &work);
    if (rc) return rc;
    char* const base = static_cast<char*>(work);
    __bf16* const planes = reinterpret_cast<__bf16*>(base);
    double* const factors = reinterpret_cast<double*>(base + factors_at);
    const int8_t* q = q_packed;
    if (pad) {
        int8_t* const to = reinterpret_cast<int8_t*>(base + codes_at);
        kh::rows::pad_rows_kernel<<<(unsigned)((N * (Kp / 16) + 255) / 256), 256, 0, d->stream>>>(
            q_packed, q_packed, 0, (int)N, (int)K, (int)Kp, to);
        rc = kh::launch_status("pad_rows");
        q = to;
    }
    const bool vec = K % 4 == 0 && kh::aligned(x, 16);
    for (int64_t i0 = 0; i0 < M && !rc; i0 += slab) {
        const int64_t m = min(slab, M - i0);
        const float* const xs = x + i0 * K;
        if (vec) split_rows_kernel<true><<<(unsigned)m, 256, 0, d->stream>>>(xs, m, (int)K, (int)Kp, planes, factors);
        else split_rows_kernel<false><<<(unsigned)m, 256, 0, d->stream>>>(xs, m, (int)K, (int)Kp, planes, factors);
        rc = kh::launch_status("split_rows");
        if (rc) break;
        const W8Out o{factors, scales, scales_n != 1, bias, out + i0 * N,
                      S > 1 ? reinterpret_cast<float*>(base + sums_at) : nullptr, xs, q_packed, K};
        const int64_t kq = pad ? Kp : K;
        rc = wide ? launch_w8<64, 128, 2>(d, planes, q, m, N, kq, Kp, S, o)
                  : launch_w8<64, 64, 2>(d, planes, q, m, N, kq, Kp, S, o);
        if (!rc && S > 1)
            rc = S == 2 ? launch_w8_sum<2>(d, m, N, o) : S == 4 ? launch_w8_sum<4>(d, m, N, o)
                                                                : launch_w8_sum<8>(d, m, N, o);
    }
    kh_free(work);  // stream-ordered: reused only by work queued after the product
    return rc;
}
