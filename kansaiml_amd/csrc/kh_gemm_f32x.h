// kh_gemm_f32x.h -- the fp32 matmul on the bf16 matrix cores.  Internal: included
// by kh_gemm_f32.hip.
//
// v_mfma_f32_32x32x2_f32 multiplies 64 values a cycle and SIMD, the bf16 forms
// 1024.  A binary32 value is exactly h + m + l, three bf16 values of 8 significand
// bits (each the rounding of what the ones before left), and of the nine
// products of two such triples six are multiplied, all exact: hh, hm, mh, hl, lh,
// mm.  The other three are below 2^-24 of the product, less than the rounding of
// one binary32 sum, and a product of sixteen k rounds six sums where the fp32
// instruction rounds eight: the error against binary64 is 0.83-0.92 of the fp32
// MFMA kernel's at every size measured (K = 64 to 4096), 0.3-0.7 where K is split.
// 4096^3: 1011 -> 792 us; 2000 x 4096 x 2048 298 -> 222; 190 x 72 x 512 52 -> 13.
//
// Two launches, and a sum of partials where K is split:
//   split_units_kernel  A and B as planes [3, M, Kp] and [3, N, Kp] (B transposed:
//                       both operands K-contiguous), zeros past K.
//   gemm_f32x_kernel    BM x BN tiles, 4 waves as 2 x 2, v_mfma_f32_32x32x16_bf16,
//                       K in steps of 32 through a ring of NS LDS stages by LDS-DMA,
//                       unrolled over the ring as gemm_i8_tile_kernel is.
//
// Range.  A unit is 32 rows of an operand by 64 k.  A unit holding a NaN or
// infinity, a magnitude above 2^50 (whose products could overflow the sums where
// binary32 would not) or a nonzero one below 2^-100 (whose parts could flush) is
// written as zeros and marked; its products are added in the epilogue by
// v_mfma_f32_32x32x2_f32 on the values as given.  A 32 x 32 block whose largest
// product is below 2^-90 is computed that way altogether.
#pragma once

#include <type_traits>

#include "kh_lanes.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kUnitRows = 32, kUnitK = 64;
constexpr int kUnitMarked = 1000, kUnitZero = -1000;  // else the exponent of the unit's largest magnitude
constexpr unsigned kMostBits = (127 + 50) << 23, kLeastBits = (127 - 100) << 23;
constexpr int kLeastExp = -90;

struct UnitStat {
    unsigned most = 0;
    bool marked = false;
    __device__ __forceinline__ void add(float v) {
        const unsigned b = __float_as_uint(v) & 0x7FFFFFFFu;
        most = max(most, b);
        marked = marked || b > kMostBits || (b != 0 && b < kLeastBits);
    }
};

__device__ __forceinline__ void split3(const float (&v)[8], bool zero, bf16x8 (&p)[3]) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const float w = zero ? 0.0f : v[u];
        const __bf16 h = (__bf16)w;
        const float r = w - (float)h;
        const __bf16 m = (__bf16)r;
        p[0][u] = h;
        p[1][u] = m;
        p[2][u] = (__bf16)(r - (float)m);
    }
}

// Workgroups 0 .. a_groups - 1 take one unit of A each (unit u of row block i /
// KT); the others 64 k x 64 columns of B, two units, transposed through LDS.  VEC:
// 16-byte loads (K, for B N, a multiple of 4 and 16-byte aligned operands).
// Addresses past the end are held inside the operand and the values cleared.
template <bool VECA, bool VECB>
__global__ __launch_bounds__(256) void split_units_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                          int M, int N, int K, int KT, int a_groups,
                                                          __bf16* __restrict__ pa, __bf16* __restrict__ pb,
                                                          int* __restrict__ ea, int* __restrict__ eb) {
    __shared__ float tile[kUnitK][65];
    __shared__ unsigned most[4], marked[4];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t Kp = (int64_t)KT * kUnitK;
    const bool is_a = (int)blockIdx.x < a_groups;
    const int id = is_a ? blockIdx.x : blockIdx.x - a_groups;
    const int blk = id / KT, u = id - blk * KT;
    UnitStat st;
    if (is_a) {
        const int row = blk * kUnitRows + (t >> 3), k = u * kUnitK + (t & 7) * 8;
        const float* const src = A + (int64_t)min(row, M - 1) * K;
        float v[8];
        if (VECA) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const f32x4 w = *reinterpret_cast<const f32x4*>(src + min(k + 4 * h, K - 4));
#pragma unroll
                for (int e = 0; e < 4; ++e) v[4 * h + e] = w[e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = src[min(k + e, K - 1)];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (row >= M || k + e >= K) v[e] = 0.0f;
            st.add(v[e]);
        }
        const unsigned m = kh::lanes::wave_max(st.most);
        const bool any = __any(st.marked);
        if (lane == 0) {
            most[wave] = m;
            marked[wave] = any;
        }
        __syncthreads();
        const unsigned mm = max(max(most[0], most[1]), max(most[2], most[3]));
        const bool mk = marked[0] | marked[1] | marked[2] | marked[3];
        if (t == 0) ea[blk * KT + u] = mk ? kUnitMarked : mm ? (int)(mm >> 23) - 127 : kUnitZero;
        if (row >= M) return;
        bf16x8 p[3];
        split3(v, mk, p);
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8*>(pa + ((int64_t)i * M + row) * Kp + k) = p[i];
        return;
    }
    const int j0 = blk * 64, k0 = u * kUnitK;
    f32x4 v[4];
    const int c4 = (t & 15) * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int k = k0 + (t >> 4) + 16 * i;
        const float* const src = B + (int64_t)min(k, K - 1) * N;
        if (VECB) {
            v[i] = *reinterpret_cast<const f32x4*>(src + min(j0 + c4, N - 4));
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[i][e] = src[min(j0 + c4 + e, N - 1)];
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int k = (t >> 4) + 16 * i;
#pragma unroll
        for (int e = 0; e < 4; ++e) tile[k][c4 + e] = k0 + k < K && j0 + c4 + e < N ? v[i][e] : 0.0f;
    }
    __syncthreads();
    // Thread t: column t / 4, k = 16 (t % 4) .. + 15.
    const int c = t >> 2, kk = (t & 3) * 16, j = j0 + c;
    float x[2][8];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            x[h][e] = tile[kk + 8 * h + e][c];
            st.add(x[h][e]);
        }
    const unsigned m = kh::lanes::wave_max(st.most);
    const bool any = __any(st.marked);
    if (lane == 0) {
        most[wave] = m;
        marked[wave] = any;
    }
    __syncthreads();
    const int half = (wave >> 1) * 2;  // waves 0, 1: columns 0 .. 31; 2, 3: 32 .. 63
    const unsigned mm = max(most[half], most[half + 1]);
    const bool mk = marked[half] | marked[half + 1];
    if (lane == 0 && !(wave & 1))
        eb[(blk * 2 + (wave >> 1)) * KT + u] = mk ? kUnitMarked : mm ? (int)(mm >> 23) - 127 : kUnitZero;
    if (j >= N) return;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        bf16x8 p[3];
        split3(x[h], mk, p);
#pragma unroll
        for (int i = 0; i < 3; ++i)
            *reinterpret_cast<bf16x8*>(pb + ((int64_t)i * N + j) * Kp + k0 + kk + 8 * h) = p[i];
    }
}

struct F32x {
    const float* A;  // as given, for marked units
    const float* B;
    const int* ea;
    const int* eb;
    const float* bias;
    float* out;      // [M, N]; or
    float* partial;  // [splits, M, N]: sums only
};

// Calls f(0), f(1), .. f(n - 1) with compile-time arguments.
template <int n, int i = 0, class F>
__device__ __forceinline__ void unroll(F&& f) {
    if constexpr (i < n) {
        f(std::integral_constant<int, i>());
        unroll<n, i + 1>(f);
    }
}

template <int BM, int BN, int NS>
__global__ __launch_bounds__(256, 1) void gemm_f32x_kernel(const __bf16* __restrict__ PA, const __bf16* __restrict__ PB,
                                                           int M, int N, int K, int KT, int kper, F32x o) {
    using namespace kh::pipe;
    constexpr int BK = 32, kTM = BM / 64, kTN = BN / 64;
    constexpr int kPlaneA = BM * 64, kPlaneB = BN * 64, kLdsB = 3 * kPlaneA, kStage = 3 * (kPlaneA + kPlaneB);
    constexpr int kAInst = BM / 64, kBInst = BN / 64;  // LDS-DMA instructions per wave and plane: 16 rows of 64 bytes
    constexpr int kLoads = 3 * (kAInst + kBInst), kTurn = NS % 2 ? 2 * NS : NS;
    static_assert(NS >= 2 && NS <= 4, "wait_loads_beyond covers up to 3 stages");
    __shared__ __attribute__((aligned(1024))) int8_t lds[NS * kStage];

    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    int tm, tn;
    tile_of(blockIdx.x, tiles_m, tiles_n, 8, tm, tn);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int rows_a = min(BM, M - tm * BM), rows_b = min(BN, N - tn * BN);
    auto swz = [](int r) { return (r >> 2) & 3; };
    const int64_t Kp = (int64_t)KT * kUnitK;
    const int kt0 = blockIdx.y * kper, kt1 = min(2 * KT, kt0 + kper);  // (kper is even: whole units)

    // Fragments: lane l reads 16 bytes (8 k) of row r + l % 32 at chunk 2 s + l / 32.
    const int fr = lane & 31, fh = lane >> 5;
    int a_off[2][kTM], b_off[2][kTN];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int a = 0; a < kTM; ++a) {
            const int r = wm * (BM / 2) + a * 32 + fr;
            a_off[s][a] = r * 64 + (((2 * s + fh) ^ swz(r)) << 4);
        }
#pragma unroll
        for (int b = 0; b < kTN; ++b) {
            const int r = wn * (BN / 2) + b * 32 + fr;
            b_off[s][b] = kLdsB + r * 64 + (((2 * s + fh) ^ swz(r)) << 4);
        }
    }
    f32x16 acc[kTM][kTN];
#pragma unroll
    for (int a = 0; a < kTM; ++a)
#pragma unroll
        for (int b = 0; b < kTN; ++b) acc[a][b] = f32x16{0};

    struct Frags {
        bf16x8 a[2][3][kTM], b[2][3][kTN];
    };
    Frags f[2];
    auto read = [&](const int8_t* base, Frags& g) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int p = 0; p < 3; ++p) {
#pragma unroll
                for (int a = 0; a < kTM; ++a)
                    g.a[s][p][a] = *reinterpret_cast<const bf16x8*>(base + p * kPlaneA + a_off[s][a]);
#pragma unroll
                for (int b = 0; b < kTN; ++b)
                    g.b[s][p][b] = *reinterpret_cast<const bf16x8*>(base + p * kPlaneB + b_off[s][b]);
            }
    };
    auto multiply = [&](const Frags& g) {
        // The smallest products first.
        constexpr int pa[6] = {1, 2, 0, 1, 0, 0}, pb[6] = {1, 0, 2, 0, 1, 0};
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int a = 0; a < kTM; ++a)
#pragma unroll
                    for (int b = 0; b < kTN; ++b)
                        acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(g.a[s][pa[q]][a], g.b[s][pb[q]][b],
                                                                            acc[a][b], 0, 0, 0);
    };
    auto meet = [&]() {
        __builtin_amdgcn_s_waitcnt(wait_imm(63, 0));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };

    // Rows past M (N) lie outside the resources: their loads return zeros.
    __amdgpu_buffer_rsrc_t ra[3], rb[3];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
        ra[p] = make_rsrc(PA + ((int64_t)p * M + (int64_t)tm * BM) * Kp, (uint32_t)rows_a * (uint32_t)Kp * 2u);
        rb[p] = make_rsrc(PB + ((int64_t)p * N + (int64_t)tn * BN) * Kp, (uint32_t)rows_b * (uint32_t)Kp * 2u);
    }
    int a_voff[kAInst], b_voff[kBInst];
#pragma unroll
    for (int i = 0; i < kAInst; ++i) {
        const int r = (wave * kAInst + i) * 16 + (lane >> 2);
        a_voff[i] = r * (int)Kp * 2 + (((lane & 3) ^ swz(r)) << 4);
    }
#pragma unroll
    for (int i = 0; i < kBInst; ++i) {
        const int r = (wave * kBInst + i) * 16 + (lane >> 2);
        b_voff[i] = r * (int)Kp * 2 + (((lane & 3) ^ swz(r)) << 4);
    }
    auto issue = [&](int kt, int slot) {
        int8_t* base = lds + slot * kStage;
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
            for (int i = 0; i < kAInst; ++i)
                lds_dma16(ra[p], base + p * kPlaneA + (wave * kAInst + i) * 1024, a_voff[i], kt * BK * 2);
#pragma unroll
            for (int i = 0; i < kBInst; ++i)
                lds_dma16(rb[p], base + kLdsB + p * kPlaneB + (wave * kBInst + i) * 1024, b_voff[i], kt * BK * 2);
        }
    };
#pragma unroll
    for (int s = 0; s < NS; ++s)
        if (kt0 + s < kt1) issue(kt0 + s, s);
    wait_loads_beyond<kLoads>(min(NS - 1, kt1 - 1 - kt0));
    meet();
    read(lds, f[0]);
    // Step j of a turn of the ring (kt = kt0 + j mod kTurn).  Steady: every stage
    // it touches exists, so nothing is tested.
    auto step = [&](int kt, auto jc, auto steady) {
        constexpr int j = decltype(jc)::value;
        constexpr bool kSteady = decltype(steady)::value;
        if constexpr (kSteady)
            __builtin_amdgcn_s_waitcnt(wait_imm((NS - 2) * kLoads, 15));
        else
            wait_loads_beyond<kLoads>(max(0, min(NS - 2, kt1 - 2 - kt)));
        meet();  // stage kt + 1 landed, stage kt read
        if (kSteady || kt + NS < kt1) issue(kt + NS, j % NS);
        if (kSteady || kt + 1 < kt1) read(lds + (j + 1) % NS * kStage, f[(j + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
        multiply(f[j & 1]);
        __builtin_amdgcn_sched_barrier(0);
    };
    int kt = kt0;
    for (; kt + kTurn + NS <= kt1; kt += kTurn)
        unroll<kTurn>([&](auto j) { step(kt + decltype(j)::value, j, std::true_type()); });
    for (; kt < kt1; kt += kTurn)
        unroll<kTurn>([&](auto j) {
            if (kt + decltype(j)::value < kt1) step(kt + decltype(j)::value, j, std::false_type());
        });

    // A block's products of unit u, by the fp32 instruction on the values as
    // given: lane half h takes k = 32 h + s in product s.
    auto add_unit = [&](f32x16& c, int64_t i0, int64_t j0, int u) {
        const float* const ar = o.A + min(i0 + fr, (int64_t)M - 1) * K;
        const int64_t j = min(j0 + fr, (int64_t)N - 1);
#pragma unroll 8
        for (int s = 0; s < 32; ++s) {
            const int k = u * kUnitK + 32 * fh + s, kc = min(k, K - 1);
            const float x = ar[kc], y = o.B[(int64_t)kc * N + j];
            c = __builtin_amdgcn_mfma_f32_32x32x2f32(k < K ? x : 0.0f, k < K ? y : 0.0f, c, 0, 0, 0);
        }
    };
    const int u0 = kt0 / 2, u1 = (kt1 + 1) / 2;
    // 32x32 result layout: register r of lane l holds row 8 (r / 4) + 4 (l / 32)
    // + r % 4, column l % 32.
#pragma unroll
    for (int a = 0; a < kTM; ++a)
#pragma unroll
        for (int b = 0; b < kTN; ++b) {
            const int64_t i0 = (int64_t)tm * BM + wm * (BM / 2) + a * 32;
            const int64_t j0 = (int64_t)tn * BN + wn * (BN / 2) + b * 32;
            if (i0 >= M || j0 >= N) continue;
            const int* const xa = o.ea + i0 / kUnitRows * KT;
            const int* const xb = o.eb + j0 / kUnitRows * KT;
            int top = 2 * kUnitZero;
            bool some = false;
            for (int u = u0 + lane; u < u1; u += 64) {
                const int p = xa[u], q = xb[u];
                some = some || p == kUnitMarked || q == kUnitMarked;
                if (p != kUnitZero && q != kUnitZero) top = max(top, p + q);
            }
            some = __any(some);
            const bool small = !__any(top >= kLeastExp) && __any(top > kUnitZero);
            if (some || small) {
                if (small) acc[a][b] = f32x16{0};
                for (int u = u0; u < u1; ++u)
                    if (small || xa[u] == kUnitMarked || xb[u] == kUnitMarked) add_unit(acc[a][b], i0, j0, u);
            }
            const int64_t j = j0 + fr;
            if (j >= N) continue;
            const float bj = o.bias && !o.partial ? o.bias[j] : 0.0f;
            float* const to = o.partial ? o.partial + (int64_t)blockIdx.y * M * N : o.out;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t i = i0 + 4 * fh + 8 * (r >> 2) + (r & 3);
                if (i < M) to[i * N + j] = o.bias && !o.partial ? acc[a][b][r] + bj : acc[a][b][r];
            }
        }
}

// The K splits' sums, in order, and the bias.  Every split's load is issued
// before the first is used; a thread takes V = 4 columns where N % 4 == 0.
template <int S, int V>
__global__ __launch_bounds__(256) void f32x_sum_kernel(const float* __restrict__ partial, int M, int N,
                                                       const float* __restrict__ bias, float* __restrict__ out) {
    typedef float fv __attribute__((ext_vector_type(V == 4 ? 4 : 2)));
    const int64_t mn = (int64_t)M * N, idx = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
    if (idx >= mn) return;
    fv p[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if constexpr (V == 4) p[s] = *reinterpret_cast<const fv*>(partial + s * mn + idx);
        else p[s].x = partial[s * mn + idx];
    }
    const int64_t j = idx % N;
#pragma unroll
    for (int u = 0; u < V; ++u) {
        float sum = p[0][u];
#pragma unroll
        for (int s = 1; s < S; ++s) sum += p[s][u];
        out[idx + u] = bias ? sum + bias[j + u] : sum;
    }
}

template <int BM, int BN, int NS>
int launch_f32x_cfg(kh::Device* d, const __bf16* pa, const __bf16* pb, int64_t M, int64_t N, int64_t K, int S,
                    const F32x& o) {
    const unsigned tiles = (unsigned)(((M + BM - 1) / BM) * ((N + BN - 1) / BN));
    const int KT = (int)((K + kUnitK - 1) / kUnitK), kper = 2 * ((KT + S - 1) / S);
    gemm_f32x_kernel<BM, BN, NS>
        <<<dim3(tiles, (unsigned)S), 256, 0, d->stream>>>(pa, pb, (int)M, (int)N, (int)K, KT, kper, o);
    int rc = kh::launch_status("gemm_f32x");
    if (rc || S == 1) return rc;
    auto sum = [&](auto sc) {
        constexpr int kS = decltype(sc)::value;
        if (N % 4 == 0)
            f32x_sum_kernel<kS, 4><<<(unsigned)((M * N / 4 + 255) / 256), 256, 0, d->stream>>>(o.partial, (int)M,
                                                                                               (int)N, o.bias, o.out);
        else
            f32x_sum_kernel<kS, 1><<<(unsigned)((M * N + 255) / 256), 256, 0, d->stream>>>(o.partial, (int)M, (int)N,
                                                                                           o.bias, o.out);
    };
    if (S == 2) sum(std::integral_constant<int, 2>());
    else if (S == 4) sum(std::integral_constant<int, 4>());
    else sum(std::integral_constant<int, 8>());
    return kh::launch_status("f32x_sum");
}

// ---------------------------------------------------------------------------
// A few rows (M <= 32): B is read once, as it lies, and the products are fp32
// FMAs -- the split above would write one and a half times what it reads.  A
// workgroup takes 4 LC columns (LC lanes of one float4 each; its 256 / LC lane
// groups take every (256 / LC)-th k) of kper rows of B, MR rows of A from LDS (k-
// major, so a k's values are one broadcast read), eight or sixteen float4 of B in
// flight a lane; the groups' sums meet in LDS.  Bound: the bytes of B.  1 x 4096 x
// 4096 341 -> 24 us (2.8 TB/s, the sum of 32 partials behind it), 16 rows 342 ->
// 32, 32 rows 344 -> 44, where the split product took 63.
// ---------------------------------------------------------------------------
constexpr int kRowsMost = 32, kRowsK = 512, kRowsSplits = 32;

template <int MR, int LC, bool VEC>
__global__ __launch_bounds__(256) void gemm_f32_rows_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                            int M, int N, int K, int kper,
                                                            const float* __restrict__ bias, float* __restrict__ out,
                                                            int partial) {
    constexpr int G = 256 / LC, U = MR <= 4 ? 16 : 8, MB = MR < 4 ? MR : 4;
    __shared__ __attribute__((aligned(16))) float xs[kRowsK * MR];
    __shared__ f32x4 red[MB][256];
    const int t = threadIdx.x, g = t / LC, c = t % LC;
    const int k0 = blockIdx.y * kper, k1 = min(K, k0 + kper);
    const int64_t j0 = (int64_t)blockIdx.x * 4 * LC + 4 * c;
    for (int i = t; i < (k1 - k0) * MR; i += 256) {
        const int m = i / (k1 - k0), k = i - m * (k1 - k0);
        xs[k * MR + m] = m < M ? A[(int64_t)m * K + k0 + k] : 0.0f;
    }
    f32x4 acc[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    __syncthreads();
    for (int k = k0 + g; k < k1; k += G * U) {
        f32x4 b[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // Rows and columns past the end read the last ones; those rows' x is 0.
            const float* const row = B + (int64_t)min(k + u * G, k1 - 1) * N;
            if (VEC) {
                b[u] = *reinterpret_cast<const f32x4*>(row + min(j0, (int64_t)N - 4));
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) b[u][e] = row[min(j0 + e, (int64_t)N - 1)];
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k + u * G >= k1) break;
            const float* const x = xs + (k + u * G - k0) * MR;
#pragma unroll
            for (int m = 0; m < MR; ++m)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[m][e] = __builtin_fmaf(x[m], b[u][e], acc[m][e]);
        }
    }
    float* const to = out + (partial ? (int64_t)blockIdx.y * M * N : 0);
#pragma unroll
    for (int m0 = 0; m0 < MR; m0 += MB) {
#pragma unroll
        for (int m = 0; m < MB; ++m) red[m][t] = acc[m0 + m];
        __syncthreads();
        // Thread t finishes row m0 + t / (4 LC) .. of column t % (4 LC).
        for (int q = t; q < MB * 4 * LC; q += 256) {
            const int m = q / (4 * LC), col = q % (4 * LC);
            float sum = 0.0f;
#pragma unroll
            for (int h = 0; h < G; ++h) sum += red[m][h * LC + col / 4][col % 4];
            const int64_t j = (int64_t)blockIdx.x * 4 * LC + col;
            if (m0 + m < M && j < N) to[(int64_t)(m0 + m) * N + j] = bias ? sum + bias[j] : sum;
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(256) void rows_sum_kernel(const float* __restrict__ partial, int S, int M, int N,
                                                       const float* __restrict__ bias, float* __restrict__ out) {
    const int64_t mn = (int64_t)M * N, idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= mn) return;
    float sum = 0.0f;
    for (int s0 = 0; s0 < S; s0 += 8) {
        float p[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) p[u] = partial[min(s0 + u, S - 1) * mn + idx];
#pragma unroll
        for (int u = 0; u < 8; ++u) sum += s0 + u < S ? p[u] : 0.0f;
    }
    out[idx] = bias ? sum + bias[idx % N] : sum;
}

int launch_f32_rows(kh::Device* d, const float* A, const float* B, float* out, const float* bias, int64_t M, int64_t N,
                    int64_t K) {
    const bool vec = N % 4 == 0 && kh::aligned(B, 16), narrow = N <= 128;
    const int64_t groups = (N + (narrow ? 63 : 255)) / (narrow ? 64 : 256);
    // Two workgroups to a CU, each at least 32 k (its lane groups' first loads)
    // and at most what its copy of A's rows holds.
    int64_t S = std::min<int64_t>({kRowsSplits, std::max<int64_t>(1, 2 * (int64_t)d->cus / groups), (K + 31) / 32});
    S = std::max<int64_t>(S, (K + kRowsK - 1) / kRowsK);
    const int kper = (int)((K + S - 1) / S);
    S = (K + kper - 1) / kper;
    void* work = nullptr;
    if (S > 1) {
        int rc = kh_alloc((size_t)S * (size_t)(M * N) * sizeof(float), &work);
        if (rc) return rc;
    }
    float* const to = S > 1 ? static_cast<float*>(work) : out;
    const dim3 grid((unsigned)groups, (unsigned)S);
    auto go = [&](auto mr) {
        constexpr int MR = decltype(mr)::value;
        const float* const b = S > 1 ? nullptr : bias;
        const int p = S > 1;
        if (narrow && vec) gemm_f32_rows_kernel<MR, 16, true><<<grid, 256, 0, d->stream>>>(A, B, (int)M, (int)N, (int)K, kper, b, to, p);
        else if (narrow) gemm_f32_rows_kernel<MR, 16, false><<<grid, 256, 0, d->stream>>>(A, B, (int)M, (int)N, (int)K, kper, b, to, p);
        else if (vec) gemm_f32_rows_kernel<MR, 64, true><<<grid, 256, 0, d->stream>>>(A, B, (int)M, (int)N, (int)K, kper, b, to, p);
        else gemm_f32_rows_kernel<MR, 64, false><<<grid, 256, 0, d->stream>>>(A, B, (int)M, (int)N, (int)K, kper, b, to, p);
    };
    if (M == 1) go(std::integral_constant<int, 1>());
    else if (M == 2) go(std::integral_constant<int, 2>());
    else if (M <= 4) go(std::integral_constant<int, 4>());
    else if (M <= 8) go(std::integral_constant<int, 8>());
    else if (M <= 16) go(std::integral_constant<int, 16>());
    else go(std::integral_constant<int, 32>());
    int rc = kh::launch_status("gemm_f32_rows");
    if (S > 1) {
        if (!rc) {
            rows_sum_kernel<<<(unsigned)((M * N + 255) / 256), 256, 0, d->stream>>>(to, (int)S, (int)M, (int)N, bias, out);
            rc = kh::launch_status("rows_sum");
        }
        kh_free(work);  // stream-ordered: reused only by work queued after the sum
    }
    return rc;
}

// The planes' and partials' pooled memory, at most.
constexpr size_t kF32xMost = (size_t)16 << 30;

// False (nothing launched) where the kernel's offsets or the memory do not
// allow it.
//
// Tiles: 128 x 128 from 1.5 of them per CU (4096^3: 64 x 64 915 us, 64 x 128 772,
// 128 x 128 718; 2000 x 4096 x 2048 254, 219, 194), 64 x 128 down to one per CU
// (2048 x 2048 x 512: 39, 34, 38), else 64 x 64 with K split until the tiles come to
// one a CU, each split keeping two units (20 x 409 x 4096 47 -> 12, 190 x 72 x 512
// 10.7 -> 9.1): four stages while a workgroup has a CU to itself, else two, three
// workgroups to a CU (1000 x 1000 x 2000, 256 tiles: 36 against 47 us).
bool launch_f32x(kh::Device* d, const float* A, const float* B, float* out, const float* bias, int64_t M, int64_t N,
                 int64_t K, int* rc) {
    const int64_t KT = (K + kUnitK - 1) / kUnitK, Kp = KT * kUnitK, cus = d->cus;
    const int64_t rows = (M + 31) / 32, cols = (N + 63) / 64;
    const int64_t t64 = ((M + 63) / 64) * cols, t64x128 = ((M + 63) / 64) * ((N + 127) / 128);
    const int64_t t128 = ((M + 127) / 128) * ((N + 127) / 128);
    if (128 * Kp * 2 > 0x7FFFFFFF || M > 0x7FFFFFFF || (rows + cols) * KT > 0x7FFFFFFF || t64 > 0x7FFFFFFF) return false;
    const bool big = 2 * t128 >= 3 * cus, wide = !big && t64x128 >= cus;
    int S = 1;
    while (!big && !wide && S < 8 && t64 * S * 2 <= cus && KT >= 4 * S) S *= 2;
    const size_t plane_a = (size_t)3 * M * Kp * 2, plane_b = (size_t)3 * N * Kp * 2;  // (multiples of 128)
    const size_t stats_at = plane_a + plane_b, stats = (size_t)((rows + 2 * cols) * KT + 3) / 4 * 4 * sizeof(int);
    const size_t sums_at = stats_at + stats, bytes = sums_at + (S > 1 ? (size_t)S * M * N * sizeof(float) : 0);
    if (bytes > kF32xMost) return false;
    void* work = nullptr;
    if (kh_alloc(bytes, &work) != KH_OK) return false;
    char* const base = static_cast<char*>(work);
    __bf16* const pa = reinterpret_cast<__bf16*>(base);
    __bf16* const pb = reinterpret_cast<__bf16*>(base + plane_a);
    int* const ea = reinterpret_cast<int*>(base + stats_at);
    int* const eb = ea + rows * KT;
    const bool va = K % 4 == 0 && kh::aligned(A, 16), vb = N % 4 == 0 && kh::aligned(B, 16);
    const unsigned grid = (unsigned)((rows + cols) * KT);
    auto split = [&](auto a, auto b) {
        split_units_kernel<decltype(a)::value, decltype(b)::value><<<grid, 256, 0, d->stream>>>(
            A, B, (int)M, (int)N, (int)K, (int)KT, (int)(rows * KT), pa, pb, ea, eb);
    };
    if (va && vb) split(std::true_type(), std::true_type());
    else if (va) split(std::true_type(), std::false_type());
    else if (vb) split(std::false_type(), std::true_type());
    else split(std::false_type(), std::false_type());
    *rc = kh::launch_status("split_units");
    if (!*rc) {
        const F32x o{A, B, ea, eb, bias, out, S > 1 ? reinterpret_cast<float*>(base + sums_at) : nullptr};
        *rc = big              ? launch_f32x_cfg<128, 128, 2>(d, pa, pb, M, N, K, 1, o)
              : wide           ? launch_f32x_cfg<64, 128, 2>(d, pa, pb, M, N, K, 1, o)
              : t64 * S <= cus ? launch_f32x_cfg<64, 64, 4>(d, pa, pb, M, N, K, S, o)
                               : launch_f32x_cfg<64, 64, 2>(d, pa, pb, M, N, K, 1, o);
    }
    kh_free(work);  // stream-ordered: reused only by work queued after the product
    return true;
}

}  // namespace
