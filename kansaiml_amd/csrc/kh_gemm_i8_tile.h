// kh_gemm_i8_tile.h -- the int8 GEMM for products that do not fill the chip
// with the ping-pong kernel's tiles, and for operands whose rows are not 16-byte
// aligned.  Internal: included by kh_gemm_i8.hip after its epilogue.
//
// * Workgroup tile BM x BN (64 or 128 each), 4 waves as 2 x 2, each
//   (BM / 2) x (BN / 2) outputs as 32x32 blocks of v_mfma_i32_32x32x32_i8.
//   Several workgroups share a CU, so one's barrier, fragment reads and
//   epilogue run under another's products.
// * K in steps of 128 bytes per row, through a ring of NS LDS stages of
//   (BM + BN) x 128 bytes.  16-byte chunk c of row r lies in slot
//   c ^ ((r >> 1) & 7): two rows span the 64 banks, so 16 consecutive rows of
//   one chunk (a quarter of a fragment read) fall on distinct banks.
// * DMA: rows 16-byte aligned (K % 16 == 0).  Operands arrive by LDS-DMA, NS
//   stages ahead.  A step waits for this wave's loads of stage k + 1 and its
//   fragment reads of stage k, meets the other waves, refills the slot of stage
//   k, reads the fragments of stage k + 1 and multiplies those of stage k.  The loop
//   is unrolled over the ring: with the stage a run-time index a step spent more
//   on addresses than on products (65 x 4096 x 4096: 13.6 us, at any depth of
//   ring; unrolled 9.6).  Chunks at k >= K get an offset past the resource and
//   read zeros.  Bound: LDS, which a step of a 64 x 64 tile writes 16 KB to and
//   reads 32 KB from (384 cycles of the ~380 it takes alone on a CU).
// * Otherwise (any K, any alignment) each thread loads its 16-byte chunks from
//   their unaligned addresses two stages ahead and writes them to LDS.  An
//   address past the operand's last 16 bytes is pulled back to them; only the
//   last stage holds such chunks and chunks past the row's end, so only there
//   are bytes shifted into place and A's bytes at k >= K cleared (B's may then
//   be anything).
// * Split K: workgroup (x, y) sums steps [y kper, (y + 1) kper) and writes its
//   int32 sums as partial y (skinny_splitk_epilogue_kernel adds them up).
#pragma once

#include "kh_rows.h"

namespace {

using kh::rows::i32x4_any;
using kh::rows::tail_bytes;

template <int BM, int BN, int NS, bool FUSED, bool DMA>
__global__ __launch_bounds__(256, (BM + BN) * 128 * NS <= 53248 ? 3 : (BM + BN) * 128 * NS <= 81920 ? 2 : 1) void gemm_i8_tile_kernel(
    const int8_t* __restrict__ A, const int8_t* __restrict__ B, int M, int N, int K, int kper, int group_m,
    Epilogue ep, unsigned* parts) {
    using namespace kh::pipe;
    constexpr int BK = 128, kTM = BM / 64, kTN = BN / 64;
    constexpr int kLdsA = BM * BK, kStage = (BM + BN) * BK;
    constexpr int kAInst = BM / 32, kBInst = BN / 32;  // 16-byte chunks per lane and stage
    constexpr int kLoads = kAInst + kBInst;
    static_assert(NS == 2 || (DMA && NS == 4), "a turn of the ring below");
    __shared__ __attribute__((aligned(1024))) int8_t lds[NS * kStage];

    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    int tm, tn;
    tile_of(blockIdx.x, tiles_m, tiles_n, group_m, tm, tn);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int rows_a = min(BM, M - tm * BM), rows_b = min(BN, N - tn * BN);
    auto swz = [](int r) { return (r >> 1) & 7; };
    const int k_steps = (K + BK - 1) / BK;
    const int kt0 = blockIdx.y * kper, kt1 = min(k_steps, kt0 + kper);

    // Fragments: lane l reads 16 bytes of row r + l % 32 at chunk 2 s + l / 32.
    // One LDS address per block and s: the stage is an immediate offset (the
    // loop below is unrolled over the ring), so a step computes no address.
    const int fr = lane & 31, fh = lane >> 5;
    int a_off[4][kTM], b_off[4][kTN];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
#pragma unroll
        for (int a = 0; a < kTM; ++a) {
            const int r = wm * (BM / 2) + a * 32 + fr;
            a_off[s][a] = r * BK + (((fh + 2 * s) ^ swz(r)) << 4);
        }
#pragma unroll
        for (int b = 0; b < kTN; ++b) {
            const int r = wn * (BN / 2) + b * 32 + fr;
            b_off[s][b] = kLdsA + r * BK + (((fh + 2 * s) ^ swz(r)) << 4);
        }
    }
    i32x16 acc[kTM][kTN];
#pragma unroll
    for (int a = 0; a < kTM; ++a)
#pragma unroll
        for (int b = 0; b < kTN; ++b) acc[a][b] = i32x16{0};

    // The fragments of a stage are read while the products of the stage before
    // run, into the other of two register sets.
    struct Frags {
        i32x4 a[4][kTM], b[4][kTN];
    };
    Frags f0, f1;
    auto read = [&](const int8_t* base, Frags& f) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
            for (int a = 0; a < kTM; ++a) f.a[s][a] = *reinterpret_cast<const i32x4*>(base + a_off[s][a]);
#pragma unroll
            for (int b = 0; b < kTN; ++b) f.b[s][b] = *reinterpret_cast<const i32x4*>(base + b_off[s][b]);
        }
    };
    auto multiply = [&](const Frags& f) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int a = 0; a < kTM; ++a)
#pragma unroll
                for (int b = 0; b < kTN; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.a[s][a], f.b[s][b], acc[a][b], 0, 0, 0);
    };
    // Ends a step's reads for this wave and meets the others: after it every
    // wave has read stage kt, and stage kt + 1 is in LDS.
    auto meet = [&]() {
        __builtin_amdgcn_s_waitcnt(wait_imm(63, 0));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };

    if constexpr (DMA) {
        // Rows past M (N) lie outside the resource: their loads return zeros.
        const __amdgpu_buffer_rsrc_t ra = make_rsrc(A + (int64_t)tm * BM * K, (uint32_t)rows_a * (uint32_t)K);
        const __amdgpu_buffer_rsrc_t rb = make_rsrc(B + (int64_t)tn * BN * K, (uint32_t)rows_b * (uint32_t)K);
        // Instruction i of this wave fills rows (wave kInst + i) 8 + l / 8,
        // slot l % 8.
        int a_voff[kAInst], b_voff[kBInst];
#pragma unroll
        for (int i = 0; i < kAInst; ++i) {
            const int r = (wave * kAInst + i) * 8 + (lane >> 3);
            a_voff[i] = r * K + (((lane & 7) ^ swz(r)) << 4);
        }
#pragma unroll
        for (int i = 0; i < kBInst; ++i) {
            const int r = (wave * kBInst + i) * 8 + (lane >> 3);
            b_voff[i] = r * K + (((lane & 7) ^ swz(r)) << 4);
        }
        constexpr int kPast = 0x7FFF0000;  // past every tile's resource (at most 128 rows of 133144 bytes)
        auto issue = [&](int kt, int slot) {
            int8_t* base = lds + slot * kStage;
            const int k0 = kt * BK;
            if (k0 + BK <= K) {
#pragma unroll
                for (int i = 0; i < kAInst; ++i) lds_dma16(ra, base + (wave * kAInst + i) * 1024, a_voff[i], k0);
#pragma unroll
                for (int i = 0; i < kBInst; ++i)
                    lds_dma16(rb, base + kLdsA + (wave * kBInst + i) * 1024, b_voff[i], k0);
            } else {
#pragma unroll
                for (int i = 0; i < kAInst; ++i) {
                    const int r = (wave * kAInst + i) * 8 + (lane >> 3);
                    const bool past = k0 + (((lane & 7) ^ swz(r)) << 4) >= K;
                    lds_dma16(ra, base + (wave * kAInst + i) * 1024, past ? kPast : a_voff[i], k0);
                }
#pragma unroll
                for (int i = 0; i < kBInst; ++i) {
                    const int r = (wave * kBInst + i) * 8 + (lane >> 3);
                    const bool past = k0 + (((lane & 7) ^ swz(r)) << 4) >= K;
                    lds_dma16(rb, base + kLdsA + (wave * kBInst + i) * 1024, past ? kPast : b_voff[i], k0);
                }
            }
        };
#pragma unroll
        for (int s = 0; s < NS; ++s)
            if (kt0 + s < kt1) issue(kt0 + s, s);
        wait_loads_beyond<kLoads>(min(NS - 1, kt1 - 1 - kt0));
        meet();
        read(lds, f0);
        // Step j of a turn of the ring (kt = kt0 + j mod NS).  Steady: every
        // stage it touches exists, so nothing is tested.
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
    } else {
        // Offsets from the tile's first row; the operand's last 16 bytes start
        // at a_last / b_last, which a short last row leaves below 0 (the launch:
        // M K and N K >= 16).
        const int8_t* const pa = A + (int64_t)tm * BM * K;
        const int8_t* const pb = B + (int64_t)tn * BN * K;
        const int a_last = (int)min((int64_t)0x7FFFFFFF, (int64_t)(M - tm * BM) * K - 16);
        const int b_last = (int)min((int64_t)0x7FFFFFFF, (int64_t)(N - tn * BN) * K - 16);
        const int ch = tid & 7;
        int ao[kAInst], bo[kBInst];
        int lds_off[kAInst > kBInst ? kAInst : kBInst];
#pragma unroll
        for (int i = 0; i < kAInst; ++i) ao[i] = min((tid >> 3) + 32 * i, rows_a - 1) * K + ch * 16;
#pragma unroll
        for (int i = 0; i < kBInst; ++i) bo[i] = min((tid >> 3) + 32 * i, rows_b - 1) * K + ch * 16;
#pragma unroll
        for (int i = 0; i < (kAInst > kBInst ? kAInst : kBInst); ++i) {
            const int r = (tid >> 3) + 32 * i;
            lds_off[i] = r * BK + ((ch ^ swz(r)) << 4);
        }
        struct Chunks {
            i32x4 a[kAInst], b[kBInst];
        };
        Chunks c0, c1;  // two stages of loads in flight
        auto load = [&](int kt, Chunks& c, auto steady) {
            const int k0 = kt * BK;
            if (decltype(steady)::value || kt < k_steps - 1) {
#pragma unroll
                for (int i = 0; i < kAInst; ++i)
                    c.a[i] = *reinterpret_cast<const i32x4_any*>(pa + k0 + (unsigned)ao[i]);
#pragma unroll
                for (int i = 0; i < kBInst; ++i)
                    c.b[i] = *reinterpret_cast<const i32x4_any*>(pb + k0 + (unsigned)bo[i]);
            } else {
                // A whole stage inside the row cannot pass the operand's end.
#pragma unroll
                for (int i = 0; i < kAInst; ++i)
                    c.a[i] = *reinterpret_cast<const i32x4_any*>(pa + min(k0 + ao[i], a_last));
#pragma unroll
                for (int i = 0; i < kBInst; ++i)
                    c.b[i] = *reinterpret_cast<const i32x4_any*>(pb + min(k0 + bo[i], b_last));
            }
        };
        auto store = [&](int kt, int8_t* base, Chunks& c, auto steady) {
            if (!decltype(steady)::value && kt == k_steps - 1) {
                const int k0 = kt * BK, n = K - k0 - ch * 16;
#pragma unroll
                for (int i = 0; i < kAInst; ++i)
                    c.a[i] = tail_bytes(c.a[i], k0 + ao[i] - min(k0 + ao[i], a_last), n);
#pragma unroll
                for (int i = 0; i < kBInst; ++i)
                    c.b[i] = tail_bytes(c.b[i], k0 + bo[i] - min(k0 + bo[i], b_last), 16);
            }
#pragma unroll
            for (int i = 0; i < kAInst; ++i) *reinterpret_cast<i32x4*>(base + lds_off[i]) = c.a[i];
#pragma unroll
            for (int i = 0; i < kBInst; ++i) *reinterpret_cast<i32x4*>(base + kLdsA + lds_off[i]) = c.b[i];
        };
        using T = std::true_type;
        using F = std::false_type;
        load(kt0, c0, F());
        if (kt0 + 1 < kt1) load(kt0 + 1, c1, F());
        store(kt0, lds, c0, F());
        if (kt0 + 2 < kt1) load(kt0 + 2, c0, F());
        meet();
        // Stage kt in slot j; `c` holds stage kt + 1, and takes kt + 3.
        // Steady: those exist and are not the row's last, so nothing is tested
        // (behind a test the compiler waits for every load in flight).
        auto step = [&](int kt, int j, Chunks& c, auto steady) {
            constexpr bool kSteady = decltype(steady)::value;
            read(lds + j * kStage, f0);
            __builtin_amdgcn_sched_barrier(0);
            if (kSteady || kt + 1 < kt1) {
                store(kt + 1, lds + (j ^ 1) * kStage, c, steady);
                if (kSteady || kt + 3 < kt1) load(kt + 3, c, steady);
            }
            __builtin_amdgcn_sched_barrier(0);
            multiply(f0);
            meet();
        };
        int kt = kt0;
        for (; kt + 5 < kt1; kt += 2) {
            step(kt, 0, c1, T());
            step(kt + 1, 1, c0, T());
        }
        for (; kt < kt1; kt += 2) {
            step(kt, 0, c1, F());
            if (kt + 1 < kt1) step(kt + 1, 1, c0, F());
        }
    }

    if (ep.acc && !ep.out) ep.acc += (int64_t)blockIdx.y * M * N;
    const int64_t row0 = (int64_t)tm * BM + wm * (BM / 2), col0 = (int64_t)tn * BN + wn * (BN / 2);
    const kh::quant::Scale none{};
    unsigned mx = 0;
#pragma unroll
    for (int a = 0; a < kTM; ++a)
#pragma unroll
        for (int b = 0; b < kTN; ++b) {
            const int64_t i0 = row0 + a * 32, j0 = col0 + b * 32;
            if (i0 + 32 <= M && j0 + 32 <= N && ep.out && !ep.acc && N <= (1 << 24)) {
                const ColEpi ce = col_epi(ep, j0 + fr);
                if (ep.sa_per_row)
                    mx = max(mx, store_block32_full<FUSED, kh::quant::kOutStore, true>(ep, i0, j0, N, lane, 0.0,
                                                                                       acc[a][b], none, ce));
                else
                    mx = max(mx, store_block32_full<FUSED, kh::quant::kOutStore>(ep, i0, j0, N, lane, ep.sa[0],
                                                                                 acc[a][b], none, ce));
            } else {
                mx = max(mx, store_block32_masked<FUSED, 8>(ep, i0 + 4 * fh, j0 + fr, M, N, acc[a][b], none));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    if (parts) {
        // Per-workgroup max |out| bits, for a following per-tensor quantize.
        unsigned* wmax = reinterpret_cast<unsigned*>(lds);
        mx = kh::quant::wave_max(mx);
        __syncthreads();  // every read of the last stage is done
        if (lane == 0) wmax[wave] = mx;
        __syncthreads();
        if (tid == 0) parts[blockIdx.x] = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
    }
}

template <int BM, int BN, int NS, bool DMA>
int launch_tile_cfg(kh::Device* d, const int8_t* A, const int8_t* B, int64_t M, int64_t N, int64_t K,
                    const Epilogue& ep, int splits, unsigned* parts) {
    const unsigned tiles = (unsigned)(((M + BM - 1) / BM) * ((N + BN - 1) / BN));
    const int steps = (int)((K + 127) / 128), kper = (steps + splits - 1) / splits;
    const dim3 grid(tiles, (unsigned)splits);
    if (ep.act != kActNone || ep.residual)
        gemm_i8_tile_kernel<BM, BN, NS, true, DMA>
            <<<grid, 256, 0, d->stream>>>(A, B, (int)M, (int)N, (int)K, kper, 8, ep, parts);
    else
        gemm_i8_tile_kernel<BM, BN, NS, false, DMA>
            <<<grid, 256, 0, d->stream>>>(A, B, (int)M, (int)N, (int)K, kper, 8, ep, parts);
    return kh::launch_status("gemm_i8_tile");
}

int64_t tiles64(int64_t M, int64_t N) { return ((M + 63) / 64) * ((N + 63) / 64); }

// Where the tiles below beat the ping-pong kernel's, which are at least 128 x
// 128 and run one or two workgroups to a CU: up to four 64 x 64 tiles per CU.
// At K = 4096: 256 tiles (M = N = 1024) 24.7 -> 10.6 us, 512 (1024 x 2048)
// 25.5 -> 17.4, 1024 (1024 x 4096) 30.0 -> 27.3.  Up to six where the 128 x 64 tiles
// come to a full round of three workgroups to a CU (768 of them: 16384 x 384 x 1536
// with a residual 22.3 -> 20.6, 4096 x 1536 x 4096 44.4 -> 39.5; 612: 1472 x 3246 x
// 3648 39.0 against 40.7); 2048 tiles (2048 x 4096 x 4096) 53.7 against 56.3.
bool tile_pays(const kh::Device* d, int64_t M, int64_t N, int64_t K) {
    if (K > 0x7FFFFFFF / 128 || M > 0x7FFFFFFF || N > 0x7FFFFFFF) return false;
    const int64_t tiles = tiles64(M, N), wide = ((M + 127) / 128) * ((N + 63) / 64), cus = d->cus;
    return tiles <= 4 * cus || (tiles <= 6 * cus && K > 512 && wide <= 3 * cus && 10 * wide >= 27 * cus);
}

int launch_pingpong(kh::Device* d, const int8_t* A, const int8_t* B, int64_t M, int64_t N, int64_t K,
                    const Epilogue& ep_in, unsigned* parts, int* nparts, int mode);

// Every product of at least 16 bytes an operand that the skinny, narrow and
// ping-pong kernels leave.
//
// Tile: 64 x 64 with four stages (two workgroups of 64 KB to a CU) up to 2.5
// tiles per CU; beyond, 128 x 64 with two (three of 48 KB), which reads a
// quarter less LDS per product: 1024 x 4096 x 4096 31.7 -> 27.3 us, 4096 x 1536
// x 4096 46.5 -> 39.5, but 1024 x 2048 x 4096 17.4 against 22.4.  K <= 512 fills no
// ring of four: 64 x 64 with two stages, three workgroups to a CU, up to three
// tiles per CU (2048 x 1152 x 384 7.8 -> 6.4, 2048 x 1536 x 384 10.3 -> 8.1; 128 x 64:
// 7.1, 9.4).  Unaligned rows take 64 x 64 (1000 x 1250 x 1001 12.4 us, where a
// byte-wise gather took 165; 128 x 64 14.4).
//
// Split K: a few tiles of a long K leave CUs idle, each a chain of K / 128 steps
// of ~0.18 us; the second launch and the partials' round trip cost ~4 us.  Split
// in two, four or eight while the tiles still fit one to a CU and keep ten
// steps: 80 x 64 x 11008 18.8 -> 10.1 us, 128 x 1536 x 11008 19.1 -> 13.4, 512 x
// 1024 x 11008 21.0 -> 18.0.  Below 48 steps it does not pay (128 x 1536 x 4096
// 9.6 against 10.5).
//
// Padded: rows that the large tiles cannot take (K no multiple of 64, or
// unaligned) are first copied to a multiple of 64 where the product is large
// enough to pay for the copy, more than 4 tiles per CU (6 for aligned rows, which
// the 128 x 64 tiles take as they lie); pooled memory, so not where the caller
// cannot allocate.
int launch_tile(kh::Device* d, const int8_t* A, const int8_t* B, int64_t M, int64_t N, int64_t K, const Epilogue& ep,
                bool may_alloc, unsigned* parts, int max_parts, int* nparts, bool* parts_done) {
    KH_REQUIRE(M <= 0x7FFFFFFF && N <= 0x7FFFFFFF && tiles64(M, N) <= 0x7FFFFFFF, "kh_gemm_i8: shape too large");
    const bool dma = K % 16 == 0 && kh::aligned(A, 16) && kh::aligned(B, 16);
    const int64_t tiles = tiles64(M, N), cus = d->cus;
    const int64_t Kp = (K + 63) / 64 * 64;
    if (may_alloc && tiles > (dma ? 6 : 4) * cus && (M + N) * (Kp / 16) / 256 < 0x7FFFFFFF) {
        void* pad = nullptr;
        int rc = kh_alloc((size_t)(M + N) * (size_t)Kp, &pad);
        if (rc) return rc;
        int8_t* const pa = static_cast<int8_t*>(pad);
        int8_t* const pb = pa + M * Kp;
        kh::rows::pad_rows_kernel<<<(unsigned)(((M + N) * (Kp / 16) + 255) / 256), 256, 0, d->stream>>>(
            A, B, (int)M, (int)N, (int)K, (int)Kp, pa);
        rc = kh::launch_status("pad_rows");
        if (!rc) {
            const bool fused = parts && ((M + 127) / 128) * ((N + 127) / 128) <= max_parts;
            rc = launch_pingpong(d, pa, pb, M, N, Kp, ep, fused ? parts : nullptr, fused ? nparts : nullptr,
                                 kh::quant::kOutStore);
            *parts_done = fused;
        }
        kh_free(pad);  // stream-ordered: reused only by work queued after the product
        return rc;
    }
    const bool brief = dma && K <= 512;
    if (dma && tiles > (brief ? 3 * cus : cus * 5 / 2)) {
        const int64_t grid = ((M + 127) / 128) * ((N + 63) / 64);
        *parts_done = parts && grid <= max_parts;
        if (*parts_done) *nparts = (int)grid;
        return launch_tile_cfg<128, 64, 2, true>(d, A, B, M, N, K, ep, 1, *parts_done ? parts : nullptr);
    }
    const int steps = (int)((K + 127) / 128);
    int S = 1;
    if (may_alloc && steps >= 48)
        while (S < 8 && tiles * S * 2 <= cus && steps >= 20 * S) S *= 2;
    if (S > 1) {
        void* partial = nullptr;
        int rc = kh_alloc((size_t)S * (size_t)(M * N) * sizeof(int32_t), &partial);
        if (rc) return rc;
        Epilogue eps = ep;
        eps.out = nullptr;
        eps.acc = static_cast<int32_t*>(partial);
        eps.act = kActNone;
        eps.residual = nullptr;
        rc = dma ? launch_tile_cfg<64, 64, 4, true>(d, A, B, M, N, K, eps, S, nullptr)
                 : launch_tile_cfg<64, 64, 2, false>(d, A, B, M, N, K, eps, S, nullptr);
        if (!rc) {
            skinny_splitk_epilogue_kernel<<<(unsigned)((M * N + 255) / 256), 256, 0, d->stream>>>(
                static_cast<const int32_t*>(partial), S, (int)M, (int)N, ep);
            rc = kh::launch_status("skinny_splitk_epilogue");
        }
        kh_free(partial);  // stream-ordered: reused only by work queued after the sum
        return rc;
    }
    *parts_done = parts && tiles <= max_parts;
    if (*parts_done) *nparts = (int)tiles;
    unsigned* const p = *parts_done ? parts : nullptr;
    return brief ? launch_tile_cfg<64, 64, 2, true>(d, A, B, M, N, K, ep, 1, p)
           : dma ? launch_tile_cfg<64, 64, 4, true>(d, A, B, M, N, K, ep, 1, p)
                 : launch_tile_cfg<64, 64, 2, false>(d, A, B, M, N, K, ep, 1, p);
}

}  // namespace
