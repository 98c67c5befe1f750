// gfx950 prefill GEMMs on three-limb bf16 products (prefill_limb.h): every grid that fills the
// device, and those that gemm_split_kernel / gemm_reg_kernel (short prompts) do not take.

#include "prefill_limb.h"

#include <type_traits>

namespace flux {
namespace {

constexpr int kLimbStage = 16;   // K values per stage
constexpr int kLimbBN = 128;     // block columns: two waves of 64 (one epilogue column group each)

// C = epilogue(A[M,K] * W[N,K]^T).  Block tile (32 TM WM) x 128, WM x 2 waves, wave tile
// (32 TM) x 64.
//
// A stage is 16 K values.  Each thread loads whole float4s of the block's rows (four lanes per
// 64-byte segment, kDepth stages ahead), splits them into limbs and writes those to LDS, each
// limb as two units (the halves of the stage) of one 16-byte word per row: a wave's operand
// reads are then contiguous, and the writes of eight rows cover all banks.  Splitting here
// rather than in a pass of its own needs no workspace and moves 4 instead of 6 bytes per value
// through L2.
//
// Stage s multiplies operands that are already in registers, reads those of stage s + 1 from
// one LDS buffer and writes the limbs of stage s + 2 to the other, so one barrier per stage
// suffices and no wave waits for LDS before its first product.  The scheduling groups deal the
// split's vector instructions, the reads and the writes out between the products, which keeps
// the matrix cores busy while the waves of a SIMD run the same code in step (8192 x 3072 x 576:
// 164 us, 175 without them).
//
// Bound by power: 8192 x 3072 x 576 takes 152 to 170 us from card to card (170 to 190 TFLOP/s of
// float32 products, 1.02 to 1.14 PFLOP/s of bf16; a large bf16 matrix product reaches 1.18), at
// 1.9 GHz with the matrix cores busy for half of it, and 110 when every value is zero.  The
// float32 instruction took 228 us there.  A second accumulator for the small
// products costs 6% of the time and takes the error against 64 bits from 3.6e-7 to 1.4e-7 at
// K = 576 (float32 instruction: 4.4e-7).
//
// kKB > 1: blockIdx.x = column tile * kKB + kb; block kb covers the kb-th part of K and writes
// its tile to partial plane kb of args.split_partials.
template <GemmEpilogue E, int WM, int TM, int kKB>
__global__ void __launch_bounds__(128 * WM, 2) gemm_limb_kernel(GemmArgs args) {
    constexpr int WN = 2, TN = 2;
    constexpr int BM = 32 * TM * WM;
    constexpr int BN = kLimbBN;
    constexpr int kThreads = 64 * WM * WN;
    constexpr int kDepth = 2;  // stages of float32 rows in flight per thread
    constexpr int kQuadsA = BM * 4 / kThreads;
    constexpr int kQuads = (BM + BN) * 4 / kThreads;
    static_assert(BM * 4 % kThreads == 0 && BN * 4 % kThreads == 0, "whole quads per thread");
    constexpr int kUnit = (BM + BN) * 16 + 128;  // A rows, then W rows; the two units on different banks
    constexpr int kLimb = 2 * kUnit;
    __shared__ __align__(16) char tile[2][kLimbs * kLimb];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN;
    const int wn = wave % WN;
    const int64_t m0 = static_cast<int64_t>(blockIdx.y) * BM;
    const int kb = kKB > 1 ? static_cast<int>(blockIdx.x % kKB) : 0;
    const int n0 = static_cast<int>(blockIdx.x / kKB) * BN;
    const int K = args.k;
    const int span = K / kKB;
    const int k_first = kb * span;

    const float* src[kQuads];
    int dst[kQuads];
#pragma unroll
    for (int i = 0; i < kQuads; ++i) {
        const int u = tid + kThreads * i;
        const int row = u >> 2, q = u & 3;
        if (i < kQuadsA) {
            const int64_t gr = m0 + row < args.m ? m0 + row : args.m - 1;
            src[i] = args.a + gr * K + k_first + 4 * q;
        } else {
            const int c = n0 + row - BM;
            src[i] = args.b + static_cast<int64_t>(b_row<E>(c < args.n ? c : args.n - 1, args.n)) * K + k_first + 4 * q;
        }
        dst[i] = (q >> 1) * kUnit + row * 16 + (q & 1) * 8;
    }
    float largest = 0.0f;

    // Two accumulators per tile: the products of the leading limbs, and the five small ones,
    // whose roundings then happen at their own magnitude.
    f32x16 acc[TM][TN], low[TM][TN];
    auto clear = [&] {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = low[i][j][r] = 0.0f;
    };
    clear();

    const int h = lane >> 5;
    const int a_rd = h * kUnit + (wm * 32 * TM + (lane & 31)) * 16;
    const int b_rd = h * kUnit + (BM + wn * 32 * TN + (lane & 31)) * 16;
    const int stages = span / kLimbStage;

    f32x4 raw[kDepth][kQuads];
    u32x4 op_a[TM][kLimbs], op_b[TN][kLimbs];
    // Stages past the last repeat it (their limbs are not read).
    auto load_quad = [&](auto set, int i, int s) {
        raw[decltype(set)::value][i] =
            *reinterpret_cast<const f32x4_u*>(src[i] + (s < stages ? s : stages - 1) * kLimbStage);
    };
    auto split_quad = [&](auto set, int i, char* buf) {
        const f32x4 v = raw[decltype(set)::value][i];
        unsigned l[kLimbs][2];
        track_max(largest, v[0], v[1]);
        track_max(largest, v[2], v[3]);
        split_pair(v[0], v[1], l[0][0], l[1][0], l[2][0]);
        split_pair(v[2], v[3], l[0][1], l[1][1], l[2][1]);
#pragma unroll
        for (int j = 0; j < kLimbs; ++j)
            *reinterpret_cast<uint2*>(buf + dst[i] + j * kLimb) = make_uint2(l[j][0], l[j][1]);
    };
    auto read_a = [&](int l, const char* buf) {
#pragma unroll
        for (int i = 0; i < TM; ++i) op_a[i][l] = *reinterpret_cast<const u32x4*>(buf + a_rd + l * kLimb + 512 * i);
    };
    auto read_b = [&](int l, const char* buf) {
#pragma unroll
        for (int j = 0; j < TN; ++j) op_b[j][l] = *reinterpret_cast<const u32x4*>(buf + b_rd + l * kLimb + 512 * j);
    };
    auto products = [&](int la, int lb) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                f32x16& c = la + lb == 0 ? acc[i][j] : low[i][j];
                c = mfma_bf16(op_a[i][la], op_b[j][lb], c);
            }
    };
    auto stage = [&](auto set, int s) {
        constexpr int c = decltype(set)::value;
        // Every limb of the next stage is read once its register's last product has issued, so
        // one set of operand registers serves two stages.
        const char* next = tile[1 - c];
        products(2, 0);
        read_a(2, next);
        products(0, 0);
        products(0, 1);
        products(0, 2);
        read_a(0, next);
        read_b(2, next);
        products(1, 0);
        read_b(0, next);
        products(1, 1);
        read_a(1, next);
        read_b(1, next);
#pragma unroll
        for (int i = 0; i < kQuads; ++i) {
            split_quad(set, i, tile[c]);
            load_quad(set, i, s + 2 + kDepth);
        }
        constexpr int kProducts = kLimbProducts * TM * TN;
        constexpr int kVector = (kQuads * 28 + kProducts - 1) / kProducts;  // about 28 per quad
#pragma unroll
        for (int q = 0; q < kProducts; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);        // one product
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);        // one LDS read
            __builtin_amdgcn_sched_group_barrier(0x002, kVector, 0);  // its share of the split
            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);        // one LDS write
        }
        lds_barrier();
    };
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
#pragma unroll
    for (int i = 0; i < kQuads; ++i) load_quad(even, i, 0);
#pragma unroll
    for (int i = 0; i < kQuads; ++i) load_quad(odd, i, 1);
#pragma unroll
    for (int i = 0; i < kQuads; ++i) {
        split_quad(even, i, tile[0]);
        load_quad(even, i, 2);
    }
#pragma unroll
    for (int i = 0; i < kQuads; ++i) {
        split_quad(odd, i, tile[1]);
        load_quad(odd, i, 3);
    }
    lds_barrier();
#pragma unroll
    for (int l = 0; l < kLimbs; ++l) {
        read_a(l, tile[0]);
        read_b(l, tile[0]);
    }
    lds_barrier();
    for (int s = 0; s < stages; s += 2) {
        stage(even, s);
        if (s + 1 < stages) stage(odd, s + 1);
    }

#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] += low[i][j];
    // Tiles on the float32 instruction: one with an infinity, or a magnitude bf16 cannot hold, and
    // one with a value that is not finite, since where the leading products overflow to one
    // infinity the small ones may overflow to the other.
    float finite[TM][TN];  // zero times every value: zero if they are finite
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            finite[i][j] = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; ++r) finite[i][j] = fmaf(acc[i][j][r], 0.0f, finite[i][j]);
        }
    bool redo = !(largest <= kLimbMax);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) redo |= finite[i][j] != 0.0f;
    // And one where bits that the limbs do not carry (limbs_drop) could show: at most 2^-134 of
    // each value, so K 2^-101 of a result while no magnitude is above 2^32, and less than 2^-26 of
    // it from K 2^-75 on.  Tiles with smaller results (an exact zero, most often) or larger values
    // look at their values first; others pay nothing for this (the smallest magnitude tracked in
    // the loop instead: gate/up at 8192 rows 158 -> 169 us, down 100 -> 111).
    float least = INFINITY;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) least = fminf(least, fabsf(acc[i][j][r]));
    if (__syncthreads_or(redo || largest > 0x1p32f || least < 0x1p-75f * static_cast<float>(span))) {
        // The rows of each quad again: their pointers, kept over the loop above, would cost the
        // 128-row tile 6% of its time.
        int u = tid;
        asm volatile("" : "+v"(u));
#pragma unroll 1
        for (int i = 0; i < kQuads; ++i, u += kThreads) {
            const int row = u >> 2;
            const int64_t gr = m0 + row < args.m ? m0 + row : args.m - 1;
            const int c = n0 + row - BM < args.n ? n0 + row - BM : args.n - 1;
            const float* at = (row < BM ? args.a + gr * K : args.b + static_cast<int64_t>(b_row<E>(c, args.n)) * K) +
                              k_first + 4 * (u & 3);
#pragma unroll 4
            for (int s = 0; s < stages; ++s) {
                const f32x4 v = *reinterpret_cast<const f32x4_u*>(at + s * kLimbStage);
                redo |= limbs_drop(v[0]) || limbs_drop(v[1]) || limbs_drop(v[2]) || limbs_drop(v[3]);
            }
        }
        redo = __syncthreads_or(redo);
    }
    if (redo) {
        clear();
#pragma unroll 1
        for (int k = k_first + 4 * h; k < k_first + span; k += 8) {
            f32x4 a[TM], b[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int64_t row = m0 + (wm * TM + i) * 32 + (lane & 31);
                a[i] = *reinterpret_cast<const f32x4_u*>(args.a + (row < args.m ? row : args.m - 1) * K + k);
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int col = n0 + (wn * TN + j) * 32 + (lane & 31);
                b[j] = *reinterpret_cast<const f32x4_u*>(
                    args.b + static_cast<int64_t>(b_row<E>(col < args.n ? col : args.n - 1, args.n)) * K + k);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][e], b[j][e], acc[i][j], 0, 0, 0);
        }
    }
    const int g0 = n0 + wn * 64;
    if (g0 >= args.n) return;
    if constexpr (kKB > 1) {
        GemmArgs plane = args;
        plane.c = args.split_partials + static_cast<int64_t>(kb) * args.m * args.n;
        gemm_epilogue<GemmEpilogue::kStore, TM>(plane, acc, m0 + wm * 32 * TM, g0, lane);
    } else {
        gemm_epilogue<E, TM>(args, acc, m0 + wm * 32 * TM, g0, lane);
    }
}

// Microseconds per stage of a grid of `blocks` blocks (fits of measured times, 24 to 3072 blocks
// at K = 576; at K = 64 to 4096 and widths of 576 to 3072 the tile chosen by them measured within
// 8% of the fastest, most within 2%): one round of 256 x 128 tiles (8 waves, one block per CU) takes 1.0 to 1.5 as it
// fills, 256 blocks of 128 x 128 (two per CU) 0.73 to 0.9 alone and 0.8 each beyond, 256 of
// 64 x 128 0.46 each and never under 0.57.
double stage_us(int rows, int64_t blocks) {
    const int64_t full = blocks / 256, rest = blocks % 256;
    const double part = static_cast<double>(rest) / 256.0;
    if (rows == 256) return 1.5 * full + (rest > 0 ? 1.0 + 0.5 * part : 0.0);
    if (rows == 128) return 0.8 * full + (rest > 0 ? (full > 0 ? 0.55 : 0.73) + 0.2 * part : 0.0);
    const double t = 0.46 * (full + (rest > 0 ? 1 : 0));
    return t < 0.57 ? 0.57 : t;
}

template <GemmEpilogue E, int kKB>
hipError_t launch_tile(const GemmArgs& args, int rows, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>((args.n + kLimbBN - 1) / kLimbBN * kKB),
                    static_cast<unsigned>((args.m + rows - 1) / rows));
    if (rows == 256)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(gemm_limb_kernel<E, 4, 2, kKB>), grid, dim3(512), 0, stream, args);
    else if (rows == 128)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(gemm_limb_kernel<E, 2, 2, kKB>), grid, dim3(256), 0, stream, args);
    else
        hipLaunchKernelGGL(HIP_KERNEL_NAME(gemm_limb_kernel<E, 2, 1, kKB>), grid, dim3(256), 0, stream, args);
    return hipGetLastError();
}

}  // namespace

// The tile and K split with the least estimated time.  Partial planes cost their reads in the
// kernel that sums them: 0.92 ps per value and plane inside a norm that reads its rows anyway,
// or a kernel of its own (3 us, and the sum's write and the residual's read too).
LimbPlan limb_plan(const GemmArgs& args, int max_parts, bool fused_reduce) {
    LimbPlan best{256, 1};
    double best_us = 1e30;
    const double values = static_cast<double>(args.m) * args.n;
    for (int parts = 1; parts <= max_parts; ++parts) {
        if (args.k % (kLimbStage * parts) != 0) continue;
        const double reduce = fused_reduce ? 0.92e-6 * parts * values
                              : parts == 1 ? 0.0
                                           : 3.0 + 0.7e-6 * (parts + 2) * values;
        for (int rows = 256; rows >= 64; rows /= 2) {
            const int64_t blocks =
                static_cast<int64_t>((args.n + kLimbBN - 1) / kLimbBN) * parts * ((args.m + rows - 1) / rows);
            const double us = stage_us(rows, blocks) * (args.k / (kLimbStage * parts)) + reduce;
            if (us < best_us) {
                best_us = us;
                best = LimbPlan{rows, parts};
            }
        }
    }
    return best;
}

hipError_t launch_limb_gemm(const GemmArgs& args, GemmEpilogue epilogue, const LimbPlan& plan, hipStream_t stream) {
    if (plan.parts == 2) return launch_tile<GemmEpilogue::kStore, 2>(args, plan.rows, stream);
    if (plan.parts == 3) return launch_tile<GemmEpilogue::kStore, 3>(args, plan.rows, stream);
    switch (epilogue) {
        case GemmEpilogue::kStore:
            return launch_tile<GemmEpilogue::kStore, 1>(args, plan.rows, stream);
        case GemmEpilogue::kResidual:
            return launch_tile<GemmEpilogue::kResidual, 1>(args, plan.rows, stream);
        case GemmEpilogue::kSwiglu:
            return launch_tile<GemmEpilogue::kSwiglu, 1>(args, plan.rows, stream);
        case GemmEpilogue::kQkvRope:
            return launch_tile<GemmEpilogue::kQkvRope, 1>(args, plan.rows, stream);
    }
    return hipErrorInvalidValue;
}

}  // namespace flux
