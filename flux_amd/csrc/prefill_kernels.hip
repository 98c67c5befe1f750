// gfx950 prefill GEMMs of short prompts on FP32 MFMA, and the launch rules of all prefill GEMMs.
//
// Reference path: csrc/native_prefill_runtime/native_prefill_runtime_cuda.cu:553-665
// (cuBLAS SGEMM linear_fp32 :285-302, QKV RoPE/cache fill kernel :124-163, SwiGLU
// csrc/packed_swiglu/packed_swiglu_cuda.cu:14-31, residual add :267-278).
//
// MI355X design: grids that fill the device take the limb GEMM (prefill_limb_kernels.hip).
// Smaller ones take, for K = 576 / 1536, a register-operand kernel or a split-K kernel whose
// waves stream private LDS rings, both of which fold the preceding RMSNorm into the QKV and
// gate/up GEMMs, or 64 x 64 tiles on a ring of LDS buffers.  The epilogues consume the
// accumulator layout directly: a wave's 64 columns are one head (columns j and j + 32 are the
// RoPE pair) or 32 gate and the 32 matching up columns.  Grids that leave CUs idle split K over
// blocks into partial planes, summed in order by a reduce kernel, or by the RMSNorm kernel that
// the next GEMM needs (split_reduce_residual_norm_kernel).

#include "flux_common.h"
#include "flux_kernels.h"
#include "prefill_common.h"

#include <cfloat>
#include <cmath>
#include <type_traits>

namespace flux {
namespace {

constexpr int kBK = 16;
constexpr int kGemmThreads = 256;

// LDS tile layout (A: BM rows, B: 128 rows; 16 floats of K per row, 64 B): the
// 16-byte piece c of row r sits at piece position c ^ ((r >> 2) & 3), so the 16
// lanes of one ds_read_b128 pass (16 consecutive rows, same piece) cover all banks.
__device__ __forceinline__ int tile_offset(int r, int c) { return r * kBK + 4 * (c ^ ((r >> 2) & 3)); }

// One global_load_lds_dwordx4: each lane copies 16 B from `src` to lds + 16 * lane.
__device__ __forceinline__ void lds_copy16(const float* src, float* lds) {
    __builtin_amdgcn_global_load_lds(src, lds, 16, 0, 0);
}

// Grids smaller than the device (short and mid-length prompts): one block per
// (32 * RT) x 64 output tile, RT = 1, 2 or 4.  Its kSplitWaves waves are RT row tiles
// of 32 times kSplitWaves / RT contiguous K ranges.  A wave streams its 32 A rows and the
// tile's 64 B rows over its K range, 16 K values (64 bytes per row) at a time, 16-byte
// pieces XOR-swizzled by (row >> 2) & 3, through a private ring of kSplitStages LDS buffers;
// while a stage's MFMAs run, the next stage's operands are already in registers and the
// kSplitStages - 2 after it are being copied.  No wave waits for another until the
// partial tiles of one row tile meet in LDS (RT < 4).  They are summed in K order (the
// result does not depend on timing), and the row tile's waves share its epilogue.
constexpr int kSplitWaves = 4;
constexpr int kSplitStages = 5;

template <int S, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (S < N) {
        f(std::integral_constant<int, S>{});
        static_for<S + 1, N>(f);
    }
}

// kStages = K / (kSplitWaves / RT * 16), fixed at compile time so the stage loop is
// straight-line code and every wait names exactly the copies it needs.
// kKB > 1 (the down projection of 113 to 128 rows): blockIdx.x = column tile * kKB + kb, and block
// kb covers the kb-th third of K; instead of the epilogue it writes its summed tile to partial
// plane kb of args.split_partials for split_reduce_residual_kernel.
template <GemmEpilogue E, int kStages, int RT, bool kNorm, int kCols, int kKB>
__global__ void __launch_bounds__(64 * kSplitWaves) gemm_split_kernel(GemmArgs args) {
    static_assert(kSplitStages == 5, "the buffers below are spelled out");
    static_assert(RT == 1 || RT == 2 || RT == 4, "row tiles per block");
    // kCols = 64 (two 32-column MFMA tiles: the RoPE / SwiGLU pair layout) or 32 (plain and
    // residual epilogues only: twice the blocks, half the MFMAs per wave).
    static_assert(kCols == 64 || (kCols == 32 && !kNorm &&
                                  (E == GemmEpilogue::kStore || E == GemmEpilogue::kResidual)),
                  "32-column tiles carry no column pairs");
    static_assert(kKB == 1 || (kCols == 32 && RT == 1), "partial planes of 32-column tiles only");
    constexpr int kTiles = kCols / 32;
    constexpr int kRows = 32 + kCols;  // A rows + B rows per stage
    constexpr int kCopies = kRows / 16;
    constexpr int kParts = kSplitWaves / RT;  // K ranges per row tile
    // One variable per ring slot: a read of one slot then never waits for copies into another.
    __shared__ __align__(16) float r0[kSplitWaves][kRows * kBK];
    __shared__ __align__(16) float r1[kSplitWaves][kRows * kBK];
    __shared__ __align__(16) float r2[kSplitWaves][kRows * kBK];
    __shared__ __align__(16) float r3[kSplitWaves][kRows * kBK];
    __shared__ __align__(16) float r4[kSplitWaves][kRows * kBK];
    __shared__ float partial[kParts > 1 ? kSplitWaves : 1][kTiles][16][64];
    __shared__ __align__(16) float norm_g[kNorm ? kHidden : 4];  // folded RMSNorm: weights of the K values
    __shared__ float norm_ss[kNorm ? kSplitWaves : 1][32];       // folded RMSNorm: sums of squares per row

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row_tile = wave % RT;
    const int part = wave / RT;
    const int64_t m0 = static_cast<int64_t>(blockIdx.y) * 32 * RT + 32 * row_tile;
    const int kb = kKB > 1 ? static_cast<int>(blockIdx.x % kKB) : 0;
    const int n0 = static_cast<int>(blockIdx.x / kKB) * kCols;
    const int K = args.k;
    constexpr int kSpan = kStages * kBK;  // this wave's K values start at (kb * kParts + part) * kSpan
    const int k_first = (kb * kParts + part) * kSpan;
    static_assert(!kNorm || kStages * kBK * kParts * kKB == kHidden, "the folded norm spans the hidden width");
    // Folded RMSNorm: the norm weights are requested before the first copies and stored to LDS
    // after them, so their latency overlaps the copies'.
    constexpr int kNormLoads = (kHidden + 64 * kSplitWaves - 1) / (64 * kSplitWaves);
    float norm_load[kNormLoads];
    if constexpr (kNorm) {
#pragma unroll
        for (int i = 0; i < kNormLoads; ++i) {
            const int k = threadIdx.x + 64 * kSplitWaves * i;
            norm_load[i] = k < kHidden ? args.norm_weight[k] : 0.0f;
        }
    }
    float ss = 0.0f;

    const float* src[kCopies];
#pragma unroll
    for (int i = 0; i < kCopies; ++i) {
        const int row = 16 * i + (lane >> 2);
        const int piece = (lane & 3) ^ ((row >> 2) & 3);
        const float* base;
        if (row < 32) {
            const int64_t ga = m0 + row < args.m ? m0 + row : args.m - 1;
            base = args.a + ga * K;
        } else {
            base = args.b + static_cast<int64_t>(b_row<E>(n0 + row - 32, args.n)) * K;
        }
        src[i] = base + k_first + 4 * piece;
    }
    auto slot = [&](auto bi) -> float* {
        constexpr int b = decltype(bi)::value % kSplitStages;
        if constexpr (b == 0) return r0[wave];
        else if constexpr (b == 1) return r1[wave];
        else if constexpr (b == 2) return r2[wave];
        else if constexpr (b == 3) return r3[wave];
        else return r4[wave];
    };
    auto issue = [&](auto st) {
        float* dst = slot(st);
#pragma unroll
        for (int i = 0; i < kCopies; ++i) lds_copy16(src[i] + decltype(st)::value * kBK, dst + i * 16 * kBK);
    };

    const int h = lane >> 5;
    const int ra = lane & 31;
    const int a_off0 = tile_offset(ra, 2 * h), a_off1 = tile_offset(ra, 2 * h + 1);
    int b_off[kTiles][2];
    f32x16 acc[kTiles];
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
        b_off[j][0] = tile_offset(32 + 32 * j + ra, 2 * h);
        b_off[j][1] = tile_offset(32 + 32 * j + ra, 2 * h + 1);
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = 0.0f;
    }
    struct Operands {
        f32x4 a[2];
        f32x4 b[kTiles][2];
        f32x4 g[2];  // folded RMSNorm: the weights of the a values
    };
    auto read = [&](auto st, Operands& o) {
        const float* t = slot(st);
        o.a[0] = *reinterpret_cast<const f32x4*>(t + a_off0);
        o.a[1] = *reinterpret_cast<const f32x4*>(t + a_off1);
        if constexpr (kNorm) {
            // This lane's K values: pieces 2h and 2h + 1 of the stage.
            const float* g = norm_g + k_first + decltype(st)::value * kBK + 8 * h;
            o.g[0] = *reinterpret_cast<const f32x4*>(g);
            o.g[1] = *reinterpret_cast<const f32x4*>(g + 4);
        }
#pragma unroll
        for (int j = 0; j < kTiles; ++j)
#pragma unroll
            for (int q = 0; q < 2; ++q) o.b[j][q] = *reinterpret_cast<const f32x4*>(t + b_off[j][q]);
    };
    // Folded RMSNorm: accumulate the squares of a stage's raw A values, then scale them by the
    // norm weights of their K indices.
    auto fold_norm = [&](Operands& o) {
        if constexpr (kNorm) {
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    ss = fmaf(o.a[q][e], o.a[q][e], ss);
                    o.a[q][e] *= o.g[q][e];
                }
        }
    };
    constexpr int kAhead = kSplitStages - 1;  // stages issued before the loop
    static_for<0, (kStages < kAhead ? kStages : kAhead)>([&](auto st) { issue(st); });
    if constexpr (kNorm) {
#pragma unroll
        for (int i = 0; i < kNormLoads; ++i) {
            const int k = threadIdx.x + 64 * kSplitWaves * i;
            if (k < kHidden) norm_g[k] = norm_load[i];
        }
        lds_barrier();  // waits for LDS traffic only, not for the copies in flight
    }
    Operands cur, nxt;
    wait_vmcnt<((kStages < kAhead ? kStages : kAhead) - 1) * kCopies>();
    read(std::integral_constant<int, 0>{}, cur);
    fold_norm(cur);
    static_for<0, kStages>([&](auto st) {
        constexpr int s = decltype(st)::value;
        // Slot (s + kAhead) % kSplitStages last held stage s - 1, whose operands were read in
        // step s - 2 and consumed in step s - 1.
        if constexpr (s + 1 < kStages) {
            constexpr int newest = s + kAhead - 1 < kStages ? s + kAhead - 1 : kStages - 1;
            wait_vmcnt<(newest - s - 1) * kCopies>();
            read(std::integral_constant<int, s + 1>{}, nxt);
        }
        if constexpr (s + kAhead < kStages) issue(std::integral_constant<int, s + kAhead>{});
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < 8; ++kk)
#pragma unroll
            for (int j = 0; j < kTiles; ++j)
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(cur.a[kk >> 2][kk & 3], cur.b[j][kk >> 2][kk & 3], acc[j],
                                                              0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        // The folded norm scales the next stage's operands once this stage's MFMAs have issued:
        // its reads have landed by then, and no MFMA in flight reads those registers.
        if constexpr (s + 1 < kStages) fold_norm(nxt);
        cur = nxt;
    });
    wait_vmcnt<0>();  // no copy may still be landing in LDS when the block retires
    if constexpr (kNorm) {
        ss += __shfl_xor(ss, 32, 64);  // the two K halves of the lane's row
        if (lane < 32) norm_ss[wave][lane] = ss;
    }
    // Inverse RMS of output row `row` (0..31) of this wave's row tile, summed over the K parts
    // in order; read after the block barrier below (kParts > 1) or this wave's own writes.
    auto row_scale = [&](int row) {
        float total = norm_ss[kNorm ? row_tile : 0][row];
#pragma unroll
        for (int p = 1; p < kParts; ++p) total += norm_ss[kNorm ? row_tile + RT * p : 0][row];
        return rms_inverse(total, kHidden, args.norm_eps);
    };
    if constexpr (kKB > 1) {
        // Partial plane kb: this block's sums over its K range.
        float* plane = args.split_partials + static_cast<int64_t>(kb) * args.m * args.n;
#pragma unroll
        for (int r = 0; r < 16; ++r) partial[wave][0][r][lane] = acc[0][r];
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 16 / kParts; ++u) {
            const int r = (16 / kParts) * part + u;
            float v = partial[row_tile][0][r][lane];
#pragma unroll
            for (int p = 1; p < kParts; ++p) v += partial[row_tile + RT * p][0][r][lane];
            const int64_t out_row = m0 + mfma32_row(lane, r);
            if (out_row < args.m) plane[out_row * args.n + n0 + (lane & 31)] = v;
        }
    } else if constexpr (kParts == 1 && kCols == 32) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int64_t out_row = m0 + mfma32_row(lane, r);
            if (out_row < args.m) gemm_store_one<E>(args, out_row, n0 + (lane & 31), acc[0][r]);
        }
    } else if constexpr (kParts == 1) {
        if constexpr (kNorm) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float inv = row_scale(mfma32_row(lane, r));
                acc[0][r] *= inv;
                acc[1][r] *= inv;
            }
        }
        const f32x16(&whole)[1][2] = reinterpret_cast<const f32x16(&)[1][kTiles]>(acc);
        gemm_epilogue<E, 1>(args, whole, m0, n0, lane);
    } else {
#pragma unroll
        for (int j = 0; j < kTiles; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) partial[wave][j][r][lane] = acc[j][r];
        __syncthreads();
        const int j = lane & 31;
#pragma unroll
        for (int u = 0; u < 16 / kParts; ++u) {
            const int r = (16 / kParts) * part + u;
            float lo = partial[row_tile][0][r][lane], hi = partial[row_tile][kTiles - 1][r][lane];
#pragma unroll
            for (int p = 1; p < kParts; ++p) {
                lo += partial[row_tile + RT * p][0][r][lane];
                hi += partial[row_tile + RT * p][kTiles - 1][r][lane];
            }
            if constexpr (kNorm) {
                const float inv = row_scale(mfma32_row(lane, r));
                lo *= inv;
                hi *= inv;
            }
            const int64_t out_row = m0 + mfma32_row(lane, r);
            if (out_row >= args.m) continue;
            if constexpr (kCols == 64) gemm_store_pair<E>(args, out_row, n0, j, lo, hi);
            else gemm_store_one<E>(args, out_row, n0 + j, lo);
        }
    }
}

// Small-M GEMM on v_mfma_f32_16x16x4f32 with the operands loaded straight into registers.
// Block = kRegWaves waves (three per SIMD), output tile (16 RT) rows x kCols columns; wave w
// sums the w-th of kRegWaves contiguous K slices (48 values at K = 576).  Lane l loads float4s
// of four consecutive K values from memory (L2): A rows l % 16 (+ 16 rt), B columns l % 16
// (+ 16 jb), K values 4 (l / 16) .. + 3 of each 16-value stage, so k-step s of the stage pairs
// component s of every operand (the MFMA's K index l / 16 stands for K value 4 (l / 16) + s).
// A ring of kDepth stages is in flight; at K = 576 it holds the whole slice, so each wave
// issues all of its loads at once and pays one memory round trip.  The LDS ring of
// gemm_split_kernel is shallower than a round trip at one wave per SIMD, and its K split
// needs a reduce kernel.  The waves' partial tiles are summed in LDS in K order and the block
// shares the epilogue.
constexpr int kRegWaves = 12;

// Scheduling barriers keep every load where it is issued: left free, the compiler sinks the
// loads to their uses (fewer live registers) and the ring is gone.
template <int kStages, int kDepth, typename Issue, typename Compute>
__device__ __forceinline__ void reg_pipeline(Issue&& issue, Compute&& compute) {
    static_for<0, (kStages < kDepth ? kStages : kDepth)>([&](auto st) { issue(st); });
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, kStages>([&](auto st) {
        compute(st);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (decltype(st)::value + kDepth < kStages) {
            issue(std::integral_constant<int, decltype(st)::value + kDepth>{});
            __builtin_amdgcn_sched_barrier(0);
        }
    });
}

template <GemmEpilogue E, int RT, int kCols, bool kNorm, int kK>
__global__ void __launch_bounds__(64 * kRegWaves) gemm_reg_kernel(GemmArgs args) {
    static_assert(kK % (kRegWaves * 16) == 0, "whole 16-value stages per wave");
    constexpr bool kPair = E == GemmEpilogue::kQkvRope || E == GemmEpilogue::kSwiglu;
    static_assert(kCols == 32 || kCols == 64 || (kCols == 16 && !kPair), "16-column blocks, column pairs in two of them");
    static_assert(!kNorm || kK == kHidden, "the folded norm spans the hidden width");
    constexpr int kJB = kCols / 16;
    constexpr int kRows = 16 * RT;
    constexpr int kStages = kK / (kRegWaves * 16);
    constexpr int kPerStage = RT + kJB + (kNorm ? 1 : 0);  // float4 loads per lane per stage
    // Ring stages: as many as 72 registers hold (three waves share a SIMD's 512 per lane).
    constexpr int kRingRegs = 72;
    constexpr int kDepthFit = kRingRegs / (4 * kPerStage) < 2 ? 2 : kRingRegs / (4 * kPerStage);
    constexpr int kDepth = kDepthFit < 9 ? kDepthFit : 9;
    __shared__ float partial[kRegWaves][kRows][kCols + 1];
    __shared__ float norm_ss[kNorm ? kRegWaves : 1][kRows];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int64_t m0 = static_cast<int64_t>(blockIdx.y) * kRows;
    // A 32-column tile of a pair epilogue is half of a 64-column group: 16 columns and the 16 that
    // they pair with, 32 further on.
    constexpr bool kHalfGroup = kPair && kCols == 32;
    const int n0 = static_cast<int>(kHalfGroup ? (blockIdx.x >> 1) * 64 : blockIdx.x * kCols);
    const int sub = kHalfGroup ? 16 * static_cast<int>(blockIdx.x & 1) : 0;
    const int kq = lane >> 4;
    const int r16 = lane & 15;
    const int k_first = wave * (kK / kRegWaves) + 4 * kq;  // this lane's first K value

    const float* a_src[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int64_t row = m0 + 16 * rt + r16;
        a_src[rt] = args.a + (row < args.m ? row : args.m - 1) * kK + k_first;
    }
    const float* b_src[kJB];
#pragma unroll
    for (int jb = 0; jb < kJB; ++jb)
        b_src[jb] = args.b + static_cast<int64_t>(b_row<E>(n0 + sub + (kHalfGroup ? 32 : 16) * jb + r16, args.n)) * kK + k_first;
    const float* g_src = kNorm ? args.norm_weight + k_first : nullptr;

    f32x4 ring_a[kDepth][RT];
    f32x4 ring_b[kDepth][kJB];
    f32x4 ring_g[kNorm ? kDepth : 1];
    auto issue = [&](auto st) {
        constexpr int s = decltype(st)::value;
        constexpr int slot = s % kDepth;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) ring_a[slot][rt] = *reinterpret_cast<const f32x4*>(a_src[rt] + 16 * s);
#pragma unroll
        for (int jb = 0; jb < kJB; ++jb) ring_b[slot][jb] = *reinterpret_cast<const f32x4*>(b_src[jb] + 16 * s);
        if constexpr (kNorm) ring_g[slot] = *reinterpret_cast<const f32x4*>(g_src + 16 * s);
    };
    f32x4 acc[RT][kJB];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int jb = 0; jb < kJB; ++jb) acc[rt][jb] = f32x4{0.f, 0.f, 0.f, 0.f};
    float ss[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) ss[rt] = 0.0f;
    auto compute = [&](auto st) {
        constexpr int slot = decltype(st)::value % kDepth;
        f32x4 a[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            a[rt] = ring_a[slot][rt];
            if constexpr (kNorm) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    ss[rt] = fmaf(a[rt][e], a[rt][e], ss[rt]);
                    a[rt][e] *= ring_g[slot][e];
                }
            }
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int jb = 0; jb < kJB; ++jb)
                    acc[rt][jb] =
                        __builtin_amdgcn_mfma_f32_16x16x4f32(a[rt][s], ring_b[slot][jb][s], acc[rt][jb], 0, 0, 0);
    };
    reg_pipeline<kStages, kDepth>(issue, compute);

    // D[row 4 (l / 16) + r][column l % 16] of each 16 x 16 block.
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int jb = 0; jb < kJB; ++jb)
#pragma unroll
            for (int r = 0; r < 4; ++r) partial[wave][16 * rt + 4 * kq + r][16 * jb + r16] = acc[rt][jb][r];
    if constexpr (kNorm) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            float v = ss[rt];
            v += __shfl_xor(v, 16, kWave);
            v += __shfl_xor(v, 32, kWave);
            if (lane < 16) norm_ss[wave][16 * rt + lane] = v;
        }
    }
    __syncthreads();
    auto total = [&](int row, int col) {
        float t = partial[0][row][col];
#pragma unroll
        for (int w = 1; w < kRegWaves; ++w) t += partial[w][row][col];
        return t;
    };
    auto inv_rms = [&](int row) {
        if constexpr (kNorm) {
            float t = norm_ss[0][row];
#pragma unroll
            for (int w = 1; w < kRegWaves; ++w) t += norm_ss[w][row];
            return rms_inverse(t, kHidden, args.norm_eps);
        } else {
            return 1.0f;
        }
    };
    if constexpr (E == GemmEpilogue::kStore || E == GemmEpilogue::kResidual) {
        for (int i = static_cast<int>(threadIdx.x); i < kRows * kCols; i += 64 * kRegWaves) {
            const int row = i / kCols, col = i % kCols;
            const int64_t out_row = m0 + row;
            if (out_row < args.m) gemm_store_one<E>(args, out_row, n0 + col, total(row, col) * inv_rms(row));
        }
    } else {
        // Column pairs j / j + 32 of the 64-column group (the RoPE pair, or gate and up).
        constexpr int kPairs = kCols / 2;
        for (int i = static_cast<int>(threadIdx.x); i < kRows * kPairs; i += 64 * kRegWaves) {
            const int row = i / kPairs, j = i % kPairs;
            const int64_t out_row = m0 + row;
            if (out_row >= args.m) continue;
            const float inv = inv_rms(row);
            gemm_store_pair<E>(args, out_row, n0, sub + j, total(row, j) * inv, total(row, j + kPairs) * inv);
        }
    }
}

// c = residual + (plane 0 + plane 1 + ...): the partial planes of a K-split GEMM (gemm_split_kernel or
// gemm_limb_kernel) in plane order, thread per output value.
template <int kPlanes>
__global__ void __launch_bounds__(256) split_reduce_residual_kernel(GemmArgs args) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int64_t plane = args.m * args.n;
    if (i >= plane) return;
    float v = args.split_partials[i];
#pragma unroll
    for (int b = 1; b < kPlanes; ++b) v += args.split_partials[b * plane + i];
    args.c[i] = args.residual[i] + v;
}

// The reduce of a K-split 576-column GEMM with the residual epilogue, folded into the RMSNorm
// of its output: c = residual + (plane 0 + plane 1 + ...) and norm_out = w * (c * inv_rms(c)).
// Wave per row, the row in registers as float4 quads; the sums run in the order of
// split_reduce_residual_kernel and the norm in that of rmsnorm_wave4_kernel, so both outputs are
// bitwise those of the reduce kernel followed by launch_rmsnorm_rows.
template <int kPlanes>
__global__ void __launch_bounds__(256) split_reduce_residual_norm_kernel(GemmArgs args, const float* __restrict__ w,
                                                                         float eps, float* __restrict__ norm_out) {
    constexpr int kQuads = 3;  // 144 quads of a 576-wide row over 64 lanes
    const int lane = threadIdx.x & 63;
    const int64_t plane = args.m * kHidden;
    for (int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6); row < args.m;
         row += static_cast<int64_t>(gridDim.x) * 4) {
        float4 v[kQuads];
        float ss = 0.0f;
#pragma unroll
        for (int j = 0; j < kQuads; ++j) {
            const int c = 4 * (lane + 64 * j);
            if (c < kHidden) {
                const float* p = args.split_partials + row * kHidden + c;
                float4 a = *reinterpret_cast<const float4*>(p);
#pragma unroll
                for (int b = 1; b < kPlanes; ++b) {
                    const float4 q = *reinterpret_cast<const float4*>(p + b * plane);
                    a = make_float4(a.x + q.x, a.y + q.y, a.z + q.z, a.w + q.w);
                }
                const float4 r = *reinterpret_cast<const float4*>(args.residual + row * kHidden + c);
                v[j] = make_float4(r.x + a.x, r.y + a.y, r.z + a.z, r.w + a.w);
                *reinterpret_cast<float4*>(args.c + row * kHidden + c) = v[j];
                ss = fmaf(v[j].x, v[j].x, ss);
                ss = fmaf(v[j].y, v[j].y, ss);
                ss = fmaf(v[j].z, v[j].z, ss);
                ss = fmaf(v[j].w, v[j].w, ss);
            }
        }
        const float inv = rms_inverse(wave_sum(ss), kHidden, eps);
#pragma unroll
        for (int j = 0; j < kQuads; ++j) {
            const int c = 4 * (lane + 64 * j);
            if (c < kHidden) {
                const float4 g = *reinterpret_cast<const float4*>(w + c);
                *reinterpret_cast<float4*>(norm_out + row * kHidden + c) =
                    make_float4(g.x * (v[j].x * inv), g.y * (v[j].y * inv), g.z * (v[j].z * inv),
                                g.w * (v[j].w * inv));
            }
        }
    }
}

// Narrow-column GEMM for the residual / plain epilogues of N = 576 outputs (o_proj,
// down): block tile 64 x 64, 4 waves in 2 x 2, wave tile 32 x 32 (one accumulator
// chain).  576 columns are 9 such tiles, so no wave computes a padded column group,
// and the 9 x (M / 64) blocks are small enough to spread evenly over the CUs.  A
// stage is 32 K values, one 128-byte line per row (16-byte pieces XOR-swizzled so a
// 16-lane read pass covers all 64 banks), streamed through a ring of four LDS buffers
// with three copies in flight, counted waits and one barrier per stage (two buffers fit
// more blocks per CU but wait on each stage's copy, and measured slower).
template <GemmEpilogue E>
__global__ void __launch_bounds__(kGemmThreads) gemm_narrow_kernel(GemmArgs args) {
    static_assert(E == GemmEpilogue::kStore || E == GemmEpilogue::kResidual, "plain epilogues only");
    constexpr int kNS = 4;
    constexpr int kRows = 64;
    constexpr int kDepth = 32;
    constexpr int kLoads = 4;  // global_load_lds per wave per stage
    __shared__ __align__(16) float a_s0[kRows * kDepth];
    __shared__ __align__(16) float a_s1[kRows * kDepth];
    __shared__ __align__(16) float a_s2[kRows * kDepth];
    __shared__ __align__(16) float a_s3[kRows * kDepth];
    __shared__ __align__(16) float b_s0[kRows * kDepth];
    __shared__ __align__(16) float b_s1[kRows * kDepth];
    __shared__ __align__(16) float b_s2[kRows * kDepth];
    __shared__ __align__(16) float b_s3[kRows * kDepth];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 1;
    const int wn = wave & 1;
    const int64_t m0 = static_cast<int64_t>(blockIdx.y) * kRows;
    const int n0 = static_cast<int>(blockIdx.x) * kRows;
    const int K = args.k;

    const float* a_src[2];
    const float* b_src[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int row = 8 * (wave + 4 * j) + (lane >> 3);
        const int piece = (lane & 7) ^ ((row >> 1) & 7);
        const int64_t ga = m0 + row < args.m ? m0 + row : args.m - 1;
        a_src[j] = args.a + ga * K + 4 * piece;
        b_src[j] = args.b + static_cast<int64_t>(n0 + row) * K + 4 * piece;
    }
    auto abuf = [&](auto bi) -> float* {
        constexpr int b = decltype(bi)::value;
        if constexpr (b == 0) return a_s0;
        else if constexpr (b == 1) return a_s1;
        else if constexpr (b == 2) return a_s2;
        else return a_s3;
    };
    auto bbuf = [&](auto bi) -> float* {
        constexpr int b = decltype(bi)::value;
        if constexpr (b == 0) return b_s0;
        else if constexpr (b == 1) return b_s1;
        else if constexpr (b == 2) return b_s2;
        else return b_s3;
    };
    const int stages = K / kDepth;
    auto issue = [&](auto bi, int st) {
        const int k0 = (st < stages ? st : stages - 1) * kDepth;
        float* as = abuf(bi);
        float* bs = bbuf(bi);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            lds_copy16(a_src[j] + k0, as + (wave + 4 * j) * 8 * kDepth);
            lds_copy16(b_src[j] + k0, bs + (wave + 4 * j) * 8 * kDepth);
        }
    };

    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    const int h = lane >> 5;
    const int ra = wm * 32 + (lane & 31);
    const int rb = wn * 32 + (lane & 31);
    int a_off[4], b_off[4];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            a_off[2 * u + q] = ra * kDepth + 4 * ((4 * u + 2 * h + q) ^ ((ra >> 1) & 7));
            b_off[2 * u + q] = rb * kDepth + 4 * ((4 * u + 2 * h + q) ^ ((rb >> 1) & 7));
        }
    auto step = [&](auto bi, int s) {
        constexpr int b = decltype(bi)::value;
        const float* as = abuf(bi);
        const float* bs = bbuf(bi);
        f32x4 av[4], bv[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            av[p] = *reinterpret_cast<const f32x4*>(as + a_off[p]);
            bv[p] = *reinterpret_cast<const f32x4*>(bs + b_off[p]);
        }
        issue(std::integral_constant<int, (b + kNS - 1) % kNS>{}, s + kNS - 1);
        if (s < stages) {
#pragma unroll
            for (int p = 0; p < 4; ++p)
#pragma unroll
                for (int kk = 0; kk < 4; ++kk)
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av[p][kk], bv[p][kk], acc, 0, 0, 0);
        }
        wait_vmcnt<(kNS - 2) * kLoads>();
        lds_barrier();
    };
    issue(std::integral_constant<int, 0>{}, 0);
    issue(std::integral_constant<int, 1>{}, 1);
    issue(std::integral_constant<int, 2>{}, 2);
    wait_vmcnt<(kNS - 2) * kLoads>();
    lds_barrier();
    for (int s = 0; s < stages; s += kNS) {
        step(std::integral_constant<int, 0>{}, s);
        step(std::integral_constant<int, 1>{}, s + 1);
        step(std::integral_constant<int, 2>{}, s + 2);
        step(std::integral_constant<int, 3>{}, s + 3);
    }
    wait_vmcnt<0>();  // no copy may still be landing in LDS when the block retires

    const int col = n0 + wn * 32 + (lane & 31);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int64_t row = m0 + wm * 32 + mfma32_row(lane, r);
        if (row >= args.m) continue;
        const int64_t i0 = row * args.n + col;
        if constexpr (E == GemmEpilogue::kResidual) {
            args.c[i0] = args.residual[i0] + acc[r];
        } else {
            args.c[i0] = acc[r];
        }
    }
}

__global__ void embedding_gather_kernel(const int64_t* ids, const float* embedding, int64_t vocab, int64_t seq,
                                        float* hidden) {
    const int64_t total = seq * (kHidden / 4);
    for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < total;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int64_t row = i / (kHidden / 4);
        const int64_t col = (i % (kHidden / 4)) * 4;
        const int64_t token = ids[row];
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (token >= 0 && token < vocab) v = *reinterpret_cast<const float4*>(embedding + token * kHidden + col);
        *reinterpret_cast<float4*>(hidden + row * kHidden + col) = v;
    }
}

}  // namespace

constexpr int64_t kSplitBlocks = 256;  // gemm_split_kernel while its grid fits the device once
constexpr int64_t kSplitKBlocks = 256;  // ... and with K split over blocks while that grid fits it too
// gemm_narrow_kernel (64 x 64 tiles over all of K) while its grid fits the device once.  It takes
// what is left then without partial planes, e.g. one layer's o_proj up to 1792 rows: a limb block
// is longer than one of its blocks there (1000 rows, K = 576: 21 against 13 us; K = 1536, 1536
// rows: 49 against 31; 500 x 1024, K = 64: 6.2 against 4.9, K = 1024: 33 against 20), and shorter
// beyond (2048 rows: 21 against 25; 49 against 57).  On two rounds of blocks it is
// even with limb tiles at K = 64 and 128 at best.
constexpr int64_t kNarrowBlocks = 256;

// Tiling of gemm_split_kernel for this GEMM (rt = 0 when it does not take it), for K = 576
// (hidden) or, plain and residual epilogues, 1536 (intermediate), while the grid fits the device once.  Plain and residual
// epilogues first try 32-column tiles (one row tile per block).  Otherwise 64-column tiles
// with the smallest row tiling that fits; shapes the 64 x 64 tile kernel takes use one row
// tile only: with more, their 9 column tiles leave too many CUs idle (measured slower at
// 1024 to 2048 rows).
struct SplitShape {
    int rt;
    int cols;
};
static SplitShape split_shape(const GemmArgs& args, GemmEpilogue epilogue) {
    const bool plain = epilogue == GemmEpilogue::kStore || epilogue == GemmEpilogue::kResidual;
    if (args.k != kHidden && !(plain && args.k == kInter)) return {0, 0};
    if (plain && (args.n / 32) * ((args.m + 31) / 32) <= kSplitBlocks) return {1, 32};
    const bool narrow_shape = plain && args.n % 128 != 0 && args.k % 32 == 0;
    for (int rt = 1; rt <= (narrow_shape ? 1 : 4); rt *= 2)
        if ((args.n / 64) * ((args.m + 32 * rt - 1) / (32 * rt)) <= kSplitBlocks) return {rt, 64};
    return {0, 0};
}

// Tiling of gemm_reg_kernel (rt = 0 when it does not take the GEMM): 16-row blocks with the
// narrowest column tile whose grid fits the device once (one block per CU).  For the GEMMs over the
// hidden width (QKV, o_proj, gate/up) 32 or 64 columns: QKV at 128 rows takes 6.8 us on 32 (half a
// column group) and 9.1 on 64, gate/up at 20 rows 7.0 and 9.7.  For the down projection
// (K = intermediate) 16 columns only, i.e. up to 112 rows: 7.1 us against gemm_split_kernel's 8.9
// (32 columns, or two rounds of 16: 9.9 and 12.2 us at 128 rows).
struct RegShape {
    int rt;
    int cols;
};
static RegShape reg_shape(const GemmArgs& args, GemmEpilogue epilogue) {
    if (args.n % 64 != 0) return {0, 0};
    const bool pair = epilogue == GemmEpilogue::kQkvRope || epilogue == GemmEpilogue::kSwiglu;
    const int64_t r16 = (args.m + 15) / 16;
    if (args.k == kInter && !pair && (args.n / 16) * r16 <= kSplitBlocks) return {1, 16};
    if (args.k != kHidden) return {0, 0};
    if ((args.n / 32) * r16 <= kSplitBlocks) return {1, 32};
    if ((args.n / 64) * r16 <= kSplitBlocks) return {1, 64};
    return {0, 0};
}

// gemm_reg_kernel and gemm_split_kernel fold an RMSNorm of the A rows into the QKV and gate/up
// GEMMs (K = hidden).
static bool split_folds_norm(const GemmArgs& args, GemmEpilogue epilogue) {
    return args.k == kHidden && (epilogue == GemmEpilogue::kQkvRope || epilogue == GemmEpilogue::kSwiglu) &&
           (reg_shape(args, epilogue).rt != 0 || split_shape(args, epilogue).rt != 0);
}

static hipError_t launch_reg(const GemmArgs& args, GemmEpilogue epilogue, RegShape shape, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>(args.n / shape.cols), static_cast<unsigned>((args.m + 16 * shape.rt - 1) /
                                                                                   (16 * shape.rt)));
    const dim3 block(64 * kRegWaves);
    const bool norm = args.norm_weight != nullptr;
#define FLUX_REG(E, COLS, NORM) \
    hipLaunchKernelGGL(HIP_KERNEL_NAME(gemm_reg_kernel<E, 1, COLS, NORM, kHidden>), grid, block, 0, stream, args)
#define FLUX_REG_PLAIN(E)                                                                                            \
    do {                                                                                                             \
        if (args.k == kInter)                                                                                        \
            hipLaunchKernelGGL(HIP_KERNEL_NAME(gemm_reg_kernel<E, 1, 16, false, kInter>), grid, block, 0, stream, args); \
        else if (shape.cols == 32) FLUX_REG(E, 32, false);                                                           \
        else FLUX_REG(E, 64, false);                                                                                 \
    } while (0)
#define FLUX_REG_PAIR(E)                                   \
    do {                                                   \
        if (shape.cols == 32 && norm) FLUX_REG(E, 32, true); \
        else if (shape.cols == 32) FLUX_REG(E, 32, false); \
        else if (norm) FLUX_REG(E, 64, true);              \
        else FLUX_REG(E, 64, false);                       \
    } while (0)
    switch (epilogue) {
        case GemmEpilogue::kStore:
            FLUX_REG_PLAIN(GemmEpilogue::kStore);
            break;
        case GemmEpilogue::kResidual:
            FLUX_REG_PLAIN(GemmEpilogue::kResidual);
            break;
        case GemmEpilogue::kSwiglu:
            FLUX_REG_PAIR(GemmEpilogue::kSwiglu);
            break;
        case GemmEpilogue::kQkvRope:
            FLUX_REG_PAIR(GemmEpilogue::kQkvRope);
            break;
    }
#undef FLUX_REG_PAIR
#undef FLUX_REG_PLAIN
#undef FLUX_REG
    return hipGetLastError();
}

// True when `parts` partial planes of this GEMM fit the caller's workspace.
static bool planes_fit(const GemmArgs& args, int parts) {
    return args.split_partials != nullptr && parts * args.m * static_cast<int64_t>(args.n) <= args.split_floats;
}

// Most K parts of a limb GEMM (its partial planes are summed by split_reduce_residual_kernel or
// split_reduce_residual_norm_kernel): residual epilogue, as many planes as fit.
static int limb_max_parts(const GemmArgs& args, GemmEpilogue epilogue) {
    if (epilogue != GemmEpilogue::kResidual) return 1;
    return planes_fit(args, kSplitBlocksK) ? kSplitBlocksK : (planes_fit(args, 2) ? 2 : 1);
}

static bool narrow_taken(const GemmArgs& args, GemmEpilogue epilogue) {
    return (epilogue == GemmEpilogue::kStore || epilogue == GemmEpilogue::kResidual) && args.k % 32 == 0 &&
           static_cast<int64_t>(args.n / 64) * ((args.m + 63) / 64) <= kNarrowBlocks;
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Whether gemm_split_kernel takes these args with K split over kSplitBlocksK blocks: 32-column tiles
// over the intermediate width whose grid fits the device once even when tripled, and the
// caller's planes hold the split.
static bool split_k_taken(const GemmArgs& args, GemmEpilogue epilogue) {
    const SplitShape shape = split_shape(args, epilogue);
    if (epilogue != GemmEpilogue::kResidual || shape.cols != 32 || args.k != kInter) return false;
    const int64_t blocks = (args.n / 32) * ((args.m + 31) / 32);
    return planes_fit(args, kSplitBlocksK) && blocks * kSplitBlocksK <= kSplitKBlocks;
}

// c = residual + the sum of `parts` partial planes.
static hipError_t launch_split_reduce(const GemmArgs& args, int parts, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>((args.m * args.n + 255) / 256));
    if (parts == 2)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(split_reduce_residual_kernel<2>), grid, dim3(256), 0, stream, args);
    else
        hipLaunchKernelGGL(HIP_KERNEL_NAME(split_reduce_residual_kernel<kSplitBlocksK>), grid, dim3(256), 0, stream,
                           args);
    return hipGetLastError();
}

static hipError_t gemm_args_valid(const GemmArgs& args, GemmEpilogue epilogue) {
    if (args.k % kBK != 0 || args.n % 64 != 0 || args.m <= 0) return hipErrorInvalidValue;
    if (epilogue == GemmEpilogue::kSwiglu && args.n % 128 != 0) return hipErrorInvalidValue;
    if (epilogue == GemmEpilogue::kQkvRope && args.n != kQKV) return hipErrorInvalidValue;
    const bool norm = args.norm_weight != nullptr;
    if (norm && !split_folds_norm(args, epilogue)) return hipErrorInvalidValue;
    return hipSuccess;
}

static hipError_t launch_gemm_split(const GemmArgs& args, GemmEpilogue epilogue, hipStream_t stream);

hipError_t launch_gemm(const GemmArgs& args, GemmEpilogue epilogue, hipStream_t stream) {
    const hipError_t valid = gemm_args_valid(args, epilogue);
    if (valid != hipSuccess) return valid;
    const RegShape reg = reg_shape(args, epilogue);
    if (reg.rt != 0) return launch_reg(args, epilogue, reg, stream);
    return launch_gemm_split(args, epilogue, stream);
}

// gemm_split_kernel and the remaining kernels of launch_gemm.
static hipError_t launch_gemm_split(const GemmArgs& args, GemmEpilogue epilogue, hipStream_t stream) {
    const bool norm = args.norm_weight != nullptr;
    const SplitShape shape = split_shape(args, epilogue);
    const int rt = shape.rt;
    if (rt != 0) {
        const bool hidden = args.k == kHidden;
        dim3 grid(static_cast<unsigned>(args.n / shape.cols), static_cast<unsigned>((args.m + 32 * rt - 1) / (32 * rt)));
        const dim3 split_block(64 * kSplitWaves);
        if (split_k_taken(args, epilogue)) {
            grid.x *= kSplitBlocksK;
            hipLaunchKernelGGL(HIP_KERNEL_NAME(gemm_split_kernel<GemmEpilogue::kResidual, 24 / kSplitBlocksK, 1, false,
                                                                 32, kSplitBlocksK>),
                               grid, split_block, 0, stream, args);
            const hipError_t st = hipGetLastError();
            return st != hipSuccess ? st : launch_split_reduce(args, kSplitBlocksK, stream);
        }
#define FLUX_SPLIT_RT(E, ST, RT, NORM, COLS)                                                                          \
    hipLaunchKernelGGL(HIP_KERNEL_NAME(gemm_split_kernel<E, ST * RT, RT, NORM, COLS, 1>), grid, split_block, 0, stream, \
                       args)
#define FLUX_SPLIT_ROWS(E, ST, NORM)                     \
    do {                                                 \
        if (rt == 1) FLUX_SPLIT_RT(E, ST, 1, NORM, 64);      \
        else if (rt == 2) FLUX_SPLIT_RT(E, ST, 2, NORM, 64); \
        else FLUX_SPLIT_RT(E, ST, 4, NORM, 64);              \
    } while (0)
#define FLUX_SPLIT_PLAIN(E)                                             \
    do {                                                                \
        if (shape.cols == 32 && hidden) FLUX_SPLIT_RT(E, 9, 1, false, 32); \
        else if (shape.cols == 32) FLUX_SPLIT_RT(E, 24, 1, false, 32);     \
        else if (hidden) FLUX_SPLIT_ROWS(E, 9, false);                     \
        else FLUX_SPLIT_ROWS(E, 24, false);                                \
    } while (0)
#define FLUX_SPLIT_PAIR(E)                  \
    do {                                    \
        if (norm) FLUX_SPLIT_ROWS(E, 9, true); \
        else FLUX_SPLIT_ROWS(E, 9, false);     \
    } while (0)
        switch (epilogue) {
            case GemmEpilogue::kStore:
                FLUX_SPLIT_PLAIN(GemmEpilogue::kStore);
                break;
            case GemmEpilogue::kResidual:
                FLUX_SPLIT_PLAIN(GemmEpilogue::kResidual);
                break;
            case GemmEpilogue::kSwiglu:
                FLUX_SPLIT_PAIR(GemmEpilogue::kSwiglu);
                break;
            case GemmEpilogue::kQkvRope:
                FLUX_SPLIT_PAIR(GemmEpilogue::kQkvRope);
                break;
        }
#undef FLUX_SPLIT_PAIR
#undef FLUX_SPLIT_PLAIN
#undef FLUX_SPLIT_ROWS
#undef FLUX_SPLIT_RT
        return hipGetLastError();
    }
    const int max_parts = limb_max_parts(args, epilogue);
    if (max_parts == 1 && narrow_taken(args, epilogue)) {
        const dim3 grid(static_cast<unsigned>(args.n / 64), static_cast<unsigned>((args.m + 63) / 64));
        if (epilogue == GemmEpilogue::kResidual)
            hipLaunchKernelGGL(HIP_KERNEL_NAME(gemm_narrow_kernel<GemmEpilogue::kResidual>), grid, dim3(kGemmThreads),
                               0, stream, args);
        else
            hipLaunchKernelGGL(HIP_KERNEL_NAME(gemm_narrow_kernel<GemmEpilogue::kStore>), grid, dim3(kGemmThreads), 0,
                               stream, args);
        return hipGetLastError();
    }
    const LimbPlan plan = limb_plan(args, max_parts, false);
    const hipError_t st = launch_limb_gemm(args, epilogue, plan, stream);
    if (st != hipSuccess || plan.parts == 1) return st;
    return launch_split_reduce(args, plan.parts, stream);
}

hipError_t launch_norm_gemm(const GemmArgs& args, const float* norm_weight, float eps, float* scratch,
                            GemmEpilogue epilogue, hipStream_t stream) {
    if (split_folds_norm(args, epilogue)) {
        GemmArgs folded = args;
        folded.norm_weight = norm_weight;
        folded.norm_eps = eps;
        return launch_gemm(folded, epilogue, stream);
    }
    const hipError_t e = launch_rmsnorm_rows(args.a, norm_weight, scratch, args.m, args.k, eps, stream);
    if (e != hipSuccess) return e;
    GemmArgs plain = args;
    plain.a = scratch;
    plain.norm_weight = nullptr;
    return launch_gemm(plain, epilogue, stream);
}

bool gemm_folds_norm(const GemmArgs& args, GemmEpilogue epilogue) { return split_folds_norm(args, epilogue); }

hipError_t launch_gemm_residual_norm(const GemmArgs& args, const float* norm_weight, float eps, float* norm_out,
                                     hipStream_t stream) {
    // The fused kernel reads and writes rows as float4: every buffer must be 16-byte aligned
    // (a norm weight that is a view into a larger tensor may not be), else the plain path runs.
    const bool fusable = args.n == kHidden && reg_shape(args, GemmEpilogue::kResidual).rt == 0 &&
                         split_shape(args, GemmEpilogue::kResidual).rt == 0 && aligned16(args.c) &&
                         aligned16(args.residual) && aligned16(args.split_partials) && aligned16(norm_weight) &&
                         aligned16(norm_out);
    const int max_parts = fusable && planes_fit(args, 1) ? limb_max_parts(args, GemmEpilogue::kResidual) : 0;
    if (max_parts == 0) {
        const hipError_t e = launch_gemm(args, GemmEpilogue::kResidual, stream);
        if (e != hipSuccess) return e;
        return launch_rmsnorm_rows(args.c, norm_weight, norm_out, args.m, static_cast<int>(args.n), eps, stream);
    }
    // One plane too: the norm reads the residual as fast as the GEMM's output, which the GEMM's
    // epilogue does not (8192 rows, o_proj: 62 + 8 us against 51 + 12).
    const LimbPlan plan = limb_plan(args, max_parts, true);
    GemmArgs planes = args;
    if (plan.parts == 1) planes.c = args.split_partials;
    const hipError_t e = launch_limb_gemm(planes, GemmEpilogue::kStore, plan, stream);
    if (e != hipSuccess) return e;
    const int64_t grid = (args.m + 3) / 4 < 65535 ? (args.m + 3) / 4 : 65535;
    if (plan.parts == 1)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(split_reduce_residual_norm_kernel<1>), dim3(static_cast<unsigned>(grid)),
                           dim3(256), 0, stream, args, norm_weight, eps, norm_out);
    else if (plan.parts == 2)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(split_reduce_residual_norm_kernel<2>), dim3(static_cast<unsigned>(grid)),
                           dim3(256), 0, stream, args, norm_weight, eps, norm_out);
    else
        hipLaunchKernelGGL(HIP_KERNEL_NAME(split_reduce_residual_norm_kernel<kSplitBlocksK>),
                           dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, args, norm_weight, eps, norm_out);
    return hipGetLastError();
}

hipError_t launch_embedding_gather(const int64_t* ids, const float* embedding, int64_t vocab, int64_t seq,
                                   float* hidden, hipStream_t stream) {
    const int64_t total = seq * (kHidden / 4);
    const int grid = static_cast<int>((total + 255) / 256 < 16384 ? (total + 255) / 256 : 16384);
    hipLaunchKernelGGL(embedding_gather_kernel, dim3(grid), dim3(256), 0, stream, ids, embedding, vocab, seq, hidden);
    return hipGetLastError();
}

}  // namespace flux
