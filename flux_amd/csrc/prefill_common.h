// Device helpers shared by the prefill kernel files: MFMA accumulator layout, the GEMM
// epilogues (RoPE + cache rows, SwiGLU, residual), LDS barriers and lane-half reductions.
#pragma once

#include "flux_common.h"
#include "flux_kernels.h"

namespace flux {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// MFMA 32x32x2 accumulator element r of lane l -> (row, col) inside the 32x32 tile.
__device__ __forceinline__ int mfma32_row(int lane, int r) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

#pragma clang fp contract(off)
__device__ __forceinline__ float rope_lo(float x, float paired, float c, float s) {
    const float a = x * c;
    const float b = (-paired) * s;
    return a + b;
}
__device__ __forceinline__ float rope_hi(float x, float paired, float c, float s) {
    const float a = x * c;
    const float b = paired * s;
    return a + b;
}
#pragma clang fp contract(fast)

// Weight row used for virtual column `col` of the B operand.
template <GemmEpilogue E>
__device__ __forceinline__ int b_row(int col, int n) {
    if constexpr (E == GemmEpilogue::kSwiglu) {
        // Column group t (64 columns) = gate rows [32t, 32t+32) then up rows [half + 32t, ...).
        const int half = n / 2;
        const int t = col >> 6;
        const int v = col & 63;
        return v < 32 ? 32 * t + v : half + 32 * t + (v - 32);
    } else {
        return col;
    }
}

// Epilogue of one wave's (32*MI) x 64 tile whose first row is row0 and whose column
// group (one head for RoPE, one gate/up pair for SwiGLU) starts at column g0.
// One output row of a wave's 64-column group: lo is column g0 + j, hi is column g0 + 32 + j.
template <GemmEpilogue E>
__device__ __forceinline__ void gemm_store_pair(const GemmArgs& args, int64_t row, int g0, int j, float lo, float hi) {
    if constexpr (E == GemmEpilogue::kStore) {
        args.c[row * args.n + g0 + j] = lo;
        args.c[row * args.n + g0 + 32 + j] = hi;
    } else if constexpr (E == GemmEpilogue::kResidual) {
        const int64_t i0 = row * args.n + g0 + j;
        args.c[i0] = args.residual[i0] + lo;
        args.c[i0 + 32] = args.residual[i0 + 32] + hi;
    } else if constexpr (E == GemmEpilogue::kSwiglu) {
        const int half = args.n / 2;
        args.c[row * half + (g0 >> 1) + j] = silu(lo) * hi;
    } else {  // kQkvRope: the column group is one head; columns j / j+32 are the RoPE pair.
        const int head = g0 / kHeadDim;
        if (head < kQHeads + kKVHeads) {
            const float* cr = args.rope_cos + row * kHeadDim;
            const float* sr = args.rope_sin + row * kHeadDim;
            const float qlo = rope_lo(lo, hi, cr[j], sr[j]);
            const float qhi = rope_hi(hi, lo, cr[j + 32], sr[j + 32]);
            float* dst = head < kQHeads
                             ? args.q_out + (static_cast<int64_t>(head) * args.m + row) * kHeadDim
                             : args.key_cache + (static_cast<int64_t>(head - kQHeads) * args.capacity + row) * kHeadDim;
            dst[j] = qlo;
            dst[j + 32] = qhi;
        } else {
            float* dst = args.value_cache +
                         (static_cast<int64_t>(head - kQHeads - kKVHeads) * args.capacity + row) * kHeadDim;
            dst[j] = lo;
            dst[j + 32] = hi;
        }
    }
}

// One output value of the plain or residual epilogue.
template <GemmEpilogue E>
__device__ __forceinline__ void gemm_store_one(const GemmArgs& args, int64_t row, int col, float v) {
    static_assert(E == GemmEpilogue::kStore || E == GemmEpilogue::kResidual, "plain epilogues only");
    const int64_t i0 = row * args.n + col;
    if constexpr (E == GemmEpilogue::kResidual) {
        args.c[i0] = args.residual[i0] + v;
    } else {
        args.c[i0] = v;
    }
}

// For 32-row subtile i, a lane holds columns j (acc[i][0]) and j + 32 (acc[i][1]) of the wave's
// 64-column group for 16 rows.  What the stores combine with (residual, RoPE rows) is loaded for
// eight rows at a time before any of them is stored: the compiler cannot move those loads over
// the stores by itself (they may alias), and row by row every pair of stores waited for a memory
// round trip (8192 x 576 x 576 with a residual: 64 us against 51 without).
template <GemmEpilogue E, int MI>
__device__ __forceinline__ void gemm_epilogue(const GemmArgs& args, const f32x16 (&acc)[MI][2], int64_t row0, int g0,
                                              int lane) {
    const int j = lane & 31;
    const int head = g0 / kHeadDim;
    const bool rotates = E == GemmEpilogue::kQkvRope && head < kQHeads + kKVHeads;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
        for (int r0 = 0; r0 < 16; r0 += 8) {
            float with[8][4];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int64_t row = row0 + 32 * i + mfma32_row(lane, r0 + u);
                const int64_t at = row < args.m ? row : args.m - 1;
                if constexpr (E == GemmEpilogue::kResidual) {
                    with[u][0] = args.residual[at * args.n + g0 + j];
                    with[u][1] = args.residual[at * args.n + g0 + j + 32];
                } else if constexpr (E == GemmEpilogue::kQkvRope) {
                    if (rotates) {
                        with[u][0] = args.rope_cos[at * kHeadDim + j];
                        with[u][1] = args.rope_cos[at * kHeadDim + j + 32];
                        with[u][2] = args.rope_sin[at * kHeadDim + j];
                        with[u][3] = args.rope_sin[at * kHeadDim + j + 32];
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int64_t row = row0 + 32 * i + mfma32_row(lane, r0 + u);
                if (row >= args.m) continue;
                const float lo = acc[i][0][r0 + u], hi = acc[i][1][r0 + u];
                if constexpr (E == GemmEpilogue::kResidual) {
                    args.c[row * args.n + g0 + j] = with[u][0] + lo;
                    args.c[row * args.n + g0 + j + 32] = with[u][1] + hi;
                } else if constexpr (E == GemmEpilogue::kQkvRope) {
                    if (rotates) {
                        float* dst = head < kQHeads
                                         ? args.q_out + (static_cast<int64_t>(head) * args.m + row) * kHeadDim
                                         : args.key_cache +
                                               (static_cast<int64_t>(head - kQHeads) * args.capacity + row) * kHeadDim;
                        dst[j] = rope_lo(lo, hi, with[u][0], with[u][2]);
                        dst[j + 32] = rope_hi(hi, lo, with[u][1], with[u][3]);
                    } else {
                        gemm_store_pair<E>(args, row, g0, j, lo, hi);
                    }
                } else {
                    gemm_store_pair<E>(args, row, g0, j, lo, hi);
                }
            }
        }
    }
}

// Waits until at most N vector-memory operations of this wave are outstanding
// (vmcnt only; the LDS and export counters are left alone).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit field");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Barrier for LDS hand-offs: this wave's LDS reads are complete and no memory access
// moves across it; global-memory copies still in flight are not waited for (each
// wave waits for its own with vmcnt where needed).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// max / sum of the values of lanes l and l ^ 32 (v_permlane32_swap: r[0] holds the
// low half's values in both halves, r[1] the high half's).
__device__ __forceinline__ float halves_max(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float halves_sum(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

}  // namespace
}  // namespace flux
