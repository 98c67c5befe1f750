// gfx950 causal GQA prefill attention (csrc/streaming_prefill_gqa/streaming_prefill_gqa_cuda.cu:
// online softmax over K/V tiles in shared memory, no score materialisation).
#include "flux_common.h"
#include "flux_kernels.h"
#include "prefill_limb.h"

#include <cmath>
#include <type_traits>

namespace flux {
namespace {

// ---------------------------------------------------------------------------
// Causal GQA prefill attention on three-limb bf16 products (prefill_limb.h).
//
// Block = (128-query tile, query head, chunk of at most attn_chunk_tiles(seq) 64-key tiles);
// 4 waves x 32 queries.  attention_limbs_kernel first splits the layer's K and V into limb
// planes in MFMA operand order.  Per 64-key tile a wave computes S^T = K Q^T as two 32 x 32 tiles
// (24 MFMAs each), then O^T += V^T P^T (12 MFMAs per 16 keys): a lane's S^T values are, in order,
// the values of its B operand of the PV product, so P is split in registers and never leaves them.
// Q is pre-scaled by scale * log2(e), so scores are already in exp2 units.
//
// K/V planes stream HBM -> LDS with global_load_lds: one K buffer, refilled with the
// next tile as soon as every wave has finished its S^T, and two V buffers, the
// next tile's copied while this tile's is read.  Each buffer is its own LDS
// variable, so reads of one never wait on copies into another.  Two blocks fit a
// CU (74 KB of LDS, 198 VGPRs), i.e. two waves per SIMD, one in its softmax while the other
// multiplies.
//
// A query tile's keys are split into chunks of attn_chunk_tiles(seq) tiles: about one
// block slot's even share of the causal work, so short prompts still spread over the device,
// and at most kMaxChunkTiles (2048 keys) for long ones.  A tile with one
// chunk writes its rows directly, longer ones write (o, m, l) partials that
// prefill_attention_merge_kernel combines
// (csrc/streaming_prefill_gqa/streaming_prefill_gqa_cuda.cu:43-460 splits the keys into
// partitions and merges them the same way).  Items (query tile, chunk) are
// launched longest first so the tail of the grid is short chunks.
//
// A wave raises its issue priority (s_setprio 1) for its MFMA blocks and drops it for the
// softmax: the SIMD's other wave then runs its softmax and LDS work in the gaps of its MFMA
// stream rather than delaying it.  Priority orders issue only; every wave still reaches every
// barrier.
//
// Bound by power, as the limb GEMMs: 8192 tokens 632 -> 405 us with the planes and the merge
// (191 TFLOP/s of float32 products, 1.15 PFLOP/s of bf16; 401 to 429 from card to card), 4096:
// 185 -> 118, 2048: 64 -> 48.7, 1024: 30.6 -> 29.1; the error against 64 bits at 8000 tokens
// 4.3e-7 -> 1.7e-7.  Blocks whose values or sums limbs cannot hold (kLimbMaxScore and what follows
// it), and prompts below kLimbAttnMinSeq, take the float32 instruction (attention_item_f32).
constexpr int kQTile = 128;
constexpr int kKTile = 64;
constexpr int kAttnThreads = 256;
// Shorter prompts pay more for splitting K and V than they gain (832 tokens: 23.3 against 20.8 us).
constexpr int64_t kLimbAttnMinSeq = 897;
constexpr int kMaxChunkTiles = 32;  // 2048 keys: 16 measured 411 us at 8192 tokens and 128 at 4096, 24 411 and 117, 32 405 and 117
constexpr int kPartialRow = kHeadDim + 4;  // o[64], m, l, 2 words of padding (16-byte rows)
constexpr int kMergeMaxChunks = 8;         // >= the chunks of any query tile up to kMaxCapacity
constexpr int kKVTileFloats = kKTile * kHeadDim;

__host__ __device__ __forceinline__ int64_t attn_q_tiles(int64_t seq) { return (seq + kQTile - 1) / kQTile; }
__host__ __device__ __forceinline__ int64_t attn_key_tiles(int64_t seq, int64_t qt) {
    const int64_t last = (qt + 1) * kQTile - 1 < seq - 1 ? (qt + 1) * kQTile - 1 : seq - 1;
    return last / kKTile + 1;
}
// Even number of key tiles that is one of `slots` even shares of the 9 heads' causal tile steps
// (query tile qt walks 2 (qt + 1) key tiles), in [2, most].  Even, because each query tile adds
// two key tiles.
__host__ __device__ __forceinline__ int64_t attn_share_tiles(int64_t seq, int64_t slots, int64_t most) {
    const int64_t q = attn_q_tiles(seq);
    const int64_t share = (kQHeads * q * (q + 1) + slots - 1) / slots;
    const int64_t even = (share + 1) / 2 * 2;
    return even < 2 ? 2 : (even > most ? most : even);
}
// Key tiles per chunk: an even share of the device's 512 block slots (256 CUs x 2 resident blocks;
// dividing over 768 instead: 52.6 against 46.9 us at 2048 tokens).  Up to 14 query tiles the chunks
// are longer than that, so that partials and limb planes together fit the workspace of
// prefill_attention_workspace_floats.
__host__ __device__ __forceinline__ int64_t attn_chunk_tiles(int64_t seq) {
    if (seq < kLimbAttnMinSeq) return 2;  // the share of any such prompt, known to the compiler
    const int64_t share = attn_share_tiles(seq, 512, kMaxChunkTiles);
    const int64_t q = attn_q_tiles(seq);
    const int64_t least = q <= 12 ? 4 : (q <= 14 ? 6 : 2);
    return share < least ? least : share;
}

// Quotients of tile counts (below 2^31) in 32 bits: every block divides before its first load, and
// 64 bits by a variable are a chain of some hundred instructions.  With this and the constant chunk
// below 897 tokens: 19.5 -> 18.4 us at 543 tokens, 22.2 -> 21.3 at 896.
__host__ __device__ __forceinline__ int64_t tile_quotient(int64_t n, int64_t d) {
    return static_cast<uint32_t>(n) / static_cast<uint32_t>(d);
}
__host__ __device__ __forceinline__ int64_t attn_chunks(int64_t seq, int64_t qt) {
    const int64_t ct = attn_chunk_tiles(seq);
    return tile_quotient(attn_key_tiles(seq, qt) + ct - 1, ct);
}
// Query tiles below attn_long_tile(seq) have a single chunk.
__host__ __device__ __forceinline__ int64_t attn_long_tile(int64_t seq) { return attn_chunk_tiles(seq) * kKTile / kQTile; }
__host__ __device__ __forceinline__ int64_t attn_max_chunks(int64_t seq) { return attn_chunks(seq, attn_q_tiles(seq) - 1); }
__host__ __device__ __forceinline__ int64_t attn_partial_slot(int64_t seq, int64_t qt, int h, int64_t c) {
    return ((qt - attn_long_tile(seq)) * kQHeads + h) * attn_max_chunks(seq) + c;
}
// Items of one head, longest first: every chunk of the last query tile, then the
// full chunks of the others (chunk-major), then their partial last chunks by
// decreasing length.  Inner query tiles have 2 (qt + 1) key tiles.
__host__ __device__ __forceinline__ int64_t attn_items(int64_t seq) {
    const int64_t q_tiles = attn_q_tiles(seq);
    int64_t n = attn_chunks(seq, q_tiles - 1);
    for (int64_t qt = 0; qt + 1 < q_tiles; ++qt) n += attn_chunks(seq, qt);
    return n;
}
__device__ __forceinline__ void attn_item(int64_t seq, int64_t i, int64_t& qt, int64_t& chunk) {
    const int64_t q_tiles = attn_q_tiles(seq);
    const int64_t ct = attn_chunk_tiles(seq);
    const int64_t last_chunks = attn_chunks(seq, q_tiles - 1);
    if (i < last_chunks) {
        qt = q_tiles - 1;
        chunk = i;
        return;
    }
    i -= last_chunks;
    // Full chunk c of inner tile qt needs 2 (qt + 1) >= ct (c + 1).
    for (int64_t c = 0;; ++c) {
        const int64_t first = ct / 2 * (c + 1) - 1;
        const int64_t count = q_tiles - 1 - first > 0 ? q_tiles - 1 - first : 0;
        if (count == 0) break;
        if (i < count) {
            qt = first + i;
            chunk = c;
            return;
        }
        i -= count;
    }
    // Partial chunks: length 2 (qt + 1) mod ct = len, longest first.
    for (int64_t len = ct - 2; len >= 2; len -= 2) {
        const int64_t r0 = len / 2 - 1;
        const int64_t count = q_tiles - 2 - r0 >= 0 ? tile_quotient(q_tiles - 2 - r0, ct / 2) + 1 : 0;
        if (i < count) {
            qt = r0 + (ct / 2) * i;
            chunk = tile_quotient(2 * (qt + 1), ct);
            return;
        }
        i -= count;
    }
    qt = 0;  // not reached for i < attn_items(seq)
    chunk = 0;
}

// LDS tiles: K rows are padded to 17 16-byte pieces (68 words), so the 32 lanes that
// read one piece of 32 consecutive rows hit distinct banks; V rows are plain (the 32
// lanes of a V read cover one whole row).  Every read is a per-lane base plus an
// immediate offset.
constexpr int kKRow = kHeadDim + 4;                    // words per padded K row
constexpr int kKTileWords = kKTile * kKRow;           // 4352
constexpr int kKCopies = kKTileWords / 256;           // 17 global_load_lds of 1 KB
constexpr int kVCopies = kKVTileFloats / 256;         // 16

// One block's item on the float32 instruction: every block of a prompt below kLimbAttnMinSeq, and
// blocks of longer ones whose values limbs cannot hold.
__device__ __forceinline__ void attention_item_f32(const float* __restrict__ q, const float* __restrict__ key_cache,
                                                const float* __restrict__ value_cache, int64_t seq, int64_t capacity,
                                                float scale, float* __restrict__ workspace,
                                                float* __restrict__ out_rows, int h, int64_t qt, int64_t chunk,
                                                float* ks, float* v0s, float* v1s) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = h / kGroup;
    const int64_t qw0 = qt * kQTile + 32 * wave;  // first query of this wave
    const int col = lane & 31;
    const int half = lane >> 5;
    const int64_t my_q = qw0 + col;

    // B operand of S^T = K Q^T: qreg[s] = Q[my_q][s + 32 half] * scale * log2(e).
    float qreg[32];
    {
        const int64_t r = my_q < seq ? my_q : seq - 1;
        const float* qp = q + (static_cast<int64_t>(h) * seq + r) * kHeadDim + 32 * half;
        const float s2 = scale * kLog2e;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const float4 v = *reinterpret_cast<const float4*>(qp + 4 * t);
            qreg[4 * t] = v.x * s2;
            qreg[4 * t + 1] = v.y * s2;
            qreg[4 * t + 2] = v.z * s2;
            qreg[4 * t + 3] = v.w * s2;
        }
    }

    const float* kg = key_cache + static_cast<int64_t>(g) * capacity * kHeadDim;
    const float* vg = value_cache + static_cast<int64_t>(g) * capacity * kHeadDim;
    const int64_t k_tiles = attn_key_tiles(seq, qt);
    const int64_t chunk_tiles = attn_chunk_tiles(seq);
    const int64_t kt_begin = chunk * chunk_tiles;
    const int64_t kt_end = kt_begin + chunk_tiles < k_tiles ? kt_begin + chunk_tiles : k_tiles;

    // Copies of key tile kt: K slot s (16 bytes) of the padded tile holds piece s % 17
    // of row s / 17 (piece 16 is padding and repeats piece 0); V slot s holds piece
    // s % 16 of row s / 16.  Copy i covers slots 64 i .. 64 i + 63; wave w issues
    // copies w, w + 4, ...  Rows past the prompt repeat its last row (they are masked).
    auto issue_k = [&](int64_t kt) {
        const int k0 = static_cast<int>(kt) * kKTile;
        const int last = static_cast<int>(seq) - 1 - k0;  // last valid row of the tile
#pragma unroll
        for (int j = 0; j < (kKCopies + 3) / 4; ++j) {
            const int i = wave + 4 * j;
            if (i < kKCopies) {
                const int slot = 64 * i + lane;
                int row = slot / 17;
                int piece = slot - 17 * row;
                piece = piece == 16 ? 0 : piece;
                row = row < last ? row : last;
                __builtin_amdgcn_global_load_lds(kg + static_cast<int64_t>(k0 + row) * kHeadDim + 4 * piece,
                                                 ks + 256 * i, 16, 0, 0);
            }
        }
    };
    auto issue_v = [&](float* vbuf, int64_t kt) {
        const int k0 = static_cast<int>(kt) * kKTile;
        const int last = static_cast<int>(seq) - 1 - k0;
#pragma unroll
        for (int j = 0; j < kVCopies / 4; ++j) {
            const int i = wave + 4 * j;
            int row = 4 * i + (lane >> 4);
            row = row < last ? row : last;
            __builtin_amdgcn_global_load_lds(vg + static_cast<int64_t>(k0 + row) * kHeadDim + 4 * (lane & 15),
                                             vbuf + 256 * i, 16, 0, 0);
        }
    };

    f32x16 o_acc[2];
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[db][r] = 0.0f;
    float m_run = -INFINITY;
    float l_run = 0.0f;

    const int seq32 = static_cast<int>(seq);
    const int qw = static_cast<int>(qw0);
    const int q_me = static_cast<int>(my_q);
    // QK of one tile: both 32-key halves when the second is visible to the wave (the
    // two accumulator chains alternate), the K operands of step t + 1 read from LDS
    // before the MFMAs of step t.
    auto qk = [&](const float* ks, f32x16* s_acc, auto both_c) {
        constexpr bool both = decltype(both_c)::value;
        const float* k0p = ks + col * kKRow + 32 * half;  // row col, dims 32 half ..
        const float* k1p = k0p + 32 * kKRow;                // row 32 + col
        f32x4 ka = *reinterpret_cast<const f32x4*>(k0p);
        f32x4 kb;
        if constexpr (both) kb = *reinterpret_cast<const f32x4*>(k1p);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            f32x4 na, nb;
            if (t < 7) {
                na = *reinterpret_cast<const f32x4*>(k0p + 4 * (t + 1));
                if constexpr (both) nb = *reinterpret_cast<const f32x4*>(k1p + 4 * (t + 1));
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s_acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(ka[e], qreg[4 * t + e], s_acc[0], 0, 0, 0);
                if constexpr (both)
                    s_acc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(kb[e], qreg[4 * t + e], s_acc[1], 0, 0, 0);
            }
            if (t < 7) {
                ka = na;
                if constexpr (both) kb = nb;
            }
        }
    };
    // One key tile: S^T from the K tile, an LDS barrier after which the K buffer is
    // refilled with the next tile, then softmax and O^T += V^T P^T from this tile's
    // V buffer.  Waves whose queries all precede the tile skip the math but not the
    // barriers.
    auto tile = [&](const float* vs, int64_t kt, int64_t kt_next) {
        const int k0 = static_cast<int>(kt) * kKTile;
        const bool active = k0 <= qw + 31;
        const bool need_mask = k0 + kKTile - 1 > qw || k0 + kKTile > seq32;
        const bool live1 = k0 + 32 <= qw + 31;  // second 32-key half visible to some query
        f32x16 s_acc[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) s_acc[kb][r] = 0.0f;
        __builtin_amdgcn_s_setprio(1);  // the MFMA block (see above the kernel)
        if (live1)
            qk(ks, s_acc, std::true_type{});
        else if (active)
            qk(ks, s_acc, std::false_type{});
        __builtin_amdgcn_s_setprio(0);
        lds_barrier();  // every wave is done with the K tile
        issue_k(kt_next);
        if (!active) return;
        // Lane holds keys k0 + 32 kb + 8 (r / 4) + 4 half + r % 4 of query my_q.
        if (!live1) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s_acc[1][r] = -INFINITY;
        }
        if (need_mask) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key = k0 + 32 * kb + 8 * (r >> 2) + 4 * half + (r & 3);
                    s_acc[kb][r] = (key <= q_me && key < seq32) ? s_acc[kb][r] : -INFINITY;
                }
            }
        }
        float tile_max = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) tile_max = fmaxf(tile_max, s_acc[kb][r]);
        tile_max = halves_max(tile_max);
        const float m_new = fmaxf(m_run, tile_max);  // finite: the first key of a chunk precedes every query
        const float alpha = fast_exp2(m_run - m_new);
        float psum = 0.0f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float p = fast_exp2(s_acc[kb][r] - m_new);
                s_acc[kb][r] = p;
                psum += p;
            }
        }
        psum = halves_sum(psum);
        l_run = l_run * alpha + psum;
        m_run = m_new;
        // alpha is exactly 1 where the running max did not move: skip the rescale
        // when that holds for every lane (multiplying by 1 would not change a bit).
        if (__any(alpha != 1.0f)) {
#pragma unroll
            for (int db = 0; db < 2; ++db) o_acc[db] *= alpha;
        }
        __builtin_amdgcn_s_setprio(1);  // the MFMA block (see above the kernel)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            if (kb == 1 && !live1) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float2 v = *reinterpret_cast<const float2*>(vs + (4 * half) * kHeadDim + 2 * col +
                                                                  (32 * kb + 8 * (r >> 2) + (r & 3)) * kHeadDim);
                o_acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(v.x, s_acc[kb][r], o_acc[0], 0, 0, 0);
                o_acc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(v.y, s_acc[kb][r], o_acc[1], 0, 0, 0);
            }
        }
        __builtin_amdgcn_s_setprio(0);
    };

    issue_k(kt_begin);
    issue_v(v0s, kt_begin);
    __builtin_amdgcn_s_waitcnt(0);
    lds_barrier();
    for (int64_t kt = kt_begin; kt < kt_end; kt += 2) {
        const int64_t n1 = kt + 1 < kt_end ? kt + 1 : kt_end - 1;
        issue_v(v1s, n1);
        tile(v0s, kt, n1);
        __builtin_amdgcn_s_waitcnt(0);  // this wave's copies of tile kt + 1 have landed
        lds_barrier();
        if (kt + 1 < kt_end) {
            const int64_t n2 = kt + 2 < kt_end ? kt + 2 : kt_end - 1;
            issue_v(v0s, n2);
            tile(v1s, kt + 1, n2);
            __builtin_amdgcn_s_waitcnt(0);
            lds_barrier();
        }
    }

    // O^T accumulator: lane holds dims 2 (8 (r / 4) + 4 half + r % 4) + db of query my_q.
    if (my_q >= seq) return;
    const bool single = attn_chunks(seq, qt) == 1;
    const float inv = single ? 1.0f / l_run : 1.0f;
    float* dst = single ? out_rows + my_q * kHidden + h * kHeadDim
                        : workspace + (attn_partial_slot(seq, qt, h, chunk) * kQTile + (my_q - qt * kQTile)) * kPartialRow;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int i = 8 * (r >> 2) + 4 * half + (r & 3);
        *reinterpret_cast<float2*>(dst + 2 * i) = make_float2(o_acc[0][r] * inv, o_acc[1][r] * inv);
    }
    if (!single && half == 0) *reinterpret_cast<float2*>(dst + kHeadDim) = make_float2(m_run, l_run);  // m in log2 units
}

// Prompts below kLimbAttnMinSeq: every block on the float32 instruction.
__global__ void __launch_bounds__(kAttnThreads) __attribute__((amdgpu_waves_per_eu(3)))
prefill_attention_f32_kernel(const float* __restrict__ q, const float* __restrict__ key_cache,
                             const float* __restrict__ value_cache, int64_t seq, int64_t capacity, float scale,
                             float* __restrict__ workspace, float* __restrict__ out_rows) {
    __shared__ __align__(16) float ks[kKTileWords];
    __shared__ __align__(16) float v0s[kKVTileFloats];
    __shared__ __align__(16) float v1s[kKVTileFloats];
    __builtin_assume(seq < kLimbAttnMinSeq);
    int64_t qt, chunk;
    attn_item(seq, blockIdx.x / kQHeads, qt, chunk);
    attention_item_f32(q, key_cache, value_cache, seq, capacity, scale, workspace, out_rows,
                       static_cast<int>(blockIdx.x % kQHeads), qt, chunk, ks, v0s, v1s);
}

// Limb planes of one layer's keys and values, so that the attention blocks copy MFMA operands
// instead of splitting every tile again.  Per KV head and 64-key tile, 24 KB of K:
// [key half][16-dim step][limb][dims 0-7 | 8-15][32 keys] x 8 values (16 bytes), and 24 KB of V:
// [key half][step][dim half][limb][lane half][32 dims] x 8 values, whose slot e holds key
// 8 (2 step + e / 4) + 4 (lane half) + e % 4 of the half: the keys whose probabilities a lane
// holds after S^T.  Block (KV head, tile); rows past the prompt repeat its last row (masked).
// flags[block] tells that a key of the tile is above kLimbMaxScore or a value above kLimbMaxValue.
constexpr int kLimbTile = kKTile * kHeadDim * 2 * kLimbs;  // bytes of one K or V tile: 24576
// Magnitudes up to which no sum of products overflows (64 of a scaled query and a key, at most 2048
// of a weight and a value), which those of small limbs could do to another sign than the whole, and
// up to which bits that limbs do not carry (at most 2^-134 of each factor, limbs_drop) change a
// score by less than 2^-66, a weight by as little, and a sum over n key tiles by less than 2^-108 n.
constexpr float kLimbMaxScore = 0x1p60f;
constexpr float kLimbMaxValue = 0x1p19f;
constexpr float kLimbSureSum = 0x1p-82f;  // per key tile: from here on that is under 2^-26 of a sum

__device__ __forceinline__ bool above(const float (&v)[8], float most) {
    float m = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; e += 2) track_max(m, v[e], v[e + 1]);
    return !(m <= most);
}

__device__ __forceinline__ void store_limbs(char* at, const float (&v)[8]) {
    const Limbs8 l = split8(f32x4{v[0], v[1], v[2], v[3]}, f32x4{v[4], v[5], v[6], v[7]});
#pragma unroll
    for (int j = 0; j < kLimbs; ++j) *reinterpret_cast<u32x4*>(at + 1024 * j) = l.limb[j];
}

__global__ void __launch_bounds__(256) attention_limbs_kernel(const float* __restrict__ key_cache,
                                                              const float* __restrict__ value_cache, int64_t seq,
                                                              int64_t capacity, char* __restrict__ k_planes,
                                                              char* __restrict__ v_planes, int* __restrict__ flags) {
    const int tiles = static_cast<int>((seq + kKTile - 1) / kKTile);
    const int g = static_cast<int>(blockIdx.x) / tiles;
    const int64_t key0 = static_cast<int64_t>(blockIdx.x % tiles) * kKTile;
    const float* kg = key_cache + static_cast<int64_t>(g) * capacity * kHeadDim;
    const float* vg = value_cache + static_cast<int64_t>(g) * capacity * kHeadDim;
    char* kp = k_planes + static_cast<int64_t>(blockIdx.x) * kLimbTile;
    char* vp = v_planes + static_cast<int64_t>(blockIdx.x) * kLimbTile;
    bool large = false;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int u = static_cast<int>(threadIdx.x) + 256 * i;
        float v[8];
        const int key = u >> 3, part = u & 7;  // eight lanes per key row
        const int64_t row = key0 + key < seq ? key0 + key : seq - 1;
        *reinterpret_cast<f32x4*>(v) = *reinterpret_cast<const f32x4*>(kg + row * kHeadDim + 8 * part);
        *reinterpret_cast<f32x4*>(v + 4) = *reinterpret_cast<const f32x4*>(kg + row * kHeadDim + 8 * part + 4);
        large |= above(v, kLimbMaxScore);
        store_limbs(kp + ((key >> 5) * 4 + (part >> 1)) * 3072 + (part & 1) * 512 + (key & 31) * 16, v);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int u = static_cast<int>(threadIdx.x) + 256 * i;
        float v[8];
        const int dim = u & 63, half = (u >> 6) & 1, step = u >> 7;  // step: 16-key group of the tile
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int64_t key = key0 + 16 * step + 8 * (e >> 2) + 4 * half + (e & 3);
            v[e] = vg[(key < seq ? key : seq - 1) * kHeadDim + dim];
        }
        large |= above(v, kLimbMaxValue);
        store_limbs(vp + (step * 2 + (dim >> 5)) * 3072 + half * 512 + (dim & 31) * 16, v);
    }
    const int any = __syncthreads_or(large);
    if (threadIdx.x == 0) flags[blockIdx.x] = any;
}

// One block's item on limb products; false, and nothing written, where it needs the float32
// instruction.
__device__ __forceinline__ bool attention_item_limbs(const float* __restrict__ q, const char* __restrict__ k_planes,
                                                    const char* __restrict__ v_planes, const int* __restrict__ flags,
                                                    int64_t seq, float scale, float* __restrict__ workspace,
                                                    float* __restrict__ out_rows, int h, int64_t qt, int64_t chunk,
                                                    char* ks, char* v0s, char* v1s, int* unsure) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = h / kGroup;
    const int64_t qw0 = qt * kQTile + 32 * wave;  // first query of this wave
    const int col = lane & 31;
    const int half = lane >> 5;
    const int64_t my_q = qw0 + col;
    const int64_t tiles = (seq + kKTile - 1) / kKTile;
    const int64_t k_tiles = attn_key_tiles(seq, qt);
    const int64_t chunk_tiles = attn_chunk_tiles(seq);
    const int64_t kt_begin = chunk * chunk_tiles;
    const int64_t kt_end = kt_begin + chunk_tiles < k_tiles ? kt_begin + chunk_tiles : k_tiles;

    // B operand of S^T = K Q^T: the limbs of Q[my_q][16 step + 8 half ..] * scale * log2(e).
    u32x4 qreg[4][kLimbs];
    {
        const int64_t r = my_q < seq ? my_q : seq - 1;
        const float* qp = q + (static_cast<int64_t>(h) * seq + r) * kHeadDim + 8 * half;
        const float s2 = scale * kLog2e;
        bool large = false;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const f32x4 lo = *reinterpret_cast<const f32x4*>(qp + 16 * t) * s2;
            const f32x4 hi = *reinterpret_cast<const f32x4*>(qp + 16 * t + 4) * s2;
            const float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            large |= above(v, kLimbMaxScore);
            const Limbs8 l = split8(lo, hi);
#pragma unroll
            for (int j = 0; j < kLimbs; ++j) qreg[t][j] = l.limb[j];
        }
        if (kt_begin + lane < kt_end) large |= flags[g * tiles + kt_begin + lane] != 0;
        if (threadIdx.x == 0) *unsure = 0;
        if (__syncthreads_or(large)) return false;
    }

    // Copies of key tile kt: 24 of 1 KB each for K and V, wave w issues w, w + 4, ...
    const char* kg = k_planes + static_cast<int64_t>(g) * tiles * kLimbTile + 16 * lane;
    const char* vg = v_planes + static_cast<int64_t>(g) * tiles * kLimbTile + 16 * lane;
    auto issue = [&](const char* planes, char* buf, int64_t kt) {
#pragma unroll
        for (int j = 0; j < kLimbTile / 4096; ++j) {
            const int i = wave + 4 * j;
            __builtin_amdgcn_global_load_lds(reinterpret_cast<const unsigned*>(planes + kt * kLimbTile + 1024 * i),
                                             reinterpret_cast<unsigned*>(buf + 1024 * i), 16, 0, 0);
        }
    };

    // O^T and its small limb products (prefill_limb.h), summed apart so that only the products
    // of the leading limbs are rounded at the size of the result.
    f32x16 o_acc[2], o_low[2];
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[db][r] = o_low[db][r] = 0.0f;
    float m_run = -INFINITY;
    float l_run = 0.0f;

    const int seq32 = static_cast<int>(seq);
    const int qw = static_cast<int>(qw0);
    const int q_me = static_cast<int>(my_q);
    // QK of 32 keys: the small products of all 64 dims first, those of the leading limbs last.
    auto qk = [&](int kb, f32x16& c) {
        const char* kp = ks + kb * 4 * 3072 + 16 * lane;
        u32x4 lead[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            lead[t] = *reinterpret_cast<const u32x4*>(kp + 3072 * t);
            const u32x4 k1 = *reinterpret_cast<const u32x4*>(kp + 3072 * t + 1024);
            const u32x4 k2 = *reinterpret_cast<const u32x4*>(kp + 3072 * t + 2048);
            c = mfma_bf16(k2, qreg[t][0], c);
            c = mfma_bf16(lead[t], qreg[t][2], c);
            c = mfma_bf16(k1, qreg[t][1], c);
            c = mfma_bf16(k1, qreg[t][0], c);
            c = mfma_bf16(lead[t], qreg[t][1], c);
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) c = mfma_bf16(lead[t], qreg[t][0], c);
    };
    // One key tile: S^T from the K tile, an LDS barrier after which the K buffer is
    // refilled with the next tile, then softmax and O^T += V^T P^T from this tile's
    // V buffer.  Waves whose queries all precede the tile skip the math but not the
    // barriers.
    auto tile = [&](const char* vs, int64_t kt, int64_t kt_next) {
        const int k0 = static_cast<int>(kt) * kKTile;
        const bool active = k0 <= qw + 31;
        const bool need_mask = k0 + kKTile - 1 > qw || k0 + kKTile > seq32;
        const bool live1 = k0 + 32 <= qw + 31;  // second 32-key half visible to some query
        f32x16 s_acc[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) s_acc[kb][r] = 0.0f;
        __builtin_amdgcn_s_setprio(1);  // the MFMA block (see above the kernel)
        if (active) qk(0, s_acc[0]);
        if (live1) qk(1, s_acc[1]);
        __builtin_amdgcn_s_setprio(0);
        lds_barrier();  // every wave is done with the K tile
        issue(kg, ks, kt_next);
        if (!active) return;
        // Lane holds keys k0 + 32 kb + 8 (r / 4) + 4 half + r % 4 of query my_q.
        if (!live1) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s_acc[1][r] = -INFINITY;
        }
        if (need_mask) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key = k0 + 32 * kb + 8 * (r >> 2) + 4 * half + (r & 3);
                    s_acc[kb][r] = (key <= q_me && key < seq32) ? s_acc[kb][r] : -INFINITY;
                }
            }
        }
        float tile_max = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) tile_max = fmaxf(tile_max, s_acc[kb][r]);
        tile_max = halves_max(tile_max);
        const float m_new = fmaxf(m_run, tile_max);  // finite: the first key of a chunk precedes every query
        const float alpha = fast_exp2(m_run - m_new);
        float psum = 0.0f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float p = fast_exp2(s_acc[kb][r] - m_new);
                s_acc[kb][r] = p;
                psum += p;
            }
        }
        psum = halves_sum(psum);
        l_run = l_run * alpha + psum;
        m_run = m_new;
        // alpha is exactly 1 where the running max did not move: skip the rescale
        // when that holds for every lane (multiplying by 1 would not change a bit).
        if (__any(alpha != 1.0f)) {
#pragma unroll
            for (int db = 0; db < 2; ++db) {
                o_acc[db] *= alpha;
                o_low[db] *= alpha;
            }
        }
        const char* vp = vs + 16 * lane;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            if (kb == 1 && !live1) continue;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const f32x16& s = s_acc[kb];
                const Limbs8 p = split8(f32x4{s[8 * t], s[8 * t + 1], s[8 * t + 2], s[8 * t + 3]},
                                        f32x4{s[8 * t + 4], s[8 * t + 5], s[8 * t + 6], s[8 * t + 7]});
                u32x4 v[2][kLimbs];
#pragma unroll
                for (int db = 0; db < 2; ++db)
#pragma unroll
                    for (int l = 0; l < kLimbs; ++l)
                        v[db][l] =
                            *reinterpret_cast<const u32x4*>(vp + ((kb * 2 + t) * 2 + db) * 3072 + 1024 * l);
                __builtin_amdgcn_s_setprio(1);
#pragma unroll
                for (int db = 0; db < 2; ++db) o_low[db] = mfma_bf16(v[db][2], p.limb[0], o_low[db]);
#pragma unroll
                for (int db = 0; db < 2; ++db) o_low[db] = mfma_bf16(v[db][0], p.limb[2], o_low[db]);
#pragma unroll
                for (int db = 0; db < 2; ++db) o_low[db] = mfma_bf16(v[db][1], p.limb[1], o_low[db]);
#pragma unroll
                for (int db = 0; db < 2; ++db) o_low[db] = mfma_bf16(v[db][1], p.limb[0], o_low[db]);
#pragma unroll
                for (int db = 0; db < 2; ++db) o_low[db] = mfma_bf16(v[db][0], p.limb[1], o_low[db]);
#pragma unroll
                for (int db = 0; db < 2; ++db) o_acc[db] = mfma_bf16(v[db][0], p.limb[0], o_acc[db]);
                __builtin_amdgcn_s_setprio(0);
            }
        }
    };

    issue(kg, ks, kt_begin);
    issue(vg, v0s, kt_begin);
    __builtin_amdgcn_s_waitcnt(0);
    lds_barrier();
    for (int64_t kt = kt_begin;; kt += 2) {
        const int64_t n1 = kt + 1 < kt_end ? kt + 1 : kt_end - 1;
        issue(vg, v1s, n1);
        tile(v0s, kt, n1);
        if (kt + 1 >= kt_end) break;
        __builtin_amdgcn_s_waitcnt(0);  // this wave's copies of tile kt + 1 have landed
        lds_barrier();
        const int64_t n2 = kt + 2 < kt_end ? kt + 2 : kt_end - 1;
        issue(vg, v0s, n2);
        tile(v1s, kt + 1, n2);
        if (kt + 2 >= kt_end) break;
        __builtin_amdgcn_s_waitcnt(0);
        lds_barrier();
    }

    // O^T accumulator: lane holds dims 32 db + 8 (r / 4) + 4 half + r % 4 of query my_q.
    // A sum below kLimbSureSum may lack bits: the smallest, exact zeros aside (those are of values
    // that are zero, or of products that float32 does not hold either).
    unsigned least = ~0u;
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            o_acc[db][r] += o_low[db][r];
            least = min(least, magnitude_key(o_acc[db][r]));
        }
    if (least < magnitude_key(kLimbSureSum * static_cast<float>(kt_end - kt_begin))) *unsure = 1;
    __builtin_amdgcn_s_waitcnt(0);  // no copy may still be landing in LDS when the block retires or starts again
    lds_barrier();
    if (*unsure != 0) return false;
    if (my_q >= seq) return true;
    const bool single = attn_chunks(seq, qt) == 1;
    const float inv = single ? 1.0f / l_run : 1.0f;
    float* dst = single ? out_rows + my_q * kHidden + h * kHeadDim
                        : workspace + (attn_partial_slot(seq, qt, h, chunk) * kQTile + (my_q - qt * kQTile)) * kPartialRow;
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
            f32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = o_acc[db][r + e] * inv;
            *reinterpret_cast<f32x4*>(dst + 32 * db + 2 * r + 4 * half) = o;
        }
    if (!single && half == 0) *reinterpret_cast<float2*>(dst + kHeadDim) = make_float2(m_run, l_run);  // m in log2 units
    return true;
}

__global__ void __launch_bounds__(kAttnThreads, 2)
prefill_attention_kernel(const float* __restrict__ q, const float* __restrict__ key_cache,
                         const float* __restrict__ value_cache, const char* __restrict__ k_planes,
                         const char* __restrict__ v_planes, const int* __restrict__ flags, int64_t seq,
                         int64_t capacity, float scale, float* __restrict__ workspace, float* __restrict__ out_rows) {
    __shared__ __align__(16) char ks[kLimbTile];
    __shared__ __align__(16) char v0s[kLimbTile];
    __shared__ __align__(16) char v1s[kLimbTile];
    __shared__ int unsure;  // some sum may lack bits that limbs do not carry
    const int h = static_cast<int>(blockIdx.x % kQHeads);
    int64_t qt, chunk;
    attn_item(seq, blockIdx.x / kQHeads, qt, chunk);
    if (!attention_item_limbs(q, k_planes, v_planes, flags, seq, scale, workspace, out_rows, h, qt, chunk, ks, v0s,
                              v1s, &unsure))
        attention_item_f32(q, key_cache, value_cache, seq, capacity, scale, workspace, out_rows, h, qt, chunk,
                           reinterpret_cast<float*>(ks), reinterpret_cast<float*>(v0s), reinterpret_cast<float*>(v1s));
}

// Combines the chunk partials of query tiles with more than one chunk.  Block
// ((qt - attn_long_tile(seq)) * 9 + h) * 8 + row group; thread t -> row 16 * group + t / 16,
// dims 4 (t % 16) .. + 3.  All chunk loads of a thread are issued before the combine.
template <int kMaxChunks>
__global__ void __launch_bounds__(kAttnThreads) prefill_attention_merge_kernel(const float* __restrict__ workspace,
                                                                               int64_t seq,
                                                                               float* __restrict__ out_rows) {
    constexpr int kRowsPerBlock = kAttnThreads / 16;
    const int64_t tile_head = blockIdx.x / (kQTile / kRowsPerBlock);
    const int64_t qt = attn_long_tile(seq) + tile_head / kQHeads;
    const int h = static_cast<int>(tile_head % kQHeads);
    const int row = static_cast<int>(blockIdx.x % (kQTile / kRowsPerBlock)) * kRowsPerBlock +
                    static_cast<int>(threadIdx.x >> 4);
    const int d = 4 * static_cast<int>(threadIdx.x & 15);
    const int64_t q0 = qt * kQTile;
    if (q0 + row >= seq) return;
    const int chunks = static_cast<int>(attn_chunks(seq, qt));
    float4 o[kMaxChunks];
    float m[kMaxChunks], l[kMaxChunks];
#pragma unroll
    for (int c = 0; c < kMaxChunks; ++c) {
        if (c < chunks) {
            const float* p = workspace + (attn_partial_slot(seq, qt, h, c) * kQTile + row) * kPartialRow;
            o[c] = *reinterpret_cast<const float4*>(p + d);
            const float2 ml = *reinterpret_cast<const float2*>(p + kHeadDim);
            m[c] = ml.x;
            l[c] = ml.y;
        } else {
            o[c] = make_float4(0.f, 0.f, 0.f, 0.f);
            m[c] = -INFINITY;
            l[c] = 0.0f;
        }
    }
    float M = -INFINITY;
#pragma unroll
    for (int c = 0; c < kMaxChunks; ++c) M = fmaxf(M, m[c]);
    float4 O = make_float4(0.f, 0.f, 0.f, 0.f);
    float L = 0.0f;
#pragma unroll
    for (int c = 0; c < kMaxChunks; ++c) {
        const float f = fast_exp2(m[c] - M);
        O.x = fmaf(o[c].x, f, O.x);
        O.y = fmaf(o[c].y, f, O.y);
        O.z = fmaf(o[c].z, f, O.z);
        O.w = fmaf(o[c].w, f, O.w);
        L = fmaf(l[c], f, L);
    }
    *reinterpret_cast<float4*>(out_rows + (q0 + row) * kHidden + h * kHeadDim + d) =
        make_float4(O.x / L, O.y / L, O.z / L, O.w / L);
}

// Short prompts: block = (32-query tile t, query head h).  The tile's causal keys are
// the 32-key chunks c = 0..t; chunk c goes to wave c % 8, and each wave runs the online
// softmax over its chunks with K, V and Q read from global memory straight into MFMA
// operands (a chunk is 16 KB of K/V, served by L2).  S^T = K Q^T and O^T += V^T P^T use
// the same operand layouts as prefill_attention_kernel.  The waves' (o, m, l) meet in
// LDS, where 512 threads combine them, so no partials leave the block and no merge
// kernel runs.  A 128-token prompt is 36 blocks of at most one chunk per wave, against 9
// blocks whose last wave walks 128 keys in the 128-query-tile kernel.
constexpr int kSmallQ = 32;
constexpr int kSmallWaves = 8;
// Measured against the 128-query-tile kernel (whole prefill, ms): 128 tokens 1.58 vs 1.81,
// 256: 1.81 vs 2.04, 512: 2.62 vs 2.71, 1024: 4.38 vs 4.36 (16 waves per block: slower
// from 512 on).
constexpr int64_t kSmallAttnMaxSeq = 512;

__global__ void __launch_bounds__(64 * kSmallWaves)
prefill_attention_small_kernel(const float* __restrict__ q, const float* __restrict__ key_cache,
                               const float* __restrict__ value_cache, int64_t seq, int64_t capacity, float scale,
                               float* __restrict__ out_rows) {
    __shared__ float o_s[kSmallWaves][kSmallQ][kHeadDim + 1];
    __shared__ float m_s[kSmallWaves][kSmallQ];
    __shared__ float l_s[kSmallWaves][kSmallQ];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int h = static_cast<int>(blockIdx.x % kQHeads);
    const int t = static_cast<int>(blockIdx.x / kQHeads);
    const int g = h / kGroup;
    const int col = lane & 31;
    const int half = lane >> 5;
    const int seq32 = static_cast<int>(seq);
    const int q_me = kSmallQ * t + col;

    // B operand of S^T = K Q^T: qreg[s] = Q[q_me][s + 32 half] * scale * log2(e).
    float qreg[32];
    {
        const int64_t r = q_me < seq32 ? q_me : seq32 - 1;
        const float* qp = q + (static_cast<int64_t>(h) * seq + r) * kHeadDim + 32 * half;
        const float s2 = scale * kLog2e;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float4 v = *reinterpret_cast<const float4*>(qp + 4 * i);
            qreg[4 * i] = v.x * s2;
            qreg[4 * i + 1] = v.y * s2;
            qreg[4 * i + 2] = v.z * s2;
            qreg[4 * i + 3] = v.w * s2;
        }
    }
    const float* kg = key_cache + static_cast<int64_t>(g) * capacity * kHeadDim;
    const float* vg = value_cache + static_cast<int64_t>(g) * capacity * kHeadDim;

    f32x16 o_acc[2];
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[db][r] = 0.0f;
    float m_run = -INFINITY;
    float l_run = 0.0f;
    for (int c = wave; c <= t; c += kSmallWaves) {
        const int k0 = kSmallQ * c;
        // A operand of S^T: this lane's key k0 + col (rows past the prompt repeat its last
        // row; they are masked), dims 32 half ..; the V operands of the chunk are requested
        // with it, before the softmax needs them.
        const int krow = k0 + col < seq32 ? k0 + col : seq32 - 1;
        const float* kp = kg + static_cast<int64_t>(krow) * kHeadDim + 32 * half;
        f32x4 kv[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) kv[i] = *reinterpret_cast<const f32x4*>(kp + 4 * i);
        float2 vv[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int key = k0 + 8 * (r >> 2) + 4 * half + (r & 3);
            const int vrow = key < seq32 ? key : seq32 - 1;
            vv[r] = *reinterpret_cast<const float2*>(vg + static_cast<int64_t>(vrow) * kHeadDim + 2 * col);
        }
        f32x16 s_acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) s_acc[r] = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                s_acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[i][e], qreg[4 * i + e], s_acc, 0, 0, 0);
        // Lane holds keys k0 + 8 (r / 4) + 4 half + r % 4 of query q_me.  Every chunk a wave
        // takes holds a key <= q_me below the prompt length (key 32 t on the diagonal), so the
        // running maximum is finite after the first chunk.
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int key = k0 + 8 * (r >> 2) + 4 * half + (r & 3);
            s_acc[r] = (key <= q_me && key < seq32) ? s_acc[r] : -INFINITY;
        }
        float tile_max = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) tile_max = fmaxf(tile_max, s_acc[r]);
        tile_max = halves_max(tile_max);
        const float m_new = fmaxf(m_run, tile_max);
        const float alpha = fast_exp2(m_run - m_new);
        float psum = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float p = fast_exp2(s_acc[r] - m_new);
            s_acc[r] = p;
            psum += p;
        }
        psum = halves_sum(psum);
        l_run = l_run * alpha + psum;
        m_run = m_new;
#pragma unroll
        for (int db = 0; db < 2; ++db) o_acc[db] *= alpha;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            o_acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv[r].x, s_acc[r], o_acc[0], 0, 0, 0);
            o_acc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv[r].y, s_acc[r], o_acc[1], 0, 0, 0);
        }
    }

    // O^T accumulator: lane holds dims 2 (8 (r / 4) + 4 half + r % 4) + db of query q_me.
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int i = 8 * (r >> 2) + 4 * half + (r & 3);
        o_s[wave][col][2 * i] = o_acc[0][r];
        o_s[wave][col][2 * i + 1] = o_acc[1][r];
    }
    if (half == 0) {
        m_s[wave][col] = m_run;
        l_s[wave][col] = l_run;
    }
    __syncthreads();
    // Thread -> query 32 t + (thread / 16), dims 4 (thread % 16) .. + 3; waves in order.
    const int qq = static_cast<int>(threadIdx.x >> 4);
    const int d = 4 * static_cast<int>(threadIdx.x & 15);
    const int qrow = kSmallQ * t + qq;
    if (qrow >= seq32) return;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < kSmallWaves; ++w) M = fmaxf(M, m_s[w][qq]);
    float4 O = make_float4(0.f, 0.f, 0.f, 0.f);
    float L = 0.0f;
#pragma unroll
    for (int w = 0; w < kSmallWaves; ++w) {
        const float mw = m_s[w][qq];
        const float f = mw == -INFINITY ? 0.0f : fast_exp2(mw - M);
        const float* ow = &o_s[w][qq][d];
        O.x = fmaf(ow[0], f, O.x);
        O.y = fmaf(ow[1], f, O.y);
        O.z = fmaf(ow[2], f, O.z);
        O.w = fmaf(ow[3], f, O.w);
        L = fmaf(l_s[w][qq], f, L);
    }
    *reinterpret_cast<float4*>(out_rows + static_cast<int64_t>(qrow) * kHidden + h * kHeadDim + d) =
        make_float4(O.x / L, O.y / L, O.z / L, O.w / L);
}

}  // namespace

// Floats of the split-key partials (a multiple of 4).
static int64_t attn_partial_floats(int64_t seq) {
    const int64_t long_tiles = attn_q_tiles(seq) - attn_long_tile(seq);
    if (long_tiles <= 0 || attn_max_chunks(seq) <= 1) return 0;
    return long_tiles * kQHeads * attn_max_chunks(seq) * kQTile * kPartialRow;
}

// Floats that the kernels use: the partials, and from kLimbAttnMinSeq on the limb planes of K and V
// and one flag per key tile.
static int64_t attn_used_floats(int64_t seq) {
    const int64_t tiles = kKVHeads * ((seq + kKTile - 1) / kKTile);
    return attn_partial_floats(seq) +
           (seq < kLimbAttnMinSeq ? 0 : tiles * (2 * kLimbTile / 4) + (tiles + 3) / 4 * 4);
}

// The size callers are told: partials of chunks of an even share of 768 slots and at most 16 key
// tiles, which covers what is used at every length (launch_prefill_attention checks it), so that
// a workspace kept from an earlier version of the library still fits.
size_t prefill_attention_workspace_floats(int64_t seq) {
    if (seq <= kSmallAttnMaxSeq) return 0;  // prefill_attention_small_kernel keeps its partials in LDS
    const int64_t ct = attn_share_tiles(seq, 768, 16);
    const int64_t q_tiles = attn_q_tiles(seq);
    const int64_t max_chunks = (attn_key_tiles(seq, q_tiles - 1) + ct - 1) / ct;
    const int64_t long_tiles = q_tiles - ct * kKTile / kQTile;
    if (long_tiles <= 0 || max_chunks <= 1) return 0;
    return static_cast<size_t>(long_tiles * kQHeads * max_chunks * kQTile * kPartialRow);
}

hipError_t launch_prefill_attention(const float* q, const float* key_cache, const float* value_cache, int64_t seq,
                                    int64_t capacity, float scale, float* workspace, float* out_rows,
                                    hipStream_t stream) {
    if (seq <= 0 || seq > capacity) return hipErrorInvalidValue;
    if (prefill_attention_workspace_floats(seq) > 0 && workspace == nullptr) return hipErrorInvalidValue;
    if (seq <= kSmallAttnMaxSeq) {
        const dim3 grid(static_cast<unsigned>((seq + kSmallQ - 1) / kSmallQ * kQHeads));
        hipLaunchKernelGGL(prefill_attention_small_kernel, grid, dim3(64 * kSmallWaves), 0, stream, q, key_cache,
                           value_cache, seq, capacity, scale, out_rows);
        return hipGetLastError();
    }
    if (attn_max_chunks(seq) > kMergeMaxChunks ||
        attn_used_floats(seq) > static_cast<int64_t>(prefill_attention_workspace_floats(seq)))
        return hipErrorInvalidValue;
    const dim3 blocks(static_cast<unsigned>(attn_items(seq) * kQHeads));
    hipError_t st = hipSuccess;
    if (seq < kLimbAttnMinSeq) {
        hipLaunchKernelGGL(prefill_attention_f32_kernel, blocks, dim3(kAttnThreads), 0, stream, q, key_cache,
                           value_cache, seq, capacity, scale, workspace, out_rows);
        st = hipGetLastError();
    } else {
        const int64_t tiles = kKVHeads * ((seq + kKTile - 1) / kKTile);
        char* k_planes = reinterpret_cast<char*>(workspace + attn_partial_floats(seq));
        char* v_planes = k_planes + tiles * kLimbTile;
        int* flags = reinterpret_cast<int*>(v_planes + tiles * kLimbTile);
        hipLaunchKernelGGL(attention_limbs_kernel, dim3(static_cast<unsigned>(tiles)), dim3(256), 0, stream, key_cache,
                           value_cache, seq, capacity, k_planes, v_planes, flags);
        st = hipGetLastError();
        if (st != hipSuccess) return st;
        hipLaunchKernelGGL(prefill_attention_kernel, blocks, dim3(kAttnThreads), 0, stream, q, key_cache, value_cache,
                           k_planes, v_planes, flags, seq, capacity, scale, workspace, out_rows);
        st = hipGetLastError();
    }
    if (st != hipSuccess) return st;
    const int64_t long_tiles = attn_q_tiles(seq) - attn_long_tile(seq);
    if (long_tiles > 0 && attn_max_chunks(seq) > 1) {
        // Registers for at most 4 or 8 chunks: fewer registers, more waves in flight.
        const dim3 grid(static_cast<unsigned>(long_tiles * kQHeads * (kQTile / (kAttnThreads / 16))));
        if (attn_max_chunks(seq) <= 4)
            hipLaunchKernelGGL(prefill_attention_merge_kernel<4>, grid, dim3(kAttnThreads), 0, stream, workspace, seq,
                               out_rows);
        else
            hipLaunchKernelGGL(prefill_attention_merge_kernel<kMergeMaxChunks>, grid, dim3(kAttnThreads), 0, stream,
                               workspace, seq, out_rows);
        st = hipGetLastError();
    }
    return st;
}

}  // namespace flux
