// Prompt forward for MI355X (gfx950): a dense Llama forward over a whole prompt.
//
// A prompt of a few thousand positions is bound by its matrix products; what a framework adds to them is traffic - the
// same activations read and written once per small operation - and launches.  In this file every stage between two
// products is one kernel: residual add + RMS norm, rotary embedding + cache append + the layouts attention reads, attention
// itself, SiLU * up, argmax.  Prompts of up to some thousand positions have their products here, too, with these stages
// inside them: mk_prefill_rows.h for up to 64 rows of models up to 2048 wide, mk_prefill_tiles.h above, mk_prefill_wide.h for
// longer prompts and wider models; the host side below chooses.  Values are
// narrowed to bf16 exactly where the plain forward narrows them (megakernels/llama.py:38-47 for the norm, :136-174 for the
// rotation), but for the norm of few rows.
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <type_traits>

#include "../../include/mk_prefill.h"

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
#define MK_LDS __attribute__((address_space(3)))
#define MK_GLOBAL __attribute__((address_space(1)))

__device__ __forceinline__ float bf16_lo(uint32_t pair) { return __builtin_bit_cast(float, pair << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t pair) { return __builtin_bit_cast(float, pair & 0xffff0000u); }
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    const f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ float round_bf16(float v) { return bf16_lo(pack_bf16(v, 0.0f)); }
__device__ __forceinline__ float bf16_f32(uint16_t v) { return __builtin_bit_cast(float, (uint32_t)v << 16); }

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int offset = 32; offset >= 1; offset /= 2) v += __shfl_xor(v, offset);
    return v;
}

// ---------------------------------------------------------------------------------------------
// Residual add + RMS norm, one block per row.  Bound by memory: two rows in, two out (the embedding
// row instead of the two where the stream starts).
// ---------------------------------------------------------------------------------------------
constexpr int kNormThreads = 256;
constexpr int kMaxHidden = 8192;
constexpr int kNormChunks = kMaxHidden / (8 * kNormThreads);  // 16-byte pieces of a row per thread, at most

// position as an index of a table of `count` rows: negative ones count from the end
__device__ __forceinline__ int64_t wrap_position(int64_t position, int count) { return position < 0 ? position + count : position; }

// an id or a position outside its table aborts the kernel
__device__ __forceinline__ void check_token(const mk_prefill_shape &s, int64_t id, int64_t position) {
    const int64_t cache_row = wrap_position(position, s.kv_max_len), rope_row = wrap_position(position, s.rope_positions);
    if (id < 0 || id >= s.vocab_size || cache_row < 0 || cache_row >= s.kv_max_len || rope_row < 0 || rope_row >= s.rope_positions)
        __builtin_trap();
}

enum NormSource { kNormAdd, kNormEmbed, kNormPlain };  // h += src; h = embed row; h as it is

template <NormSource SOURCE>
__global__ __launch_bounds__(kNormThreads) void norm_kernel(mk_prefill_shape s, const int64_t *ids, const int64_t *positions,
                                                            const uint16_t *src, const uint16_t *weight, uint16_t *h, uint16_t *x) {
    const int row = blockIdx.x, hid = s.hidden_size, pieces = hid / 8;
    const uint16_t *add = src + (size_t)row * hid;
    if constexpr (SOURCE == kNormEmbed) {
        const int64_t id = ids[row];
        check_token(s, id, positions[row % s.seq]);
        add = src + (size_t)id * hid;
    }
    uint16_t *const h_row = h + (size_t)row * hid;
    u32x4 v[kNormChunks];
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < kNormChunks; i++) {
        const int at = (int)threadIdx.x + i * kNormThreads;
        if (at >= pieces) break;
        v[i] = *(const u32x4 *)((SOURCE == kNormPlain ? h_row : add) + (size_t)at * 8);
        if constexpr (SOURCE == kNormAdd) {
            const u32x4 old = *(const u32x4 *)(h_row + (size_t)at * 8);
#pragma unroll
            for (int j = 0; j < 4; j++) v[i][j] = pack_bf16(bf16_lo(old[j]) + bf16_lo(v[i][j]), bf16_hi(old[j]) + bf16_hi(v[i][j]));
        }
        if constexpr (SOURCE != kNormPlain) *(u32x4 *)(h_row + (size_t)at * 8) = v[i];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float lo = bf16_lo(v[i][j]), hi = bf16_hi(v[i][j]);
            sum += lo * lo;
            sum += hi * hi;
        }
    }
    __shared__ float wave_sums[kNormThreads / 64];
    sum = wave_sum(sum);
    if (threadIdx.x % 64 == 0) wave_sums[threadIdx.x / 64] = sum;
    __syncthreads();
    sum = 0.0f;
#pragma unroll
    for (int w = 0; w < kNormThreads / 64; w++) sum += wave_sums[w];
    const float scale = rsqrtf(sum / (float)hid + s.rms_norm_eps);
#pragma unroll
    for (int i = 0; i < kNormChunks; i++) {
        const int at = (int)threadIdx.x + i * kNormThreads;
        if (at >= pieces) break;
        const u32x4 w = *(const u32x4 *)(weight + (size_t)at * 8);
        u32x4 out;
#pragma unroll
        for (int j = 0; j < 4; j++)
            out[j] = pack_bf16(bf16_lo(w[j]) * round_bf16(bf16_lo(v[i][j]) * scale), bf16_hi(w[j]) * round_bf16(bf16_hi(v[i][j]) * scale));
        *(u32x4 *)(x + (size_t)row * hid + (size_t)at * 8) = out;
    }
}

// ---------------------------------------------------------------------------------------------
// Rotary embedding, cache append, and the layouts attention reads.  One block per 64 positions of one
// head (query, key or value).  Keys are copied to [KVH, padded, D] because the cache rows of a prompt need
// not be consecutive.  Values are transposed to [KVH, D, padded] with the positions of every group of 16 in
// the order 0-3, 8-11, 4-7, 12-15: the order in which attention's probabilities leave the matrix cores, so
// that its second product reads both operands without exchanging lanes.  Padding positions hold zeros.
// ---------------------------------------------------------------------------------------------
constexpr int kPosTile = 64;

__device__ __forceinline__ int slot_in_group(int position) {  // place of a position within its group of 16
    return (position & 3) | ((position & 4) << 1) | ((position & 8) >> 1);
}

template <int D>
__global__ __launch_bounds__(256) void rope_kernel(mk_prefill_shape s, int padded, const uint16_t *qkv, const int64_t *positions,
                                                   const float *rope_cos, const float *rope_sin, uint16_t *k_cache, uint16_t *v_cache,
                                                   uint16_t *q, uint16_t *keys, uint16_t *values_t) {
    constexpr int kPieces = D / 8;
    const int H = s.num_attention_heads, KVH = s.num_kv_heads;
    const int head = blockIdx.y, batch = blockIdx.z, first = blockIdx.x * kPosTile;
    const size_t qkv_row = (size_t)(H + 2 * KVH) * D;
    const bool is_value = head >= H + KVH;
    const int kv_head = is_value ? head - H - KVH : head - H;
    __shared__ uint16_t tile[D][kPosTile + 8];
    for (int i = threadIdx.x; i < kPosTile * kPieces; i += 256) {
        const int p = i / kPieces, piece = i % kPieces, seq_at = first + p;
        u32x4 v = {0, 0, 0, 0};
        if (seq_at < s.seq) {
            const int64_t position = positions[seq_at];
            const uint16_t *src = qkv + ((size_t)batch * s.seq + seq_at) * qkv_row + (size_t)head * D;
            v = *(const u32x4 *)(src + piece * 8);
            if (!is_value) {
                const size_t rope_row = (size_t)wrap_position(position, s.rope_positions) * D + piece * 8;
                u32x4 other = v;
                if (!s.interleaved) other = *(const u32x4 *)(src + (piece * 8 + D / 2) % D);
                const bool upper = piece * 8 >= D / 2;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const f32x2 c = *(const f32x2 *)(rope_cos + rope_row + 2 * j), sn = *(const f32x2 *)(rope_sin + rope_row + 2 * j);
                    const float lo = bf16_lo(v[j]), hi = bf16_hi(v[j]);
                    float part_lo = -hi, part_hi = lo;
                    if (!s.interleaved) {
                        part_lo = upper ? bf16_lo(other[j]) : -bf16_lo(other[j]);
                        part_hi = upper ? bf16_hi(other[j]) : -bf16_hi(other[j]);
                    }
                    v[j] = pack_bf16(lo * c.x + part_lo * sn.x, hi * c.y + part_hi * sn.y);
                }
            }
            if (head < H) {
                *(u32x4 *)(q + (((size_t)batch * s.seq + seq_at) * H + head) * D + piece * 8) = v;
            } else {
                uint16_t *const cache = is_value ? v_cache : k_cache;
                const size_t cache_row = (size_t)batch * s.kv_max_len + (size_t)wrap_position(position, s.kv_max_len);
                *(u32x4 *)(cache + (cache_row * KVH + kv_head) * D + piece * 8) = v;
            }
        }
        if (is_value) {
            const int slot = (p & ~15) | slot_in_group(p & 15);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                tile[piece * 8 + 2 * j][slot] = (uint16_t)v[j];
                tile[piece * 8 + 2 * j + 1][slot] = (uint16_t)(v[j] >> 16);
            }
        } else if (head >= H) {
            *(u32x4 *)(keys + (((size_t)batch * KVH + kv_head) * padded + seq_at) * D + piece * 8) = v;
        }
    }
    if (!is_value) return;
    __syncthreads();
    for (int i = threadIdx.x; i < D * (kPosTile / 8); i += 256) {
        const int d = i / (kPosTile / 8), piece = i % (kPosTile / 8);
        *(u32x4 *)(values_t + (((size_t)batch * KVH + kv_head) * D + d) * padded + first + piece * 8) = *(const u32x4 *)&tile[d][piece * 8];
    }
}

// ---------------------------------------------------------------------------------------------
// Causal attention.  A block works on one KV head and QB query positions: its waves are the four query
// heads of the KV head times QB / 32 groups of 32 positions, and share the K and V tiles of 64 positions,
// which go from memory straight into LDS (double-buffered, 16-byte pieces swizzled so that the reads of a
// wave are spread over all banks).
//
// The scores are computed transposed, S^T = K Q^T: a query position is then a lane (lane % 32) and its
// scores lie in that lane's registers, so the maximum and the sum over a tile need one exchange between
// the two halves of the wave instead of a tree over lanes, rescaling the output is one factor per lane, and
// the probabilities are already in the operand layout of O^T = V^T P^T.
//
// Bound by the vector units, not by the matrix cores, at head_dim 64: 2048 scores take 512 clocks of matrix
// work per wave and about 900 of vector work (the exponential alone 512).
// ---------------------------------------------------------------------------------------------
constexpr int kKeyTile = 64;

__device__ __forceinline__ float half_exchange_max(float v) {
    uint32_t a = __builtin_bit_cast(uint32_t, v), b = a;
    // written in assembly: the compiler's builtin for this instruction returns the first result twice
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    return fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
}
__device__ __forceinline__ float half_exchange_sum(float v) {
    uint32_t a = __builtin_bit_cast(uint32_t, v), b = a;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    return __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b);
}

// 16 bytes per lane from memory into LDS at `dst` (the same in every lane) + 16 * lane
__device__ __forceinline__ void load_to_lds(const void *src, MK_LDS void *dst) {
    __builtin_amdgcn_global_load_lds((const MK_GLOBAL void *)src, dst, 16, 0, 0);
}

// Two waves per SIMD are asked for because LDS allows no more blocks at head_dim 128 and the compiler, left to itself,
// spread one wave's values over all 512 registers with copies between the two halves of the file: 2048 positions, 32 heads
// of 128: 88 us without, 56.5 with the bound; 777 positions of heads of 64: 18.0 and 15.2.
template <int D, int WAVES>
__global__ __launch_bounds__(WAVES * 64, 2) void attention_kernel(mk_prefill_shape s, int padded, float scale, const uint16_t *q,
                                                               const uint16_t *keys, const uint16_t *values_t, uint16_t *out) {
    constexpr int kGqa = 4, kQueries = 32 * WAVES / kGqa, kThreads = WAVES * 64;
    constexpr int kKeyPieces = D / 8, kTileBytes = kKeyTile * D * 2, kPieces = kTileBytes / 16;
    constexpr int kDepthSteps = D / 16, kOutTiles = D / 32;
    static_assert(kPieces % kThreads == 0, "every thread moves whole pieces");
    __shared__ alignas(16) unsigned char lds[2][2][kTileBytes];  // [buffer][keys, values]

    const int H = s.num_attention_heads, KVH = s.num_kv_heads, seq = s.seq;
    const int kv_head = blockIdx.x % KVH, batch = blockIdx.y, tiles = (seq + kQueries - 1) / kQueries;
    // A tile's work grows with its position.  The first half of the blocks takes the heavy tiles in
    // descending order, the second the light ones in ascending order: blocks that share a CU add up to the
    // same work, and where there are more blocks than the chip holds, the light ones come last.
    const int order = blockIdx.x / KVH, heavy = (tiles + 1) / 2;
    const int tile = order < heavy ? tiles - 1 - order : order - heavy;
    const int wave = (int)threadIdx.x / 64, lane = (int)threadIdx.x % 64, half = lane / 32;
    const int head = kv_head * kGqa + wave % kGqa;
    const int q_first = tile * kQueries + wave / kGqa * 32, q_at = q_first + lane % 32;
    const int key_tiles = (min(tile * kQueries + kQueries, seq) + kKeyTile - 1) / kKeyTile;
    const unsigned char *const key_src = (const unsigned char *)(keys + ((size_t)batch * KVH + kv_head) * padded * D);
    const unsigned char *const value_src = (const unsigned char *)(values_t + ((size_t)batch * KVH + kv_head) * D * padded);

    auto request = [&](int t, int buffer) {
#pragma unroll
        for (int i = 0; i < kPieces / kThreads; i++) {
            const int wave_at = i * kThreads + wave * 64, at = wave_at + lane;
            const int row = at / kKeyPieces, piece = (at % kKeyPieces) ^ (kKeyPieces == 8 ? (row >> 1) & 7 : row & 15);
            load_to_lds(key_src + ((size_t)t * kKeyTile + row) * (D * 2) + piece * 16, (MK_LDS void *)&lds[buffer][0][wave_at * 16]);
            const int vrow = at / 8, vpiece = (at % 8) ^ ((vrow >> 1) & 7);
            load_to_lds(value_src + (size_t)vrow * padded * 2 + (size_t)t * (kKeyTile * 2) + vpiece * 16, (MK_LDS void *)&lds[buffer][1][wave_at * 16]);
        }
    };
    request(0, 0);

    bf16x8 query[kDepthSteps];
    {
        const uint16_t *const src = q + (((size_t)batch * seq + min(q_at, seq - 1)) * H + head) * D + half * 8;
#pragma unroll
        for (int i = 0; i < kDepthSteps; i++) query[i] = *(const bf16x8 *)(src + i * 16);
    }
    f32x16 acc[kOutTiles];
#pragma unroll
    for (int i = 0; i < kOutTiles; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][r] = 0.0f;
    float maximum = -INFINITY, sum = 0.0f;

    for (int t = 0; t < key_tiles; t++) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (t + 1 < key_tiles) request(t + 1, (t + 1) & 1);
        if (t * kKeyTile > q_first + 31) continue;  // wholly above the diagonal for this wave
        const unsigned char *const key_tile = lds[t & 1][0], *const value_tile = lds[t & 1][1];

        f32x16 score[2];
#pragma unroll
        for (int sub = 0; sub < 2; sub++) {
#pragma unroll
            for (int r = 0; r < 16; r++) score[sub][r] = 0.0f;
            const int row = sub * 32 + lane % 32, swizzle = kKeyPieces == 8 ? (row >> 1) & 7 : row & 15;
#pragma unroll
            for (int i = 0; i < kDepthSteps; i++) {
                const bf16x8 key = *(const bf16x8 *)(key_tile + row * (D * 2) + ((2 * i + half) ^ swizzle) * 16);
                score[sub] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(key, query[i], score[sub], 0, 0, 0);
            }
        }
        if (t * kKeyTile + kKeyTile - 1 > q_first) {
#pragma unroll
            for (int sub = 0; sub < 2; sub++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int key_at = t * kKeyTile + sub * 32 + 8 * (r / 4) + 4 * half + r % 4;
                    if (key_at > q_at) score[sub][r] = -INFINITY;
                }
        }
        float tile_max = score[0][0];
#pragma unroll
        for (int sub = 0; sub < 2; sub++)
#pragma unroll
            for (int r = 0; r < 16; r++) tile_max = fmaxf(tile_max, score[sub][r]);
        const float next = fmaxf(maximum, half_exchange_max(tile_max));
        if (__any(next > maximum)) {
            const float shrink = exp2f((maximum - next) * scale);
            sum *= shrink;
#pragma unroll
            for (int i = 0; i < kOutTiles; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][r] *= shrink;
            maximum = next;
        }
        const float offset = maximum * scale;
        uint32_t prob[2][8];
#pragma unroll
        for (int sub = 0; sub < 2; sub++)
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const float a = __builtin_amdgcn_exp2f(fmaf(score[sub][r], scale, -offset));
                const float b = __builtin_amdgcn_exp2f(fmaf(score[sub][r + 1], scale, -offset));
                sum += a;
                sum += b;
                prob[sub][r / 2] = pack_bf16(a, b);
            }
#pragma unroll
        for (int step = 0; step < 4; step++) {
            const u32x4 words = {prob[step / 2][step % 2 * 4], prob[step / 2][step % 2 * 4 + 1], prob[step / 2][step % 2 * 4 + 2],
                                 prob[step / 2][step % 2 * 4 + 3]};
            const bf16x8 p = __builtin_bit_cast(bf16x8, words);
#pragma unroll
            for (int i = 0; i < kOutTiles; i++) {
                const int row = i * 32 + lane % 32;
                const bf16x8 value = *(const bf16x8 *)(value_tile + row * (kKeyTile * 2) + ((2 * step + half) ^ ((row >> 1) & 7)) * 16);
                acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(value, p, acc[i], 0, 0, 0);
            }
        }
    }
    if (q_at >= seq) return;
    const float inverse = 1.0f / half_exchange_sum(sum);
    uint16_t *const dst = out + (((size_t)batch * seq + q_at) * H + head) * D;
#pragma unroll
    for (int i = 0; i < kOutTiles; i++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const u32x2 pairs = {pack_bf16(acc[i][4 * g] * inverse, acc[i][4 * g + 1] * inverse),
                                 pack_bf16(acc[i][4 * g + 2] * inverse, acc[i][4 * g + 3] * inverse)};
            *(u32x2 *)(dst + i * 32 + 8 * g + 4 * half) = pairs;
        }
}

// ---------------------------------------------------------------------------------------------
// SiLU(gate) * up, with the gate's activation narrowed to bf16 before the product.  Bound by memory.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ float silu(float g) { return g / (1.0f + expf(-g)); }

__global__ __launch_bounds__(256) void silu_mul_kernel(size_t pieces, const uint16_t *gate, const uint16_t *up, uint16_t *out) {
    const size_t at = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (at >= pieces) return;
    const u32x4 g = *(const u32x4 *)(gate + at * 8), u = *(const u32x4 *)(up + at * 8);
    u32x4 o;
#pragma unroll
    for (int j = 0; j < 4; j++)
        o[j] = pack_bf16(round_bf16(silu(bf16_lo(g[j]))) * bf16_lo(u[j]), round_bf16(silu(bf16_hi(g[j]))) * bf16_hi(u[j]));
    *(u32x4 *)(out + at * 8) = o;
}

// ---------------------------------------------------------------------------------------------
// First maximum of every row of logits: the row's values as integers that order like the values, a NaN
// above everything, with the complement of the index below them, so that the largest key is the answer.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t order_bits(uint32_t bf16) {
    if ((bf16 & 0x7fffu) > 0x7f80u) return 0xffffu;
    if (bf16 == 0x8000u) bf16 = 0;  // minus zero equals zero
    return (bf16 & 0x8000u) ? ~bf16 & 0xffffu : bf16 | 0x8000u;
}

// the block's largest key to ids[blockIdx.x], as an index
template <int THREADS>
__device__ __forceinline__ void write_best(uint64_t best, int64_t *ids) {
#pragma unroll
    for (int offset = 32; offset >= 1; offset /= 2) {
        const uint64_t other = __shfl_xor(best, offset);
        best = other > best ? other : best;
    }
    __shared__ uint64_t of_wave[THREADS / 64];
    if (threadIdx.x % 64 == 0) of_wave[threadIdx.x / 64] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < THREADS / 64; w++) best = of_wave[w] > best ? of_wave[w] : best;
        ids[blockIdx.x] = (int64_t)(uint32_t)~(uint32_t)best;
    }
}

__global__ __launch_bounds__(1024) void argmax_kernel(int vocab, const uint16_t *logits, int64_t *ids) {
    const uint16_t *const row = logits + (size_t)blockIdx.x * vocab;
    uint64_t best = 0;
    for (int at = (int)threadIdx.x; at < vocab / 8; at += 1024) {
        const u32x4 v = *(const u32x4 *)(row + (size_t)at * 8);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint64_t key = (uint64_t)order_bits((v[j / 2] >> (j % 2 * 16)) & 0xffffu) << 32 | (uint32_t)~(uint32_t)(at * 8 + j);
            best = key > best ? key : best;
        }
    }
    write_best<1024>(best, ids);
}

#include "mk_prefill_rows.h"
#include "mk_prefill_tiles.h"
#include "mk_prefill_wide.h"

// ---------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------
thread_local char g_error[256];

int fail(int code, const char *format, ...) {
    va_list args;
    va_start(args, format);
    vsnprintf(g_error, sizeof g_error, format, args);
    va_end(args);
    return code;
}
int launched(const char *what) {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : fail(-5, "%s: %s", what, hipGetErrorString(e));
}
int check_shape(const mk_prefill_shape *s) {
    if (!s) return fail(-1, "no shape");
    if (s->batch < 1 || s->seq < 1 || s->batch > 65535 || (int64_t)s->batch * s->seq > (1 << 22)) return fail(-2, "batch %d x seq %d", s->batch, s->seq);
    if (s->head_dim != 64 && s->head_dim != 128) return fail(-2, "head_dim %d: 64 or 128", s->head_dim);
    if (s->num_kv_heads < 1 || s->num_attention_heads != 4 * s->num_kv_heads) return fail(-2, "four query heads per KV head");
    if (s->hidden_size < 8 || s->hidden_size % 8 || s->hidden_size > kMaxHidden) return fail(-2, "hidden_size %d", s->hidden_size);
    if (s->intermediate_size < 8 || s->intermediate_size % 8) return fail(-2, "intermediate_size %d", s->intermediate_size);
    if (s->vocab_size < 8 || s->vocab_size % 8) return fail(-2, "vocab_size %d", s->vocab_size);
    if (s->kv_max_len < 1 || s->rope_positions < 1) return fail(-2, "empty cache or rope table");
    return 0;
}
template <typename... P>
int check(const mk_prefill_shape *s, const P *...pointers) {
    if (int rc = check_shape(s)) return rc;
    return (... && pointers) ? 0 : fail(-2, "null device pointer");
}
int padded_seq(int seq) { return (seq + kPosTile - 1) / kPosTile * kPosTile; }

template <int D>
int launch_attention(const mk_prefill_shape &s, const uint16_t *q, const uint16_t *keys, const uint16_t *values_t, uint16_t *out, hipStream_t stream) {
    const float scale = 1.44269504088896341f / sqrtf((float)D);
    const int padded = padded_seq(s.seq);
    // Eight waves share a tile's loads among 64 positions; four leave twice as many blocks, which matters while there are
    // fewer than two blocks of eight per CU.  32 heads of 64, four and eight waves, us: 512 positions (64 blocks of eight)
    // 10.9 and 14.5, 2048 (256) 33.6 and 44.3, 3500 (440) 76.5 and 75.1, 6000 (752) 198 and 192, 8192 (1024) 347 and 359;
    // heads of 128: 2048 53 and 65, 3500 144 and 137, 6000 344 and 351, 8192 606 and 592.
    if ((int64_t)s.batch * s.num_kv_heads * ((s.seq + 63) / 64) >= 512) {
        const dim3 grid((s.seq + 63) / 64 * s.num_kv_heads, s.batch);
        attention_kernel<D, 8><<<grid, 512, 0, stream>>>(s, padded, scale, q, keys, values_t, out);
    } else {
        const dim3 grid((s.seq + 31) / 32 * s.num_kv_heads, s.batch);
        attention_kernel<D, 4><<<grid, 256, 0, stream>>>(s, padded, scale, q, keys, values_t, out);
    }
    return launched("attention");
}

// ---- few rows: the whole forward, products included ----

// Blocks over which K is split.  A block reads all of X's rows once per column tile, so with a long K the 128 blocks of a
// 2048-wide product spend their time on X: 32 rows, K = 8192: 16.4 us whole, 12.2 us as two tiles a block and K in four.
// The blocks' meeting costs 3 us, too much for a short K (K = 2048: 4.9 and 7.4).
int rows_split(int k) { return k >= 6144 ? 4 : 1; }

template <int MT, int NT, int WAVES, int STAGES, int EPI, bool NORM>
int launch_rows(const RowsArgs &a, int split, const char *what, hipStream_t stream) {
    const int width = EPI == kRowsSilu ? NT * 8 : NT * 16, bytes = RowsLds<MT, NT, WAVES, STAGES, NORM>::bytes(a.k);
    auto *kernel = a.past ? rows_kernel<MT, NT, WAVES, STAGES, EPI, NORM, true> : rows_kernel<MT, NT, WAVES, STAGES, EPI, NORM, false>;
    const hipError_t e = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return fail(-5, "%s: %d bytes of LDS: %s", what, bytes, hipGetErrorString(e));
    kernel<<<dim3((a.n + width - 1) / width, split), WAVES * 64, bytes, stream>>>(a);
    return launched(what);
}
// Two tiles a block of four waves.  (One stage for more than 32 rows: 60 rows 1043 us, 1023 with two.)
template <int MT, int EPI, bool NORM>
int launch_rows_wide(const RowsArgs &a, int split, const char *what, hipStream_t stream) {
    return launch_rows<MT, 2, 4, 2, EPI, NORM>(a, split, what, stream);
}
// Four tiles a block where there are enough columns (LM head, gate and up): a block reads X once, and with two tiles X's
// bytes from L2 are as many as W's from memory.  Whole forwards of the 1B layers, us, two and four tiles: 12 rows 860 and
// 843, 32 rows 925 and 898, 60 rows 1146 and 1073.  Gate and up have two where blocks of four are no more than half the CUs: whole
// forwards of eight layers, 32 rows, us, two and four tiles, 5120 columns (160 blocks of four) 342 and 331, 4096 columns 274 and
// 284, 2048 columns 189 and 203; 64 rows 442 and 415, 340 and 341, 224 and 239.
constexpr int kRowsFar = 4, kRowsFarBlocks = 129;
template <int MT, int EPI>
int launch_rows_far(const RowsArgs &a, const char *what, hipStream_t stream) {
    if constexpr (EPI == kRowsSilu)
        if ((a.n + kRowsFar * 8 - 1) / (kRowsFar * 8) < kRowsFarBlocks) return launch_rows<MT, 2, 4, MT == 4 ? 1 : 2, EPI, true>(a, 1, what, stream);
    return launch_rows<MT, kRowsFar, 4, 1, EPI, true>(a, 1, what, stream);
}
// One tile a block: where there is at most one block per CU it has eight waves, so that the CU has enough loads in flight.
// More blocks than CUs only queries, keys and values can have (above 4096 columns: heads wider than the hidden state).
template <int MT, int EPI, bool NORM>
int launch_rows_narrow(const RowsArgs &a, const char *what, hipStream_t stream) {
    if constexpr (!NORM)
        if (rows_split(a.k) > 1) return launch_rows_wide<MT, EPI, NORM>(a, rows_split(a.k), what, stream);
    if constexpr (EPI == kRowsRope)
        if (a.n / 16 > 256) return launch_rows<MT, 1, 4, 1, EPI, NORM>(a, 1, what, stream);
    return launch_rows<MT, 1, 8, MT == 4 ? 1 : 2, EPI, NORM>(a, 1, what, stream);
}
template <int NT, int EPI, bool NORM>
int launch_rows(const RowsArgs &a, const char *what, hipStream_t stream) {
    if constexpr (NT == 1) {
        if (a.rows <= 16) return launch_rows_narrow<1, EPI, NORM>(a, what, stream);
        if (a.rows <= 32) return launch_rows_narrow<2, EPI, NORM>(a, what, stream);
        return launch_rows_narrow<4, EPI, NORM>(a, what, stream);
    } else {
        if (a.rows <= 16) return launch_rows_far<1, EPI>(a, what, stream);
        if (a.rows <= 32) return launch_rows_far<2, EPI>(a, what, stream);
        return launch_rows_far<4, EPI>(a, what, stream);
    }
}

// Weights that one forward uses once go past the caches, unless the last-level cache (256 MiB) holds about all of the model's, for
// the next forward.  Whole forwards, 32 rows, us, through the caches and past them: the 1B architecture (2.5 GB) 896 and 865, 1024
// wide with ten layers (371 MB) 336 and 327, eight (310 MB) 279 and 272, seven (280 MB) 238 and 240, five (219 MB) 157 and 179.
constexpr int64_t kRowsCached = 280 << 20;
bool rows_past(const mk_prefill_shape &s, int layers) {
    const int64_t heads = (int64_t)s.num_attention_heads * s.head_dim, kv = (int64_t)s.num_kv_heads * s.head_dim;
    return 2 * s.hidden_size * (layers * (2 * heads + 2 * kv + 3ll * s.intermediate_size) + s.vocab_size) > kRowsCached;
}

// the workspace of the forward for few rows, in elements of 2 bytes; every part a multiple of 16 bytes
struct RowsWorkspace {
    size_t q, attn, prod, keys, values_t, arrived, best, partial, total;  // values_t and arrived: zero at the start
    explicit RowsWorkspace(const mk_prefill_shape &s) {
        const size_t rows = (size_t)s.batch * s.seq, heads = rows * s.num_attention_heads * s.head_dim;
        const size_t kv = (size_t)s.batch * s.num_kv_heads * s.head_dim * padded_seq(s.seq);
        q = 0;
        attn = q + heads;
        prod = attn + heads;
        keys = prod + rows * s.intermediate_size;
        values_t = keys + kv;
        arrived = values_t + kv;
        best = arrived + (s.hidden_size / 32 + 3) / 4 * 4 * 2;
        partial = best + (rows * ((s.vocab_size + kRowsFar * 16 - 1) / (kRowsFar * 16)) + 1) / 2 * 2 * 4;
        const size_t sums = (rows <= 16 ? 16 : rows <= 32 ? 32 : 64) * (size_t)s.hidden_size;  // of one part of K
        const int split = max(rows_split(s.intermediate_size), rows_split(s.num_attention_heads * s.head_dim));
        total = partial + (split > 1 ? split * sums * 2 : 0);
    }
};
// Whether the whole forward is this library's, products included.  The limit of 2048 columns is none of the kernels', of
// speed or of accuracy: at 4096 columns and 32 layers these products are faster than the library's up to 512 rows (32 rows
// 3904 us and 4513, 128 rows 5547 and 7384, 512 rows 9933 and 10673; 777 rows 15522 and 14592), and either way the hidden
// states are 1.56 % of their norm from the forward without roundings.  It is there because so deep a model passes any change
// of an order of sums on to what it decodes behind the prompt: over 18 prompts of 16 to 120 tokens the decoded hidden state
// is 2.51 to 3.02 % of its norm (mean 2.88) from the plain forward's where the products are the library's, 2.83 to 3.10 %
// (mean 2.96) where they are these; the plain forward's itself is 3.1 % from the one without roundings.  The route that stays
// nearer to the plain forward is kept, by little.
// It is depth that amplifies, not width; deeper models of up to 2048 columns than 16 layers have not been measured.
bool whole_covers(const mk_prefill_shape &s) {
    return s.hidden_size <= 2048 && s.hidden_size % 64 == 0 && s.intermediate_size % 64 == 0;
}
bool rows_covers(const mk_prefill_shape &s) { return whole_covers(s) && (int64_t)s.batch * s.seq <= kRowsMax; }
// Narrow tiles alone, for what wide_covers leaves: from some thousand rows on the library's products are the faster ones.  Whole
// forwards of eight layers, intermediate size four times the width, vocabulary 32768, library's products and tiles, us:
//   2048 wide: 512 rows 1237 and 1176, 768 rows 1542 and 1555, 1024 rows 1808 and 1712, 1536 rows 2291 and 2567
//   1024 wide: 1024 rows 1130 and 889, 2048 rows 1471 and 1365, 3000 rows 1886 and 1950, 4096 rows 2308 and 2430
//    512 wide: 2048 rows 1150 and 866, 3000 rows 1268 and 1282, 4096 rows 1564 and 1536, 8192 rows 2664 and 2885
//    256 wide: 2048 rows 1131 and 672, 4096 rows 1187 and 1180, 8192 rows 2016 and 2215
//     64 wide: 4096 rows 1129 and 981, 8192 rows 1636 and 1782, 32768 rows 7208 and 8451
bool tiles_cover(const mk_prefill_shape &s) {
    const int64_t rows = (int64_t)s.batch * s.seq;
    return whole_covers(s) && rows <= 4096 && rows * s.hidden_size <= 1 << 21;
}
// Wide tiles (mk_prefill_wide.h) beside the narrower ones.  Whole forwards, us, narrow tiles or the library's products, and wide:
//   1B architecture: 253 rows 1752 and 1752, 320 rows 2132 and 2034, 777 rows 2971 and 2829, 1024 rows 3325 and 3191 (tiles);
//     1100 rows 4343 and 4100, 1500 rows 4782 and 4601, 2048 rows 5879 and 5329, 4096 rows 10982 and 10181 (library)
//   8B architecture: 520 rows 11889 and 11437, 640 rows 12608 and 12239, 777 rows 15119 and 13540, 2048 rows 28328 and 26686,
//     2300 rows 31529 and 34397, 2600 rows 44288 and 38257, 3000 rows 41329 and 43537, 4096 rows 53581 and 54067 (library)
// Prompts of up to 512 rows of wide models are the library's for the reason above.
// The lines for other widths, from whole forwards of four or eight layers with vocabularies of 32768, us, library's products (or
// narrow tiles, up to 2^21 values of a narrow model) and wide.  Which one wins depends on how the rounds of both fit:
//   up to 2048 wide: 512 wide 4096 rows 1528 and 1386, 1024 wide 2049 rows 1624 and 1444, 1536 wide 2300 rows 2405 and 2442, 4096
//     rows 3866 and 3444.  Beyond 4096 rows 2048 wide 5000 rows 6572 and 6392, 8192 rows 10414 and 10181: not crossed, but not
//     looked at for narrower models or the whole architecture.
//   2049 to 3071 wide: 2304 wide 560 rows 1751 and 1521, 1024 rows 2445 and 2311, but 1300 rows 2591 and 2811, 1536 rows 2922 and
//     3110; 2560 wide 700 rows 2124 and 2021, but 1100 rows 2599 and 2876
//   3072 to 4096 wide: 3072 wide 513 rows 1842 and 1648, 1300 rows 3113 and 3073, 2048 rows 3969 and 3855; 3584 wide 513 rows 1635 and
//     1578, 2048 rows 5236 and 3773; the worst of 60 sizes 3840 wide, 1100 rows, 1.07 times the library's
//   wider: 5120 wide 650 rows 2152 and 2006, 1024 rows 2802 and 2681, but 1650 rows 4275 and 4717; 6144 wide 560 rows 3521 and 3040,
//     but 2048 rows 8005 and 8422; 7168 wide 560 rows 3237 and 3509 (five row tiles fill five eighths of the chip), 777 rows 4660 and
//     3984, but 1400 rows 5965 and 6993; 8192 wide 560 rows 4447 and 4574, 777 rows 6070 and 5707, but 1536 rows 9203 and 10004
bool wide_covers(const mk_prefill_shape &s) {
    const int64_t rows = (int64_t)s.batch * s.seq;
    const int hid = s.hidden_size;
    const int least = hid <= 2048 ? 257 : hid <= 6144 ? 513 : 641, most = hid <= 2048 ? 4096 : hid >= 3072 && hid <= 4096 ? 2048 : 1024;
    return hid % 64 == 0 && s.intermediate_size % 64 == 0 && hid >= 256 && rows >= least && rows <= most
        && (int64_t)s.batch * s.kv_max_len < INT32_MAX
        // (offsets of 32 bits within a tile's rows, of K as of the columns)
        && s.intermediate_size <= kWideMostColumns && s.num_kv_heads <= 1 << 10;
}

// ---- more rows: tiles, narrow and wide ----

// The shapes a product can be tiled in, with what a stage of 64 elements of K takes (us, measured with as many blocks as
// there are slots) and how many blocks the chip holds at once.
struct TileShape {
    int rows, columns, slots;
    float stage_us;
};
constexpr TileShape kTileShapes[] = {
    {64, 128, 256, 0.42f},   // four stages in LDS: the least time for one tile
    {128, 128, 256, 0.62f},  // four stages
    {128, 128, 512, 1.05f},  // two stages, two blocks a CU
    {256, 256, 256, 1.40f},  // square_kernel: the most work per byte of LDS
    {128, 256, 256, 0.84f},  // flat_kernel
};
constexpr int kSquare = 3, kFlat = 4, kWideLeastK = 4 * kTileK;
struct TilePlan {
    int shape, split, m_tiles, n_tiles;
    float us;
};
// The plan with the least estimated time: rounds of blocks, 3 us to start and end, and for a split of K the blocks' meeting
// and their sums' way through memory.  (rows 253: 2048 x 8192 estimated 25, measured 24.3 in 64 x 128 x 4 parts against
// 52.9 whole; rows 777: 16384 x 2048 estimated 48, measured 51.4 in 256 x 256.)  Rounds are those of the XCD with the most
// column tiles, as column tile n is XCD n % 8's: 12 of them are two for four XCDs and one for the others.  (Counted over the
// whole chip, plans were chosen that took a round more: whole forwards of eight layers, us, 1536 wide 2300 rows 2763 -> 2442,
// 2304 wide 560 rows 1744 -> 1521, 2048 wide 2300 rows 3317 -> 3220.)  The residual epilogue has no 256 x 256: its products are
// narrow, and 128 x 256 fills the chip twice as soon.
TilePlan tile_plan(TileEpilogue epilogue, int rows, int n, int k, bool wide) {
    const int columns = epilogue == kTileSilu ? 2 * n : n;
    const bool whole = epilogue == kTileSilu || epilogue == kTileArgmax;  // no split of K
    TilePlan best{};
    for (int shape = 0; shape <= (wide ? kFlat : kSquare); shape++) {
        const TileShape &t = kTileShapes[shape];
        if ((shape == kSquare && epilogue == kTileResidual) || (shape >= kSquare && k < kWideLeastK)) continue;
        // (a product of more columns reaches this without wide_covers, too)
        if (shape == kSquare && epilogue == kTileSilu && n > kWideMostColumns) continue;
        const int m_tiles = (rows + t.rows - 1) / t.rows, n_tiles = (columns + t.columns - 1) / t.columns, stages = k / kTileK;
        for (int split = 1; split <= 8; split *= 2) {
            if (split > 1 && (whole || stages / split < 8 || shape == kSquare)) break;
            const int64_t tiles = (int64_t)((n_tiles + 7) / 8) * m_tiles * split, slots = t.slots / 8;  // of the fullest XCD
            const int64_t rounds = (tiles + slots - 1) / slots;
            // more sums than fit one round of blocks cost more than the estimate (3000 rows of an 8B model's layers)
            if (wide && split > 1 && rounds > 1) break;
            const float meeting = split > 1 ? 3.0f + (float)split * rows * columns * 8 / 3e6f : 0.0f;
            float full = (float)rounds;
            // halves of tiles in a last round that they fit, which square_kernel has but for rotation
            if (wide && shape == kSquare && epilogue != kTileRope && tiles % slots && tiles % slots <= slots / 2) full -= 0.35f;
            const float us = full * ((stages + split - 1) / split) * t.stage_us + 3.0f + meeting;
            if (best.split == 0 || us < best.us) best = {shape, split, m_tiles, n_tiles, us};
        }
    }
    return best;
}
// the five products of a layer and of the head
struct Plans {
    TilePlan qkv, o, up, down, head;
    explicit Plans(const mk_prefill_shape &s) {
        const bool wide = wide_covers(s);
        const int rows = s.batch * s.seq, heads = s.num_attention_heads * s.head_dim, kv = s.num_kv_heads * s.head_dim;
        qkv = tile_plan(kTileRope, rows, heads + 2 * kv, s.hidden_size, wide);
        o = tile_plan(kTileResidual, rows, s.hidden_size, heads, wide);
        up = tile_plan(kTileSilu, rows, s.intermediate_size, s.hidden_size, wide);
        down = tile_plan(kTileResidual, rows, s.hidden_size, s.intermediate_size, wide);
        head = tile_plan(kTileArgmax, rows, s.vocab_size, s.hidden_size, wide);
    }
    int get(int product, int32_t plan[4]) const {
        if (product < 0 || product > 4) return fail(-2, "product %d", product);
        const TilePlan &p = (&qkv)[product];
        plan[0] = p.shape, plan[1] = kTileShapes[p.shape].rows, plan[2] = kTileShapes[p.shape].columns, plan[3] = p.split;
        return 0;
    }
};

template <typename Kernel>
int launch_lds(Kernel *kernel, dim3 grid, int threads, int bytes, const TileArgs &a, const char *what, hipStream_t stream) {
    const hipError_t e = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return fail(-5, "%s: %d bytes of LDS: %s", what, bytes, hipGetErrorString(e));
    kernel<<<grid, threads, bytes, stream>>>(a);
    return launched(what);
}
template <int WN, int MT, int STAGES, int EPI>
int launch_tiles(const TileArgs &a, dim3 grid, const char *what, hipStream_t stream) {
    return launch_lds(tile_kernel<WN, MT, 2, STAGES, EPI>, grid, WN * 128, STAGES * (MT * 64 + WN * 64) * kTileK * 2, a, what, stream);
}
template <int EPI>
int launch_tiles(const TileArgs &a, const TilePlan &plan, const char *what, hipStream_t stream) {
    const dim3 grid(8 * ((plan.n_tiles + 7) / 8) * plan.m_tiles, plan.split);
    switch (plan.shape) {
    case 0: return launch_tiles<2, 1, 4, EPI>(a, grid, what, stream);
    case 1: return launch_tiles<2, 2, 4, EPI>(a, grid, what, stream);
    case 2: return launch_tiles<2, 2, 2, EPI>(a, grid, what, stream);
    case kFlat: return launch_lds(flat_kernel<EPI>, grid, 512, kFlatBytes, a, what, stream);
    }
    if constexpr (EPI != kTileResidual) return launch_lds(square_kernel<EPI>, dim3(256), 512, kSquareBytes, a, what, stream);
    else return fail(-2, "%s: no such tiles", what);
}

// The workspace, in elements of 2 bytes, as in RowsWorkspace.
struct TilesWorkspace {
    size_t x, q, attn, prod, keys, values_t, arrived, best, partial, total;
    TilesWorkspace(const mk_prefill_shape &s, const Plans &plans) {
        const size_t rows = (size_t)s.batch * s.seq, heads = rows * s.num_attention_heads * s.head_dim;
        const size_t kv = (size_t)s.batch * s.num_kv_heads * s.head_dim * padded_seq(s.seq);
        x = 0;
        q = x + rows * s.hidden_size;
        attn = q + heads;
        prod = attn + heads;
        keys = prod + rows * s.intermediate_size;
        values_t = keys + kv;
        arrived = values_t + kv;
        size_t counters = 0, sums = 0;
        for (const TilePlan &plan : {plans.qkv, plans.o, plans.down}) {
            if (plan.split == 1) continue;
            const size_t tiles = (size_t)plan.m_tiles * plan.n_tiles;
            counters = max(counters, tiles);
            sums = max(sums, tiles * plan.split * kTileShapes[plan.shape].rows * kTileShapes[plan.shape].columns);
        }
        best = arrived + (counters + 3) / 4 * 4 * 2;
        partial = best + ((s.vocab_size + 255) / 256 * 4 * rows + 1) / 2 * 2 * 4;
        total = partial + sums * 2;
    }
};

__global__ __launch_bounds__(256) void zero_kernel(u32x4 *dst, int pieces) {
    for (int i = blockIdx.x * 256 + threadIdx.x; i < pieces; i += gridDim.x * 256) dst[i] = u32x4{0, 0, 0, 0};
}

int rows_forward(const mk_prefill_shape &s, const mk_prefill_model &w, const int64_t *ids, const int64_t *positions, uint16_t *h,
                 uint16_t *workspace, int64_t *out_ids, hipStream_t stream);
int tiles_forward(const mk_prefill_shape &s, const mk_prefill_model &w, const Plans &plans, const int64_t *ids, const int64_t *positions,
                  uint16_t *h, uint16_t *workspace, int64_t *out_ids, hipStream_t stream);

int check_model(const mk_prefill_shape *shape, const mk_prefill_model *model, const int64_t *ids, const int64_t *positions, const uint16_t *h,
                const uint16_t *workspace, const int64_t *out_ids) {
    if (int rc = check(shape, ids, positions, h, workspace, out_ids)) return rc;
    if (!model) return fail(-1, "no model");
    const mk_prefill_model &m = *model;
    if (int rc = check(shape, m.embed, m.attn_norm, m.qkv, m.o, m.mlp_norm, m.gate, m.up, m.down, m.final_norm, m.head, m.rope_cos, m.rope_sin, m.k_cache, m.v_cache)) return rc;
    if (m.num_layers < 1 || m.cache_batch < shape->batch) return fail(-2, "no layers, or a cache of fewer sequences than the call");
    return 0;
}

}  // namespace

extern "C" {

int64_t mk_prefill_workspace_bytes(const mk_prefill_shape *shape) {
    if (int rc = check_shape(shape)) return rc;
    if (rows_covers(*shape)) return (int64_t)RowsWorkspace(*shape).total * 2;
    return wide_covers(*shape) || tiles_cover(*shape) ? (int64_t)TilesWorkspace(*shape, Plans(*shape)).total * 2 : 0;
}

int mk_prefill_forward(const mk_prefill_shape *shape, const mk_prefill_model *model, const int64_t *ids, const int64_t *positions,
                       uint16_t *h, uint16_t *workspace, int64_t *out_ids, void *stream) {
    if (int rc = check_model(shape, model, ids, positions, h, workspace, out_ids)) return rc;
    if (rows_covers(*shape)) return rows_forward(*shape, *model, ids, positions, h, workspace, out_ids, (hipStream_t)stream);
    if (wide_covers(*shape) || tiles_cover(*shape)) return tiles_forward(*shape, *model, Plans(*shape), ids, positions, h, workspace, out_ids, (hipStream_t)stream);
    return fail(-2, "%d x %d rows of %d, %d: not a call that the whole forward takes", shape->batch, shape->seq, shape->hidden_size, shape->intermediate_size);
}

int mk_prefill_tile_plan(const mk_prefill_shape *shape, int product, int32_t plan[4]) {
    if (int rc = check(shape, plan)) return rc;
    if (rows_covers(*shape) || !(wide_covers(*shape) || tiles_cover(*shape)))
        return fail(-2, "%d x %d rows of %d: not tiled", shape->batch, shape->seq, shape->hidden_size);
    return Plans(*shape).get(product, plan);
}

int64_t mk_prefill_wide_workspace_bytes(const mk_prefill_shape *shape) {
    if (int rc = check_shape(shape)) return rc;
    return wide_covers(*shape) ? mk_prefill_workspace_bytes(shape) : 0;
}

int mk_prefill_wide_forward(const mk_prefill_shape *shape, const mk_prefill_model *model, const int64_t *ids, const int64_t *positions,
                            uint16_t *h, uint16_t *workspace, int64_t *out_ids, void *stream) {
    if (int rc = check_shape(shape)) return rc;
    if (!wide_covers(*shape)) return fail(-2, "%d x %d rows of %d, %d: not a call of wide tiles", shape->batch, shape->seq, shape->hidden_size, shape->intermediate_size);
    return mk_prefill_forward(shape, model, ids, positions, h, workspace, out_ids, stream);
}

int mk_prefill_wide_plan(const mk_prefill_shape *shape, int product, int32_t plan[4]) {
    if (int rc = check(shape, plan)) return rc;
    if (!wide_covers(*shape)) return fail(-2, "%d x %d rows of %d: no wide tiles", shape->batch, shape->seq, shape->hidden_size);
    return mk_prefill_tile_plan(shape, product, plan);
}

int mk_prefill_padded_seq(int seq) { return padded_seq(seq); }

int mk_prefill_embed(const mk_prefill_shape *shape, const int64_t *ids, const int64_t *positions, const uint16_t *embed,
                     const uint16_t *norm_weight, uint16_t *h, uint16_t *x, void *stream) {
    if (int rc = check(shape, ids, positions, embed, norm_weight, h, x)) return rc;
    norm_kernel<kNormEmbed><<<shape->batch * shape->seq, kNormThreads, 0, (hipStream_t)stream>>>(*shape, ids, positions, embed, norm_weight, h, x);
    return launched("embed");
}

int mk_prefill_add_norm(const mk_prefill_shape *shape, const uint16_t *y, const uint16_t *norm_weight, uint16_t *h, uint16_t *x, void *stream) {
    if (int rc = check(shape, y, norm_weight, h, x)) return rc;
    norm_kernel<kNormAdd><<<shape->batch * shape->seq, kNormThreads, 0, (hipStream_t)stream>>>(*shape, nullptr, nullptr, y, norm_weight, h, x);
    return launched("add_norm");
}

int mk_prefill_rope(const mk_prefill_shape *shape, const uint16_t *qkv, const int64_t *positions, const float *rope_cos,
                    const float *rope_sin, uint16_t *k_cache, uint16_t *v_cache, uint16_t *q, uint16_t *keys,
                    uint16_t *values_t, void *stream) {
    if (int rc = check(shape, qkv, positions, rope_cos, rope_sin, k_cache, v_cache, q, keys, values_t)) return rc;
    const int padded = padded_seq(shape->seq);
    const dim3 grid(padded / kPosTile, shape->num_attention_heads + 2 * shape->num_kv_heads, shape->batch);
    auto *kernel = shape->head_dim == 64 ? rope_kernel<64> : rope_kernel<128>;
    kernel<<<grid, 256, 0, (hipStream_t)stream>>>(*shape, padded, qkv, positions, rope_cos, rope_sin, k_cache, v_cache, q, keys, values_t);
    return launched("rope");
}

int mk_prefill_attention(const mk_prefill_shape *shape, const uint16_t *q, const uint16_t *keys, const uint16_t *values_t,
                         uint16_t *out, void *stream) {
    if (int rc = check(shape, q, keys, values_t, out)) return rc;
    return shape->head_dim == 64 ? launch_attention<64>(*shape, q, keys, values_t, out, (hipStream_t)stream)
                                 : launch_attention<128>(*shape, q, keys, values_t, out, (hipStream_t)stream);
}

int mk_prefill_silu_mul(const mk_prefill_shape *shape, const uint16_t *gate, const uint16_t *up, uint16_t *out, void *stream) {
    if (int rc = check(shape, gate, up, out)) return rc;
    const size_t pieces = (size_t)shape->batch * shape->seq * shape->intermediate_size / 8;
    silu_mul_kernel<<<(unsigned)((pieces + 255) / 256), 256, 0, (hipStream_t)stream>>>(pieces, gate, up, out);
    return launched("silu_mul");
}

int mk_prefill_argmax(const mk_prefill_shape *shape, const uint16_t *logits, int64_t *ids, void *stream) {
    if (int rc = check(shape, logits, ids)) return rc;
    argmax_kernel<<<shape->batch * shape->seq, 1024, 0, (hipStream_t)stream>>>(shape->vocab_size, logits, ids);
    return launched("argmax");
}

const char *mk_prefill_last_error(void) { return g_error; }

}  // extern "C"

namespace {

int rows_forward(const mk_prefill_shape &s, const mk_prefill_model &w, const int64_t *ids, const int64_t *positions, uint16_t *h,
                 uint16_t *workspace, int64_t *out_ids, hipStream_t stream) {
    const RowsWorkspace at(s);
    const int rows = s.batch * s.seq, H = s.num_attention_heads, KVH = s.num_kv_heads, D = s.head_dim, hid = s.hidden_size, inter = s.intermediate_size;
    uint16_t *const q = workspace + at.q, *const attn = workspace + at.attn, *const prod = workspace + at.prod;
    uint16_t *const keys = workspace + at.keys, *const values_t = workspace + at.values_t;
    uint64_t *const best = (uint64_t *)(workspace + at.best);

    const int value_pieces = (int)((at.best - at.values_t) / 8);  // with the arrivals behind them
    rows_embed_kernel<<<rows + (value_pieces + 1023) / 1024, 256, 0, stream>>>(s, rows, ids, positions, w.embed, h, (u32x4 *)values_t, value_pieces);
    if (int rc = launched("embed")) return rc;

    RowsArgs base{};
    base.s = s, base.rows = rows, base.padded = padded_seq(s.seq), base.positions = positions, base.past = rows_past(s, w.num_layers);
    base.rope_cos = w.rope_cos, base.rope_sin = w.rope_sin, base.keys = keys, base.values_t = values_t, base.best = best;
    base.arrived = (int *)(workspace + at.arrived), base.partial = (float *)(workspace + at.partial);
    const size_t qkv_rows = (size_t)(H + 2 * KVH) * D, cache_layer = (size_t)w.cache_batch * s.kv_max_len * KVH * D;
    for (int layer = 0; layer < w.num_layers; layer++) {
        RowsArgs a = base;
        a.n = (int)qkv_rows, a.k = hid, a.x = h, a.norm_weight = w.attn_norm + (size_t)layer * hid, a.w0 = w.qkv + layer * qkv_rows * hid, a.out = q;
        a.k_cache = w.k_cache + layer * cache_layer, a.v_cache = w.v_cache + layer * cache_layer;
        if (int rc = launch_rows<1, kRowsRope, true>(a, "qkv", stream)) return rc;
        if (int rc = mk_prefill_attention(&s, q, keys, values_t, attn, stream)) return rc;
        a = base;
        a.n = hid, a.k = H * D, a.x = attn, a.w0 = w.o + (size_t)layer * hid * H * D, a.out = h;
        if (int rc = launch_rows<1, kRowsResidual, false>(a, "o", stream)) return rc;
        a = base;
        a.n = inter, a.k = hid, a.x = h, a.norm_weight = w.mlp_norm + (size_t)layer * hid, a.out = prod;
        a.w0 = w.gate + (size_t)layer * inter * hid, a.w1 = w.up + (size_t)layer * inter * hid;
        if (int rc = launch_rows<kRowsFar, kRowsSilu, true>(a, "gate and up", stream)) return rc;
        a = base;
        a.n = hid, a.k = inter, a.x = prod, a.w0 = w.down + (size_t)layer * hid * inter, a.out = h;
        if (int rc = launch_rows<1, kRowsResidual, false>(a, "down", stream)) return rc;
    }
    RowsArgs a = base;
    a.n = s.vocab_size, a.k = hid, a.x = h, a.norm_weight = w.final_norm, a.w0 = w.head;
    if (int rc = launch_rows<kRowsFar, kRowsArgmax, true>(a, "head", stream)) return rc;
    rows_best_kernel<<<rows, 256, 0, stream>>>((s.vocab_size + kRowsFar * 16 - 1) / (kRowsFar * 16), best, out_ids);
    return launched("best");
}

int tiles_forward(const mk_prefill_shape &s, const mk_prefill_model &w, const Plans &plans, const int64_t *ids, const int64_t *positions,
                  uint16_t *h, uint16_t *workspace, int64_t *out_ids, hipStream_t stream) {
    const TilesWorkspace at(s, plans);
    const int rows = s.batch * s.seq, H = s.num_attention_heads, KVH = s.num_kv_heads, D = s.head_dim, hid = s.hidden_size, inter = s.intermediate_size;
    uint16_t *const x = workspace + at.x, *const q = workspace + at.q, *const attn = workspace + at.attn, *const prod = workspace + at.prod;
    uint16_t *const keys = workspace + at.keys, *const values_t = workspace + at.values_t;
    uint64_t *const best = (uint64_t *)(workspace + at.best);

    const int pieces = (int)((at.best - at.values_t) / 8);  // the padding of the values, and the arrivals
    zero_kernel<<<min((pieces + 1023) / 1024, 1024), 256, 0, stream>>>((u32x4 *)values_t, pieces);
    if (int rc = launched("zero")) return rc;
    if (int rc = mk_prefill_embed(&s, ids, positions, w.embed, w.attn_norm, h, x, stream)) return rc;

    TileArgs base{};
    base.s = s, base.rows = rows, base.padded = padded_seq(s.seq), base.positions = positions;
    base.rope_cos = w.rope_cos, base.rope_sin = w.rope_sin, base.keys = keys, base.values_t = values_t, base.best = best;
    base.arrived = (int *)(workspace + at.arrived), base.partial = (float *)(workspace + at.partial);
    const size_t qkv_rows = (size_t)(H + 2 * KVH) * D, cache_layer = (size_t)w.cache_batch * s.kv_max_len * KVH * D;
    auto norm = [&](const uint16_t *weight) {
        norm_kernel<kNormPlain><<<rows, kNormThreads, 0, stream>>>(s, nullptr, nullptr, nullptr, weight, h, x);
        return launched("norm");
    };
    for (int layer = 0; layer < w.num_layers; layer++) {
        TileArgs a = base;
        a.n = (int)qkv_rows, a.k = hid, a.x = x, a.w0 = w.qkv + layer * qkv_rows * hid, a.out = q;
        a.k_cache = w.k_cache + layer * cache_layer, a.v_cache = w.v_cache + layer * cache_layer;
        if (int rc = launch_tiles<kTileRope>(a, plans.qkv, "qkv", stream)) return rc;
        if (int rc = mk_prefill_attention(&s, q, keys, values_t, attn, stream)) return rc;
        a = base;
        a.n = hid, a.k = H * D, a.x = attn, a.w0 = w.o + (size_t)layer * hid * H * D, a.out = h;
        if (int rc = launch_tiles<kTileResidual>(a, plans.o, "o", stream)) return rc;
        if (int rc = norm(w.mlp_norm + (size_t)layer * hid)) return rc;
        a = base;
        a.n = inter, a.k = hid, a.x = x, a.out = prod;
        a.w0 = w.gate + (size_t)layer * inter * hid, a.w1 = w.up + (size_t)layer * inter * hid;
        if (int rc = launch_tiles<kTileSilu>(a, plans.up, "gate and up", stream)) return rc;
        a = base;
        a.n = hid, a.k = inter, a.x = prod, a.w0 = w.down + (size_t)layer * hid * inter, a.out = h;
        if (int rc = launch_tiles<kTileResidual>(a, plans.down, "down", stream)) return rc;
        if (int rc = norm(layer + 1 == w.num_layers ? w.final_norm : w.attn_norm + (size_t)(layer + 1) * hid)) return rc;
    }
    TileArgs a = base;
    a.n = s.vocab_size, a.k = hid, a.x = x, a.w0 = w.head;
    if (int rc = launch_tiles<kTileArgmax>(a, plans.head, "head", stream)) return rc;
    tile_best_kernel<<<(rows + 15) / 16, 1024, 0, stream>>>(rows, plans.head.n_tiles * (kTileShapes[plans.head.shape].columns / 64), best, out_ids);
    return launched("best");
}

}  // namespace
