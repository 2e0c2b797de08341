// The prompt forward's matrix products for few rows (a one-line prompt): every product is a stream of its weights.
//
// With M rows a weight element is used M times, so up to some hundred rows the time is the weights' bytes over the
// memory rate plus what each launch adds.  Both ends shape the kernel below:
//   * a block owns 16 to 64 output columns and its waves split K, so that even a 2048-wide product has 128 blocks with
//     every wave's loads in flight at once.  Both operands go from memory straight into LDS in whole lines (a wave: eight
//     rows of 128 bytes), each wave into a ring of its own, so the loop has no barrier; the partial sums meet in LDS.
//     Loaded into registers in the order of v_mfma_f32_16x16x32_bf16 instead, every 16 lanes touch 16 lines and the L1
//     takes 64 clocks an instruction: 2048 x 8192 with 32 rows 27.2 us against 16.4, 8192 x 2 x 2048 21.5 against 16.3.
//   * the operations between two products are the products' own prologues and epilogues - RMS norm, rotary embedding and
//     cache append, residual add, SiLU * up, argmax - so a layer is five launches.
// The norm needs no pass of its own: sum_k W[n,k] (h_k s w_k) = s sum_k W[n,k] (h_k w_k), and every block reads all of h
// anyway, so it sums the squares on the way and scales the finished sums.  (One rounding, of h_k w_k, where the plain
// forward has two.)
// 32 rows of a 2.5 GB model: 2225 us as library products with Python launches, 860 to 870 here (its bytes at the rate of a
// copy, 4.9 TB/s: 507; at that of reads alone, 7.0 TB/s: 353).  60 rows: 1023.  More loads in flight (three or four stages,
// twice the waves) change none of it: what is left is five launches a layer, each with its start from cold.
// (Weights go past the caches there; through them, as those of a model that the last-level cache holds, 896.)
// The blocks of a product read X again and again from L2 (M * K * 2 bytes each): the reason for the limit of kRowsMax.
constexpr int kRowsMax = 64;

enum RowsEpilogue { kRowsRope, kRowsResidual, kRowsSilu, kRowsArgmax };

struct RowsArgs {
    mk_prefill_shape s;
    int rows, n, k, padded;
    bool past;                                  // whether the weights go past the caches
    const uint16_t *x, *norm_weight, *w0, *w1;  // x [rows, k]; w0 (and w1: up beside gate) [n, k]
    uint16_t *out;                              // residual: h, in place; SiLU: [rows, n]; rope: q [rows, H D]
    const int64_t *positions;
    const float *rope_cos, *rope_sin;
    uint16_t *k_cache, *v_cache, *keys, *values_t;
    uint64_t *best;                             // argmax: [rows, blocks]
    // K split over gridDim.y blocks (not with a norm): their sums, [gridDim.x, gridDim.y, NT, MT, 64] of four, and how
    // many of a column tile's blocks have arrived (zero between launches)
    float *partial;
    int *arrived;
};

__device__ __forceinline__ uint32_t order_bits(uint32_t bf16);
__device__ __forceinline__ float silu(float g);

// W row that lane `r` of the block's tile `t` holds (SiLU: the first half of the tiles are gate's, the others up's)
template <int NT, int EPI>
__device__ __forceinline__ int rows_weight_row(const RowsArgs &a, int t, int r) {
    const int first = EPI == kRowsSilu ? (blockIdx.x * (NT / 2) + t % (NT / 2)) * 16 : (blockIdx.x * NT + t) * 16, D = a.s.head_dim;
    if (EPI == kRowsRope && !a.s.interleaved && first < (a.s.num_attention_heads + a.s.num_kv_heads) * D) {
        // the two members of a rotary pair are half a head apart: eight columns of each half
        return first / D * D + first % D / 2 + (r & 7) + (r >> 3) * (D / 2);
    }
    return EPI == kRowsArgmax || EPI == kRowsSilu ? min(first + r, a.n - 1) : first + r;
}

// The fragments of COUNT tiles, 2048 bytes apart, read and waited for in one block of assembly: before an ordinary read of
// LDS the compiler waits for every load into LDS that is still in flight.
template <int COUNT>
__device__ __forceinline__ void rows_read(u32x4 (&v)[COUNT], uint32_t at) {
    static_assert(COUNT >= 2 && COUNT <= 8);
#define MK_READ(n, from, offset) "ds_read_b128 %" #n ", %" #from " offset:" #offset "\n\t"
    if constexpr (COUNT == 2)
        asm volatile(MK_READ(0, 2, 0) MK_READ(1, 2, 2048) "s_waitcnt lgkmcnt(0)" : "=&v"(v[0]), "=&v"(v[1]) : "v"(at) : "memory");
    else if constexpr (COUNT == 3)
        asm volatile(MK_READ(0, 3, 0) MK_READ(1, 3, 2048) MK_READ(2, 3, 4096) "s_waitcnt lgkmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]) : "v"(at) : "memory");
    else if constexpr (COUNT == 4)
        asm volatile(MK_READ(0, 4, 0) MK_READ(1, 4, 2048) MK_READ(2, 4, 4096) MK_READ(3, 4, 6144) "s_waitcnt lgkmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]) : "v"(at) : "memory");
    else if constexpr (COUNT == 5)
        asm volatile(MK_READ(0, 5, 0) MK_READ(1, 5, 2048) MK_READ(2, 5, 4096) MK_READ(3, 5, 6144) MK_READ(4, 5, 8192) "s_waitcnt lgkmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]) : "v"(at) : "memory");
    else if constexpr (COUNT == 6)
        asm volatile(MK_READ(0, 6, 0) MK_READ(1, 6, 2048) MK_READ(2, 6, 4096) MK_READ(3, 6, 6144) MK_READ(4, 6, 8192) MK_READ(5, 6, 10240)
                     "s_waitcnt lgkmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]) : "v"(at) : "memory");
    else
        asm volatile(MK_READ(0, 8, 0) MK_READ(1, 8, 2048) MK_READ(2, 8, 4096) MK_READ(3, 8, 6144) MK_READ(4, 8, 8192) MK_READ(5, 8, 10240)
                     MK_READ(6, 8, 12288) MK_READ(7, 8, 14336) "s_waitcnt lgkmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7]) : "v"(at) : "memory");
#undef MK_READ
}
// ... and the norm weights of the two halves of a step
__device__ __forceinline__ void rows_read_norm(u32x4 (&v)[2], uint32_t at) {
    asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:64\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1]) : "v"(at) : "memory");
}

// The sums of four columns of q, k or v of one row (a wave: 16 rows, 16 columns from `first` on), rotated, to where
// attention and the cache keep them.
__device__ __forceinline__ void rows_rope(const RowsArgs &a, int first, int row, int g, f32x4 sum) {
    const int D = a.s.head_dim, H = a.s.num_attention_heads, KVH = a.s.num_kv_heads, head = first / D;
    const bool is_value = head >= H + KVH;
    const int kv_head = is_value ? head - H - KVH : head - H;
    const bool split = !a.s.interleaved && !is_value;
    // first of the thread's four columns within the head
    const int d = split ? first % D / 2 + 4 * (g & 1) + (g >> 1) * (D / 2) : first % D + 4 * g;
    const int at = min(row, a.rows - 1), batch = at / a.s.seq, seq_at = at % a.s.seq;
    const int64_t position = a.positions[seq_at];
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = round_bf16(sum[j]);
    if (!is_value) {
        float other[4];
        if (split) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float partner = __shfl_xor(v[j], 32);  // with every lane active
                other[j] = g >= 2 ? partner : -partner;
            }
        } else {
#pragma unroll
            for (int j = 0; j < 4; j += 2) other[j] = -v[j + 1], other[j + 1] = v[j];
        }
        const size_t rope_at = (size_t)wrap_position(position, a.s.rope_positions) * D + d;
        const f32x4 c = *(const f32x4 *)(a.rope_cos + rope_at), sn = *(const f32x4 *)(a.rope_sin + rope_at);
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = v[j] * c[j] + other[j] * sn[j];
    }
    if (row >= a.rows) return;
    const u32x2 pairs = {pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
    if (head < H) {
        *(u32x2 *)(a.out + ((size_t)row * H + head) * D + d) = pairs;
        return;
    }
    const size_t cache_row = (size_t)batch * a.s.kv_max_len + (size_t)wrap_position(position, a.s.kv_max_len);
    *(u32x2 *)((is_value ? a.v_cache : a.k_cache) + (cache_row * KVH + kv_head) * D + d) = pairs;
    if (is_value) {
        uint16_t *const dst = a.values_t + (((size_t)batch * KVH + kv_head) * D + d) * a.padded + (seq_at & ~15) + slot_in_group(seq_at & 15);
#pragma unroll
        for (int j = 0; j < 4; j++) dst[(size_t)j * a.padded] = (uint16_t)(pairs[j / 2] >> (j % 2 * 16));
    } else {
        *(u32x2 *)(a.keys + (((size_t)batch * KVH + kv_head) * a.padded + seq_at) * D + d) = pairs;
    }
}

__device__ __forceinline__ void store_through(uint64_t *dst, float lo, float hi) {
    const f32x2 v = {lo, hi};
    __hip_atomic_store((MK_GLOBAL uint64_t *)dst, __builtin_bit_cast(uint64_t, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ f32x2 load_past(const uint64_t *src) {
    return __builtin_bit_cast(f32x2, __hip_atomic_load((const MK_GLOBAL uint64_t *)src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

template <int MT, int NT, int WAVES, int STAGES, bool NORM>
struct RowsLds {
    static constexpr int kStep = (NT + MT) * 2048, kRing = WAVES * STAGES * kStep;
    static constexpr int bytes(int k) { return kRing + (NORM ? (k / 64 + WAVES * 8 - 1) / (WAVES * 8) * WAVES * 1024 : 0); }
};

template <int MT, int NT, int WAVES, int STAGES, int EPI, bool NORM, bool PAST>
__global__ __launch_bounds__(WAVES * 64) void rows_kernel(RowsArgs a) {
    typedef RowsLds<MT, NT, WAVES, STAGES, NORM> Lds;
    constexpr int kLoads = (NT + MT) * 2;  // load instructions of a step
    static_assert(STAGES <= 2, "the wait for all loads but the last step's");
    extern __shared__ __align__(16) unsigned char lds[];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), lane = (int)threadIdx.x % 64, r = lane % 16, g = lane / 16;
    const int first_step = a.k / 64 * blockIdx.y / gridDim.y, steps = a.k / 64 * (blockIdx.y + 1) / gridDim.y - first_step;
    const int mine = (steps - wave + WAVES - 1) / WAVES;

    unsigned char *const ring = lds + wave * (STAGES * Lds::kStep);
    unsigned char *const norm_lds = lds + Lds::kRing + wave * ((steps + WAVES * 8 - 1) / (WAVES * 8) * 1024);
    f32x4 acc[NT][MT];
    float square[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) {
        square[m] = 0.0f;
#pragma unroll
        for (int t = 0; t < NT; t++) acc[t][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    if (mine > 0) {
        if constexpr (NORM) {
            for (int i = 0; i < mine; i += 8) {
                const int step = first_step + wave + min(i + lane / 8, mine - 1) * WAVES;
                load_to_lds(a.norm_weight + step * 64 + lane % 8 * 8, (MK_LDS void *)(norm_lds + i * 128));
            }
        }
        // a load instruction moves eight rows of 128 bytes; 16-byte pieces swizzled as they are read
        const int load_row = lane / 8;
        const uint16_t *src[kLoads];
#pragma unroll
        for (int j = 0; j < kLoads; j++) {
            const int row = j % 2 * 8 + load_row, piece = (lane % 8) ^ ((row >> 1) & 7), t = j / 2;
            const uint16_t *const base = t >= NT ? a.x + (size_t)min((t - NT) * 16 + row, a.rows - 1) * a.k
                                                 : (EPI == kRowsSilu && t >= NT / 2 ? a.w1 : a.w0) + (size_t)rows_weight_row<NT, EPI>(a, t, row) * a.k;
            src[j] = base + (first_step + wave) * 64 + piece * 8;
        }
        auto request = [&](int i) {
            unsigned char *const slot = ring + i % STAGES * Lds::kStep;
#pragma unroll
            for (int j = 0; j < kLoads; j++) {
                constexpr int kPast = PAST ? 2 : 0;
                const MK_GLOBAL void *const from = (const MK_GLOBAL void *)(src[j] + (size_t)i * (WAVES * 64));
                MK_LDS void *const to = (MK_LDS void *)(slot + j * 1024);
                if (j < 2 * NT) __builtin_amdgcn_global_load_lds(from, to, 16, 0, kPast);
                else __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
            }
        };
        const uint32_t read_at = (uint32_t)(uintptr_t)(MK_LDS unsigned char *)ring + r * 128, swizzle = (r >> 1) & 7;
        const uint32_t norm_at = (uint32_t)(uintptr_t)(MK_LDS unsigned char *)norm_lds + g * 16;
#pragma unroll
        for (int p = 0; p < STAGES; p++)
            if (p < mine) request(p);
        for (int i = 0; i < mine; i++) {
            // a wave reads only what it has loaded itself: no barrier, only its own loads' arrival, oldest first
            const int newer = mine - 1 - i;
            if (newer >= STAGES - 1) asm volatile("s_waitcnt vmcnt(%0)" ::"i"((STAGES - 1) * kLoads) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            const uint32_t slot = read_at + i % STAGES * Lds::kStep;
            u32x4 frag[2][NT + MT], norm[2];
            if constexpr (NORM) rows_read_norm(norm, norm_at + i * 128);
#pragma unroll
            for (int half = 0; half < 2; half++) rows_read(frag[half], slot + (((half * 4 + g) ^ swizzle) * 16));
            __builtin_amdgcn_sched_barrier(0);
            if (i + STAGES < mine) request(i + STAGES);
#pragma unroll
            for (int half = 0; half < 2; half++)
#pragma unroll
                for (int m = 0; m < MT; m++) {
                    u32x4 x = frag[half][NT + m];
                    if constexpr (NORM) {
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            const float lo = bf16_lo(x[j]), hi = bf16_hi(x[j]);
                            square[m] = fmaf(lo, lo, square[m]);
                            square[m] = fmaf(hi, hi, square[m]);
                            x[j] = pack_bf16(lo * bf16_lo(norm[half][j]), hi * bf16_hi(norm[half][j]));
                        }
                    }
#pragma unroll
                    for (int t = 0; t < NT; t++)
                        acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, frag[half][t]),
                                                                            __builtin_bit_cast(bf16x8, x), acc[t][m], 0, 0, 0);
                }
        }
    }
    __syncthreads();
    f32x4 *const part = (f32x4 *)lds;                                 // [WAVES][NT][MT][64]
    float *const squares = (float *)(lds + WAVES * NT * MT * 1024);   // [WAVES][MT][16]
#pragma unroll
    for (int m = 0; m < MT; m++) {
#pragma unroll
        for (int t = 0; t < NT; t++) part[((wave * NT + t) * MT + m) * 64 + lane] = acc[t][m];
        if constexpr (NORM) {
            square[m] += __shfl_xor(square[m], 16);
            square[m] += __shfl_xor(square[m], 32);
            if (g == 0) squares[(wave * MT + m) * 16 + r] = square[m];
        }
    }
    __syncthreads();

    // one thread of the first MT waves: four neighbouring columns (4 g ...) of one row, of every tile
    const int m = wave, row = m * 16 + r;
    f32x4 sum[NT];
    float total = 0.0f;
    if (wave < MT) {
#pragma unroll
        for (int t = 0; t < NT; t++) {
            sum[t] = part[(t * MT + m) * 64 + lane];
#pragma unroll
            for (int w = 1; w < WAVES; w++) sum[t] += part[((w * NT + t) * MT + m) * 64 + lane];
        }
        if constexpr (NORM)
#pragma unroll
            for (int w = 0; w < WAVES; w++) total += squares[(w * MT + m) * 16 + r];
    }
    if (!NORM && gridDim.y > 1) {
        // The last block of a column tile to arrive adds all their sums, in the order of K whichever came last.  The XCDs
        // have L2 caches of their own: sums are stored through them and loaded past them, stores waited for before the
        // arrival is counted.
        uint64_t *const sums = (uint64_t *)a.partial + (size_t)blockIdx.x * gridDim.y * NT * MT * 128;
        if (wave < MT) {
#pragma unroll
            for (int t = 0; t < NT; t++) {
                uint64_t *const dst = sums + ((size_t)(blockIdx.y * NT + t) * MT + m) * 128 + lane;
                store_through(dst, sum[t][0], sum[t][1]);
                store_through(dst + 64, sum[t][2], sum[t][3]);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        __syncthreads();  // also: the last reads of `part`
        int *const last = (int *)lds;
        if (threadIdx.x == 0) {
            const int before = __hip_atomic_fetch_add((MK_GLOBAL int *)a.arrived + blockIdx.x, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *last = before + 1 == (int)gridDim.y;
            if (*last) __hip_atomic_store((MK_GLOBAL int *)a.arrived + blockIdx.x, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (!*last) return;
        if (wave < MT) {
#pragma unroll
            for (int t = 0; t < NT; t++) sum[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            for (int y = 0; y < (int)gridDim.y; y++)
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const uint64_t *const src = sums + ((size_t)(y * NT + t) * MT + m) * 128 + lane;
                    const f32x2 lo = load_past(src), hi = load_past(src + 64);
                    sum[t] += f32x4{lo.x, lo.y, hi.x, hi.y};
                }
        }
    }
    if (wave >= MT) return;

    if constexpr (NORM) {
        const float scale = rsqrtf(total / (float)a.k + a.s.rms_norm_eps);
#pragma unroll
        for (int t = 0; t < NT; t++) sum[t] *= scale;
    }
    const bool valid = row < a.rows;
    if constexpr (EPI == kRowsResidual) {
        if (!valid) return;
#pragma unroll
        for (int t = 0; t < NT; t++) {
            u32x2 *const dst = (u32x2 *)(a.out + (size_t)row * a.n + (blockIdx.x * NT + t) * 16 + 4 * g);
            const u32x2 old = *dst;
            u32x2 next;
#pragma unroll
            for (int j = 0; j < 2; j++)
                next[j] = pack_bf16(bf16_lo(old[j]) + round_bf16(sum[t][2 * j]), bf16_hi(old[j]) + round_bf16(sum[t][2 * j + 1]));
            *dst = next;
        }
    } else if constexpr (EPI == kRowsSilu) {
        if (!valid) return;
#pragma unroll
        for (int t = 0; t < NT / 2; t++) {
            const int column = (blockIdx.x * (NT / 2) + t) * 16 + 4 * g;
            if (column >= a.n) continue;
            u32x2 next;
#pragma unroll
            for (int j = 0; j < 2; j++)
                next[j] = pack_bf16(round_bf16(silu(round_bf16(sum[t][2 * j]))) * round_bf16(sum[NT / 2 + t][2 * j]),
                                    round_bf16(silu(round_bf16(sum[t][2 * j + 1]))) * round_bf16(sum[NT / 2 + t][2 * j + 1]));
            *(u32x2 *)(a.out + (size_t)row * a.n + column) = next;
        }
    } else if constexpr (EPI == kRowsArgmax) {
        uint64_t best = 0;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int column = (blockIdx.x * NT + t) * 16 + 4 * g + j;
                const uint64_t key = (uint64_t)order_bits(pack_bf16(sum[t][j], 0.0f) & 0xffffu) << 32 | (uint32_t)~(uint32_t)column;
                if (column < a.n && key > best) best = key;
            }
#pragma unroll
        for (int offset = 16; offset <= 32; offset *= 2) {
            const uint64_t other = __shfl_xor(best, offset);
            best = other > best ? other : best;
        }
        if (valid && g == 0) a.best[(size_t)row * gridDim.x + blockIdx.x] = best;
    } else {
#pragma unroll
        for (int t = 0; t < NT; t++) rows_rope(a, (blockIdx.x * NT + t) * 16, row, g, sum[t]);
    }
}

// Embedding rows, and zeros in the transposed values: the layers write the same positions of them, and attention
// multiplies those of the padding by zero.
__global__ __launch_bounds__(256) void rows_embed_kernel(mk_prefill_shape s, int rows, const int64_t *ids, const int64_t *positions,
                                                         const uint16_t *embed, uint16_t *h, u32x4 *values_t, int value_pieces) {
    if ((int)blockIdx.x >= rows) {
        for (int i = ((int)blockIdx.x - rows) * 256 + (int)threadIdx.x; i < value_pieces; i += ((int)gridDim.x - rows) * 256)
            values_t[i] = u32x4{0, 0, 0, 0};
        return;
    }
    const int row = blockIdx.x, pieces = s.hidden_size / 8;
    const int64_t id = ids[row], position = positions[row % s.seq];
    check_token(s, id, position);
    for (int i = threadIdx.x; i < pieces; i += 256)
        *(u32x4 *)(h + (size_t)row * s.hidden_size + (size_t)i * 8) = *(const u32x4 *)(embed + (size_t)id * s.hidden_size + (size_t)i * 8);
}

__global__ __launch_bounds__(256) void rows_best_kernel(int blocks, const uint64_t *best_of_block, int64_t *ids) {
    uint64_t best = 0;
    for (int i = threadIdx.x; i < blocks; i += 256) {
        const uint64_t key = best_of_block[(size_t)blockIdx.x * blocks + i];
        best = key > best ? key : best;
    }
    write_best<256>(best, ids);
}
