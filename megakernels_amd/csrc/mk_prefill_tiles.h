// The prompt forward's matrix products for more rows than kRowsMax: y = x w^T in tiles, with the operations that follow a
// product (rotary embedding and cache append, residual add, SiLU * up, argmax) in its epilogue.
//
// K goes through a ring of LDS stages of 64 elements, filled by loads that go from memory straight into LDS (eight rows of
// 128 bytes a wave; 16-byte pieces swizzled so that a wave's reads spread over all banks) and stay in flight across the one
// barrier of a stage: each wave waits for its own loads of the next stage, then meets the others.  A wave reads the operands
// of its next stage before it multiplies the current one's, also across that barrier.  Operands are swapped (w first), so that
// a lane holds four neighbouring columns of one row: rotary pairs and gate and up of one output lie in one lane.
constexpr int kTileK = 64;

enum TileEpilogue { kTileRope, kTileResidual, kTileSilu, kTileArgmax };

struct TileArgs {
    mk_prefill_shape s;
    int rows, n, k, padded;      // n: columns of the product (of gate alone for SiLU)
    const uint16_t *x, *w0, *w1; // x [rows, k]; w0 (and w1: up beside gate) [n, k]
    uint16_t *out;               // residual: h, in place; SiLU: [rows, n]; rope: q [rows, H D]
    const int64_t *positions;
    const float *rope_cos, *rope_sin;
    uint16_t *k_cache, *v_cache, *keys, *values_t;
    uint64_t *best;              // argmax: [groups of 64 columns, rows]
    // K split over gridDim.y blocks: their sums, [tile, gridDim.y, threads] of what a thread holds, and how many of a
    // tile's blocks have arrived (zero between launches)
    float *partial;
    int *arrived;
};

// Row of w that lies at row `r` of a block's w tile.  Tiles of 32 rows alternate between what a lane has to hold side by
// side: gate and up; the two halves of a head, where rotary pairs are half a head apart.
template <int TILE_N, int EPI>
__device__ __forceinline__ const uint16_t *tile_weight_row(const TileArgs &a, int n_tile, int r) {
    if constexpr (EPI == kTileSilu) {
        const int row = min(n_tile * (TILE_N / 2) + r / 64 * 32 + r % 32, a.n - 1);
        return (r / 32 % 2 ? a.w1 : a.w0) + (size_t)row * a.k;
    }
    int row = n_tile * TILE_N + r;
    if (EPI == kTileRope && !a.s.interleaved && a.s.head_dim == 128 && row < (a.s.num_attention_heads + a.s.num_kv_heads) * 128)
        row += -(r % 128) + r % 32 + r % 128 / 64 * 32 + r / 32 % 2 * 64;
    return a.w0 + (size_t)min(row, a.n - 1) * a.k;
}

// 64 columns of q, k or v from `first` on, of one row (two lanes, half of every eight columns each), rotated, to where
// attention and the cache keep them.  `acc0`, `acc1`: the two tiles of 32 columns.
__device__ __forceinline__ void tile_rope(const TileArgs &a, int row, int first, int half, const f32x16 &acc0, const f32x16 &acc1) {
    const int D = a.s.head_dim, H = a.s.num_attention_heads, KVH = a.s.num_kv_heads;
    const int batch = row / a.s.seq, seq_at = row % a.s.seq, head = first / D, in_head = first % D;
    const bool is_value = head >= H + KVH, halves = !a.s.interleaved && !is_value;
    if (head >= H + 2 * KVH) return;
    const int kv_head = is_value ? head - H - KVH : head - H;
    const int64_t position = a.positions[seq_at];
    const size_t rope_row = (size_t)wrap_position(position, a.s.rope_positions) * D;
    const size_t cache_row = (size_t)batch * a.s.kv_max_len + (size_t)wrap_position(position, a.s.kv_max_len);
    uint16_t *const row_dst = head < H ? a.out + ((size_t)row * H + head) * D : (is_value ? a.v_cache : a.k_cache) + (cache_row * KVH + kv_head) * D;
    uint16_t *const key_dst = a.keys + (((size_t)batch * KVH + kv_head) * a.padded + seq_at) * D;
    uint16_t *const value_dst = a.values_t + ((size_t)batch * KVH + kv_head) * D * a.padded + (seq_at & ~15) + slot_in_group(seq_at & 15);
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int d = (halves ? in_head / 2 + t * (D / 2) : in_head + t * 32) + 8 * q + 4 * half;
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = round_bf16(t ? acc1[4 * q + j] : acc0[4 * q + j]);
            if (!is_value) {
                const f32x4 c = *(const f32x4 *)(a.rope_cos + rope_row + d), sn = *(const f32x4 *)(a.rope_sin + rope_row + d);
                float other[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float pair = t ? acc1[(4 * q + j) ^ 1] : acc0[(4 * q + j) ^ 1], across = t ? acc0[4 * q + j] : acc1[4 * q + j];
                    const float partner = round_bf16(halves ? across : pair);
                    other[j] = (halves ? t == 1 : j % 2 == 1) ? partner : -partner;
                }
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = v[j] * c[j] + other[j] * sn[j];
            }
            const u32x2 pairs = {pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
            *(u32x2 *)(row_dst + d) = pairs;
            if (is_value)
#pragma unroll
                for (int j = 0; j < 4; j++) value_dst[(size_t)(d + j) * a.padded] = (uint16_t)(pairs[j / 2] >> (j % 2 * 16));
            else if (head >= H)
                *(u32x2 *)(key_dst + d) = pairs;
        }
}

// 2 x WN waves of MT x NT tiles of 32 x 32
template <int WN, int MT, int NT, int STAGES, int EPI>
__global__ __launch_bounds__(WN * 128, 2) void tile_kernel(TileArgs a) {
    constexpr int kRows = MT * 64, kTileN = WN * NT * 32, kThreads = WN * 128, kWaves = WN * 2;
    constexpr int kStage = (kRows + kTileN) * kTileK * 2, kLoads = kStage / 1024 / kWaves;  // bytes; load instructions of a wave
    extern __shared__ __align__(16) unsigned char lds[];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), lane = (int)threadIdx.x % 64;
    const int wave_m = wave / WN, wave_n = wave % WN, half = lane / 32;

    // Blocks go to the XCDs in turn.  Column tile n is XCD n % 8's, whose blocks walk its column tiles eight row tiles at a
    // time, so that the tiles of x and w that are in use at once fit its L2.
    const int m_tiles = (a.rows + kRows - 1) / kRows, n_tiles = ((EPI == kTileSilu ? 2 * a.n : a.n) + kTileN - 1) / kTileN;
    const int n_of_xcd = (n_tiles + 7) / 8, xcd = blockIdx.x % 8, local = blockIdx.x / 8;
    const int m_group = local / (n_of_xcd * 8), in_group = local % (n_of_xcd * 8), group_rows = min(8, m_tiles - m_group * 8);
    const int n_tile = in_group / group_rows * 8 + xcd, m_tile = m_group * 8 + in_group % group_rows;
    if (n_tile >= n_tiles || in_group / group_rows >= n_of_xcd) return;
    const int first_step = a.k / kTileK * blockIdx.y / gridDim.y, steps = a.k / kTileK * (blockIdx.y + 1) / gridDim.y - first_step;

    const uint16_t *src[kLoads];
#pragma unroll
    for (int j = 0; j < kLoads; j++) {
        const int row = (j * kWaves + wave) * 8 + lane / 8, piece = (lane % 8) ^ ((row >> 1) & 7);
        const uint16_t *const base = row < kTileN ? tile_weight_row<kTileN, EPI>(a, n_tile, row)
                                                  : a.x + (size_t)min(m_tile * kRows + row - kTileN, a.rows - 1) * a.k;
        src[j] = base + first_step * kTileK + piece * 8;
    }
    auto request = [&](int i) {
        unsigned char *const stage = lds + i % STAGES * kStage;
#pragma unroll
        for (int j = 0; j < kLoads; j++) load_to_lds(src[j] + i * kTileK, (MK_LDS void *)(stage + (j * kWaves + wave) * 1024));
    };
    f32x16 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[m][t][r] = 0.0f;
    const int w_row = wave_n * (NT * 32) + lane % 32, x_row = wave_m * (MT * 32) + lane % 32, swizzle = (lane >> 1) & 7;
    auto read = [&](int i, int step, bf16x8 (&w)[NT], bf16x8 (&x)[MT]) {
        const unsigned char *const stage = lds + i % STAGES * kStage + ((2 * step + half) ^ swizzle) * 16;
#pragma unroll
        for (int t = 0; t < NT; t++) w[t] = *(const bf16x8 *)(stage + (w_row + t * 32) * 128);
#pragma unroll
        for (int m = 0; m < MT; m++) x[m] = *(const bf16x8 *)(stage + (kTileN + x_row + m * 32) * 128);
    };
    auto multiply = [&](const bf16x8 (&w)[NT], const bf16x8 (&x)[MT]) {
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int t = 0; t < NT; t++) acc[m][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[t], x[m], acc[m][t], 0, 0, 0);
    };
    // this wave's loads of stage `i` have arrived, and then every wave's
    auto arrive = [&](int i) {
        const int newer = min(steps - 1 - i, STAGES - 2);
        if (STAGES > 3 && newer == 2) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(2 * kLoads) : "memory");
        else if (STAGES > 2 && newer == 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(kLoads) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    static_assert(STAGES >= 2 && STAGES <= 4);
    request(0);
#pragma unroll
    for (int p = 1; p < STAGES - 1; p++)
        if (p < steps) request(p);
    arrive(0);
    if (STAGES - 1 < steps) request(STAGES - 1);
    // In the steady state no branch divides a stage, and the next operands' reads are put between the products: a wave
    // issues in order, and all its reads at once would hold its products back for as long as LDS takes to accept them.
    auto steady_arrive = [&]() {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"((STAGES - 2) * kLoads) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    int i = 0;
    // few products per operand: read a whole stage ahead
    bf16x8 w[2][4][NT], x[2][4][MT];
    auto stage = [&](int at, auto odd_, auto steady) {
        constexpr int odd = decltype(odd_)::value;
        if constexpr (steady) {
            steady_arrive();  // every wave has read stage `at`, too
            request(at + STAGES);
        } else if (at + 1 < steps) {
            arrive(at + 1);
            if (at + STAGES < steps) request(at + STAGES);
        }
        if (steady || at + 1 < steps)
#pragma unroll
            for (int step = 0; step < 4; step++) read(at + 1, step, w[1 - odd][step], x[1 - odd][step]);
#pragma unroll
        for (int step = 0; step < 4; step++) multiply(w[odd][step], x[odd][step]);
        if constexpr (steady) {
#pragma unroll
            for (int p = 0; p < 2 * MT * NT; p++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);                // MFMA
                __builtin_amdgcn_sched_group_barrier(0x100, MT * NT == 2 ? 3 : 2, 0);  // LDS read
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
#pragma unroll
    for (int step = 0; step < 4; step++) read(0, step, w[0][step], x[0][step]);
    for (; i + 1 + STAGES < steps; i += 2) {
        stage(i, std::integral_constant<int, 0>{}, std::true_type{});
        stage(i + 1, std::integral_constant<int, 1>{}, std::true_type{});
    }
    for (; i < steps; i += 2) {
        stage(i, std::integral_constant<int, 0>{}, std::false_type{});
        if (i + 1 < steps) stage(i + 1, std::integral_constant<int, 1>{}, std::false_type{});
    }
    __syncthreads();

    if (gridDim.y > 1) {
        // the last block of a tile to arrive adds all their sums in the order of K (the XCDs' L2 caches are not coherent:
        // stored through them, loaded past them, stores waited for before the arrival is counted)
        const int tile = m_tile * n_tiles + n_tile;
        uint64_t *const sums = (uint64_t *)a.partial + (size_t)tile * gridDim.y * (MT * NT * 8 * kThreads) + threadIdx.x;
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int r = 0; r < 16; r += 2)
                    store_through(sums + ((size_t)blockIdx.y * (MT * NT * 8) + (m * NT + t) * 8 + r / 2) * kThreads, acc[m][t][r], acc[m][t][r + 1]);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();  // also: the last reads of the ring
        int *const last = (int *)lds;
        if (threadIdx.x == 0) {
            const int before = __hip_atomic_fetch_add((MK_GLOBAL int *)a.arrived + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *last = before + 1 == (int)gridDim.y;
            if (*last) __hip_atomic_store((MK_GLOBAL int *)a.arrived + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (!*last) return;
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[m][t][r] = 0.0f;
        for (int y = 0; y < (int)gridDim.y; y++)
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int r = 0; r < 16; r += 2) {
                        const f32x2 v = load_past(sums + ((size_t)y * (MT * NT * 8) + (m * NT + t) * 8 + r / 2) * kThreads);
                        acc[m][t][r] += v.x, acc[m][t][r + 1] += v.y;
                    }
    }

#pragma unroll
    for (int m = 0; m < MT; m++) {
        const int row = m_tile * kRows + wave_m * (MT * 32) + m * 32 + lane % 32;
        const bool valid = row < a.rows;
        if constexpr (EPI == kTileResidual) {
            if (!valid) continue;
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int column = n_tile * kTileN + wave_n * (NT * 32) + t * 32 + 8 * q + 4 * half;
                    if (column >= a.n) continue;
                    u32x2 *const dst = (u32x2 *)(a.out + (size_t)row * a.n + column);
                    const u32x2 old = *dst;
                    u32x2 next;
#pragma unroll
                    for (int j = 0; j < 2; j++)
                        next[j] = pack_bf16(bf16_lo(old[j]) + round_bf16(acc[m][t][4 * q + 2 * j]),
                                            bf16_hi(old[j]) + round_bf16(acc[m][t][4 * q + 2 * j + 1]));
                    *dst = next;
                }
        } else if constexpr (EPI == kTileSilu) {
            if (!valid) continue;
#pragma unroll
            for (int t = 0; t < NT; t += 2)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int column = n_tile * (kTileN / 2) + wave_n * (NT * 16) + t * 16 + 8 * q + 4 * half;
                    if (column >= a.n) continue;
                    u32x2 next;
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        const int r = 4 * q + 2 * j;
                        next[j] = pack_bf16(round_bf16(silu(round_bf16(acc[m][t][r]))) * round_bf16(acc[m][t + 1][r]),
                                            round_bf16(silu(round_bf16(acc[m][t][r + 1]))) * round_bf16(acc[m][t + 1][r + 1]));
                    }
                    *(u32x2 *)(a.out + (size_t)row * a.n + column) = next;
                }
        } else if constexpr (EPI == kTileArgmax) {
            uint64_t best = 0;
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int column = n_tile * kTileN + wave_n * (NT * 32) + t * 32 + 8 * (r / 4) + 4 * half + r % 4;
                    const uint64_t key = (uint64_t)order_bits(pack_bf16(acc[m][t][r], 0.0f) & 0xffffu) << 32 | (uint32_t)~(uint32_t)column;
                    if (column < a.n && key > best) best = key;
                }
            const uint64_t other = __shfl_xor(best, 32);
            best = other > best ? other : best;
            if (valid && half == 0) a.best[(size_t)(n_tile * WN + wave_n) * a.rows + row] = best;
        } else {
            if (!valid) continue;
#pragma unroll
            for (int t = 0; t < NT; t += 2) tile_rope(a, row, n_tile * kTileN + wave_n * (NT * 32) + t * 32, half, acc[m][t], acc[m][t + 1]);
        }
    }
}

// A row's best key of all groups of 64 columns: 16 rows a block (a line of keys), 64 slices of the groups.  (64 rows a block
// left most of the chip idle: 777 rows of 2004 groups 51 us.)
__global__ __launch_bounds__(1024) void tile_best_kernel(int rows, int groups, const uint64_t *best_of_group, int64_t *ids) {
    __shared__ uint64_t of_wave[16][16];
    const int slice = (int)threadIdx.x / 16, in_block = (int)threadIdx.x % 16, row = blockIdx.x * 16 + in_block;
    uint64_t best = 0;
    for (int i = slice; i < groups; i += 64) {
        const uint64_t key = best_of_group[(size_t)i * rows + min(row, rows - 1)];
        best = key > best ? key : best;
    }
#pragma unroll
    for (int offset = 16; offset <= 32; offset *= 2) {
        const uint64_t other = __shfl_xor(best, offset);
        best = other > best ? other : best;
    }
    if (threadIdx.x % 64 < 16) of_wave[threadIdx.x / 64][in_block] = best;
    __syncthreads();
    if (threadIdx.x >= 16 || row >= rows) return;
    for (int w = 1; w < 16; w++) best = of_wave[w][in_block] > best ? of_wave[w][in_block] : best;
    ids[row] = (int64_t)(uint32_t)~(uint32_t)best;
}
