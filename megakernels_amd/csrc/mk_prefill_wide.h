// The prompt forward's matrix products where there are enough rows and columns for wide tiles: y = x w^T on
// v_mfma_f32_16x16x32_bf16, eight waves a block, with the same epilogues as mk_prefill_tiles.h.
//
// Both kernels run their two waves of a SIMD in turn: the waves form two groups of four, one on each SIMD, and one group
// lives a barrier behind the other.  While a group multiplies (16 instructions, 256 clocks, with its waves' priority
// raised), the other reads its next operands from LDS and requests later ones, then they change places.  Left to
// themselves, the waves of the former 256 x 256 kernel met at one barrier a stage and read at the same time: 1.23 PFLOP/s
// over whole rounds of tiles; in turn 1.56 (4096 x 16384 x 2048 without its stores).
//
// Operands go from memory straight into a ring in LDS that is filled as it is used, in pieces of one group's phase, five to
// seven phases ahead: a piece's place is requested again two phases after it was read, when the group behind has read it,
// too (its reads are waited for before it multiplies, one phase after it asked for them).  All waits count requests
// (vmcnt), so nothing drains between phases.
//
// Rows of 128 bytes (64 elements of K) lie in LDS with their 16-byte pieces swizzled by the row, so that 16 lanes read all
// banks.  w comes first in the product: a lane holds four neighbouring columns of one row, and w's rows are laid out so
// that a lane's fragments make two runs of eight columns, 32 columns apart (gate and up for SiLU; the two halves of a head
// where rotary pairs are half a head apart).

// row of w that lies at row `r` of the 64 of a wave: fragment r / 16, four columns of lane group r % 16 / 4
__device__ __forceinline__ int wide_column(int r) { return r / 32 * 32 + r % 16 / 4 * 8 + r / 16 % 2 * 4 + r % 4; }

// `r` of the tile's 256 columns, as an offset into the tile's rows of w (for SiLU: of gate or up)
template <int EPI>
__device__ __forceinline__ int wide_weight_row(const TileArgs &a, int n_tile, int r) {
    const int column = r / 64 * 64 + wide_column(r % 64);
    if (EPI == kTileSilu) return column / 64 * 32 + column % 32;
    // heads of 128 whose pairs are half a head apart: 32 columns of each half
    if (EPI == kTileRope && !a.s.interleaved && a.s.head_dim == 128 && n_tile * 256 + column < (a.s.num_attention_heads + a.s.num_kv_heads) * 128)
        return column / 128 * 128 + column % 128 / 64 * 32 + column % 64 / 32 * 64 + column % 32;
    return column;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)bytes, 0x00020000);
}
// Offsets have 32 bits, and kOutside, where nothing is stored, is one beyond every buffer that is written: 256 rows of at most
// this many columns of two bytes.
constexpr int kWideMostColumns = 1 << 20;
constexpr uint32_t kOutside = 0x80000000u;
static_assert(256ll * kWideMostColumns * 2 <= kOutside);

// a phase of the other group lies between two of these
__device__ __forceinline__ void wide_meet() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
}
// all but the `NEWER` newest requests of this wave have arrived, then every wave's; then this wave's reads of LDS
template <int NEWER>
__device__ __forceinline__ void wide_operands() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(NEWER) : "memory");
    wide_meet();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// tile `local` of the list of XCD `xcd` (which has column tiles n % 8 = xcd, eight row tiles at a time, so that the tiles of
// x and w in use at once share its L2); n < 0: there is none
struct WideTile {
    int m, n;
};
__device__ __forceinline__ WideTile wide_tile(int local, int xcd, int m_tiles, int n_tiles) {
    const int n_of_xcd = (n_tiles - xcd + 7) / 8;
    if (local >= n_of_xcd * m_tiles) return {0, -1};
    const int m_group = local / (n_of_xcd * 8), in_group = local - m_group * (n_of_xcd * 8), group_rows = min(8, m_tiles - m_group * 8);
    return {m_group * 8 + in_group % group_rows, in_group / group_rows * 8 + xcd};
}

__device__ __forceinline__ u32x4 pack8(const f32x4 &lo, const f32x4 &hi) {
    return u32x4{pack_bf16(lo[0], lo[1]), pack_bf16(lo[2], lo[3]), pack_bf16(hi[0], hi[1]), pack_bf16(hi[2], hi[3])};
}

// A value that the compiler takes for another one from here on: what is computed from it is not moved in front of the main
// loop, whose registers are full, to be fetched back from scratch memory behind an epilogue's stores.
template <class T>
__device__ __forceinline__ T here(T scalar) {
    asm volatile("" : "+s"(scalar));
    return scalar;
}
__device__ __forceinline__ int here_of_lane(int value) {
    asm volatile("" : "+v"(value));
    return value;
}

// The rotary tables' lines of 128 rows, in LDS: [cos, sin][row][D], the 16-byte pieces of a line swizzled by the row.  A lane
// rotates what it holds of one row, and its neighbour holds another row: 64 separate pieces of the tables a load.  Straight
// from memory these loads alone took 19 of the 80 us of 4096 x 3072 x 2048; moved into LDS in whole lines, once for all the
// heads of a tile, 4.  Behind them the rows' places in the cache: loaded where they are used, behind the stores of other
// rows, each would wait for those to complete.
constexpr int kTableRows = 128;
template <class RowOf>
__device__ __forceinline__ void wide_tables(const TileArgs &a, unsigned char *lds, int wave, int lane, RowOf row_of) {
    const int D = here(a.s.head_dim), seq = here(a.s.seq), pieces = D / 4, lines = 64 / pieces, count = kTableRows / 8 / lines;  // lines a request, requests a wave
    const int in_line = lane % pieces;
    int64_t position[8];
#pragma unroll
    for (int i = 0; i < 8; i++)
        position[i] = a.positions[min(row_of((wave * count + i % count) * lines + lane / pieces), a.rows - 1) % seq];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        if (i >= count) break;
        const int line = (wave * count + i) * lines + lane / pieces;
        const size_t from = (size_t)wrap_position(position[i], a.s.rope_positions) * D + (in_line ^ (line & 15)) * 4;
        if (in_line == 0) ((int *)(lds + 2 * kTableRows * D * 4))[line] = (int)wrap_position(position[i], a.s.kv_max_len);
        MK_LDS unsigned char *const dst = (MK_LDS unsigned char *)lds + (wave * count + i) * 1024;
        load_to_lds(a.rope_cos + from, (MK_LDS void *)dst);
        load_to_lds(a.rope_sin + from, (MK_LDS void *)(dst + kTableRows * D * 4));
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
}

// What the lanes of a wave hold of 64 columns of four groups of 16 rows (group i: rows row_of(i), one row a lane, whose tables
// are line line + i * 16; v(i)[run][j]: columns run * 32 + g * 8 + j * 4 ...) to where attention and the cache keep it.
template <class RowOf, class Values>
__device__ __forceinline__ void wide_rope(const TileArgs &a, const unsigned char *tables, int first, int g, int line, RowOf row_of, Values v) {
    const int D = here(a.s.head_dim), H = a.s.num_attention_heads, KVH = a.s.num_kv_heads, seq = here(a.s.seq);
    const uint64_t k_cache = here((uint64_t)a.k_cache), v_cache = here((uint64_t)a.v_cache);
    const int head = first / D, in_head = first % D;
    if (head >= H + 2 * KVH) return;
    const bool is_value = head >= H + KVH, interleaved = a.s.interleaved != 0, halves = !interleaved && !is_value;
    const int kv_head = is_value ? head - H - KVH : head - H;
    const int d0 = (halves ? in_head / 2 : in_head) + g * 8, d1 = d0 + (halves ? D / 2 : 32);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const unsigned char *const cosines = tables + (line + i * 16) * D * 4, *const sines = cosines + kTableRows * D * 4;
        u32x4 out[2];
#pragma unroll
        for (int run = 0; run < 2; run++) {
            if (is_value) {
                out[run] = pack8(v(i)[run][0], v(i)[run][1]);
                continue;
            }
            f32x4 rotated[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int piece = (((run ? d1 : d0) / 4 + j) ^ (line & 15)) * 16;
                const f32x4 c = *(const f32x4 *)(cosines + piece), sn = *(const f32x4 *)(sines + piece);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float pair = v(i)[run][j][e ^ 1], across = v(i)[1 - run][j][e];
                    const float partner = round_bf16(interleaved ? pair : across);
                    rotated[j][e] = round_bf16(v(i)[run][j][e]) * c[e] + ((interleaved ? e % 2 == 1 : run == 1) ? partner : -partner) * sn[e];
                }
            }
            out[run] = pack8(rotated[0], rotated[1]);
        }
        const int row = row_of(i);
        if (row >= a.rows) continue;
        if (head < H) {
            uint16_t *const dst = a.out + ((size_t)row * H + head) * D;
            *(u32x4 *)(dst + d0) = out[0], *(u32x4 *)(dst + d1) = out[1];
            continue;
        }
        const int batch = row / seq, seq_at = row - batch * seq;
        const size_t cache_row = (size_t)batch * a.s.kv_max_len + ((const int *)(tables + 2 * kTableRows * D * 4))[line + i * 16];
        uint16_t *const cache = (uint16_t *)(is_value ? v_cache : k_cache) + (cache_row * KVH + kv_head) * D;
        *(u32x4 *)(cache + d0) = out[0], *(u32x4 *)(cache + d1) = out[1];
        const size_t padded_head = (size_t)batch * KVH + kv_head;
        if (is_value) {
            uint16_t *const values = a.values_t + (padded_head * D + d0) * a.padded + (seq_at & ~15) + slot_in_group(seq_at & 15);
#pragma unroll
            for (int j = 0; j < 16; j++) values[(size_t)(j / 8 * 32 + j % 8) * a.padded] = (uint16_t)(out[j / 8][j % 8 / 2] >> (j % 2 * 16));
        } else {
            uint16_t *const keys = a.keys + (padded_head * a.padded + seq_at) * D;
            *(u32x4 *)(keys + d0) = out[0], *(u32x4 *)(keys + d1) = out[1];
        }
    }
}

// h += y
__device__ __forceinline__ u32x4 wide_add(const u32x4 &old, const f32x4 (&v)[2]) {
    const u32x4 add = pack8(v[0], v[1]);
    u32x4 next;
#pragma unroll
    for (int j = 0; j < 4; j++) next[j] = pack_bf16(bf16_lo(old[j]) + bf16_lo(add[j]), bf16_hi(old[j]) + bf16_hi(add[j]));
    return next;
}

// SiLU(gate) * up of eight columns of one row.  The exponential and the reciprocal are the instructions, not the library's exp
// and an IEEE division, which made a tile's epilogue longer than two tiles of K.  The gate is a bf16 and so is the result: for
// each of the 65536 gates, infinities and NaN among them, it is bit for bit that of silu() (before it is narrowed the two are
// up to 2.1e-7 and 1.3e-7 of the value off).  Without the step that refines the reciprocal one gate differs.  Whole forwards, us,
// with silu() and with this: 1B architecture 777 rows 3036 and 3005, 4096 rows 10692 and 10486; 8B 2048 rows 27709 and 27385.
__device__ __forceinline__ float fast_silu(float g) {
    // log2 e in two parts: a bf16 times the first is exact, and the second moves the power by less than a thousandth
    const float at = fminf(g, 64.0f), power = __builtin_amdgcn_exp2f(at * -1.44268798828125f);
    // (1 + exp(-g)) / 4: its reciprocal is no subnormal number, which the instruction would flush, for any finite power
    const float quarter = fmaf(power, fmaf(at, -4.8884951e-6f * 0.25f, 0.25f), 0.25f);
    const float y = __builtin_amdgcn_rcpf(quarter), off = fminf(fmaf(-quarter, y, 1.0f), 1.0f);  // (1: where the power is infinite and y 0)
    return g * 0.25f * fmaf(off, y, y);
}
__device__ __forceinline__ u32x4 wide_silu(const f32x4 (&v)[2][2]) {
    const u32x4 gate = pack8(v[0][0], v[0][1]), up = pack8(v[1][0], v[1][1]);
    u32x4 out;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t s = pack_bf16(fast_silu(bf16_lo(gate[j])), fast_silu(bf16_hi(gate[j])));
        out[j] = pack_bf16(bf16_lo(s) * bf16_lo(up[j]), bf16_hi(s) * bf16_hi(up[j]));
    }
    return out;
}

// The best key of 64 columns of every row, to a.best.  Keys of two words cost a dozen instructions a value.  Where a row's
// largest value is positive and none is a NaN, a word holds the bf16 value and below it the column counted from the end, and
// orders like its integer: two and a half instructions a value.
template <int GROUPS, class RowOf, class Values>
__device__ __forceinline__ void wide_best(const TileArgs &a, int first, int g, RowOf row_of, Values v) {
    int32_t largest[GROUPS];
    uint32_t negative = 0;
#pragma unroll
    for (int i = 0; i < GROUPS; i++) {
        largest[i] = 0;
#pragma unroll
        for (int run = 0; run < 2; run++) {
            const u32x4 pairs = pack8(v(i)[run][0], v(i)[run][1]);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t behind = 7 - j * 2 + (1 - run) * 32;  // minus g * 8: added for the row's best
                const uint32_t lo = pairs[j] << 16 | behind, hi = (pairs[j] & 0xffff0000u) | (behind - 1);
                largest[i] = max(largest[i], max((int32_t)lo, (int32_t)hi));
                negative = max(negative, max(lo, hi));
            }
        }
        largest[i] += (3 - g) * 8;  // at most 63 below the value
    }
    bool simple = negative <= 0xff80ffffu;
#pragma unroll
    for (int offset = 16; offset <= 32; offset *= 2)
#pragma unroll
        for (int i = 0; i < GROUPS; i++) largest[i] = max(largest[i], __shfl_xor(largest[i], offset));
#pragma unroll
    for (int i = 0; i < GROUPS; i++) simple &= row_of(i) >= a.rows || (largest[i] > 0xffff && largest[i] <= 0x7f80ffff);
    const bool all_simple = !__any(!simple);
    uint64_t *const dst = a.best + (size_t)(first / 64) * a.rows;
#pragma unroll
    for (int i = 0; i < GROUPS; i++) {
        uint64_t best = (uint64_t)order_bits((uint32_t)largest[i] >> 16) << 32 | (uint32_t)~(uint32_t)(first + 63 - (largest[i] & 0xffff));
        if (!all_simple) {
            best = 0;
#pragma unroll
            for (int run = 0; run < 2; run++)
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int column = first + run * 32 + g * 8 + e;
                    const uint64_t key = (uint64_t)order_bits(pack_bf16(v(i)[run][e / 4][e % 4], 0.0f) & 0xffffu) << 32 | (uint32_t)~(uint32_t)column;
                    if (column < a.n && key > best) best = key;
                }
#pragma unroll
            for (int offset = 16; offset <= 32; offset *= 2) {
                const uint64_t other = __shfl_xor(best, offset);
                best = other > best ? other : best;
            }
        }
        if (g == 0 && row_of(i) < a.rows) dst[row_of(i)] = best;
    }
}

// ---- 256 x 256: waves of 128 rows x 64 columns, in quarters of 64 x 32; as many blocks as CUs, each with its list of tiles ----
//
// A tile of 64 elements of K is four pieces of 16 KB (columns 0-31 of every wave, the tile's upper 128 rows, columns 32-63, the
// lower 128 rows) and four phases.  The ring holds nine: seven ahead, one being read, one that the group behind may still be
// reading; and it runs on across tiles, so that a tile's first operands arrive while the one before is finished.  At least four
// tiles of K.
// Products alone, output in bf16: 4096 x 16384 x 2048 198 us past the caches (the library 188), 176 without the stores, 1.56 PFLOP/s; 8192^3
// 721 us (the library 681).  With what follows, 4096 rows: gate, up and SiLU 201 us (the library's products and a pass over
// them 225), queries, keys and values with their rotation 64 (62), LM head with argmax 1467 (1817).
//
// Half a tile (128 rows) is two of the four phases and takes 0.65 of its time.  Where no more than half of an XCD's blocks
// would have a tile in the last round, every block has half of one; and a tile whose lower rows are past the end is its upper
// half.  Whole forwards, us: 8B architecture 2048 rows (gate and up: 3.5 rounds) 27180 -> 26750, 1B 1300 rows 4546 -> 4418.
constexpr int kSquarePieces = 9, kSquareBytes = kSquarePieces * 16384;
enum SquareRows { kAllRows, kUpperRows, kLowerRows };
struct SquareItem {
    int m, n;  // n < 0: there is none
    SquareRows rows;
};
// item `local` of the list of XCD `xcd`, which `blocks` blocks work on (a product that is narrower than the chip has halves on
// the XCDs with fewer tiles while the others work on whole ones, which is no gain: 4096 x 3072 64 -> 66 us, so rotation has none)
template <int EPI>
__device__ __forceinline__ SquareItem square_item(int local, int xcd, int m_tiles, int n_tiles, int blocks, int rows) {
    const int tiles = (n_tiles - xcd + 7) / 8 * m_tiles, whole = tiles / blocks * blocks, left = tiles - whole;
    const bool halves = EPI != kTileRope && local >= whole && 2 * left <= blocks;
    const WideTile t = wide_tile(halves ? whole + (local - whole) / 2 : local, xcd, m_tiles, n_tiles);
    const bool upper_only = rows - t.m * 256 <= 128;
    if (halves && (local - whole) % 2) return {t.m, upper_only ? -1 : t.n, kLowerRows};
    return {t.m, t.n, halves || upper_only ? kUpperRows : kAllRows};
}

template <int EPI>
__global__ __launch_bounds__(512, 2) void square_kernel(TileArgs a) {
    constexpr int kAhead = 2 * (kSquarePieces - 3);                // a wave's requests beyond a piece that is needed next
    constexpr int kStores = EPI == kTileSilu ? 8 : 0;              // stores of a wave after a tile, at least
    constexpr int kColumns = EPI == kTileSilu ? 128 : 256;
    extern __shared__ __align__(16) unsigned char lds[];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), lane = (int)threadIdx.x % 64;
    const int wave_m = wave / 4, wave_n = wave % 4, r16 = lane % 16, g = lane / 16;
    const int m_tiles = (a.rows + 255) / 256, n_tiles = (a.n + kColumns - 1) / kColumns, k_tiles = a.k / kTileK;
    const int xcd = blockIdx.x % 8, blocks = gridDim.x / 8;
    const uint32_t k_bytes = (uint32_t)a.k * 2;
    int local = blockIdx.x / 8;
    SquareItem item = square_item<EPI>(local, xcd, m_tiles, n_tiles, blocks, a.rows);
    if (item.n < 0) return;

    // a request of a wave moves eight rows of 128 bytes; two requests a piece
    uint32_t x_off[2][2], w_off[2][2];
    __amdgpu_buffer_rsrc_t x_buffer, w_buffer[2];
    int k_at = 0, put = 0, get = 0;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int row = wave * 16 + j * 8 + lane / 8, piece = (lane % 8) ^ ((row >> 1) & 7);
#pragma unroll
        for (int half = 0; half < 2; half++) x_off[half][j] = (uint32_t)(half * 128 + row) * k_bytes + piece * 16;
    }
    auto point = [&](const SquareItem &t) {
        x_buffer = buffer_of(a.x + (size_t)t.m * 256 * a.k, (uint32_t)min(256, a.rows - t.m * 256) * k_bytes);
        const size_t first = (size_t)t.n * kColumns;
        const uint32_t bytes = (uint32_t)min(kColumns, a.n - t.n * kColumns) * k_bytes;
        w_buffer[0] = buffer_of(a.w0 + first * a.k, bytes);
        if constexpr (EPI == kTileSilu) w_buffer[1] = buffer_of(a.w1 + first * a.k, bytes);
        else w_buffer[1] = w_buffer[0];
#pragma unroll
        for (int half = 0; half < 2; half++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int row = wave * 16 + j * 8 + lane / 8, piece = (lane % 8) ^ ((row >> 1) & 7);
                w_off[half][j] = (uint32_t)wide_weight_row<EPI>(a, t.n, row / 32 * 64 + half * 32 + row % 32) * k_bytes + piece * 16;
            }
        k_at = 0;
    };
    auto request_x = [&](const uint32_t (&off)[2], int at) {
        MK_LDS unsigned char *const dst = (MK_LDS unsigned char *)lds + put + wave * 2048;
#pragma unroll
        for (int j = 0; j < 2; j++) __builtin_amdgcn_raw_ptr_buffer_load_lds(x_buffer, (MK_LDS void *)(dst + j * 1024), 16, off[j], at, 0, 0);
        put = put + 16384 == kSquareBytes ? 0 : put + 16384;
    };
    auto request_w = [&](auto run_, int at) {
        constexpr int run = decltype(run_)::value;
        MK_LDS unsigned char *const dst = (MK_LDS unsigned char *)lds + put + wave * 2048;
#pragma unroll
        for (int j = 0; j < 2; j++) __builtin_amdgcn_raw_ptr_buffer_load_lds(w_buffer[run], (MK_LDS void *)(dst + j * 1024), 16, w_off[run][j], at, 0, 0);
        put = put + 16384 == kSquareBytes ? 0 : put + 16384;
    };
    f32x4 acc[2][4][2][2];  // [half of the rows][16 rows][run][four columns]
    bf16x8 x[4][2], w[2][2][2];
    const uint32_t swizzle = (r16 >> 1) & 7, step0 = (g ^ swizzle) * 16, step1 = ((4 + g) ^ swizzle) * 16;
    const uint32_t x_at = (wave_m * 64 + r16) * 128, w_at = (wave_n * 32 + r16) * 128;
    auto read_x = [&]() {
        const unsigned char *const base = lds + get + x_at;
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int i = 0; i < 4; i++) x[i][s] = *(const bf16x8 *)(base + i * 2048 + (s ? step1 : step0));
        get = get + 16384 == kSquareBytes ? 0 : get + 16384;
    };
    auto read_w = [&](auto run_) {
        constexpr int run = decltype(run_)::value;
        const unsigned char *const base = lds + get + w_at;
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int j = 0; j < 2; j++) w[run][j][s] = *(const bf16x8 *)(base + j * 2048 + (s ? step1 : step0));
        get = get + 16384 == kSquareBytes ? 0 : get + 16384;
    };
    auto multiply = [&](auto half_, auto run_) {
        constexpr int half = decltype(half_)::value, run = decltype(run_)::value;
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    acc[half][i][run][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[run][j][s], x[i][s], acc[half][i][run][j], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
        wide_meet();
    };
    constexpr std::integral_constant<int, 0> c0{};
    constexpr std::integral_constant<int, 1> c1{};
    auto k_tile = [&](auto newer_) {
        constexpr int newer = decltype(newer_)::value;
        read_x(), request_w(c0, k_at), wide_operands<newer>(), multiply(c0, c0);
        read_w(c1), request_x(x_off[0], k_at), wide_operands<newer>(), multiply(c0, c1);
        read_x(), request_w(c1, k_at), wide_operands<newer>(), multiply(c1, c0);
        read_w(c0), request_x(x_off[1], k_at), wide_operands<newer>(), multiply(c1, c1);
        k_at += 128;
    };
    // the ring is filled and its first piece read: the second group a barrier behind
    auto begin = [&]() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        wide_meet();
        if (wave_m) wide_meet();
        read_w(c0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // its place is requested again in the next phase but one of the other group
    };
    auto end = [&]() {  // the groups side by side again, nothing on its way to LDS
        if (!wave_m) wide_meet();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };
    // HALVES halves of the item's rows from half `at` on, to where they belong
    auto finish = [&](auto halves_, int at) {
        constexpr int HALVES = decltype(halves_)::value;
        const int lane_of = here_of_lane(lane), g = lane_of / 16, r16 = lane_of % 16;
        const int first = item.n * 256 + wave_n * 64, top = item.m * 256 + at * 128;
        auto row_of = [&](int i) { return top + i / 4 * 128 + wave_m * 64 + i % 4 * 16 + r16; };
        auto values = [&](int i) -> const f32x4(&)[2][2] { return acc[i / 4][i % 4]; };
        if constexpr (EPI == kTileRope) {
            // the tables take the ring's place, 128 rows at a time
#pragma unroll
            for (int half = 0; half < HALVES; half++) {
                wide_tables(a, lds, wave, lane_of, [&](int line) { return top + half * 128 + line; });
                wide_rope(a, lds, first, g, wave_m * 64 + r16, [&](int i) { return row_of(half * 4 + i); },
                          [&](int i) -> const f32x4(&)[2][2] { return acc[half][i]; });
                __syncthreads();
            }
        } else if constexpr (EPI == kTileSilu) {
            // a lane without a row or column stores outside the buffer: the count of stores is the same.  (Past the caches these
            // stores are over sooner, but the next product reads what they wrote: whole forwards of 1300 rows of the 1B
            // architecture 4127 us, 4082 through them, 4096 rows 9705 and 9593, 2048 rows of the 8B one 26340 and 25830.)
            const __amdgpu_buffer_rsrc_t out = buffer_of(a.out + (size_t)item.m * 256 * a.n, (uint32_t)min(256, a.rows - item.m * 256) * a.n * 2);
            const int column = first / 2 + g * 8;
#pragma unroll
            for (int i = 0; i < HALVES * 4; i++)
                __builtin_amdgcn_raw_buffer_store_b128(wide_silu(values(i)), out, column < a.n ? ((uint32_t)(row_of(i) - item.m * 256) * a.n + column) * 2 : kOutside, 0, 0);
        } else {
            wide_best<HALVES * 4>(a, first, g, row_of, values);
        }
    };
    bool begun = false;
    while (true) {
#pragma unroll
        for (int i = 0; i < 32; i++) ((f32x4 *)acc)[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        // (the compiler is told that these are the same for the whole wave, and the buffers are made anew for every item: once it
        // took them for the lanes' own, every request became a loop over the lanes' addresses)
        item = {__builtin_amdgcn_readfirstlane(item.m), __builtin_amdgcn_readfirstlane(item.n), (SquareRows)__builtin_amdgcn_readfirstlane(item.rows)};
        put = __builtin_amdgcn_readfirstlane(put), get = __builtin_amdgcn_readfirstlane(get);
        local = __builtin_amdgcn_readfirstlane(local) + blocks;
        const SquareItem next = square_item<EPI>(local, xcd, m_tiles, n_tiles, blocks, a.rows);
        // rotation needs LDS, and half a tile uses the ring in another order: the ring does not run on across those
        const bool goes_on = EPI != kTileRope && item.rows == kAllRows && next.n >= 0 && next.rows == kAllRows;
        if (item.rows == kAllRows) {
            point(item);
            if (!begun) {
                put = get = 0;
#pragma unroll
                for (int t = 0; t < 2; t++) request_w(c0, t * 128), request_x(x_off[0], t * 128), request_w(c1, t * 128), request_x(x_off[1], t * 128);
                begin();
            }
            k_at = 256;
            // the stores of the tile before are newer than what this tile's first phases need
            k_tile(std::integral_constant<int, kAhead + kStores>{});
            for (int k = 1; k < k_tiles - 2; k++) k_tile(std::integral_constant<int, kAhead>{});
            // the last two request the next tile's first; where there is none, this one's again, which nobody reads
            point(goes_on ? next : item);
            k_tile(std::integral_constant<int, kAhead>{});
            k_tile(std::integral_constant<int, kAhead>{});
            if (!goes_on) end();
            finish(std::integral_constant<int, 2>{}, 0);
        } else {
            // per tile of K: one piece of rows, then both of columns, the second already the next tile's; three tiles ahead, past
            // the end of K too, where nobody reads what arrives (of a buffer's last row zeros: its range check counts `at`, too)
            uint32_t off[2];
#pragma unroll
            for (int j = 0; j < 2; j++) off[j] = item.rows == kLowerRows ? x_off[1][j] : x_off[0][j];
            point(item);
            put = get = 0;
            request_w(c0, 0), request_x(off, 0), request_w(c1, 0), request_w(c0, 128), request_x(off, 128), request_w(c1, 128), request_w(c0, 256);
            begin();
            for (int k = 0; k < k_tiles; k++) {
                read_x(), request_x(off, k_at + 256), wide_operands<8>(), multiply(c0, c0);
                read_w(c1), read_w(c0), request_w(c1, k_at + 256), request_w(c0, k_at + 384), wide_operands<10>(), multiply(c0, c1);
                k_at += 128;
            }
            end();
            finish(std::integral_constant<int, 1>{}, item.rows == kLowerRows);
        }
        if (next.n < 0) return;
        begun = goes_on;
        item = next;
    }
}

// ---- 128 x 256: a tile's K is split between the two groups, which add their sums at the end ----
//
// Each group takes 32 of every 64 elements of K, with waves of 128 rows x 64 columns as above: tiles half as large for as few
// reads of LDS per product.  (Waves of 64 x 64 would need a third more than LDS delivers beside the matrix cores.)  The ring
// holds three tiles of 64 elements of K, requested three phases ahead; a block's share is at least three.
// Products alone, when a phase read eight fragments and the next four: 4096 x 2048 x 8192 113 us, 1.22 PFLOP/s (the library
// 110), 4096 x 2048 x 2048 35 (33), 2048 x 4096 x 14336 201 (206).  With six and six the whole forward of 4096 tokens of the 1B
// architecture went from 9890 to 9732 us.  777 x 2048 x 8192 with K in four parts: 43 us, 46 as 128 x 128 in two.
// K may also be split over gridDim.y blocks, whose sums meet in memory as in tile_kernel.
constexpr int kFlatStage = 49152, kFlatBytes = 3 * kFlatStage;

template <int EPI>
__global__ __launch_bounds__(512, 2) void flat_kernel(TileArgs a) {
    constexpr int kColumns = EPI == kTileSilu ? 128 : 256;
    extern __shared__ __align__(16) unsigned char lds[];  // [stage][rows 16 KB, columns 32 KB]
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), lane = (int)threadIdx.x % 64;
    const int group = wave / 4, wave_n = wave % 4, r16 = lane % 16, g = lane / 16;
    const int m_tiles = (a.rows + 127) / 128, n_tiles = (a.n + kColumns - 1) / kColumns;
    const uint32_t k_bytes = (uint32_t)a.k * 2;
    const WideTile tile = wide_tile(blockIdx.x / 8, blockIdx.x % 8, m_tiles, n_tiles);
    if (tile.n < 0) return;
    const int first_step = a.k / kTileK * blockIdx.y / gridDim.y, steps = a.k / kTileK * (blockIdx.y + 1) / gridDim.y - first_step;

    const __amdgpu_buffer_rsrc_t x_buffer = buffer_of(a.x + (size_t)tile.m * 128 * a.k, (uint32_t)min(128, a.rows - tile.m * 128) * k_bytes);
    const uint32_t w_bytes = (uint32_t)min(kColumns, a.n - tile.n * kColumns) * k_bytes;
    const __amdgpu_buffer_rsrc_t w0_buffer = buffer_of(a.w0 + (size_t)tile.n * kColumns * a.k, w_bytes);
    const __amdgpu_buffer_rsrc_t w1_buffer = EPI == kTileSilu ? buffer_of(a.w1 + (size_t)tile.n * kColumns * a.k, w_bytes) : w0_buffer;
    uint32_t x_off[2], w_off[4];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int row = j * 64 + wave * 8 + lane / 8;
        x_off[j] = (uint32_t)row * k_bytes + ((lane % 8) ^ ((row >> 1) & 7)) * 16;
    }
    // a wave's requests: eight rows each of four fragments of 16, the first two and the last two being the two runs
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int row = wave / 2 * 64 + j * 16 + wave % 2 * 8 + lane / 8;
        w_off[j] = (uint32_t)wide_weight_row<EPI>(a, tile.n, row) * k_bytes + ((lane % 8) ^ ((row >> 1) & 7)) * 16;
    }
    // places in the ring of tile t, t + 1 and t + 2 of K (that of t is t + 3's, too), and requests to them
    int place = 0, next_place = kFlatStage, far_place = 2 * kFlatStage;
    auto request_rows = [&](int t, int to, int half) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(x_buffer, (MK_LDS void *)((MK_LDS unsigned char *)lds + to + half * 8192 + wave * 1024), 16, x_off[half],
                                                 (first_step + t) * 128, 0, 0);
    };
    auto request_columns = [&](int t, int to, auto run_) {
        constexpr int run = decltype(run_)::value;
#pragma unroll
        for (int j = run * 2; j < run * 2 + 2; j++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(run ? w1_buffer : w0_buffer,
                                                     (MK_LDS void *)((MK_LDS unsigned char *)lds + to + 16384 + wave / 2 * 8192 + j * 2048 + wave % 2 * 1024), 16,
                                                     w_off[j], (first_step + t) * 128, 0, 0);
    };
    f32x4 acc[2][4][2][2];
#pragma unroll
    for (int i = 0; i < 32; i++) ((f32x4 *)acc)[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    bf16x8 x[4], first_run[2][2], second_run[2];  // first run of columns: of even and odd tiles of K
    const uint32_t at = r16 * 128 + ((group * 4 + g) ^ ((r16 >> 1) & 7)) * 16;
    auto read_x = [&](int half) {
        const unsigned char *const base = lds + place + half * 8192 + at;
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = *(const bf16x8 *)(base + i * 2048);
    };
    auto read_w = [&](int from, int run, bf16x8 (&to)[2]) {
        const unsigned char *const base = lds + from + 16384 + wave_n * 8192 + run * 4096 + at;
#pragma unroll
        for (int j = 0; j < 2; j++) to[j] = *(const bf16x8 *)(base + j * 2048);
    };
    auto multiply = [&](auto half_, auto odd_) {
        constexpr int half = decltype(half_)::value, odd = decltype(odd_)::value;
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                acc[half][i][j / 2][j % 2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(j < 2 ? first_run[odd][j] : second_run[j - 2], x[i], acc[half][i][j / 2][j % 2], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
        wide_meet();
    };
    constexpr std::integral_constant<int, 0> c0{};
    constexpr std::integral_constant<int, 1> c1{};
    // The first run of a tile's columns is read a phase early, so that both phases of a tile read six fragments.  LEFT: tiles
    // of K that follow, where they are few.
    request_columns(0, place, c0);
    request_rows(0, place, 0), request_columns(0, place, c1);
    request_rows(0, place, 1), request_columns(1, next_place, c0);
    request_rows(1, next_place, 0), request_columns(1, next_place, c1);
    request_rows(1, next_place, 1), request_columns(2, far_place, c0);
    asm volatile("s_waitcnt vmcnt(9)" ::: "memory");
    wide_meet();
    if (group) wide_meet();
    auto k_tile = [&](int t, auto odd_, auto left_) {
        constexpr int odd = decltype(odd_)::value, left = decltype(left_)::value;
        constexpr std::integral_constant<int, odd> parity{};
        read_x(0), read_w(place, 1, second_run);
        if constexpr (left >= 2) request_rows(t + 2, far_place, 0), request_columns(t + 2, far_place, c1);
        wide_operands<left >= 2 ? 9 : left == 1 ? 4 : 0>(), multiply(c0, parity);
        read_x(1);
        if constexpr (left >= 1) read_w(next_place, 0, first_run[1 - odd]);
        if constexpr (left >= 2) request_rows(t + 2, far_place, 1);
        if constexpr (left >= 3) request_columns(t + 3, place, c0);
        wide_operands<left >= 3 ? 9 : left == 2 ? 7 : left == 1 ? 1 : 0>(), multiply(c1, parity);
        const int passed = place;
        place = next_place, next_place = far_place, far_place = passed;
    };
    constexpr std::integral_constant<int, 3> many{};
    int t = 0;
    if (steps % 2 == 0) {  // an odd number before the last three
        read_w(place, 0, first_run[1]);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        k_tile(t++, c1, many);
    } else {
        read_w(place, 0, first_run[0]);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    for (; t + 3 < steps; t += 2) k_tile(t, c0, many), k_tile(t + 1, c1, many);
    k_tile(t, c0, std::integral_constant<int, 2>{});
    k_tile(t + 1, c1, c1);
    k_tile(t + 2, c0, c0);
    if (!group) wide_meet();

    const int first = tile.n * 256 + wave_n * 64;
    auto row_of = [&](int i) { return tile.m * 128 + group * 64 + i * 16 + r16; };
    // the residual stream's values arrive while the groups' sums meet
    const __amdgpu_buffer_rsrc_t h_buffer = buffer_of(a.out + (size_t)tile.m * 128 * a.n, (uint32_t)min(128, a.rows - tile.m * 128) * a.n * 2);
    u32x4 old[8];
    auto h_off = [&](int i) {
        const int column = first + i % 2 * 32 + g * 8;
        return column < a.n ? ((uint32_t)(row_of(i / 2) - tile.m * 128) * a.n + column) * 2 : kOutside;
    };
    auto load_residual = [&]() {
#pragma unroll
        for (int i = 0; i < 8; i++) old[i] = __builtin_amdgcn_raw_buffer_load_b128(h_buffer, h_off(i), 0, 0);
    };
    if (EPI == kTileResidual && gridDim.y == 1) load_residual();
    // each group hands over the half of the rows that the other finishes, and adds the other's sums of its own
    f32x4 *const other = (f32x4 *)lds;
    f32x4 sum[4][2][2];
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const f32x4 lower = acc[0][i / 4][i / 2 % 2][i % 2], upper = acc[1][i / 4][i / 2 % 2][i % 2];
        other[(wave * 16 + i) * 64 + lane] = group ? lower : upper;
        sum[i / 4][i / 2 % 2][i % 2] = group ? upper : lower;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; i++) sum[i / 4][i / 2 % 2][i % 2] += other[((wave ^ 4) * 16 + i) * 64 + lane];

    if (gridDim.y > 1) {
        // the last block of a tile to arrive adds all their sums in the order of K, as in tile_kernel
        // (16 bytes a lane where that kernel moves 8: sc1, past the XCDs' L2 caches)
        const int index = tile.m * n_tiles + tile.n;
        constexpr int kPast = 16;
        const __amdgpu_buffer_rsrc_t sums = buffer_of(a.partial + (size_t)index * gridDim.y * 32768, gridDim.y * 131072);
#pragma unroll
        for (int i = 0; i < 16; i++)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, sum[i / 4][i / 2 % 2][i % 2]), sums, (blockIdx.y * 16 + i) * 8192 + threadIdx.x * 16, 0, kPast);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();  // also: the last reads of `other`
        int *const last = (int *)lds;
        if (threadIdx.x == 0) {
            const int before = __hip_atomic_fetch_add((MK_GLOBAL int *)a.arrived + index, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *last = before + 1 == (int)gridDim.y;
            if (*last) __hip_atomic_store((MK_GLOBAL int *)a.arrived + index, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (!*last) return;
#pragma unroll
        for (int i = 0; i < 16; i++) sum[i / 4][i / 2 % 2][i % 2] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int y = 0; y < (int)gridDim.y; y++)
#pragma unroll
            for (int i = 0; i < 16; i++)
                sum[i / 4][i / 2 % 2][i % 2] += __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(sums, (y * 16 + i) * 8192 + threadIdx.x * 16, 0, kPast));
    }
    if constexpr (EPI == kTileRope) {
        __syncthreads();  // the last reads of LDS
        wide_tables(a, lds, wave, lane, [&](int line) { return tile.m * 128 + line; });
        wide_rope(a, lds, first, g, group * 64 + r16, row_of, [&](int i) -> const f32x4(&)[2][2] { return sum[i]; });
    } else if constexpr (EPI == kTileArgmax) {
        wide_best<4>(a, first, g, row_of, [&](int i) -> const f32x4(&)[2][2] { return sum[i]; });
    } else if constexpr (EPI == kTileSilu) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (row_of(i) < a.rows && first / 2 + g * 8 < a.n) *(u32x4 *)(a.out + (size_t)row_of(i) * a.n + first / 2 + g * 8) = wide_silu(sum[i]);
    } else {
        if (gridDim.y > 1) load_residual();
#pragma unroll
        for (int i = 0; i < 8; i++) __builtin_amdgcn_raw_buffer_store_b128(wide_add(old[i], sum[i / 2][i % 2]), h_buffer, h_off(i), 0, 0);
    }
}
