// Matrix products with many rows (prompts): C = A . W^T for bfloat16 A [M, K] (row-major) and the same packed
// weight the streaming kernel reads ([N/16][K/32][4][16][8]), on v_mfma_f32_16x16x32_bf16.
//
// A workgroup of 8 waves (two on every SIMD) owns a 256 x 256 tile of C, a wave 128 x 64 of it (8 x 4 MFMA tiles,
// 128 accumulator registers); or a tile of 192, 160 or 128 rows (a wave 6, 5 or 4 row tiles), where tiles of 256
// rows would leave many compute units without one. k is walked in stages of 64. A stage's 256 rows of A and of W (64 KB) are brought
// into LDS slots (two of A, three of W) by direct global-to-LDS loads, 1 KB a wave-wide instruction: of A 8 rows of 128 bytes
// (whole cache lines: with half lines, 64 bytes of 16 rows, the loads alone take a quarter longer), of W a piece as
// it lies in memory. A row's eight 16-byte chunks are stored at places exchanged by (row / 2), so that the 64 lanes
// of an operand read (row = lane % 16, chunk = 4 step + lane / 16) fall on all banks.
// A wave holds the operands of two k steps of 32 in registers: while it multiplies one step's (32 products), the
// next step's 12 reads from LDS are issued between the products, one after every second, and a stage's eight loads likewise
// (tiled_operands.h): a compute unit takes a load in 16 cycles, and asked for in one go, as before, 64 of them held the
// products up for a third of a stage. The reads and the products are volatile asm, which pins their order;
// the compiler neither sees the reads (and so orders nothing against the loads in flight) nor moves the products.
// Bound by the matrix units at the clock the power cap leaves (65 % busy, 1.94 GHz; products alone 2.0 PFLOP/s), the instructions beside them and a tile's
// start and end: loads alone take 0.7 us a stage of 1.5, and no wait for them or for the workgroup shows. So loads go through buffer descriptors
// (one instruction and a place in LDS instead of a 64-bit address each), and the first two stages of a workgroup's next tile are on their way
// while a tile's results are made and stored. Gated, before and after, 1.03 to 1.05 times as fast: 8192 x 37888 x 3584 1633 -> 1575 us (1.41 PFLOP/s), 16301 rows
// 3230 -> 3109, 2048 rows 439 -> 418, 8192 x 16384 x 2048 425 -> 404, 3584 rows 199 -> 189, 2048 x 9728 x 896 37.0 -> 35.2; float32, 2048 x 3584 x 18944 in two
// parts 225 -> 210. Four waves of 128 x 128, accumulators in the other half of the registers: the stages 5 % faster still, a tile's start and
// end, with nothing beside a wave that waits, 2 us longer (2048 x 9728 x 896 39.0). Two tiles at a time are more than the scalar registers hold: 16 to 30 of
// them wait in lanes of a vector register in the gated forms, 38 to 42 in that of queries, keys and values, 0 to 4 in the others; three are read back in the
// block of a tile's first stage, the others between tiles, none in the loop of the stages.
// Workgroups are numbered so that the 32 that run together on one of the 8 XCDs (each with a second-level cache of
// its own) own about 4 x 8 neighbouring tiles of C, and so share their rows of A and of W there, and so that every
// XCD gets the same number of tiles.
#include "cache_layout.h"
#include "common.h"
#include "microllm_hip.h"
#include "tiled_operands.h"

namespace mll {

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int kTileN = 256;
constexpr int kPieceElements = 512;                       // of W: 16 rows x 32 k in MFMA operand order, 1 KB
constexpr int kPackedStep = 1024;                         // from a tile's first k step to its second in a slot
constexpr int kSuperM = 4, kSuperN = 8;                   // tiles of C that run together on an XCD

// EPILOGUE: 0 = float32 [M, N]; 1 = bfloat16 [M, N]; 2 = bfloat16 [M, N / 2] = silu(even rows of W) * (odd rows);
// 3 = queries, keys and values: bias, rotation, queries to `store.q_out`, keys and values into their pages (W's rows
// in rotary pair order; see MllQkvStore); 5 = 2 with GELU; 7 = 2 with clamped gates, from the float32 sums (`limit`, `slope`).
// WM: a workgroup's tile of C has 32 WM rows (a wave WM row tiles of 16), 4 to 8: fewer where 256 rows a tile would
// leave many compute units without one.
// With epilogue 0 the stages of k may be dealt to gridDim.y workgroups, each writing its own [M, N] of partial sums.
template <int EPILOGUE, int WM>
__global__ __launch_bounds__(kTiledThreads, 1) void gemm_tiled_kernel(const bf16* __restrict__ a, const bf16* __restrict__ w_packed,
                                                                      void* __restrict__ out, int m, int n, int k, int n_tiles,
                                                                      int k_steps, int m_blocks, int n_blocks, int whole_rows,
                                                                      MllQkvStore store, float limit, float slope) {
    static_assert(WM >= 4 && WM <= kMaxWaveTilesM, "a wave takes 4 to 8 row tiles");
    constexpr int TILE_M = 32 * WM;
    constexpr int A_LOADS = 4 * WM;                       // a stage of A: 2 WM pieces of 16 rows, two loads of 8 rows each
    constexpr int A_TURNS = (A_LOADS + kTiledWaves - 1) / kTiledWaves;
    // Two slots of A, each [2 WM pieces of 16 rows][row][8 places of 16 bytes], the row's chunk c of 8 elements at place c ^ (row / 2); then three of W, each
    // [16 tiles][2 k steps][1 KB in MFMA operand order]. While stages are multiplied the direct loads alone write this memory and the asm reads alone read
    // it. Gated results pass through the last slot as rows, while the next tile's first two stages are on their way into the others.
    __shared__ __align__(kSlotsAlign) bf16 slots[kStageElements];

    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int col = lane % 16, quad = lane / 16;
    const int wave_m = wave / 4, wave_n = wave % 4;        // which (16 WM) x 64 of the tile

    // Workgroups 8 apart in number run on one XCD, 32 of them at a time. The tiles of C are put in a row, blocks of
    // 4 x 8 neighbouring tiles after one another (down the rows of C first, narrower at the edges), and every XCD
    // takes an equal stretch of that row: the workgroups that run together there own neighbouring tiles, and no XCD
    // has more than one tile more than another.
    const int tiles = m_blocks * n_blocks;
    const int per_xcd = (tiles + 7) / 8;
    struct Place {
        int m_block, n_block;       // m_block < 0: none
    };
    auto place_of = [&](int index) __attribute__((always_inline)) {
        const int place = (blockIdx.x % 8) * per_xcd + index;
        if (index >= per_xcd || place >= tiles) return Place{-1, 0};
        const int column = place / (m_blocks * kSuperN);                       // of blocks, kSuperN tiles wide
        const int width = min(kSuperN, n_blocks - column * kSuperN);
        const int in_column = place - column * m_blocks * kSuperN;
        const int block = in_column / (kSuperM * width);                       // in the column, kSuperM tiles high
        const int height = min(kSuperM, m_blocks - block * kSuperM);
        const int in_block = in_column - block * kSuperM * width;
        return Place{block * kSuperM + in_block % height, column * kSuperN + in_block / height};
    };

    // What this wave copies per stage, through buffer descriptors: a load is then one instruction beside its place in LDS, where a global one
    // works out a 64-bit address (135 -> 60 vector and scalar instructions a stage of 64 products). Of A the loads wave, wave + 8, ... of the stage's
    // 4 WM: load i brings 8 rows (half h = i % 2 of piece i / 2; lane L: row L / 8 of the 8, place L % 8 of the row). Tiles of 160 rows have loads for
    // half the waves' third turn: the others repeat their second, the same bytes to the same place, since no wave may pass a load over
    // (tiled_operands.h). Of W tiles 2 * wave and 2 * wave + 1, a k step an instruction.
    auto a_load = [&](int turn) __attribute__((always_inline)) {
        const int load = wave + turn * kTiledWaves;
        return A_LOADS % kTiledWaves == 0 || load < A_LOADS ? load : load - kTiledWaves;
    };
    constexpr int kNowhere = 0x7fffffff;        // past what the descriptors hold
    __amdgpu_buffer_rsrc_t a_rsrc, w_rsrc;
    int a_offset[A_TURNS], w_offset[kWTurns / 2];    // of the lane's 16 bytes from the block's first row or tile, at stage 0, in bytes
    auto describe = [&](Place at) __attribute__((always_inline)) {
        const int m0 = at.m_block * TILE_M, n_tile0 = at.n_block * (kTileN / 16);
        a_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(a) + static_cast<int64_t>(m0) * k, 0, kNowhere, kBufferFlags);
#pragma unroll
        for (int t = 0; t < A_TURNS; ++t) {
            const int load = a_load(t);
            const int row_in_piece = 8 * (load % 2) + lane / 8;
            const int row = min((load / 2) * 16 + row_in_piece, m - 1 - m0);           // rows past the end repeat the last one
            a_offset[t] = (row * k + ((lane % 8) ^ (row_in_piece / 2)) * 8) * 2;
        }
        w_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(w_packed) + static_cast<int64_t>(n_tile0) * k_steps * kPieceElements, 0, kNowhere,
                                                   kBufferFlags);
#pragma unroll
        for (int p = 0; p < kWTurns / 2; ++p)
            w_offset[p] = min(wave * (kWTurns / 2) + p, n_tiles - 1 - n_tile0) * k_steps * (kPieceElements * 2) + lane * 16;
    };
    const int all_stages = (k_steps + 1) / 2;
    const int stages_per_split = (all_stages + gridDim.y - 1) / gridDim.y;
    const int first_stage = blockIdx.y * stages_per_split;
    const int stages = min(all_stages, first_stage + stages_per_split);
    auto copy_a = [&](int turn, int stage, unsigned slot) __attribute__((always_inline)) {
        // (arguments are worked out before the call: with a captured array's subscript in it the host pass drops the kernel's stub without a word)
        bf16* place = slots + slot * kSlotElements + a_load(turn) * 512;
        const int at = a_offset[turn];
        __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, place, 16, at, stage * 128, 0, 0);
    };
    auto copy_w = [&](int turn, int stage, unsigned slot) __attribute__((always_inline)) {      // turn: which of the wave's two tiles and k steps
        const int p = turn / 2, h = turn % 2;
        bf16* place = slots + (kASlots + slot) * kSlotElements + (wave * (kWTurns / 2) + p) * 1024 + h * 512;
        const int at = w_offset[p], from = 2 * stage + h < k_steps ? (2 * stage + h) * (kPieceElements * 2) : kNowhere;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, place, 16, at, from, 0, 0);
    };
    // The stage of an odd number's last k step has no second one: the lanes that would bring its half of a row of A ask past the descriptor's end from
    // then on, as the loads of its pieces of W do, and get zeros. (Zeros on both sides: an infinity in a row's last elements times a zero would be no
    // number.) Once a tile, by asm so that it stays a branch: a choice at every load is four vector instructions a stage (2048 x 37888 x 3584 gated 425 -> 431 us).
    auto last_comes = [&]() __attribute__((always_inline)) {
        if (2 * stages - 1 != k_steps) return;
        const bool second_half = ((lane % 8) ^ (4 * (wave % 2) + lane / 16)) >= 4;      // the lane's chunk, the same in every load of the wave
        const int past = second_half ? static_cast<int>(0x80000000u) : 0;
#pragma unroll
        for (int t = 0; t < A_TURNS; ++t) asm volatile("v_or_b32 %0, %0, %1" : "+v"(a_offset[t]) : "v"(past));
    };
    // Where the lane reads its operands: row `col` of a piece, chunk 4 step + quad at its place.
    const unsigned base = lds_address(slots);
    const unsigned a_row = base + wave_m * WM * 2048 + col * 128;
    const unsigned a_step0 = a_row + ((quad ^ (col / 2)) * 16), a_step1 = a_row + (((4 + quad) ^ (col / 2)) * 16);
    const unsigned w_lane = base + kASlots * kSlotBytes + wave_n * kWaveTilesN * 2048 + lane * 16;

    constexpr bool GATED = EPILOGUE == 2 || EPILOGUE == 5 || EPILOGUE == 7;
    constexpr int STORES = GATED ? WM : 0;         // of a wave that stores a whole gated tile
    int index = blockIdx.x / 8;
    Place at = place_of(index), next;
    if (at.m_block < 0) return;
    const bool any = EPILOGUE != 0 || first_stage < stages;      // a part of the reduction may be empty
    if (any) {
        describe(at);
        begin_stages<A_TURNS>(first_stage, stages, copy_a, copy_w, last_comes);
    }
    bool stored = false;      // whether the wave issued STORES stores after the tile's first loads
    for (;; at = next) {
        index += gridDim.x / 8;
        next = place_of(index);
        const int m0 = at.m_block * TILE_M, n_tile0 = at.n_block * (kTileN / 16), n_block = at.n_block;
        floatx4 acc[kWaveTilesN][WM];     // acc[nt][mt][i] = C[m = mt*16 + col][n = nt*16 + quad*4 + i] of the wave's part
        if (any) {
            multiply_stages<kPackedStep, WM, A_TURNS, STORES>(acc, first_stage, stages, stored, a_step0, a_step1, w_lane, w_lane, copy_a, copy_w, last_comes);
            if (GATED || next.m_block >= 0) workgroup_meets();        // every wave is done with the slots
            if (next.m_block >= 0) {
                describe(next);
                begin_stages<A_TURNS>(first_stage, stages, copy_a, copy_w, last_comes);
            }
        } else {
#pragma unroll
            for (int nt = 0; nt < kWaveTilesN; ++nt)
#pragma unroll
                for (int mt = 0; mt < WM; ++mt) acc[nt][mt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        stored = false;

        if constexpr (EPILOGUE == 3) {
            // The lane's 4 columns of a tile lie in one head (head_dim is a multiple of 16). In a query or key head
            // columns 2p and 2p + 1 hold dims p and p + n_freq, the two that rotate together, so the lane's columns are
            // dims p, p + n_freq, p + 1, p + 1 + n_freq with p even: two neighbours in each half, stored as one word
            // each. Dims beyond the rotated ones, and values, are in place.
            const CacheLayout layout(store.kv_heads, store.page_size, store.head_dim);
#pragma unroll
            for (int nt = 0; nt < kWaveTilesN; ++nt) {
                const int column = (n_tile0 + wave_n * kWaveTilesN + nt) * 16 + quad * 4;
                if (column >= n) continue;
                const int head = column / store.head_dim, within = column % store.head_dim;
                const bool is_query = head < store.heads;
                const bool is_value = head >= store.heads + store.kv_heads;
                const bool rotate = !is_value && within + 3 < 2 * store.n_freq;        // both pairs or, n_freq being even here, none
                const int pair = within / 2;
                // dims of the lane's four results, in the order of the accumulator
                int dim[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) dim[i] = rotate ? pair + i / 2 + (i % 2) * store.n_freq : within + i;
                float bias[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                if (store.bias) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) bias[i] = store.bias[head * store.head_dim + dim[i]];
                }
#pragma unroll
                for (int mt = 0; mt < WM; ++mt) {
                    const int row = m0 + wave_m * (WM * 16) + mt * 16 + col;
                    if (row >= m) continue;
                    float y[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) y[i] = acc[nt][mt][i] + bias[i];
                    if (rotate) {
                        const floatx4 cs = *reinterpret_cast<const floatx4*>(store.cos_sin + (static_cast<int64_t>(row) * store.n_freq + pair) * 2);
                        const float x0 = y[0], x1 = y[1], x2 = y[2], x3 = y[3];
                        y[0] = rotate_first(x0, x1, cs[0], cs[1]);
                        y[1] = rotate_second(x0, x1, cs[0], cs[1]);
                        y[2] = rotate_first(x2, x3, cs[2], cs[3]);
                        y[3] = rotate_second(x2, x3, cs[2], cs[3]);
                    }
                    // y[0], y[2] are neighbours in dim (dim[0], dim[0] + 1) when rotated, and so are y[1], y[3]
                    bf16x2 low, high;
                    if (rotate) {
                        low[0] = static_cast<__bf16>(y[0]); low[1] = static_cast<__bf16>(y[2]);
                        high[0] = static_cast<__bf16>(y[1]); high[1] = static_cast<__bf16>(y[3]);
                    } else {
                        low[0] = static_cast<__bf16>(y[0]); low[1] = static_cast<__bf16>(y[1]);
                        high[0] = static_cast<__bf16>(y[2]); high[1] = static_cast<__bf16>(y[3]);
                    }
                    const int low_dim = dim[0], high_dim = rotate ? dim[1] : dim[2];
                    if (is_query) {
                        bf16* q_row = static_cast<bf16*>(store.q_out) + (static_cast<int64_t>(row) * store.heads + head) * store.head_dim;
                        *reinterpret_cast<bf16x2*>(q_row + low_dim) = low;
                        *reinterpret_cast<bf16x2*>(q_row + high_dim) = high;
                        continue;
                    }
                    if (!store.slot_mapping) continue;
                    const int slot = store.slot_mapping[row];
                    if (slot < 0) continue;
                    const int page = slot / store.page_size, offset = slot % store.page_size;
                    if (!is_value) {
                        bf16* pages = static_cast<bf16*>(store.k_cache);        // two neighbouring dims are neighbours in a page of keys
                        *reinterpret_cast<bf16x2*>(pages + layout.k_at(page, head - store.heads, offset, low_dim)) = low;
                        *reinterpret_cast<bf16x2*>(pages + layout.k_at(page, head - store.heads, offset, high_dim)) = high;
                    } else {
                        bf16* pages = static_cast<bf16*>(store.v_cache);        // and 8 elements apart in a page of values
                        const int kv_head = head - store.heads - store.kv_heads;
#pragma unroll
                        for (int i = 0; i < 4; ++i) pages[layout.v_at(page, kv_head, offset, within + i)] = from_float<bf16>(y[i]);
                    }
                }
            }
            if (next.m_block < 0) return;
            continue;
        }
        auto gated = [&](float gate, float up) {
            return EPILOGUE == 7 ? gated_value_fast(gate, up, kActClampedGlu, limit, slope) : gate_fast<EPILOGUE == 5>(gate) * up;
        };
        if constexpr (GATED) {
            if (whole_rows) {
                const int row0 = m0 + wave_m * (WM * 16), column = n_block * kResultColumns + wave_n * 32 + (lane % 4) * 8;
                stored = m0 + TILE_M <= m && (n_block + 1) * kResultColumns <= n / 2;
                const unsigned place = base + (kASlots + 2) * kSlotBytes + wave * (kResultRows * kResultBytes);
                const unsigned word_at = place + col * kResultBytes + (col / 4) * 16 + quad * 4;      // of tile 0; tile nt's chunk is exchanged with it
                bf16* to = static_cast<bf16*>(out) + static_cast<int64_t>(row0 + lane / 4) * (n / 2) + column;
                auto put_tiles = [&](auto mt) __attribute__((always_inline)) {
                    constexpr int MT = decltype(mt)::value;
#pragma unroll
                    for (int nt = 0; nt < kWaveTilesN; ++nt) {
                        bf16x2 two;
#pragma unroll
                        for (int i = 0; i < 2; ++i) two[i] = static_cast<__bf16>(gated(acc[nt][MT][2 * i], acc[nt][MT][2 * i + 1]));
                        put_result<MT % 4 * 16 * kResultBytes>(word_at ^ (nt * 16), __builtin_bit_cast(unsigned, two));
                    }
                };
                auto half = [&](auto first_tile) __attribute__((always_inline)) {
                    constexpr int FIRST = decltype(first_tile)::value, COUNT = WM - FIRST < 4 ? WM - FIRST : 4;
                    put_tiles(std::integral_constant<int, FIRST>{});
                    if constexpr (COUNT > 1) put_tiles(std::integral_constant<int, FIRST + (COUNT > 1)>{});
                    if constexpr (COUNT > 2) put_tiles(std::integral_constant<int, FIRST + 2 * (COUNT > 2)>{});
                    if constexpr (COUNT > 3) put_tiles(std::integral_constant<int, FIRST + 3 * (COUNT > 3)>{});
                    uintx4 piece[4];
                    get_results(piece, place, lane);      // 16 rows each; those past COUNT are stored by nobody
                    if (stored) {
#pragma unroll
                        for (int i = 0; i < COUNT; ++i) *reinterpret_cast<uintx4*>(to + static_cast<int64_t>((FIRST + i) * 16) * (n / 2)) = piece[i];
                    } else {
#pragma unroll
                        for (int i = 0; i < COUNT; ++i)
                            if (row0 + (FIRST + i) * 16 + lane / 4 < m && column < n / 2)
                                *reinterpret_cast<uintx4*>(to + static_cast<int64_t>((FIRST + i) * 16) * (n / 2)) = piece[i];
                    }
                };
                half(std::integral_constant<int, 0>{});
                if constexpr (WM > 4) half(std::integral_constant<int, 4>{});
                if (next.m_block < 0) return;
                continue;
            }
        }
#pragma unroll
        for (int mt = 0; mt < WM; ++mt) {
            const int row = m0 + wave_m * (WM * 16) + mt * 16 + col;
            if (row >= m) continue;
#pragma unroll
            for (int nt = 0; nt < kWaveTilesN; ++nt) {
                const int column = (n_tile0 + wave_n * kWaveTilesN + nt) * 16 + quad * 4;
                if (EPILOGUE == 0) {
                    float* target = static_cast<float*>(out) + (static_cast<int64_t>(blockIdx.y) * m + row) * n + column;
                    if (column + 3 < n && n % 4 == 0) {
                        *reinterpret_cast<floatx4*>(target) = acc[nt][mt];
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            if (column + i < n) target[i] = acc[nt][mt][i];
                    }
                } else if (EPILOGUE == 1) {
                    bf16* target = static_cast<bf16*>(out) + static_cast<int64_t>(row) * n + column;
                    if (column + 3 < n && n % 4 == 0) {
                        bf16x4 four;
#pragma unroll
                        for (int i = 0; i < 4; ++i) four[i] = static_cast<__bf16>(acc[nt][mt][i]);
                        *reinterpret_cast<bf16x4*>(target) = four;
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            if (column + i < n) target[i] = from_float<bf16>(acc[nt][mt][i]);
                    }
                } else {
                    bf16* target = static_cast<bf16*>(out) + static_cast<int64_t>(row) * (n / 2) + column / 2;
                    if (column + 3 < n && n % 4 == 0) {
                        bf16x2 two;
#pragma unroll
                        for (int i = 0; i < 2; ++i) two[i] = static_cast<__bf16>(gated(acc[nt][mt][2 * i], acc[nt][mt][2 * i + 1]));
                        *reinterpret_cast<bf16x2*>(target) = two;
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; i += 2)
                            if (column + i < n) target[i / 2] = from_float<bf16>(gated(acc[nt][mt][i], acc[nt][mt][i + 1]));
                    }
                }
            }
        }
        if (next.m_block < 0) return;
    }
}

template <int EPILOGUE, int WM>
static int launch_tiled_rows(const void* a, const void* w_packed, void* out, int m, int n, int k, int splits, hipStream_t stream,
                             const MllQkvStore& store, float limit, float slope) {
    const int n_tiles = (n + 15) / 16, k_steps = k / 32;
    const int m_blocks = (m + 32 * WM - 1) / (32 * WM), n_blocks = (n + kTileN - 1) / kTileN;
    // As many workgroups as run at once go from tile to tile; parts of the reduction are workgroups of their own.
    const int all = 8 * ((m_blocks * n_blocks + 7) / 8);
    const dim3 grid(splits > 1 ? all : min(all, 256), splits);
    const int whole_rows = n % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;      // of a gated result: pieces of 16 bytes
    gemm_tiled_kernel<EPILOGUE, WM><<<grid, kTiledThreads, 0, stream>>>(static_cast<const bf16*>(a), static_cast<const bf16*>(w_packed),
                                                                        out, m, n, k, n_tiles, k_steps, m_blocks, n_blocks, whole_rows, store, limit, slope);
    return check_launch("gemm_tiled");
}

// How many rows a workgroup's tile gets: the height that is done first, if every round of 256 workgroups takes a time of rows + 256. 2048 x 4608
// in tiles of 256 rows is 144 tiles, a round in which 112 compute units have none; in tiles of 160 rows 234. The model is that of a stage's loads, which
// bounded this kernel when it was drawn; the products that bound it now would say rows plus less. It is kept because what it chooses was measured again and
// because the rules of who takes a product (how full its rounds are) are drawn by it: over 8 weights from 1152 x 896 to 37888 x 3584 and 16 numbers of rows
// from 128 to 8192 its height takes 1.005 times the best one's time on the mean gated, 1.003 in float32, and in 8 of the 128 sizes 1.04 to 1.10 times (2560 x 9728 x
// 896, 1792 x 13824 x 4096, 8192 x 4608 x 3584); rows + 64 would be within 1.02 everywhere.
// Every output's additions are the same whatever the height.
static int choose_tile_rows(int m, int n, int splits) {
    const int n_blocks = (n + kTileN - 1) / kTileN;
    int best = 256;
    int64_t best_cost = -1;
    for (int rows : {256, 192, 160, 128}) {
        const int64_t blocks = static_cast<int64_t>((m + rows - 1) / rows) * n_blocks * splits;
        const int64_t cost = ((blocks + 255) / 256) * (rows + kTileN);
        if (best_cost < 0 || cost < best_cost) best = rows, best_cost = cost;
    }
    return best;
}

template <int EPILOGUE>
static int launch_tiled(const void* a, const void* w_packed, void* out, int m, int n, int k, int splits, int tile_rows,
                        hipStream_t stream, const MllQkvStore& store = MllQkvStore{}, float limit = 0.0f, float slope = 0.0f) {
    if (tile_rows == 0) tile_rows = choose_tile_rows(m, n, splits);
    switch (tile_rows) {
        case 256: return launch_tiled_rows<EPILOGUE, 8>(a, w_packed, out, m, n, k, splits, stream, store, limit, slope);
        case 192: return launch_tiled_rows<EPILOGUE, 6>(a, w_packed, out, m, n, k, splits, stream, store, limit, slope);
        case 160: return launch_tiled_rows<EPILOGUE, 5>(a, w_packed, out, m, n, k, splits, stream, store, limit, slope);
        case 128: return launch_tiled_rows<EPILOGUE, 4>(a, w_packed, out, m, n, k, splits, stream, store, limit, slope);
        default: return fail("gemm_tiled: a tile has 256, 192, 160 or 128 rows (0: chosen here)");
    }
}

}  // namespace mll

using namespace mll;

extern "C" int mll_tiled_tile_rows(int m, int n, int splits) { return choose_tile_rows(m, n, splits < 1 ? 1 : splits); }

extern "C" int mll_gemm_tiled(const void* a, const void* w_packed, void* out, int epilogue, int m, int n, int k,
                              int splits, int tile_rows, hipStream_t stream) {
    MLL_REQUIRE(m >= 0 && n > 0 && k > 0, "gemm_tiled: sizes must be positive");
    MLL_REQUIRE(k % 32 == 0, "gemm_tiled: k must be a multiple of 32");
    MLL_REQUIRE(splits >= 1 && splits <= 64 && (splits == 1 || epilogue == 0), "gemm_tiled: only the float32 epilogue takes k in parts");
    MLL_REQUIRE(static_cast<int64_t>(kTileN) * k < (int64_t{1} << 30), "gemm_tiled: k is too long");
    MLL_REQUIRE((epilogue != 2 && epilogue != 5) || n % 2 == 0, "gemm_tiled: the gated epilogue needs an even number of weight rows");
    MLL_REQUIRE(reinterpret_cast<uintptr_t>(a) % 16 == 0, "gemm_tiled: the activations must be 16-byte aligned");
    if (m == 0) return 0;
    switch (epilogue) {
        case 0: return launch_tiled<0>(a, w_packed, out, m, n, k, splits, tile_rows, stream);
        case 1: return launch_tiled<1>(a, w_packed, out, m, n, k, splits, tile_rows, stream);
        case 2: return launch_tiled<2>(a, w_packed, out, m, n, k, splits, tile_rows, stream);
        case 5: return launch_tiled<5>(a, w_packed, out, m, n, k, splits, tile_rows, stream);
        default: return fail("gemm_tiled: unknown epilogue");
    }
}

extern "C" int mll_gemm_tiled_clamped(const void* a, const void* w_packed, void* out, int m, int n, int k, float limit, float slope,
                                      int tile_rows, hipStream_t stream) {
    MLL_REQUIRE(m >= 0 && n > 0 && n % 2 == 0 && k > 0 && k % 32 == 0, "gemm_tiled_clamped: an even number of weight rows, k a multiple of 32");
    MLL_REQUIRE(static_cast<int64_t>(kTileN) * k < (int64_t{1} << 30), "gemm_tiled_clamped: k is too long");
    MLL_REQUIRE(reinterpret_cast<uintptr_t>(a) % 16 == 0, "gemm_tiled_clamped: the activations must be 16-byte aligned");
    MLL_REQUIRE(limit > 0.0f, "gemm_tiled_clamped: the limit must be positive");
    if (m == 0) return 0;
    return launch_tiled<7>(a, w_packed, out, m, n, k, 1, tile_rows, stream, MllQkvStore{}, limit, slope);
}

extern "C" int mll_gemm_tiled_qkv(const void* a, const void* w_packed, int m, int k, const MllQkvStore* store, int tile_rows,
                                  hipStream_t stream) {
    MLL_REQUIRE(store != nullptr, "gemm_tiled_qkv: no store");
    MLL_REQUIRE(m >= 0 && k > 0 && k % 32 == 0, "gemm_tiled_qkv: k must be a positive multiple of 32");
    MLL_REQUIRE(static_cast<int64_t>(kTileN) * k < (int64_t{1} << 30), "gemm_tiled_qkv: k is too long");
    MLL_REQUIRE(store->heads > 0 && store->kv_heads >= 0 && store->head_dim > 0 && store->head_dim % 16 == 0,
                "gemm_tiled_qkv: head_dim must be a multiple of 16");
    MLL_REQUIRE(store->n_freq >= 0 && store->n_freq % 2 == 0 && 2 * store->n_freq <= store->head_dim,
                "gemm_tiled_qkv: the number of rotary pairs must be even and at most head_dim / 2");
    MLL_REQUIRE(store->n_freq == 0 || (store->cos_sin && reinterpret_cast<uintptr_t>(store->cos_sin) % 16 == 0),
                "gemm_tiled_qkv: rotation needs a 16-byte aligned cos/sin table");
    MLL_REQUIRE(store->q_out && reinterpret_cast<uintptr_t>(store->q_out) % 4 == 0, "gemm_tiled_qkv: no place for the queries");
    MLL_REQUIRE(!store->slot_mapping || (store->k_cache && store->v_cache && store->page_size > 0 && store->page_size % 16 == 0),
                "gemm_tiled_qkv: a slot mapping needs both caches and pages of a multiple of 16 positions");
    MLL_REQUIRE(reinterpret_cast<uintptr_t>(a) % 16 == 0, "gemm_tiled_qkv: the activations must be 16-byte aligned");
    if (m == 0) return 0;
    const int n = (store->heads + 2 * store->kv_heads) * store->head_dim;
    return launch_tiled<3>(a, w_packed, nullptr, m, n, k, 1, tile_rows, stream, *store);
}
