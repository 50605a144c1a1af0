// Matrix products with few rows (decoding): C = A . W^T for bfloat16 A [M <= 64, K] and a weight that was
// packed once, at load time, into the order the MFMA consumes it, so that a wave streams its 16 rows of W as
// consecutive 1 KB pieces. The kernel is bound by reading W once from HBM.
//
// Packed layout: [N/16][K/32][quad 0..3][row 0..15][8 elements]; lane (row + 16 * quad) of a wave reads its
// 16 bytes of piece (n_tile, k_step) at byte offset lane * 16: the A operand of v_mfma_f32_16x16x32_bf16.
// The product is computed transposed (C^T = W . A^T): the activations are the B operand, 16 rows per tile.
// A workgroup owns NT tiles of W; its waves (1 to 16, see skinny_waves) take a run of the k steps each and their sums
// are added in wave order through LDS: the result is the same in every run and does not depend on the other rows of A.
#include "cache_layout.h"
#include "common.h"
#include "microllm_hip.h"

#include <type_traits>

namespace mll {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int uintx4 __attribute__((ext_vector_type(4)));


constexpr int kNonTemporal = 2;
constexpr int kChunk = 4;     // k steps a wave takes in a row, then skips what the other waves take

union Piece {
    bf16x8 v;
    uintx4 raw;
};

// The value of the lane ROWS * steps places further on within every 16 lanes, wrapping round.
template <int ROWS>
__device__ inline unsigned turn_lanes(unsigned value, int steps) {
    const int v = static_cast<int>(value);
    switch (steps) {        // a constant after unrolling; 0x120 + r: row_ror by r lanes
        case 1: return static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, v, 0x120 + 16 - ROWS, 0xf, 0xf, false));
        case 2: return static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, v, 0x120 + (2 * ROWS < 16 ? 16 - 2 * ROWS : 1), 0xf, 0xf, false));
        case 3: return static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, v, 0x120 + (3 * ROWS < 16 ? 16 - 3 * ROWS : 1), 0xf, 0xf, false));
        default: return value;
    }
}

// EPILOGUE: 0 = float32 [M, N]; 1 = bfloat16 [M, N]; 2 = bfloat16 [M, N / 2] = silu(even rows of W) * (odd rows).
// 3 = the q/k/v projection of an attention layer finished in place: bias, rotation of the position, queries to
// `q_out`, keys and values into their pages (at most 16 rows; see MllQkvStore). 4 = the product is added to the
// float32 residual stream and the sum, times the next norm's weight, is written as the next product's input,
// with each workgroup's share of the rows' sums of squares (at most 16 rows; see MllResidualNorm).
// 5 = 2 with the tanh form of gelu for silu. 6 = bfloat16 [M, N] = gelu_tanh(product) * the token's columns of a side
// table (at most 16 rows; see MllSideTable). 7 = 2 with the clamped form (gated_value in common.h; at most 16 rows).
// Whatever the epilogue, a row of the product is first multiplied by the factor that MllRowScale describes,
// if one is given (at most 16 rows).
// W is read past the caches (non-temporal loads): a step reads every weight once, and all of them together are far
// more than the caches hold. Measured on MI355X inside the decode step, against ordinary loads for weights under 64 MB:
// 7B sizes +1 % at batch 8, +1.6 % at batch 1, +0.7 % at batch 64; 0.5B sizes +4 % at batch 1, the same otherwise.
// HALF: a workgroup owns 8 rows of W instead of 16 (half a tile), for weights whose tiles alone would leave compute
// units idle: a wave's A operand holds the 8 rows at one k step in its first 8 rows and at the next step in its last 8,
// and the B operand 8 rows of the activations at the first step and again at the next, so that the product's upper left
// 8 x 8 is the even step's and its lower right 8 x 8 the odd step's; the other two quarters are read by nobody. MT counts
// 8 rows of the activations then. SPLIT (more than 16 rows, and epilogue 3): the same sums in the same order with whole tiles. FAR: 64-bit addresses
// and loads under conditions, for reductions beyond what a descriptor's 32-bit offsets reach.
template <int MT, int NT, int EPILOGUE, bool SCALED, int GROUP, int HALF, bool SPLIT, bool FAR>
__global__ __launch_bounds__(1024) void gemm_skinny_kernel(
    const bf16* __restrict__ a, const bf16* __restrict__ w_packed, void* __restrict__ out,
    int m, int n, int k, int n_tiles, int k_steps, MllSkinnyExtras extras) {
    extern __shared__ float reduce_shared[];
    const MllQkvStore& store = extras.store;   // [waves][NT * MT][64 lanes][4]
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int waves = blockDim.x / kWave;
    const int col = lane % 16, quad = lane / 16;
    constexpr int TILE = HALF ? 8 : 16;         // columns of the result a tile has, and rows of A a group of MT
    const int tile0 = blockIdx.x * NT;          // in halves of tiles with HALF, as is n_tiles
    const int token = HALF ? col % 8 : col;     // the row of A (of 8 or 16) that the lane's accumulators belong to
    const bool mine = !HALF || (col < 8 && quad < 2);       // whether they are results

    constexpr int SETS = SPLIT ? 2 : 1;         // sums of even and of odd steps apart
    floatx4 sums[SETS][NT][MT];
#pragma unroll
    for (int set = 0; set < SETS; ++set)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) sums[set][nt][mt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    // The waves take runs of kChunk k steps in turn, so that a workgroup reads one stretch of W at a time. Operands come
    // through buffer descriptors, whose loads give zeros past the end of what they describe: no branch stands between two
    // loads, so the compiler counts those in flight instead of waiting for all of them. A wave keeps two blocks of loads
    // on their way; with few steps a wave everything is asked for at once, before the epilogue's own loads.
    constexpr int kPast = 0x7ffffff0, kPastRow = 0x40000000;       // offsets past the end of every descriptor here
    constexpr bool kHolds = EPILOGUE == 3 || EPILOGUE == 4 || EPILOGUE == 6;     // the epilogue holds values of its own meanwhile
    // loads of W a tile and block: what stays in 128 registers beside the sums and those values
    constexpr int DEPTH = HALF ? HALF * kChunk / 2 : (MT + NT <= 3) ? (kHolds && NT == 2 && GROUP <= (EPILOGUE == 3 ? 2 : 1) ? 2 : 4) : MT <= 2 ? 2 : 1;
    __amdgpu_buffer_rsrc_t w_rsrc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const bool live = tile0 + nt < n_tiles;
        const int whole = (live ? tile0 + nt : tile0) / (HALF ? 2 : 1);
        w_rsrc[nt] = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(w_packed) + static_cast<int64_t>(whole) * k_steps * 512, 0,
                                                       live ? k_steps * 1024 : 0, kBufferFlags);
    }
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(a), 0, m * k * 2, kBufferFlags);
    // Whole tiles and one group of rows: an A load brings GROUP steps of 16 / GROUP rows instead of one step of 16 (rows
    // of which most may be none): lane `col` of 16 reads row col % (16 / GROUP) at step col / (16 / GROUP) of the group. Step u's
    // operand is the loaded one turned by u * 16 / GROUP lanes; what then lies in the columns past the rows belongs to
    // other steps and goes into columns of the product that nobody reads. GROUP 1 (9 to 16 rows): two steps are read at a
    // time: lanes 0..7 of every 16 read rows 0..7 (then 8..15) at one step and lanes 8..15 the same rows at the next, so
    // that a load touches whole 128-byte lines of 8 rows instead of half lines of 16; lanes 8 apart then exchange what the
    // other needs. With HALF that same load is the operand as it is.
    constexpr bool PAIRED = MT == 1 && GROUP == 1 && !HALF;
    constexpr int GROUP_ROWS = HALF ? 8 : 16 / GROUP;
    const bool upper = col >= 8;
    // Where a lane reads W and A at step 0; for a row that is none, past the end (and with every step's offset added to it).
    const int w_at = HALF ? (col / 8) * 1024 + quad * 256 + (tile0 % 2) * 128 + (col % 8) * 16 : lane * 16;
    const int a_lane = (HALF ? (col / 8) * 64 : GROUP > 1 ? (col / GROUP_ROWS) * 64 : PAIRED && upper ? 64 : 0) + quad * 16;
    int a_row[MT == 1 ? 2 : MT], a_at[MT == 1 ? 2 : MT];
#pragma unroll
    for (int i = 0; i < (MT == 1 ? 2 : MT); ++i) {
        a_row[i] = HALF ? i * 8 + token : GROUP > 1 ? col % GROUP_ROWS : PAIRED ? (col & 7) + 8 * i : i * 16 + col;
        a_at[i] = a_row[i] < m ? a_row[i] * k * 2 + a_lane : kPastRow;
    }
    const int k_left = k - quad * 8 - (HALF || GROUP > 1 ? col / GROUP_ROWS : (PAIRED && upper)) * 32;     // a lane reads A at steps below this many elements

    auto load_w = [&](int nt, int step) -> uintx4 {
        if constexpr (FAR) {
            const bool there = tile0 + nt < n_tiles && step + (HALF ? col / 8 : 0) < k_steps;
            const int64_t at = (static_cast<int64_t>((tile0 + nt) / (HALF ? 2 : 1)) * k_steps + step) * 1024 + w_at;
            return there ? *reinterpret_cast<const uintx4*>(reinterpret_cast<const char*>(w_packed) + at) : uintx4{0u, 0u, 0u, 0u};
        } else {
            return __builtin_amdgcn_raw_buffer_load_b128(w_rsrc[nt], w_at + step * 1024, 0, kNonTemporal);
        }
    };
    auto load_a = [&](int i, int step) -> uintx4 {
        if constexpr (FAR) {
            const bool there = a_row[i] < m && static_cast<int64_t>(step) * 32 < k_left;
            const int64_t at = static_cast<int64_t>(a_row[i]) * k * 2 + a_lane + static_cast<int64_t>(step) * 64;
            return there ? *reinterpret_cast<const uintx4*>(reinterpret_cast<const char*>(a) + at) : uintx4{0u, 0u, 0u, 0u};
        } else {
            return __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, step * 32 < k_left ? a_at[i] + step * 64 : kPast, 0, 0);
        }
    };
    auto load = [&](int block, Piece (&w_piece)[DEPTH][NT], Piece (&a_piece)[DEPTH][MT]) {
#pragma unroll
        for (int u = 0; u < DEPTH; ++u) {
            const int run = HALF ? block * HALF + u / (kChunk / 2) : block * DEPTH / kChunk;     // the wave's run of steps, and the step in it
            const int within = HALF ? u % (kChunk / 2) * 2 : block * DEPTH % kChunk + u;
            const int step = (run * waves + wave) * kChunk + within;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                w_piece[u][nt].raw = load_w(nt, step);
            if constexpr (GROUP > 1 && !HALF) {
                if (u % GROUP == 0)
                    a_piece[u][0].raw = load_a(0, step);
            } else if constexpr (PAIRED) {
                // a_piece[u] of an even u: rows 0..7 (both steps of the pair); of the odd u after it: rows 8..15
                const int pair = step - (u & 1);
                a_piece[u][0].raw = load_a(u & 1, pair);
            } else {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    a_piece[u][mt].raw = load_a(mt, step);
            }
        }
    };
    auto multiply = [&](Piece (&w_piece)[DEPTH][NT], Piece (&a_piece)[DEPTH][MT], auto block) {     // block: of the two, the even or the odd one
        if constexpr (GROUP > 1 && !HALF) {
#pragma unroll
            for (int u = 0; u < DEPTH; ++u)
                if (u % GROUP != 0) {
                    const uintx4 loaded = a_piece[u - u % GROUP][0].raw;
#pragma unroll
                    for (int i = 0; i < 4; ++i) a_piece[u][0].raw[i] = turn_lanes<GROUP_ROWS>(loaded[i], u % GROUP);
                }
        } else if constexpr (PAIRED) {
            // low = rows 0..7 at the pair's first step (lanes 0..7) and its second (lanes 8..15), high = rows
            // 8..15 likewise. The first step's operand: own low | the partner's high; the second's: the partner's
            // low | own high.
#pragma unroll
            for (int u = 0; u < DEPTH; u += 2) {
                const uintx4 low = a_piece[u][0].raw, high = a_piece[u + 1][0].raw;
                uintx4 low_swapped, high_swapped;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    low_swapped[i] = turn_lanes<8>(low[i], 1);
                    high_swapped[i] = turn_lanes<8>(high[i], 1);
                }
                a_piece[u][0].raw = upper ? high_swapped : low;
                a_piece[u + 1][0].raw = upper ? high : low_swapped;
            }
        }
#pragma unroll
        for (int u = 0; u < DEPTH; ++u)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    floatx4& sum = sums[(decltype(block)::value * DEPTH + u) % SETS][nt][mt];
                    sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w_piece[u][nt].v, a_piece[u][mt].v, sum, 0, 0, 0);
                }
    };
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    Piece w_even[DEPTH][NT], w_odd[DEPTH][NT], a_even[DEPTH][MT], a_odd[DEPTH][MT];
    load(0, w_even, a_even);
    load(1, w_odd, a_odd);

    // What the epilogue reads beside the product is on its way while the weight streams. The sums of squares for the
    // rows' factors (SCALED) go straight from memory into LDS, behind the waves' slots: [m][stride] as it lies in
    // memory, 1 KB per wave-wide load: buffer loads, since a global load into LDS is encoded as a flat one, and while one may be
    // under way the compiler waits for all loads of the weight instead of the block it multiplies.
    float* factor_shared = reduce_shared + static_cast<size_t>(waves - 1) * NT * MT * kWave * 4;
    if (SCALED && wave == 0) {
        const int count = m * extras.scale.stride;                  // floats; stride is a multiple of 4
        const auto sums_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(extras.scale.sumsq), 0, count * 4, kBufferFlags);
        for (int first = 0; first < count; first += 256) {
            const int index = first + lane * 4;
            if (index < count)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(sums_rsrc, factor_shared + first, 16, index * 4, 0, 0, 0);
        }
    }
    // Epilogue 3: the lane's 4 columns lie in one head (head_dim is a multiple of 16). In a query or key head the weight's
    // rows were ordered so that columns 2p and 2p + 1 hold dims p and p + n_freq: the two that rotate together. Where
    // every value goes is worked out here too (a null pointer: nowhere), since divisions by run-time sizes take as long
    // as the sums after them.
    float bias_first[NT][2], bias_second[NT][2];
    float2 cos_sin[NT][MT][2];
    bf16* target_first[NT][MT][2];
    bf16* target_second[NT][MT][2];
    bool rotates[NT][2];
    if (EPILOGUE == 3 && wave == 0) {
        int slot[MT], page[MT], place[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int row = mt * TILE + token;
            slot[mt] = store.slot_mapping && row < m ? store.slot_mapping[row] : -1;
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int column = (tile0 + nt) * TILE + quad * 4;
            const int head = column / store.head_dim, within = column % store.head_dim;
            const bool is_query = head < store.heads, is_value = head >= store.heads + store.kv_heads;
            const bool live = mine && column < n;
            int first[2], second[2];
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const bool rotate = !is_value && within + 2 * half < 2 * store.n_freq;
                rotates[nt][half] = rotate;
                const int pair = (within + 2 * half) / 2;
                first[half] = rotate ? pair : within + 2 * half;
                second[half] = rotate ? pair + store.n_freq : within + 2 * half + 1;
                bias_first[nt][half] = (live && store.bias) ? store.bias[head * store.head_dim + first[half]] : 0.0f;
                bias_second[nt][half] = (live && store.bias) ? store.bias[head * store.head_dim + second[half]] : 0.0f;
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const int row = mt * TILE + token;
                    cos_sin[nt][mt][half] = make_float2(1.0f, 0.0f);
                    if (live && rotate && row < m)
                        cos_sin[nt][mt][half] = reinterpret_cast<const float2*>(store.cos_sin)[static_cast<int64_t>(row) * store.n_freq + pair];
                }
            }
            const CacheLayout layout(store.kv_heads, store.page_size, store.head_dim);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const int row = mt * TILE + token;
                if (nt == 0) {
                    page[mt] = slot[mt] >= 0 ? slot[mt] / store.page_size : 0;
                    place[mt] = slot[mt] >= 0 ? slot[mt] % store.page_size : 0;
                }
                bf16* q_row = static_cast<bf16*>(store.q_out) + (static_cast<int64_t>(row) * store.heads + head) * store.head_dim;
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    bf16* to_first = nullptr;
                    bf16* to_second = nullptr;
                    if (live && row < m) {
                        if (is_query) {
                            to_first = q_row + first[half];
                            to_second = q_row + second[half];
                        } else if (slot[mt] >= 0 && !is_value) {
                            bf16* pages = static_cast<bf16*>(store.k_cache);
                            to_first = pages + layout.k_at(page[mt], head - store.heads, place[mt], first[half]);
                            to_second = pages + layout.k_at(page[mt], head - store.heads, place[mt], second[half]);
                        } else if (slot[mt] >= 0) {
                            bf16* pages = static_cast<bf16*>(store.v_cache);
                            const int kv_head = head - store.heads - store.kv_heads;
                            to_first = pages + layout.v_at(page[mt], kv_head, place[mt], first[half]);
                            to_second = pages + layout.v_at(page[mt], kv_head, place[mt], second[half]);
                        }
                    }
                    target_first[nt][mt][half] = to_first;
                    target_second[nt][mt][half] = to_second;
                }
            }
        }
    }
    float h_before[NT][MT][4], norm_weight[NT][4];
    if (EPILOGUE == 4 && wave == 0) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int column = (tile0 + nt) * TILE + quad * 4 + i;
                norm_weight[nt][i] = mine && column < n ? extras.residual.norm_weight[column] : 0.0f;
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const int row = mt * TILE + token;
                    h_before[nt][mt][i] = mine && row < m && column < n ? extras.residual.h[static_cast<int64_t>(row) * n + column] : 0.0f;
                }
            }
    }

    float side[NT][MT][4];
    if (EPILOGUE == 6 && wave == 0) {
        const MllSideTable& table = extras.side;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int id = mt * TILE + token < m ? table.ids[mt * TILE + token] : 0;
            const bool known = id >= 0 && id < table.vocab;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int column = (tile0 + nt) * TILE + quad * 4 + i;
                    const int64_t at = static_cast<int64_t>(id) * table.stride + table.column_at + column;
                    side[nt][mt][i] = known ? 0.0f : NAN;
                    if (known && mine && column < n)
                        side[nt][mt][i] = table.dtype == kF32 ? static_cast<const float*>(table.rows)[at] : to_float(static_cast<const bf16*>(table.rows)[at]);
                }
        }
    }

    // No branch around a load, for the same reason; a block past the last step costs no memory access.
    constexpr int kBlockSteps = HALF ? HALF * kChunk : DEPTH;
    const int blocks = (k_steps + waves * kChunk - 1) / (waves * kChunk) * kChunk;     // steps of the wave with the most, whole runs
    for (int done = 2 * kBlockSteps; done < blocks; done += 2 * kBlockSteps) {
        multiply(w_even, a_even, even);
        load(done / kBlockSteps, w_even, a_even);
        __builtin_amdgcn_sched_barrier(0);      // else the loads sink below the next products, behind their waits
        multiply(w_odd, a_odd, odd);
        load(done / kBlockSteps + 1, w_odd, a_odd);
        __builtin_amdgcn_sched_barrier(0);
    }
    multiply(w_even, a_even, even);
    multiply(w_odd, a_odd, odd);

    floatx4 (&acc)[NT][MT] = sums[0];
    if constexpr (HALF != 0 || SPLIT) {         // the even steps' sums and the odd ones'
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[nt][mt][i] += SPLIT ? sums[SETS - 1][nt][mt][i] : __shfl(acc[nt][mt][i], (lane + 40) % kWave, kWave);
    }

    // The factor of row `col`: the four lanes of a row take every fourth run of four sums; the order of the
    // additions is fixed by the number of sums. Formed while other waves may still be waiting for their weights.
    float row_factor[MT];
    if (SCALED && wave == 0) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // the loads into LDS have landed (the wave issued them itself)
        floatx4 parts = floatx4{0.0f, 0.0f, 0.0f, 0.0f};      // four sums side by side, then the four together
        if (col < m) {
            const float* squares = factor_shared + col * extras.scale.stride;
#pragma unroll 4
            for (int run = quad; 4 * run < extras.scale.groups; run += 4) {
                floatx4 four = *reinterpret_cast<const floatx4*>(squares + 4 * run);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (4 * run + i >= extras.scale.groups) four[i] = 0.0f;
                parts += four;
            }
        }
        float part = (parts[0] + parts[1]) + (parts[2] + parts[3]);
        part = sum_lanes_16_apart(part);
        const float factor = 1.0f / sqrtf(part / static_cast<float>(extras.scale.width) + extras.scale.eps);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) row_factor[mt] = HALF ? __shfl(factor, mt * 8 + token, kWave) : factor;
    }

    // The waves' sums, added in wave order by wave 0; several slots are read at a time, as many as stay in registers beside what
    // the epilogue holds.
    constexpr int kAtATime = NT * MT >= 6 ? 1 : NT * MT >= 3 || (kHolds && NT * MT == 2) ? 2 : 4;
    if (waves > 1) {
        floatx4* slots = reinterpret_cast<floatx4*>(reduce_shared);
        if (wave > 0) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) slots[((wave - 1) * NT * MT + nt * MT + mt) * kWave + lane] = acc[nt][mt];
        }
        __syncthreads();
        if (wave > 0) return;
        for (int first = 0; first < waves - 1; first += kAtATime) {
            floatx4 part[kAtATime][NT][MT];
#pragma unroll
            for (int i = 0; i < kAtATime; ++i) {
                const int other = min(first + i, waves - 2);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) part[i][nt][mt] = slots[(other * NT * MT + nt * MT + mt) * kWave + lane];
            }
#pragma unroll
            for (int i = 0; i < kAtATime; ++i)
                if (first + i < waves - 1) {
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) acc[nt][mt] += part[i][nt][mt];
                }
        }
    }

    // acc[nt][mt][i] = C[row mt * TILE + token][column (tile0 + nt) * TILE + quad * 4 + i] in the lanes that hold results
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int n_tile = tile0 + nt;
        if (n_tile >= n_tiles) continue;       // the same for every lane of the wave
        float squares[MT];                     // epilogue 4: this lane's share of its rows' sums of squares over the tile
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            squares[mt] = 0.0f;
            const int row = mt * TILE + token;
            if (row >= m || !mine) continue;
            if (SCALED) acc[nt][mt] *= row_factor[mt];
            if (EPILOGUE == 4) {
                const MllResidualNorm& residual = extras.residual;
                const int column = n_tile * TILE + quad * 4;
                float* h_row = residual.h + static_cast<int64_t>(row) * n;
                bf16* x_row = static_cast<bf16*>(residual.x_out) + static_cast<int64_t>(row) * n;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (column + i >= n) continue;
                    const float value = h_before[nt][mt][i] + acc[nt][mt][i];
                    h_row[column + i] = value;
                    x_row[column + i] = from_float<bf16>(value * norm_weight[nt][i]);
                    squares[mt] += value * value;
                }
            } else if (EPILOGUE == 0) {
                float* target = static_cast<float*>(out) + static_cast<int64_t>(row) * n;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int column = n_tile * TILE + quad * 4 + i;
                    if (column < n) target[column] = acc[nt][mt][i];
                }
            } else if (EPILOGUE == 1) {
                bf16* target = static_cast<bf16*>(out) + static_cast<int64_t>(row) * n;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int column = n_tile * TILE + quad * 4 + i;
                    if (column < n) target[column] = from_float<bf16>(acc[nt][mt][i]);
                }
            } else if (EPILOGUE == 6) {
                bf16* target = static_cast<bf16*>(out) + static_cast<int64_t>(row) * n;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int column = n_tile * TILE + quad * 4 + i;
                    if (column < n) target[column] = from_float<bf16>(activate(acc[nt][mt][i], kActGeluTanh) * side[nt][mt][i]);
                }
            } else if (EPILOGUE == 7) {
                bf16* target = static_cast<bf16*>(out) + static_cast<int64_t>(row) * (n / 2);
#pragma unroll
                for (int i = 0; i < 4; i += 2) {
                    const int column = n_tile * (TILE / 2) + quad * 2 + i / 2;
                    if (column < n / 2)
                        target[column] = from_float<bf16>(gated_value_fast(acc[nt][mt][i], acc[nt][mt][i + 1], kActClampedGlu, extras.glu_limit, extras.glu_slope));
                }
            } else if (EPILOGUE == 2 || EPILOGUE == 5) {
                bf16* target = static_cast<bf16*>(out) + static_cast<int64_t>(row) * (n / 2);
#pragma unroll
                for (int i = 0; i < 4; i += 2) {
                    const int column = n_tile * (TILE / 2) + quad * 2 + i / 2;
                    if (column < n / 2) target[column] = from_float<bf16>(gate_fast<EPILOGUE == 5>(acc[nt][mt][i]) * acc[nt][mt][i + 1]);
                }
            } else {
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    const float x1 = acc[nt][mt][2 * half] + bias_first[nt][half], x2 = acc[nt][mt][2 * half + 1] + bias_second[nt][half];
                    const float c = cos_sin[nt][mt][half].x, sn = cos_sin[nt][mt][half].y;
                    if (target_first[nt][mt][half] != nullptr) {
                        *target_first[nt][mt][half] = from_float<bf16>(rotates[nt][half] ? rotate_first(x1, x2, c, sn) : x1);
                        *target_second[nt][mt][half] = from_float<bf16>(rotates[nt][half] ? rotate_second(x1, x2, c, sn) : x2);
                    }
                }
            }
        }
        if (EPILOGUE == 4) {
            // The row's sum over the tile's columns: the lanes of a row, in a fixed order. One entry per tile of W (or
            // half of one), so that the sums do not depend on how many tiles a workgroup takes.
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const float over_tile = sum_lanes_16_apart(squares[mt]);
                const int row = mt * TILE + token;
                if (quad == 0 && mine && row < m) extras.residual.sumsq_out[static_cast<int64_t>(row) * extras.residual.sumsq_stride + n_tile] = over_tile;
            }
        }
    }
}

// Weights of at most this many tiles of 16 rows are read in halves of tiles: a compute unit brings about 45 GB/s from
// memory however much it asks for, so that 56 of them take 4.5 us for 7 MB and 112 take 3.5 (a kernel that only reads).
// Product of 896 x 4864 at one row: 7.1 us with the whole tiles of before, 6.7 with whole tiles in this kernel, 5.2 in halves; 2048 x 8192:
// 11.2, 9.5, 8.3. Above that line the activations, which every workgroup reads, cost more than the halves
// give (224 tiles, 3584 x 18944 at 8 rows: 26 us, in halves 36).
constexpr int kHalfTiles = 128;
static bool in_halves(int n_tiles) { return n_tiles <= kHalfTiles; }

// Waves a workgroup: 16 k steps a wave, so that a wave asks for all it needs at once without asking past the end, at most
// 16 waves and about eight thousand over the whole launch. A function of (n, k) alone, like the split of k it implies.
// From 9 waves on a compute unit holds one workgroup whatever their number: more are taken where the waves' runs, of which the main
// loop takes two rounds at a time, then fill their rounds better by an eighth. 520 tiles of 8192 with 15 and 16 waves at 1, 8, 12
// and 16 rows 27.2 and 25.8 us, 30.8 and 28.8, 36.4 and 32.0, 41.8 and 36.7; 576 of 11008 with 14 and 16 at 12 rows 49.2 and 46.1; but
// 640 of 11008, as well filled with 12 as with 16, 39.7 and 42.6 at 8.
static int skinny_waves(int n_tiles, int k_steps) {
    const int waves = max(1, min(min(16, 8192 / n_tiles), (k_steps + 15) / 16));
    if (waves <= 8) return waves;
    const auto slots = [k_steps](int count) { return ((k_steps + count * kChunk - 1) / (count * kChunk) + 1) / 2 * count; };
    int best = waves;
    for (int more = waves + 1; more <= 16; ++more)
        if (slots(more) < slots(best)) best = more;
    return 9 * slots(best) <= 8 * slots(waves) ? best : waves;
}

template <int MT, int NT, int EPILOGUE, int GROUP, int HALF, bool SPLIT, bool FAR = false>
static void launch_one(const bf16* a, const bf16* w, void* out, int m, int n, int k, int n_tiles,
                       int k_steps, const MllSkinnyExtras& extras, hipStream_t stream) {
    const int waves = skinny_waves(n_tiles, k_steps);
    const int units = HALF ? (n + 7) / 8 : n_tiles;
    const int groups = (units + NT - 1) / NT;
    size_t lds = waves > 1 ? static_cast<size_t>(waves - 1) * NT * MT * kWave * sizeof(floatx4) : 0;
    if (MT * (HALF ? 8 : 16) <= 16 && extras.scale.sumsq != nullptr) {
        lds += (static_cast<size_t>(m) * extras.scale.stride * sizeof(float) + 1023) / 1024 * 1024;
        gemm_skinny_kernel<MT, NT, EPILOGUE, (MT * (HALF ? 8 : 16) <= 16), GROUP, HALF, SPLIT, FAR><<<groups, waves * kWave, lds, stream>>>(
            a, w, out, m, n, k, units, k_steps, extras);
    } else {
        gemm_skinny_kernel<MT, NT, EPILOGUE, false, GROUP, HALF, SPLIT, FAR><<<groups, waves * kWave, lds, stream>>>(
            a, w, out, m, n, k, units, k_steps, extras);
    }
}

// Up to 16 rows: halves of tiles (with few steps a wave both blocks in flight hold one run of steps, else two), or
// whole tiles with as many steps an A load as the rows allow. Queries, keys and values of 9 to 16 rows of a weight in halves take whole
// tiles and the same sums: their places are worked out for every group of 8 rows, which halves would double (12 rows of
// 1536 x 1024 5.7 and 5.3 us, of 768 x 512 4.8 and 4.3).
template <int NT, int EPILOGUE>
static void launch_few(const bf16* a, const bf16* w, void* out, int m, int n, int k, int n_tiles,
                       int k_steps, const MllSkinnyExtras& extras, hipStream_t stream) {
    if constexpr (NT == 1) {
        if (in_halves(n_tiles)) {
            const bool few_steps = k_steps <= 2 * kChunk * skinny_waves(n_tiles, k_steps);
            if (m <= 8 && few_steps) launch_one<1, 1, EPILOGUE, 1, 1, false>(a, w, out, m, n, k, n_tiles, k_steps, extras, stream);
            else if (m <= 8) launch_one<1, 1, EPILOGUE, 1, 2, false>(a, w, out, m, n, k, n_tiles, k_steps, extras, stream);
            else if constexpr (EPILOGUE == 3) launch_one<1, 1, EPILOGUE, 1, 0, true>(a, w, out, m, n, k, n_tiles, k_steps, extras, stream);
            else launch_one<2, 1, EPILOGUE, 1, 1, false>(a, w, out, m, n, k, n_tiles, k_steps, extras, stream);
            return;
        }
    }
    if (m <= 4) launch_one<1, NT, EPILOGUE, 4, 0, false>(a, w, out, m, n, k, n_tiles, k_steps, extras, stream);
    else if (m <= 8) launch_one<1, NT, EPILOGUE, 2, 0, false>(a, w, out, m, n, k, n_tiles, k_steps, extras, stream);
    else launch_one<1, NT, EPILOGUE, 1, 0, false>(a, w, out, m, n, k, n_tiles, k_steps, extras, stream);
}

// Reductions whose byte offsets (64 rows of the activations) pass what descriptors reach: 16 rows at a time, the same sums.
constexpr int kWidestNear = 1 << 23;
template <int EPILOGUE>
static void launch_far(const bf16* a, const bf16* w, void* out, int m, int n, int k, int n_tiles, int k_steps, const MllSkinnyExtras& extras,
                       hipStream_t stream) {
    const int64_t row_bytes = EPILOGUE == 0 ? 4ll * n : EPILOGUE == 1 || EPILOGUE == 6 ? 2ll * n : n;
    for (int first = 0; first < m; first += 16) {
        const int rows = min(16, m - first);
        const bf16* a_ = a + static_cast<int64_t>(first) * k;
        void* out_ = static_cast<char*>(out) + first * row_bytes;
        if (in_halves(n_tiles) && rows <= 8) launch_one<1, 1, EPILOGUE, 1, 1, false, true>(a_, w, out_, rows, n, k, n_tiles, k_steps, extras, stream);
        else if (in_halves(n_tiles)) launch_one<2, 1, EPILOGUE, 1, 1, false, true>(a_, w, out_, rows, n, k, n_tiles, k_steps, extras, stream);
        else launch_one<1, 1, EPILOGUE, 1, 0, false, true>(a_, w, out_, rows, n, k, n_tiles, k_steps, extras, stream);
    }
}

// 17 to 64 rows: what gemm_medium is for; kept for callers of the entry. 64 rows of 896 x 4864 22 us, 3584 x 18944 100, 37888 x
// 3584 102 (with two steps a block and four slots read at a time, which spilled up to 670 registers, 81, 163 and 190).
template <int MT, int NT, int EPILOGUE>
static void launch_many(const bf16* a, const bf16* w, void* out, int m, int n, int k, int n_tiles,
                        int k_steps, const MllSkinnyExtras& extras, hipStream_t stream) {
    // Narrow weights: one tile a workgroup, so that its two sets of sums stay in registers beside the loads.
    if (in_halves(n_tiles)) launch_one<MT, 1, EPILOGUE, 1, 0, true>(a, w, out, m, n, k, n_tiles, k_steps, extras, stream);
    else launch_one<MT, NT, EPILOGUE, 1, 0, false>(a, w, out, m, n, k, n_tiles, k_steps, extras, stream);
}

// Tiles of W a workgroup takes: two where enough workgroups are left, so that every piece of A is used twice (MI355X, one
// against two: 1024 tiles of 2048 at 8 rows 12.4 and 11.9, at one row 12.5 and 12.5; 2368 tiles of 3584 at 8 rows 43.1 and 41.9; four
// tiles a workgroup were slower), and where one a workgroup would leave a second round of the 256 compute units half empty, of
// 257 to 512 tiles: 288 tiles of 3584 at 1, 8 and 16 rows 9.1 and 8.9, 10.5 and 9.8, 13.3 and 11.1, of 8192 18.0 and 15.9,
// 20.4 and 18.1, 26.0 and 20.5; 512 tiles of 3584 11.5 and 11.4, 11.5 and 11.0, 13.9 and 11.9, at 4 rows 10.9 and 11.2; 608 tiles of
// 3584 13.4 and 15.7, 14.8 and 16.4, 18.6 and 19.0. With fewer than 48 steps it makes no difference. Above three rounds, 768 tiles, two are better
// again from few rows on: 769 to 1023 tiles at 8, 12 and 16 rows, 864 of 2560 14.2 and 13.2, 18.4 and 14.8, 19.7 and 15.3, of 5120 29.8 and
// 25.8, 37.0 and 29.1, 40.9 and 30.5, 1008 of 3584 19.7 and 19.2, 21.9 and 19.7, 24.3 and 20.5 (864 of 5120 at 5 rows 27.8 and 25.1, at 4
// 26.8 and 24.7, but 960 24.9 and 24.5 and 864 of 896 7.0 and 7.1); 768 of 3584 15.9 and 17.3, 17.5 and 18.3, 19.1 and 19.3, of 2560 at
// 16 rows 17.3 and 15.1. So are they from 13 rows on where a workgroup has 9 waves or more, which leave a compute unit room for no other: 640
// tiles of 5120 at 12 and 16 rows 25.6 and 25.2, 28.8 and 26.6, of 8192 37.3 and 38.6, 41.1 and 40.2. The q/k/v epilogue holds
// so much that few rows lose: 288 tiles of 3584 at 1, 5, 8 and 16 rows 9.7 and 11.6, 10.1 and 10.7, 11.1 and 10.8, 12.7 and 11.1.
template <int EPILOGUE>
static int tiles_per_group(int m, int n_tiles, int k_steps) {
    if (m > 32) return 2;
    if (m > 16) return n_tiles >= 2048 ? 2 : 1;
    if (n_tiles >= 2048 || (m > 4 && n_tiles > (m > 12 ? 767 : 768))) return 2;
    if (m > 12 && n_tiles > 512 && skinny_waves(n_tiles, k_steps) > 8) return 2;
    const bool half_a_round = n_tiles > 256 && n_tiles <= (m > 4 ? 512 : 384) && k_steps >= 48;
    return half_a_round && (EPILOGUE != 3 || m > 5) ? 2 : 1;
}

template <int EPILOGUE>
static int launch_skinny(const void* a, const void* w_packed, void* out, int m, int n, int k,
                         const MllSkinnyExtras& extras, hipStream_t stream) {
    const int n_tiles = (n + 15) / 16;
    const int k_steps = (k + 31) / 32;
    const bf16* a_ = static_cast<const bf16*>(a);
    const bf16* w_ = static_cast<const bf16*>(w_packed);
    const int m_tiles = (m + 15) / 16;
    const bool two = tiles_per_group<EPILOGUE>(m, n_tiles, k_steps) == 2;
    if (k > kWidestNear) {
        launch_far<EPILOGUE>(a_, w_, out, m, n, k, n_tiles, k_steps, extras, stream);
    } else if (m_tiles == 1) {
        if (two) launch_few<2, EPILOGUE>(a_, w_, out, m, n, k, n_tiles, k_steps, extras, stream);
        else launch_few<1, EPILOGUE>(a_, w_, out, m, n, k, n_tiles, k_steps, extras, stream);
    } else if constexpr (EPILOGUE == 3 || EPILOGUE == 4 || EPILOGUE == 6 || EPILOGUE == 7) {
        return fail("gemm_skinny: this epilogue takes at most 16 rows");
    } else if (m_tiles == 2) {
        if (two) launch_many<2, 2, EPILOGUE>(a_, w_, out, m, n, k, n_tiles, k_steps, extras, stream);
        else launch_many<2, 1, EPILOGUE>(a_, w_, out, m, n, k, n_tiles, k_steps, extras, stream);
    } else if (m_tiles == 3) {
        launch_many<3, 2, EPILOGUE>(a_, w_, out, m, n, k, n_tiles, k_steps, extras, stream);
    } else if (m_tiles == 4) {
        launch_many<4, 2, EPILOGUE>(a_, w_, out, m, n, k, n_tiles, k_steps, extras, stream);
    } else {
        return fail("gemm_skinny: more than 64 rows");
    }
    return check_launch("gemm_skinny");
}

}  // namespace mll

using namespace mll;

static int check_scale(const MllRowScale* scale, int m) {
    if (scale == nullptr || scale->sumsq == nullptr) return 0;
    MLL_REQUIRE(m <= 16, "gemm_skinny: a row factor needs at most 16 rows");
    MLL_REQUIRE(scale->groups > 0 && scale->width > 0 && scale->eps >= 0.0f, "gemm_skinny: bad row factor description");
    MLL_REQUIRE(scale->stride >= scale->groups && scale->stride % 4 == 0 && reinterpret_cast<uintptr_t>(scale->sumsq) % 16 == 0,
                "gemm_skinny: the rows of sums must be 16-byte aligned");
    MLL_REQUIRE(scale->stride <= 512, "gemm_skinny: a row factor from more than 512 sums (a norm wider than 8192)");
    return 0;
}

extern "C" int mll_gemm_skinny(const void* a, const void* w_packed, void* out, int epilogue, int m, int n, int k,
                               const MllRowScale* scale, hipStream_t stream) {
    MLL_REQUIRE(m >= 0 && m <= 64, "gemm_skinny: takes at most 64 rows");
    MLL_REQUIRE(n > 0 && k > 0 && k % 8 == 0, "gemm_skinny: k must be a positive multiple of 8");
    MLL_REQUIRE((epilogue != 2 && epilogue != 5) || n % 2 == 0, "gemm_skinny: the gated epilogue needs an even number of weight rows");
    if (check_scale(scale, m) != 0) return 1;
    if (m == 0) return 0;
    MllSkinnyExtras extras{};
    if (scale) extras.scale = *scale;
    switch (epilogue) {
        case 0: return launch_skinny<0>(a, w_packed, out, m, n, k, extras, stream);
        case 1: return launch_skinny<1>(a, w_packed, out, m, n, k, extras, stream);
        case 2: return launch_skinny<2>(a, w_packed, out, m, n, k, extras, stream);
        case 5: return launch_skinny<5>(a, w_packed, out, m, n, k, extras, stream);
        default: return fail("gemm_skinny: unknown epilogue");
    }
}

extern "C" int mll_gemm_skinny_clamped(const void* a, const void* w_packed, void* out, int m, int n, int k, float limit, float slope,
                                       hipStream_t stream) {
    MLL_REQUIRE(m >= 0 && m <= 16, "gemm_skinny_clamped: takes at most 16 rows");
    MLL_REQUIRE(n > 0 && n % 2 == 0 && k > 0 && k % 8 == 0, "gemm_skinny_clamped: an even number of weight rows, k a multiple of 8");
    MLL_REQUIRE(limit > 0.0f, "gemm_skinny_clamped: the limit must be positive");
    if (m == 0) return 0;
    MllSkinnyExtras extras{};
    extras.glu_limit = limit;
    extras.glu_slope = slope;
    return launch_skinny<7>(a, w_packed, out, m, n, k, extras, stream);
}

extern "C" int mll_gemm_skinny_side(const void* a, const void* w_packed, void* out, int m, int n, int k, const MllSideTable* side,
                                    hipStream_t stream) {
    MLL_REQUIRE(side != nullptr && side->rows && side->ids, "gemm_skinny_side: a side table and the rows' ids are needed");
    MLL_REQUIRE(m >= 0 && m <= 16, "gemm_skinny_side: takes at most 16 rows");
    MLL_REQUIRE(n > 0 && k > 0 && k % 8 == 0, "gemm_skinny_side: k must be a positive multiple of 8");
    MLL_REQUIRE(side->dtype == kF32 || side->dtype == kBF16, "gemm_skinny_side: unknown dtype of the side table");
    MLL_REQUIRE(side->vocab > 0 && side->column_at >= 0 && side->column_at + n <= side->stride,
                "gemm_skinny_side: the columns lie outside the table's rows");
    if (m == 0) return 0;
    MllSkinnyExtras extras{};
    extras.side = *side;
    return launch_skinny<6>(a, w_packed, out, m, n, k, extras, stream);
}

extern "C" int mll_gemm_skinny_qkv(const void* a, const void* w_packed, int m, int k, const MllQkvStore* store,
                                   const MllRowScale* scale, hipStream_t stream) {
    MLL_REQUIRE(store != nullptr, "gemm_skinny_qkv: no epilogue description");
    MLL_REQUIRE(m >= 0 && m <= 16, "gemm_skinny_qkv: takes at most 16 rows");
    MLL_REQUIRE(k > 0 && k % 8 == 0, "gemm_skinny_qkv: k must be a positive multiple of 8");
    MLL_REQUIRE(store->heads > 0 && store->kv_heads >= 0, "gemm_skinny_qkv: bad head counts");
    MLL_REQUIRE(store->head_dim >= 16 && store->head_dim % 16 == 0, "gemm_skinny_qkv: head_dim must be a multiple of 16");
    MLL_REQUIRE(store->n_freq >= 0 && 2 * store->n_freq <= store->head_dim, "gemm_skinny_qkv: more rotary pairs than dims");
    MLL_REQUIRE(store->n_freq == 0 || store->cos_sin, "gemm_skinny_qkv: rotation needs the table of cos and sin");
    MLL_REQUIRE(store->q_out, "gemm_skinny_qkv: the query output is needed");
    MLL_REQUIRE(!store->slot_mapping || (store->k_cache && store->v_cache && store->page_size > 0 && store->page_size % 16 == 0),
                "gemm_skinny_qkv: writing pages needs both caches and a page size that is a multiple of 16");
    if (check_scale(scale, m) != 0) return 1;
    if (m == 0) return 0;
    const int n = (store->heads + 2 * store->kv_heads) * store->head_dim;
    MllSkinnyExtras extras{};
    extras.store = *store;
    if (scale) extras.scale = *scale;
    return launch_skinny<3>(a, w_packed, nullptr, m, n, k, extras, stream);
}

extern "C" int mll_skinny_sum_columns(int n) { return in_halves((n + 15) / 16) ? 8 : 16; }

extern "C" int mll_gemm_skinny_residual(const void* a, const void* w_packed, int m, int n, int k,
                                        const MllResidualNorm* residual, const MllRowScale* scale, hipStream_t stream) {
    MLL_REQUIRE(residual != nullptr && residual->h && residual->norm_weight && residual->x_out && residual->sumsq_out,
                "gemm_skinny_residual: the residual stream, the norm's weight and both outputs are needed");
    MLL_REQUIRE(m >= 0 && m <= 16, "gemm_skinny_residual: takes at most 16 rows");
    MLL_REQUIRE(n > 0 && k > 0 && k % 8 == 0, "gemm_skinny_residual: k must be a positive multiple of 8");
    const int columns = mll_skinny_sum_columns(n);
    MLL_REQUIRE(residual->sumsq_stride >= (n + columns - 1) / columns, "gemm_skinny_residual: the rows of sums are too short");
    if (check_scale(scale, m) != 0) return 1;
    if (m == 0) return 0;
    MllSkinnyExtras extras{};
    extras.residual = *residual;
    if (scale) extras.scale = *scale;
    return launch_skinny<4>(a, w_packed, nullptr, m, n, k, extras, stream);
}
