// Matrix products with 17 to 64 rows (decoding many requests, short portions of prompts): C = A . W^T for
// bfloat16 A [M, K] (row-major) and the packed weight the streaming kernel reads ([N/16][K/32][4][16][8]).
// Still bound by reading W once from HBM, but with this many rows the activations a wave needs per piece of W
// are several times the piece: here the 4 or 8 waves of a workgroup walk the same k steps, each over its own one
// or two tiles of W, and share the activations through LDS (8 k steps at a time, double buffered, loaded straight
// into it by all waves together). A wave keeps two stages of its tiles in registers: one on its way while
// the other is multiplied. All loads go through buffer descriptors, which return zeros past their end: a load
// under a condition would make the compiler wait for all loads before it.
//
// A workgroup takes so many tiles that the workgroups fill the compute units evenly (see balanced_tiles): of
// 37888 x 3584 10 a workgroup, 237 of them, where 16 would leave 108 of the 256 units without one. 64 rows of it
// 66.1 -> 51.7 us (the reads alone take 40), of 152064 x 3584 214.6 -> 205.3 us (155), 32 rows of 9728 x 896 10.3 -> 7.4 us (now 6.4),
// of 896 x 4864 7.2 -> 5.4 us (4.9), of 1152 x 896 5.0 -> 3.5 us (2.9). With 64 rows the products and the reads of LDS take about as
// long as W's way, and the stages' barriers keep them from covering each other whole.
//
// Where W has too few tiles to fill the GPU this way, k is split over `splits` workgroups (grid y), each of
// which writes its own float32 partial sum [split][M][N]; the consumer adds them in order. Which k steps a
// sum holds, and in which order, depends on (n, k, splits) alone: a row's result does not depend on the
// other rows, nor on the tiles a workgroup takes.
#include "common.h"
#include "microllm_hip.h"

#include <type_traits>

namespace mll {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int uintx4 __attribute__((ext_vector_type(4)));

namespace medium {

constexpr int kStepsPerStage = 8;    // k steps of activations in one LDS buffer, and of W in one batch of loads
constexpr int kMostTiles = 16;       // two a wave of 8
constexpr unsigned kPast = 0x40000000;   // an offset past the end of every descriptor here
constexpr int kMostSteps = static_cast<int>(kPast) / (kMostTiles * 1024);      // so that a workgroup's tiles end before it
constexpr int kNonTemporal = 2;      // W is read once a step: past the caches
constexpr int kArithmetic = 0xf;     // to sched_barrier: vector, scalar and matrix instructions

union Piece {
    bf16x8 v;
    uintx4 raw;
};

// EPILOGUE: 0 = float32 [splits][M, N]; 1 = bfloat16 [M, N]; 2 = bfloat16 [M, N / 2] = silu(even rows of W) * (odd
// rows). 1 and 2 need splits == 1. A workgroup takes `tiles` tiles of W, a wave its wave-th and (NT = 2) that kWaves on. FAR: 64-bit
// addresses and loads under conditions, for reductions beyond what a descriptor's 32-bit offsets reach.
template <int MT, int NT, int kWaves, int EPILOGUE, bool FAR>
__global__ __launch_bounds__(kWaves * kWave) void gemm_medium_kernel(
    const bf16* __restrict__ a, const bf16* __restrict__ w_packed, void* __restrict__ out,
    int m, int n, int k, int n_tiles, int k_steps, int steps_per_split, int tiles) {
    constexpr int kStagePieces = MT * kStepsPerStage;             // pieces of A in a buffer, 1 KB each
    constexpr int kPiecesPerWave = kStagePieces / kWaves;
    // Two buffers, [pair of k steps][MT * 16 rows][8 places of 16 bytes]: 128 bytes of a row, whose chunk c is at place c ^ (row / 2). Two variables,
    // so that the compiler knows which of them a load into LDS fills.
    __shared__ uintx4 buffer_even[kStagePieces * kWave], buffer_odd[kStagePieces * kWave];

    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int col = lane % 16, quad = lane / 16;
    const int tile0 = blockIdx.x * tiles;
    const int live_tiles = min(tiles, n_tiles - tile0);
    const int first_step = blockIdx.y * steps_per_split;
    const int end_step = min(k_steps, first_step + steps_per_split);
    const int n_stages = (end_step - first_step + kStepsPerStage - 1) / kStepsPerStage;

    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16*>(w_packed) + static_cast<int64_t>(tile0) * k_steps * 512, 0, live_tiles * k_steps * 1024, kBufferFlags);
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(a), 0, m * k * 2, kBufferFlags);
    unsigned w_at[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        w_at[nt] = wave + kWaves * nt < live_tiles ? static_cast<unsigned>((wave + kWaves * nt) * k_steps * 1024 + lane * 16) : kPast;
        asm("" : "+v"(w_at[nt]));       // else the choice becomes a branch around the loads
    }
    // This wave's share of a buffer: pieces wave, wave + kWaves, ... of 8 rows of 128 bytes (a pair of k steps). A piece is a load straight into LDS, of
    // whole lines (in MFMA operand order, 64 bytes of 16 rows a load by way of registers, every line was asked for twice: 64 rows of
    // 37888 x 3584 gated 54.9 -> 51.3 us, 3584 x 18944 31.1 -> 30.2, 9728 x 896 gated 9.0 -> 7.8, 896 x 4864 6.9 -> 5.9, 32 rows 47.2 -> 46.7, 25.4 -> 25.3, 6.5 -> 6.2
    // and 5.1 -> 4.7; 16 weights at 17 to 64 rows 1.05 times as fast on the mean, none slower. Without the activations' loads 49.8 and 28.4 us.)
    constexpr int kOctets = 2 * MT;      // groups of 8 rows
    int a_at[kPiecesPerWave], a_left[kPiecesPerWave];      // where the lane reads at step 0, and below how many elements from there its steps begin
#pragma unroll
    for (int j = 0; j < kPiecesPerWave; ++j) {
        const int piece = wave + kWaves * j, row = piece % kOctets * 8 + lane / 8, chunk = (lane % 8) ^ (row % 16 / 2), element = piece / kOctets * 64 + chunk * 8;
        a_at[j] = (row * k + element) * 2;
        a_left[j] = row < m ? (FAR && end_step == k_steps ? k : min(k, end_step * 32)) - element : 0;
    }

    auto load_w = [&](Piece (&pieces)[kStepsPerStage][NT], int stage_number) {
        const int step = first_step + stage_number * kStepsPerStage;
#pragma unroll
        for (int u = 0; u < kStepsPerStage; ++u) {
            const unsigned at = step + u < end_step ? static_cast<unsigned>(step + u) * 1024 : kPast;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                if constexpr (FAR) {
                    const int tile = wave + kWaves * nt;
                    const bf16* from = w_packed + (static_cast<int64_t>(tile0 + tile) * k_steps + step + u) * 512 + lane * 8;
                    pieces[u][nt].raw = tile < live_tiles && step + u < end_step ? *reinterpret_cast<const uintx4*>(from) : uintx4{0u, 0u, 0u, 0u};
                } else {
                    pieces[u][nt].raw = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, w_at[nt] + at, 0, kNonTemporal);
                }
            }
        }
    };
    auto load_share = [&](uintx4* buffer, int stage_number) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < kPiecesPerWave; ++j) {
            const int step = first_step + stage_number * kStepsPerStage;
            uintx4* place = buffer + (wave + kWaves * j) * kWave;
            const bool there = static_cast<int64_t>(step) * 32 < a_left[j];
            if constexpr (FAR) {
                const int piece = wave + kWaves * j, row = piece % kOctets * 8 + lane / 8, chunk = (lane % 8) ^ (row % 16 / 2);
                const bf16* from = a + static_cast<int64_t>(row) * k + static_cast<int64_t>(step) * 32 + piece / kOctets * 64 + chunk * 8;
                place[lane] = there ? *reinterpret_cast<const uintx4*>(from) : uintx4{0u, 0u, 0u, 0u};
            } else {
                const int at = there ? a_at[j] + step * 64 : static_cast<int>(kPast);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, place, 16, at, 0, 0, 0);
            }
        }
        // share_landed counts what was issued after the share: only arithmetic may pass from one side of this place to the other.
        __builtin_amdgcn_sched_barrier(kArithmetic);
    };
    // The share that was asked for before the last `LATER` loads has landed, the wave's reads of the other buffer have arrived, and the workgroup meets.
    auto share_landed = [&]() __attribute__((always_inline)) {
        if constexpr (FAR) {
            __syncthreads();
        } else {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NT * kStepsPerStage) : "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
    };

    floatx4 acc[NT][MT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    // With one tile a wave a step's activations are read from LDS while the step before is multiplied: left alone, the compiler reads them one or two
    // ahead of their products (48 rows of 1152 x 896 3.46 -> 3.25 us, 64 rows of 9728 x 896 8.9 -> 8.5, of 3584 x 3584 9.67 -> 9.35). With two there
    // are twice as many products to cover a read, and the order it chooses is the better one (32 rows of 37888 x 3584 44.3, 44.9 this way).
    const int a_place[2] = {col * 8 + (quad ^ (col / 2)), col * 8 + ((4 + quad) ^ (col / 2))};      // of a pair's first step and its second
    auto multiply = [&](const Piece (&pieces)[kStepsPerStage][NT], const uintx4* buffer) __attribute__((always_inline)) {
        Piece a_piece[2][MT];
        auto read = [&](int u) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) a_piece[u % 2][mt].raw = buffer[(u / 2 * MT + mt) * (2 * kWave) + a_place[u % 2]];
        };
        if constexpr (NT == 1) read(0);
#pragma unroll
        for (int u = 0; u < kStepsPerStage; ++u) {
            if constexpr (NT == 1) {
                if (u + 1 < kStepsPerStage) read(u + 1);
                __builtin_amdgcn_sched_barrier(0);
            } else {
                read(u);
            }
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pieces[u][nt].v, a_piece[u % 2][mt].v, acc[nt][mt], 0, 0, 0);
            if constexpr (NT == 1) __builtin_amdgcn_sched_barrier(0);
        }
    };

    // The activations of a stage are asked for before its tiles: loads come back in order, and the buffer must not wait
    // for the tiles. A buffer was last read in the stage before the one that fills it, and the workgroup has met since.
    Piece w_even[kStepsPerStage][NT], w_odd[kStepsPerStage][NT];
    load_share(buffer_even, 0);
    load_w(w_even, 0);
    __builtin_amdgcn_sched_barrier(0);
    share_landed();
    // Two stages a round, and what is left of an odd number after the rounds: were the loop left between the two, the compiler would think that it
    // comes round with the odd tiles' loads on their way, and wait for all loads at the start of every round (17 rows of 9728 x 896
    // 6.84 -> 5.87 us, of 3584 x 18944 23.8 -> 22.7, 64 rows of 1152 x 896 4.37 -> 3.64, of 896 x 4864 7.05 -> 6.67, of 37888 x 3584 50.6 -> 50.3).
    int s = 0;
    for (; s + 1 < n_stages; s += 2) {
        load_share(buffer_odd, s + 1);
        load_w(w_odd, s + 1);
        __builtin_amdgcn_sched_barrier(0);      // else the loads sink below the products, behind their waits
        multiply(w_even, buffer_even);
        share_landed();
        load_share(buffer_even, s + 2);
        load_w(w_even, s + 2);
        __builtin_amdgcn_sched_barrier(0);
        multiply(w_odd, buffer_odd);
        share_landed();
    }
    if (s < n_stages) multiply(w_even, buffer_even);

    // acc[nt][mt][i] = C[row mt*16 + col][column n_tile*16 + quad*4 + i]
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        if (wave + kWaves * nt >= live_tiles) continue;
        const int n_tile = tile0 + wave + kWaves * nt;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int row = mt * 16 + col;
            if (row >= m) continue;
            if (EPILOGUE == 0) {
                float* target = static_cast<float*>(out) + (static_cast<int64_t>(blockIdx.y) * m + row) * n;
                const int column = n_tile * 16 + quad * 4;
                if (column + 3 < n && n % 4 == 0) {
                    *reinterpret_cast<floatx4*>(target + column) = acc[nt][mt];
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (column + i < n) target[column + i] = acc[nt][mt][i];
                }
            } else if (EPILOGUE == 1) {
                bf16* target = static_cast<bf16*>(out) + static_cast<int64_t>(row) * n;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int column = n_tile * 16 + quad * 4 + i;
                    if (column < n) target[column] = from_float<bf16>(acc[nt][mt][i]);
                }
            } else {
                bf16* target = static_cast<bf16*>(out) + static_cast<int64_t>(row) * (n / 2);
#pragma unroll
                for (int i = 0; i < 4; i += 2) {
                    const int column = n_tile * 8 + quad * 2 + i / 2;
                    if (column < n / 2) target[column] = from_float<bf16>(gate_fast<EPILOGUE == 5>(acc[nt][mt][i]) * acc[nt][mt][i + 1]);
                }
            }
        }
    }
}

// The tiles of W a workgroup takes, at most `most`: so that the compute units' rounds times what a round takes (its tiles, and the
// activations' copy, which costs about two) come to the least. 64 rows of 37888 x 3584 with 10 tiles 51.7 us, with 5 69.2 and
// with 4 74.5. `parts`: the splits that hold stages; the others store zeros, which costs a little where they begin a round of their own
// (4864 in 16 splits of whole stages fills ten: counted as 16, 4608 x 4864 at 17 and 64 rows took 14.2 and 21.9 us, now 11.7 and 17.8). Above
// 8 tiles a workgroup's registers leave a compute unit room for no other. Where a workgroup has few stages (one or two, up to four where it
// would take 16 tiles) and there is work for several rounds, its first loads then stand in the open; up to 32 rows 8 tiles and two workgroups a unit are
// better: 32 rows of 20480 x 1536 with 8, 12 and 16 tiles 14.4, 18.8 and 16.6, of 11008 x 2048 13.3, 14.7 and 15.9, of 152064 x 64 14.9, 19.9 and
// 17.1, 17 of 8192 x 8192 27.4, 28.5 and 30.1; but 64 rows of 20480 x 1536 21.0, 24.7 and 21.1, 17 of 11008 x 8192 in four
// stages with 8 and 11 tiles 36.4 and 32.9, of 16384 x 8192 in eight with 8 and 16 47.7 and 43.7.
static int balanced_tiles(int n_tiles, int splits, int parts, int stages, int row_tiles, int most) {
    constexpr int kUnits = 256, kCopy = 2, kFewStages = 2, kSeveralRounds = 12 * kUnits;
    int best = 1, least = 0x7fffffff;
    for (int tiles = 1; tiles <= most; ++tiles) {
        const int64_t groups = static_cast<int64_t>((n_tiles + tiles - 1) / tiles), rounds = (groups * parts + kUnits - 1) / kUnits;
        const int64_t cost = rounds * (tiles + kCopy) + (groups * splits > rounds * kUnits ? 2 * kCopy : 0);
        if (cost < least) {
            best = tiles;
            least = static_cast<int>(cost);
        }
    }
    const bool few_stages = parts > 1 ? stages <= kFewStages || (best == 16 && stages <= 2 * kFewStages) : stages == 1;
    if (row_tiles <= 2 && few_stages && static_cast<int64_t>(n_tiles) * parts >= kSeveralRounds) return min(8, most);
    return best;
}

// Each split takes whole stages, so that the stages of a sum begin at the same k whatever the split.
static int stages_of_a_split(int k, int splits) {
    const int stages = ((k + 31) / 32 + kStepsPerStage - 1) / kStepsPerStage;
    return (stages + splits - 1) / splits;
}

static int tiles_of(int m, int n, int k, int splits, int most) {
    const int each = stages_of_a_split(k, splits), parts = (stages_of_a_split(k, 1) + each - 1) / each;
    return (k + 31) / 32 > kMostSteps ? 4 : balanced_tiles((n + 15) / 16, splits, parts, each, (m + 15) / 16, most);
}

template <int MT, int EPILOGUE>
static void launch_rows(const bf16* a, const bf16* w, void* out, int m, int n, int k, int most_tiles, int splits, hipStream_t stream) {
    const int n_tiles = (n + 15) / 16, k_steps = (k + 31) / 32;
    const int steps_per_split = stages_of_a_split(k, splits) * kStepsPerStage;
    const bool far = k_steps > kMostSteps;
    const int tiles = tiles_of(m, n, k, splits, most_tiles);
    const dim3 grid((n_tiles + tiles - 1) / tiles, splits);
    const auto launch = [&](auto tiles_a_wave, auto waves) {
        constexpr int kWaves = decltype(waves)::value;
        gemm_medium_kernel<MT, decltype(tiles_a_wave)::value, kWaves, EPILOGUE, false><<<grid, kWaves * kWave, 0, stream>>>(
            a, w, out, m, n, k, n_tiles, k_steps, steps_per_split, tiles);
    };
    using std::integral_constant;
    if (far) {
        gemm_medium_kernel<MT, 1, 4, EPILOGUE, true><<<grid, 4 * kWave, 0, stream>>>(a, w, out, m, n, k, n_tiles, k_steps, steps_per_split, tiles);
        return;
    }
    // Four waves where there are no more tiles (64 rows of 9728 x 896, 3 tiles a workgroup: 11.7 -> 9.6 us, now 8.5). Four waves of up to four
    // tiles each read LDS half as often, but hold too much: 64 rows of 37888 x 3584 51.7 -> 55.6 us.
    if (tiles <= 4) launch(integral_constant<int, 1>{}, integral_constant<int, 4>{});
    else if (tiles <= 8) launch(integral_constant<int, 1>{}, integral_constant<int, 8>{});
    else launch(integral_constant<int, 2>{}, integral_constant<int, 8>{});
}

template <int EPILOGUE>
static int launch_medium(const void* a, const void* w_packed, void* out, int m, int n, int k, int most_tiles, int splits, hipStream_t stream) {
    const bf16* a_ = static_cast<const bf16*>(a);
    const bf16* w_ = static_cast<const bf16*>(w_packed);
    switch ((m + 15) / 16) {
        case 1: launch_rows<1, EPILOGUE>(a_, w_, out, m, n, k, most_tiles, splits, stream); break;
        case 2: launch_rows<2, EPILOGUE>(a_, w_, out, m, n, k, most_tiles, splits, stream); break;
        case 3: launch_rows<3, EPILOGUE>(a_, w_, out, m, n, k, most_tiles, splits, stream); break;
        case 4: launch_rows<4, EPILOGUE>(a_, w_, out, m, n, k, most_tiles, splits, stream); break;
        default: return fail("gemm_medium: more than 64 rows");
    }
    return check_launch("gemm_medium");
}

}  // namespace medium
}  // namespace mll

using namespace mll;

extern "C" int mll_gemm_medium_tiles(int m, int n, int k, int tiles_per_wave, int waves, int splits) {
    return medium::tiles_of(m, n, k, splits, tiles_per_wave * waves);
}

extern "C" int mll_gemm_medium(const void* a, const void* w_packed, void* out, int epilogue, int m, int n, int k,
                               int tiles_per_wave, int waves, int splits, hipStream_t stream) {
    MLL_REQUIRE(m >= 0 && m <= 64, "gemm_medium: takes at most 64 rows");
    MLL_REQUIRE(n > 0 && k > 0 && k % 8 == 0, "gemm_medium: k must be a positive multiple of 8");
    MLL_REQUIRE(tiles_per_wave == 1 || tiles_per_wave == 2, "gemm_medium: a wave takes one or two tiles of the weight");
    MLL_REQUIRE(waves == 4 || waves == 8, "gemm_medium: workgroups of 4 or 8 waves");
    MLL_REQUIRE(splits >= 1 && splits <= 64, "gemm_medium: between 1 and 64 splits of k");
    MLL_REQUIRE(epilogue == 0 || splits == 1, "gemm_medium: only float32 partial sums can be split over k");
    MLL_REQUIRE((epilogue != 2 && epilogue != 5) || n % 2 == 0, "gemm_medium: the gated epilogue needs an even number of weight rows");
    MLL_REQUIRE(reinterpret_cast<uintptr_t>(a) % 16 == 0, "gemm_medium: the activations must be 16-byte aligned");
    if (m == 0) return 0;
    switch (epilogue) {
        case 0: return medium::launch_medium<0>(a, w_packed, out, m, n, k, tiles_per_wave * waves, splits, stream);
        case 1: return medium::launch_medium<1>(a, w_packed, out, m, n, k, tiles_per_wave * waves, splits, stream);
        case 2: return medium::launch_medium<2>(a, w_packed, out, m, n, k, tiles_per_wave * waves, splits, stream);
        case 5: return medium::launch_medium<5>(a, w_packed, out, m, n, k, tiles_per_wave * waves, splits, stream);
        default: return fail("gemm_medium: unknown epilogue");
    }
}
