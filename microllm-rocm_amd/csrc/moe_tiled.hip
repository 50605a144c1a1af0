// The chosen experts' products for many (token, choice) pairs, in large tiles: the pairs lie in the order of their experts
// (moe_sort_kernel in moe.hip), and a workgroup of 8 waves takes up to 256 pairs of one expert and 256 rows of its weight, with the main loop of
// gemm_tiled.hip: stages of 64 of the reduction by direct loads into LDS slots (two of A, three of W), the operands of a k step read from
// LDS between the products of the step before. Here both sides are rows of memory, 8 rows of 128 bytes a load, and A's rows are taken from
// wherever their tokens lie. Bound by the products of a stage with what stands between them (1.5 us; gemm_tiled.hip) and by a tile's beginning and end, which
// nothing overlaps: as many workgroups as compute units go from tile to tile, and the height of the tiles is chosen so that their rounds are done
// first (an expert's last pairs take a tile of 192 or 128 rows where that is enough). 3117 tokens with 4 of 16 experts of 2048 x 2048 and 4
// ids that return their input: 426 -> 343 us with gate, up, down and the sort (tiles of 256 by a workgroup each 401), 0.73 PFLOP/s; loads
// through buffer descriptors, 16 experts without those ids, 352 -> 348 to 360 -> 352.
// The tiles of all experts stand in a row, an expert after another, its columns one after another and down the rows first; every XCD takes
// an equal stretch, so that the workgroups that run together there share an expert's rows and neighbouring rows of its weight.
// A result's additions are those of moe_grouped_kernel in the same order, so a pair's bits do not depend on which of the two it meets.
#include "common.h"
#include "microllm_hip.h"
#include "moe_tiled.h"
#include "tiled_operands.h"

namespace mll {

namespace {

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

constexpr int kTileCols = 256;              // rows of the weight in a tile
constexpr int kComputeUnits = 256;
constexpr int kHeights[3] = {256, 192, 128};    // pairs of a tile, at most

struct Tiling {
    int height, tiles;       // tiles of pairs over all experts
};
struct TileOfExpert {
    int expert, first_row, rows, column;
};

// The height of which all tiles are done first, if every round of the compute units takes as long as a stage's loads (rows + columns). A
// lane an expert, 64 at a time.
__device__ inline Tiling choose_tiling(const int32_t* __restrict__ offsets, int experts, int n_blocks, int lane) {
    int tiles[3] = {0, 0, 0};
    for (int base = 0; base < experts; base += kWave) {
        const int e = base + lane;
        const int count = e < experts ? offsets[e + 1] - offsets[e] : 0;
#pragma unroll
        for (int i = 0; i < 3; ++i) tiles[i] += (count + kHeights[i] - 1) / kHeights[i];
    }
    Tiling best = {0, 0};
    int64_t least = 0;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        for (int offset = kWave / 2; offset > 0; offset >>= 1) tiles[i] += __shfl_xor(tiles[i], offset, kWave);
        const int64_t cost = (static_cast<int64_t>(tiles[i]) * n_blocks + kComputeUnits - 1) / kComputeUnits * (kHeights[i] + kTileCols);
        if (i == 0 || cost < least) {
            best = Tiling{kHeights[i], tiles[i]};
            least = cost;
        }
    }
    return Tiling{__builtin_amdgcn_readfirstlane(best.height), __builtin_amdgcn_readfirstlane(best.tiles)};
}

// The tile at a place of the row of all tiles (which has one there).
__device__ inline TileOfExpert tile_at(int place, const int32_t* __restrict__ offsets, int experts, int n_blocks, int height, int lane) {
    TileOfExpert found = {0, 0, 0, 0};
    int before = 0;         // tiles of the experts so far
    for (int base = 0; base < experts; base += kWave) {
        const int e = base + lane;
        const int begin = e < experts ? offsets[e] : 0, count = e < experts ? offsets[e + 1] - begin : 0;
        const int tiles = (count + height - 1) / height;
        int up_to_me = tiles;
        for (int offset = 1; offset < kWave; offset <<= 1) {
            const int theirs = __shfl_up(up_to_me, offset, kWave);
            if (lane >= offset) up_to_me += theirs;
        }
        const int last = (before + up_to_me) * n_blocks, first = last - tiles * n_blocks;
        const unsigned long long here = __ballot(place >= first && place < last);
        if (here != 0) {
            const int owner = __ffsll(here) - 1;
            const int within = place - __shfl(first, owner, kWave), high = __shfl(tiles, owner, kWave);
            const int row = within % high * height;
            found.expert = __builtin_amdgcn_readfirstlane(base + owner);
            found.first_row = __builtin_amdgcn_readfirstlane(__shfl(begin, owner, kWave) + row);
            found.rows = __builtin_amdgcn_readfirstlane(min(height, __shfl(count, owner, kWave) - row));
            found.column = __builtin_amdgcn_readfirstlane(within / high);
            break;
        }
        before += __shfl(up_to_me, kWave - 1, kWave);
    }
    return found;
}

// FORM as in moe_grouped_kernel: 1 gated, 2 one inner weight, 0 down. The products of a tile of up to 32 WM pairs.
template <int FORM, int WM>
__device__ __attribute__((always_inline)) inline void tile_products(bf16* slots, const TileOfExpert& tile, const bf16* __restrict__ a,
                                                                    const bf16* __restrict__ w, const int32_t* __restrict__ order,
                                                                    const float* __restrict__ weights, int n_out, int k, void* __restrict__ out,
                                                                    int top, int n_tokens, int weight_on_input, int from_tokens,
                                                                    const MllExpertForm& form) {
    constexpr bool GATED = FORM == 1;
    constexpr int A_TURNS = WM / 2;        // loads of 8 rows a wave and stage
    constexpr int W_TURNS = 4;
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int col = lane % 16, quad = lane / 16;
    const int wave_m = wave / 4, wave_n = wave % 4;
    // A gated tile holds 128 gate rows and the 128 up rows that belong to them: of a wave's four tiles of 16 two are gate's and two up's.
    const int column0 = tile.column * (GATED ? kTileCols / 2 : kTileCols);
    const bf16* w_expert = w + static_cast<int64_t>(tile.expert) * (GATED ? 2 * n_out : n_out) * k;

    // Load i of a stage brings rows 8 i .. 8 i + 7 of the tile, lane L chunk (L % 8) ^ (row / 2) of row L / 8 of them; a wave takes
    // the loads wave, wave + 8, ... Rows past the end repeat the last one.
    const int row_in_piece = 8 * (wave % 2) + lane / 8;
    const int chunk = ((lane % 8) ^ (row_in_piece / 2)) * 8;
    unsigned a_from[A_TURNS], w_from[W_TURNS];         // bytes from `a` and from the expert's weight: 32 bits, which the caller has checked
#pragma unroll
    for (int t = 0; t < A_TURNS; ++t) {
        const int row = tile.first_row + min((wave + t * kTiledWaves) * 8 + lane / 8, tile.rows - 1);
        a_from[t] = (static_cast<unsigned>(from_tokens ? order[row] / top : row) * static_cast<unsigned>(k) + chunk) * 2;
    }
#pragma unroll
    for (int t = 0; t < W_TURNS; ++t) {
        const int row = (wave + t * kTiledWaves) * 8 + lane / 8;       // 64 of a wave's columns of C, 16 a tile
        int w_row;
        if (GATED) {
            const int column = min(column0 + row / 64 * 32 + row % 32, n_out - 1);
            w_row = row % 64 < 32 ? column : n_out + column;
        } else {
            w_row = min(column0 + row, n_out - 1);
        }
        w_from[t] = (static_cast<unsigned>(w_row) * static_cast<unsigned>(k) + chunk) * 2;
    }
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(a), 0, 0xffffffff, kBufferFlags);
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(w_expert), 0, 0xffffffff, kBufferFlags);
    auto copy_a = [&](int turn, int stage, unsigned slot) __attribute__((always_inline)) {
        bf16* place = slots + slot * kSlotElements + wave * 512;
        const unsigned at = a_from[turn];
        __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, place + turn * (kTiledWaves * 512), 16, at, stage * 128, 0, 0);
    };
    auto copy_w = [&](int turn, int stage, unsigned slot) __attribute__((always_inline)) {
        bf16* place = slots + (kASlots + slot) * kSlotElements + wave * 512;
        const unsigned at = w_from[turn];
        __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, place + turn * (kTiledWaves * 512), 16, at, stage * 128, 0, 0);
    };
    const unsigned base = lds_address(slots);
    const unsigned step0 = col * 128 + ((quad ^ (col / 2)) * 16), step1 = col * 128 + (((4 + quad) ^ (col / 2)) * 16);
    const unsigned a_at = base + wave_m * WM * 2048, w_at = base + kASlots * kSlotBytes + wave_n * kWaveTilesN * 2048;

    floatx4 acc[kWaveTilesN][WM];     // acc[nt][mt][i] = C[pair mt*16 + col][weight row nt*16 + quad*4 + i] of the wave's part
    const auto last_comes = [] {};      // reductions are whole stages
    begin_stages<A_TURNS>(0, k / 64, copy_a, copy_w, last_comes);
    multiply_stages<0, WM, A_TURNS, 0>(acc, 0, k / 64, false, a_at + step0, a_at + step1, w_at + step0, w_at + step1, copy_a, copy_w, last_comes);

    if constexpr (GATED) {
        workgroup_meets();
        const int row0 = wave_m * (WM * 16), column = column0 + wave_n * 32 + (lane % 4) * 8;
        const unsigned place = base + (kASlots + 2) * kSlotBytes + wave * (kResultRows * kResultBytes);
        const unsigned words_at = place + col * kResultBytes + (((quad / 2) ^ (col / 4)) * 16) + (quad % 2) * 8;
        bf16* to = static_cast<bf16*>(out) + static_cast<int64_t>(tile.first_row + row0 + lane / 4) * n_out + column;
        auto put_tiles = [&](auto mt) __attribute__((always_inline)) {
            constexpr int MT = decltype(mt)::value;
#pragma unroll
            for (int nt = 0; nt < kWaveTilesN / 2; ++nt) {
                bf16x4 four;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    four[i] = static_cast<__bf16>(gated_value_fast(acc[nt][MT][i], acc[nt + 2][MT][i], form.activation, form.limit, form.slope));
                put_result<MT % 4 * 16 * kResultBytes>(words_at ^ (nt * 32), __builtin_bit_cast(uint64_t, four));
            }
        };
        auto half = [&](auto first_tile) __attribute__((always_inline)) {
            constexpr int FIRST = decltype(first_tile)::value, COUNT = WM - FIRST < 4 ? WM - FIRST : 4;
            put_tiles(std::integral_constant<int, FIRST>{});
            put_tiles(std::integral_constant<int, FIRST + 1>{});
            if constexpr (COUNT > 2) put_tiles(std::integral_constant<int, FIRST + 2 * (COUNT > 2)>{});
            if constexpr (COUNT > 3) put_tiles(std::integral_constant<int, FIRST + 3 * (COUNT > 3)>{});
            uintx4 piece[4];
            get_results(piece, place, lane);
#pragma unroll
            for (int i = 0; i < COUNT; ++i)
                if (row0 + (FIRST + i) * 16 + lane / 4 < tile.rows && column < n_out)
                    *reinterpret_cast<uintx4*>(to + static_cast<int64_t>((FIRST + i) * 16) * n_out) = piece[i];
        };
        half(std::integral_constant<int, 0>{});
        if constexpr (WM > 4) half(std::integral_constant<int, 4>{});
        return;
    }
#pragma unroll
    for (int mt = 0; mt < WM; ++mt) {
        const int row = wave_m * (WM * 16) + mt * 16 + col;
        if (row >= tile.rows) continue;
        const int sorted = tile.first_row + row;
        if constexpr (FORM == 0) {
            const int pair = order[sorted];
            const float factor = weight_on_input ? 1.0f : weights[pair];
            float* to = static_cast<float*>(out) + (static_cast<int64_t>(pair % top) * n_tokens + pair / top) * n_out;
#pragma unroll
            for (int nt = 0; nt < kWaveTilesN; ++nt) {
                const int column = column0 + wave_n * 64 + nt * 16 + quad * 4;      // four columns or none: n_out is a multiple of 8
                if (column < n_out) *reinterpret_cast<floatx4*>(to + column) = acc[nt][mt] * factor;
            }
        } else {
            bf16* to = static_cast<bf16*>(out) + static_cast<int64_t>(sorted) * n_out;
#pragma unroll
            for (int nt = 0; nt < kWaveTilesN; ++nt) {
                const int column = column0 + wave_n * 64 + nt * 16 + quad * 4;
                bf16x4 four;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    four[i] = static_cast<__bf16>(activate(acc[nt][mt][i], form.activation));
                if (column < n_out) *reinterpret_cast<bf16x4*>(to + column) = four;
            }
        }
    }
}

}  // namespace

template <int FORM>
__global__ __launch_bounds__(kTiledThreads, 1) void moe_tiled_kernel(const bf16* __restrict__ a, const bf16* __restrict__ w,
                                                                     const int32_t* __restrict__ offsets, const int32_t* __restrict__ order,
                                                                     const float* __restrict__ weights, int n_out, int k, void* __restrict__ out,
                                                                     int top, int n_tokens, int weight_on_input, int from_tokens,
                                                                     const bf16* __restrict__ x, MllExpertForm form) {
    __shared__ __align__(kSlotsAlign) bf16 slots[kStageElements];
    constexpr int kOutputsATile = FORM == 1 ? kTileCols / 2 : kTileCols;
    const int lane = threadIdx.x % kWave;
    const int n_blocks = (n_out + kOutputsATile - 1) / kOutputsATile;
    const Tiling tiling = choose_tiling(offsets, form.experts, n_blocks, lane);
    // Workgroups 8 apart in number run on one XCD: an equal stretch of the tiles each, whose workgroups go along it together.
    const int all = tiling.tiles * n_blocks, per_xcd = (all + 7) / 8;
    for (int index = blockIdx.x / 8; index < per_xcd; index += gridDim.x / 8) {
        const int place = blockIdx.x % 8 * per_xcd + index;
        if (place >= all) break;        // the same for every thread of the workgroup
        const TileOfExpert tile = tile_at(place, offsets, form.experts, n_blocks, tiling.height, lane);
        workgroup_meets();      // every wave is done with the slots of the tile before
        if (tile.rows > 192) tile_products<FORM, 8>(slots, tile, a, w, order, weights, n_out, k, out, top, n_tokens, weight_on_input, from_tokens, form);
        else if (tile.rows > 128) tile_products<FORM, 6>(slots, tile, a, w, order, weights, n_out, k, out, top, n_tokens, weight_on_input, from_tokens, form);
        else if (tile.rows > 0) tile_products<FORM, 4>(slots, tile, a, w, order, weights, n_out, k, out, top, n_tokens, weight_on_input, from_tokens, form);
    }
    if (FORM != 0 || form.identity == 0) return;
    // The pairs of ids that return their input stand behind the experts': their inputs times their weights, eight columns a thread.
    const int first = offsets[form.experts], last = offsets[form.experts + form.identity];
    const int pieces = n_out / 8;       // n_out is a multiple of 8
    const int64_t count = static_cast<int64_t>(last - first) * pieces;
    for (int64_t index = static_cast<int64_t>(blockIdx.x) * kTiledThreads + threadIdx.x; index < count; index += static_cast<int64_t>(gridDim.x) * kTiledThreads) {
        const int pair = order[first + static_cast<int>(index / pieces)], column = static_cast<int>(index % pieces) * 8;
        const float weight = weights[pair];
        const uintx4 given = *reinterpret_cast<const uintx4*>(x + static_cast<int64_t>(pair / top) * n_out + column);
        floatx4* to = reinterpret_cast<floatx4*>(static_cast<float*>(out) + (static_cast<int64_t>(pair % top) * n_tokens + pair / top) * n_out + column);
        floatx4 values[2];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            values[i / 2][2 * i % 4] = __builtin_bit_cast(float, given[i] << 16) * weight;
            values[i / 2][(2 * i + 1) % 4] = __builtin_bit_cast(float, given[i] & 0xffff0000u) * weight;
        }
        to[0] = values[0];
        to[1] = values[1];
    }
}

template <int FORM>
static int launch_form(const bf16* a, const bf16* w, const int32_t* offsets, const int32_t* order, const float* weights, int n_out, int k, void* out,
                       int top, int n_tokens, int weight_on_input, int from_tokens, const bf16* x, const MllExpertForm& form, hipStream_t stream) {
    const int columns = FORM == 1 ? kTileCols / 2 : kTileCols;
    // as many workgroups as run at once, fewer where there cannot be as many tiles (every expert's last one may hold one pair)
    const int64_t most = (static_cast<int64_t>(n_tokens) * top / kHeights[2] + form.experts) * ((n_out + columns - 1) / columns);
    MLL_REQUIRE(most < (1ll << 31), "moe_tiled: too many tiles");
    const int groups = static_cast<int>(most < kComputeUnits ? (most + 7) / 8 * 8 : kComputeUnits);
    moe_tiled_kernel<FORM><<<groups, kTiledThreads, 0, stream>>>(
        a, w, offsets, order, weights, n_out, k, out, top, n_tokens, weight_on_input, from_tokens, x, form);
    return check_launch("moe_tiled");
}

int launch_moe_tiled(int form_number, const bf16* a, const bf16* w, const int32_t* offsets, const int32_t* order, const float* weights, int n_out,
                     int k, void* out, int top, int n_tokens, int weight_on_input, int from_tokens, const bf16* x, const MllExpertForm& form,
                     hipStream_t stream) {
    switch (form_number) {
        case 1: return launch_form<1>(a, w, offsets, order, weights, n_out, k, out, top, n_tokens, weight_on_input, from_tokens, x, form, stream);
        case 2: return launch_form<2>(a, w, offsets, order, weights, n_out, k, out, top, n_tokens, weight_on_input, from_tokens, x, form, stream);
        default: return launch_form<0>(a, w, offsets, order, weights, n_out, k, out, top, n_tokens, weight_on_input, from_tokens, x, form, stream);
    }
}

}  // namespace mll
