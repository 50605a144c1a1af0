// Paged attention, one wave per (query token, head) or per (query token, head, chunk of keys): the plain path
// that every dtype and every head size can take, and the float32 path's only attention.
//
// A query's keys are cut into chunks of 128 at absolute positions. Within a chunk the keys are reduced in tiles
// of 64, also at absolute positions, with a running maximum and sum; the chunks' results are then merged one
// after the other, lowest positions first. Both happen in a fixed order that depends on the query's position
// and its window alone, so a query's result does not depend on the step's cut, the batch or the pages, to the
// last bit. Two ways to run this give the same bits: one wave walks all chunks of its row and merges as it goes
// (steps with many rows: portions of prompts), or one wave per chunk leaves its result in a workspace and a
// second kernel merges them (steps with few rows, whose keys would otherwise be walked by a handful of waves).
// Sums that decide bits are written with explicit fused multiply-adds, so that both kernels round alike.
//
// Runs of 16 tokens of one request in steps with many rows (prompts) take a third kernel in float32, which does the
// same operations in the same order on the matrix units: a float32 MFMA of gfx950 gives, element by element, the bits of
// fused multiply-adds in ascending order of its terms (gemm_f32.hip).
#include <type_traits>

#include "cache_layout.h"
#include "common.h"
#include "microllm_hip.h"

namespace mll {

constexpr int kRowwiseMaxHeadDim = 512;
constexpr int kRowwiseChunk = 128;      // keys; a multiple of the tiles of 64
// How many query heads of a kv head a wave takes in the float32 kernels: 0 lets the launch choose by how many waves
// the step then still has (rowwise_heads_a_wave); tests and measurements force 1 to 8 with mll_rowwise_heads_a_wave.
static int forced_heads_a_wave = 0;
constexpr int64_t kRowwiseWavesWanted = 4096;      // four a SIMD: fewer leave the loads' latency in the open

__device__ inline void load_eight(const float* from, float (&to)[8]) {
    const float4 low = *reinterpret_cast<const float4*>(from);
    const float4 high = *reinterpret_cast<const float4*>(from + 4);
    to[0] = low.x, to[1] = low.y, to[2] = low.z, to[3] = low.w;
    to[4] = high.x, to[5] = high.y, to[6] = high.z, to[7] = high.w;
}

__device__ inline void load_eight(const bf16* from, float (&to)[8]) {
    union { uint4 raw; bf16 values[8]; } piece;
    piece.raw = *reinterpret_cast<const uint4*>(from);
#pragma unroll
    for (int i = 0; i < 8; ++i) to[i] = to_float(piece.values[i]);
}

// What a row needs to walk its keys.
template <typename T>
struct RowwiseRow {
    const T* k_cache;
    const T* v_cache;
    const int32_t* table;
    int kv_head, head_dim, page_size, lane;
    int low, position;      // the keys the query sees
    float scale;
};

// The keys [first, last] of one chunk (all visible, in one chunk): maximum, sum of exp(score - maximum) and the
// weighted sum of values (dims lane, lane + 64, ...), from zero. q_shared holds the query.
template <typename T, int DIMS>
__device__ inline void attend_chunk(const RowwiseRow<T>& row, const CacheLayout& layout, const float* q_shared,
                                    float* p_shared, int64_t (*v_shared)[kWave], int first, int last, float& chunk_max,
                                    float& chunk_sum, float (&acc)[DIMS]) {
    const int lane = row.lane;
#pragma unroll
    for (int i = 0; i < DIMS; ++i) acc[i] = 0.0f;
    chunk_max = -INFINITY;
    chunk_sum = 0.0f;
    for (int tile = (first / kWave) * kWave; tile <= last; tile += kWave) {
        const int key = tile + lane;
        const bool visible = key >= first && key <= last;
        float score = -INFINITY;
        int64_t v_place = 0, v_place_last = 0;
        if (visible) {
            const int64_t page = row.table[key / row.page_size];
            const int offset = key % row.page_size;
            const T* k_tile = row.k_cache + layout.k_tile(page, row.kv_head, offset / 16) + (offset % 16) * 8;
            // Values lie as [dim / 32][position / 8][dim % 32][position % 8], a last block of 16 dims as
            // [position / 8][16][8] (cache_layout.h): the share of the place that the key's group of 8 positions
            // has, for either kind of block; the dim's share is added below.
            const int64_t v_tile = layout.v_tile(page, row.kv_head, offset / 16);
            v_place = v_tile + ((offset % 16) / 8) * 256;
            v_place_last = v_tile + ((offset % 16) / 8) * 128;
            float dot = 0.0f;
            const int whole = row.head_dim / 8 * 8;
            for (int d = 0; d < whole; d += 8) {      // keys lie as [dim / 8][position][dim % 8]
                float k[8];
                load_eight(k_tile + (d / 8) * 128, k);
#pragma unroll
                for (int i = 0; i < 8; ++i) dot = __fmaf_rn(q_shared[d + i], k[i], dot);
            }
            for (int d = whole; d < row.head_dim; ++d) dot = __fmaf_rn(q_shared[d], to_float(k_tile[(d / 8) * 128 + d % 8]), dot);
            score = __fmul_rn(dot, row.scale);
        }
        const float new_max = fmaxf(chunk_max, wave_max(score));      // every tile holds a visible key
        const float p = visible ? expf(score - new_max) : 0.0f;
        const float rescale = expf(chunk_max - new_max);               // exp(-inf) = 0 on the first tile
        chunk_sum = __fmaf_rn(chunk_sum, rescale, wave_sum(p));
        chunk_max = new_max;

        __syncthreads();      // the previous tile's readers are done
        p_shared[lane] = p;
        v_shared[0][lane] = v_place;
        v_shared[1][lane] = v_place_last;
        __syncthreads();
        const int begin = max(first - tile, 0);
        const int end = min(last - tile, kWave - 1);
#pragma unroll
        for (int i = 0; i < DIMS; ++i) {
            const int d = lane + i * kWave;
            if (d < row.head_dim) {
                const int of_dim = layout.v_in_tile(0, d);
                const int64_t* places = v_shared[layout.v_in_tile(8, d) - of_dim == 256 ? 0 : 1];
                float value = __fmul_rn(acc[i], rescale);
                // Eight positions lie side by side: one read brings a dim's values of a group of 8 keys, of which the
                // visible ones are added in the order of the keys (the others may be stale memory: never multiplied).
                for (int group = begin / 8; group <= end / 8; ++group) {
                    const int from = max(begin, 8 * group), to = min(end, 8 * group + 7);
                    float v[8];
                    load_eight(row.v_cache + places[from] + of_dim, v);
#pragma unroll
                    for (int r = 0; r < 8; ++r)
                        if (8 * group + r >= from && 8 * group + r <= to) value = __fmaf_rn(p_shared[8 * group + r], v[r], value);
                }
                acc[i] = value;
            }
        }
    }
}

// (maximum, sum, values) of the chunks so far, and one more chunk: the same arithmetic wherever chunks are merged.
__device__ inline void merge_scales(float so_far_max, float chunk_max, float& new_max, float& keep, float& add) {
    new_max = fmaxf(so_far_max, chunk_max);
    keep = so_far_max == -INFINITY ? 0.0f : expf(so_far_max - new_max);
    add = expf(chunk_max - new_max);
}

__device__ inline float merged(float so_far, float keep, float chunk, float add) {
    return __fmaf_rn(so_far, keep, __fmul_rn(chunk, add));
}

// ---- runs of 16 tokens on the matrix units -----------------------------------------------------------------------
typedef float floatx4 __attribute__((ext_vector_type(4)));
constexpr int kRunTokens = 16;
constexpr int kMostRuns = 3;             // stretches of a block
constexpr int64_t kRunsWork = 50000000;  // tokens * heads * head size * keys: 100 tokens of one request, 28 heads of 128, 40 million, take 26 us a wave a token and 31 so
// Tokens a request, on average, from which a step's stretches are worth a launch of their own beside the kernels for the rest, by
// how many keys the step reaches (28 heads of 128, a wave a token and so): 32 requests of 33 and 48 new tokens 75 and 86 us, 103
// and 62; 128 of 16 after 500 1383 and 391; 32 of 12 after 500 235 and 105, of 6 175 and 220.
static int64_t runs_from(int64_t keys) { return keys < kWave ? 40 : keys < 4 * kWave ? 16 : 8; }

// The tokens 16 * block .. + 15 of the step in stretches of places of one request in a row: bit i is set where token i begins
// one. Tokens that only pad the step, or lie past its end, begin one each and belong to none (`none`).
struct TokenRuns {
    unsigned begins, none;
    int most;       // stretches with which the block is taken
    __device__ int end_of(int begin) const {      // where the stretch that begins there ends
        const unsigned after = begins & ~((2u << begin) - 1);
        return after ? __ffs(after) - 1 : kRunTokens;
    }
    // A wave on the matrix units takes as long for one token as for 16, 22 + 0.17 ns a key over the whole GPU (28 heads of 128), a wave a
    // token 1.7 + 0.044: the more keys, the shorter a stretch may be.
    __device__ bool taken() const { return __popc(begins & ~none) <= most; }
};
__device__ inline TokenRuns token_runs(const int32_t* seq_of_token, const int32_t* positions, int block, int n_tokens) {
    const int at = static_cast<int>(threadIdx.x) % kRunTokens;
    const int token = min(block * kRunTokens + at, n_tokens - 1), before = max(token - 1, 0);
    const int seq = seq_of_token[token];
    const bool none = block * kRunTokens + at >= n_tokens || seq < 0;
    const bool begins = none || at == 0 || seq_of_token[before] != seq || positions[before] + 1 != positions[token];
    TokenRuns runs;
    runs.begins = static_cast<unsigned>(__ballot(begins)) & 0xffffu;
    runs.none = static_cast<unsigned>(__ballot(none)) & 0xffffu;
    const int position = none ? 0 : positions[token];
    runs.most = __ballot(position >= 4 * kWave) != 0 ? kMostRuns : __ballot(position >= kWave) != 0 ? 2 : 1;
    return runs;
}

// DIMS: dims a lane holds (head_dim <= 64 * DIMS). MODE 0: one wave per (token, head) walks all chunks. MODE 1: one wave per (token, head, chunk) writes
// part_o[row][slot][dim] and part_ml[row][slot] = (maximum, sum), slot counting from the row's first chunk.
template <typename T, int MODE, int DIMS>
__global__ __launch_bounds__(kWave) void paged_attention_rowwise_kernel(
    const T* __restrict__ q, const T* __restrict__ k_cache, const T* __restrict__ v_cache,
    const int32_t* __restrict__ block_table, int table_width, const int32_t* __restrict__ seq_of_token,
    const int32_t* __restrict__ positions, T* __restrict__ out, float* __restrict__ part_o,
    float* __restrict__ part_ml, int max_chunks, float scale, int window, int heads, int kv_heads, int head_dim,
    int page_size, int runs_apart) {
    __shared__ float q_shared[kRowwiseMaxHeadDim];
    __shared__ float p_shared[kWave];
    __shared__ int64_t v_shared[2][kWave];
    const CacheLayout layout(kv_heads, page_size, head_dim);

    const int token = blockIdx.x;
    const int head = blockIdx.y;
    const int lane = threadIdx.x;
    const int seq = seq_of_token[token];
    if (seq < 0) return;      // a row that only pads the step to a fixed shape: its output stays as it is
    if (MODE == 0 && runs_apart && token_runs(seq_of_token, positions, token / kRunTokens, gridDim.x).taken()) return;
    const int position = positions[token];
    const int low = window > 0 ? max(0, position - window + 1) : 0;
    const int first_chunk = low / kRowwiseChunk, last_chunk = position / kRowwiseChunk;
    if (MODE == 1 && first_chunk + static_cast<int>(blockIdx.z) > last_chunk) return;

    RowwiseRow<T> row;
    row.k_cache = k_cache;
    row.v_cache = v_cache;
    row.table = block_table + static_cast<int64_t>(seq) * table_width;
    row.kv_head = head / (heads / kv_heads);
    row.head_dim = head_dim;
    row.page_size = page_size;
    row.lane = lane;
    row.low = low;
    row.position = position;
    row.scale = scale;

    const T* q_row = q + (static_cast<int64_t>(token) * heads + head) * head_dim;
    for (int d = lane; d < head_dim; d += kWave) q_shared[d] = to_float(q_row[d]);
    __syncthreads();

    float acc[DIMS];
    float chunk_max, chunk_sum;
    if (MODE == 1) {
        const int chunk = first_chunk + blockIdx.z;
        attend_chunk(row, layout, q_shared, p_shared, v_shared, max(low, chunk * kRowwiseChunk),
                     min(position, chunk * kRowwiseChunk + kRowwiseChunk - 1), chunk_max, chunk_sum, acc);
        const int64_t slot = (static_cast<int64_t>(token) * heads + head) * max_chunks + blockIdx.z;
#pragma unroll
        for (int i = 0; i < DIMS; ++i) {
            const int d = lane + i * kWave;
            if (d < head_dim) part_o[slot * head_dim + d] = acc[i];
        }
        if (lane == 0) {
            part_ml[slot * 2] = chunk_max;
            part_ml[slot * 2 + 1] = chunk_sum;
        }
        return;
    }

    float total[DIMS];
#pragma unroll
    for (int i = 0; i < DIMS; ++i) total[i] = 0.0f;
    float total_max = -INFINITY, total_sum = 0.0f;
    for (int chunk = first_chunk; chunk <= last_chunk; ++chunk) {
        attend_chunk(row, layout, q_shared, p_shared, v_shared, max(low, chunk * kRowwiseChunk),
                     min(position, chunk * kRowwiseChunk + kRowwiseChunk - 1), chunk_max, chunk_sum, acc);
        float new_max, keep, add;
        merge_scales(total_max, chunk_max, new_max, keep, add);
        total_sum = merged(total_sum, keep, chunk_sum, add);
#pragma unroll
        for (int i = 0; i < DIMS; ++i) total[i] = merged(total[i], keep, acc[i], add);
        total_max = new_max;
    }
    T* out_row = out + (static_cast<int64_t>(token) * heads + head) * head_dim;
    const float inverse = 1.0f / total_sum;
#pragma unroll
    for (int i = 0; i < DIMS; ++i) {
        const int d = lane + i * kWave;
        if (d < head_dim) out_row[d] = from_float<T>(__fmul_rn(total[i], inverse));
    }
}

// MODE 1 for GW query heads of one kv head in one wave: a chunk's keys and values are read once and used for all of
// them (with 7 query heads a kv head the plain kernel reads every key 7 times, and it is those reads that bound it
// when a step has many rows of long requests). Head by head the operations and their order are those of
// attend_chunk: the dot products in ascending dims, the tile's maximum and sum over the wave, the values in the
// order of the keys; only what is independent of the head (addresses, loads) is done once. Writes what MODE 1 writes,
// bit for bit. Head sizes up to 64 * DIMS <= 128.
// MODE as in the kernel for one head a wave: 0 walks all chunks of the row and merges as it goes (out), 1 takes the chunk
// blockIdx.z and leaves its result in the workspace (part_o, part_ml). runs_apart (MODE 0, both kernels): tokens that
// paged_attention_rowwise_runs_kernel takes are passed over.
template <typename T, int MODE, int DIMS, int GW>
__global__ __launch_bounds__(kWave) void paged_attention_rowwise_heads_kernel(
    const T* __restrict__ q, const T* __restrict__ k_cache, const T* __restrict__ v_cache,
    const int32_t* __restrict__ block_table, int table_width, const int32_t* __restrict__ seq_of_token,
    const int32_t* __restrict__ positions, T* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml,
    int max_chunks, float scale, int window, int heads, int kv_heads, int head_dim, int page_size, int runs_apart) {
    __shared__ float q_shared[GW][64 * DIMS];
    __shared__ float p_shared[GW][kWave];
    __shared__ int64_t v_shared[2][kWave];
    const CacheLayout layout(kv_heads, page_size, head_dim);
    const int token = blockIdx.x;
    const int lane = threadIdx.x;
    const int group = heads / kv_heads;
    const int waves_of_group = (group + GW - 1) / GW;            // the group's last wave may have fewer heads
    const int kv_head = blockIdx.y / waves_of_group;
    const int first_in_group = (blockIdx.y % waves_of_group) * GW;
    const int first_head = kv_head * group + first_in_group;
    const int heads_here = min(GW, group - first_in_group);      // heads past them repeat the last one and write nothing
    const int seq = seq_of_token[token];
    if (seq < 0) return;
    if (MODE == 0 && runs_apart && token_runs(seq_of_token, positions, token / kRunTokens, gridDim.x).taken()) return;
    const int position = positions[token];
    const int low = window > 0 ? max(0, position - window + 1) : 0;
    const int first_chunk = low / kRowwiseChunk, last_chunk = position / kRowwiseChunk;
    if (MODE == 1 && first_chunk + static_cast<int>(blockIdx.z) > last_chunk) return;
    const int32_t* table = block_table + static_cast<int64_t>(seq) * table_width;
#pragma unroll
    for (int g = 0; g < GW; ++g) {
        const T* q_row = q + (static_cast<int64_t>(token) * heads + first_head + min(g, heads_here - 1)) * head_dim;
        for (int d = lane; d < head_dim; d += kWave) q_shared[g][d] = to_float(q_row[d]);
    }
    __syncthreads();

    float acc[GW][DIMS], chunk_max[GW], chunk_sum[GW];
    // The keys [first, last] of one chunk, from zero: attend_chunk for every head of the wave.
    auto attend = [&](int first, int last) __attribute__((always_inline)) {
#pragma unroll
    for (int g = 0; g < GW; ++g) {
        chunk_max[g] = -INFINITY;
        chunk_sum[g] = 0.0f;
#pragma unroll
        for (int i = 0; i < DIMS; ++i) acc[g][i] = 0.0f;
    }
    for (int tile = (first / kWave) * kWave; tile <= last; tile += kWave) {
        const int key = tile + lane;
        const bool visible = key >= first && key <= last;
        float dot[GW];
#pragma unroll
        for (int g = 0; g < GW; ++g) dot[g] = 0.0f;
        int64_t v_place = 0, v_place_last = 0;
        if (visible) {
            const int64_t page = table[key / page_size];
            const int offset = key % page_size;
            const T* k_tile = k_cache + layout.k_tile(page, kv_head, offset / 16) + (offset % 16) * 8;
            const int64_t v_tile = layout.v_tile(page, kv_head, offset / 16);
            v_place = v_tile + ((offset % 16) / 8) * 256;
            v_place_last = v_tile + ((offset % 16) / 8) * 128;
            const int whole = head_dim / 8 * 8;
#pragma unroll 4
            for (int d = 0; d < whole; d += 8) {
                float k[8];
                load_eight(k_tile + (d / 8) * 128, k);
#pragma unroll
                for (int g = 0; g < GW; ++g)
#pragma unroll
                    for (int i = 0; i < 8; ++i) dot[g] = __fmaf_rn(q_shared[g][d + i], k[i], dot[g]);
            }
            for (int d = whole; d < head_dim; ++d) {
                const float k = to_float(k_tile[(d / 8) * 128 + d % 8]);
#pragma unroll
                for (int g = 0; g < GW; ++g) dot[g] = __fmaf_rn(q_shared[g][d], k, dot[g]);
            }
        }
        float rescale[GW];
        __syncthreads();      // the previous tile's readers are done
#pragma unroll
        for (int g = 0; g < GW; ++g) {
            const float score = visible ? __fmul_rn(dot[g], scale) : -INFINITY;
            const float new_max = fmaxf(chunk_max[g], wave_max(score));
            const float p = visible ? expf(score - new_max) : 0.0f;
            rescale[g] = expf(chunk_max[g] - new_max);
            chunk_sum[g] = __fmaf_rn(chunk_sum[g], rescale[g], wave_sum(p));
            chunk_max[g] = new_max;
            p_shared[g][lane] = p;
        }
        v_shared[0][lane] = v_place;
        v_shared[1][lane] = v_place_last;
        __syncthreads();
        const int begin = max(first - tile, 0);
        const int end = min(last - tile, kWave - 1);
#pragma unroll
        for (int i = 0; i < DIMS; ++i) {
            const int d = lane + i * kWave;
            if (d < head_dim) {
                const int of_dim = layout.v_in_tile(0, d);
                const int64_t* places = v_shared[layout.v_in_tile(8, d) - of_dim == 256 ? 0 : 1];
                float value[GW];
#pragma unroll
                for (int g = 0; g < GW; ++g) value[g] = __fmul_rn(acc[g][i], rescale[g]);
                for (int eight = begin / 8; eight <= end / 8; ++eight) {
                    const int from = max(begin, 8 * eight), to = min(end, 8 * eight + 7);
                    float v[8];
                    load_eight(v_cache + places[from] + of_dim, v);
#pragma unroll
                    for (int g = 0; g < GW; ++g)
#pragma unroll
                        for (int r = 0; r < 8; ++r)
                            if (8 * eight + r >= from && 8 * eight + r <= to) value[g] = __fmaf_rn(p_shared[g][8 * eight + r], v[r], value[g]);
                }
#pragma unroll
                for (int g = 0; g < GW; ++g) acc[g][i] = value[g];
            }
        }
    }
    };

    if (MODE == 1) {
        const int chunk = first_chunk + blockIdx.z;
        attend(max(low, chunk * kRowwiseChunk), min(position, chunk * kRowwiseChunk + kRowwiseChunk - 1));
#pragma unroll
        for (int g = 0; g < GW; ++g) {
            if (g >= heads_here) break;
            const int64_t slot = (static_cast<int64_t>(token) * heads + first_head + g) * max_chunks + blockIdx.z;
#pragma unroll
            for (int i = 0; i < DIMS; ++i) {
                const int d = lane + i * kWave;
                if (d < head_dim) part_o[slot * head_dim + d] = acc[g][i];
            }
            if (lane == 0) {
                part_ml[slot * 2] = chunk_max[g];
                part_ml[slot * 2 + 1] = chunk_sum[g];
            }
        }
        return;
    }
    float total[GW][DIMS], total_max[GW], total_sum[GW];
#pragma unroll
    for (int g = 0; g < GW; ++g) {
        total_max[g] = -INFINITY;
        total_sum[g] = 0.0f;
#pragma unroll
        for (int i = 0; i < DIMS; ++i) total[g][i] = 0.0f;
    }
    for (int chunk = first_chunk; chunk <= last_chunk; ++chunk) {
        attend(max(low, chunk * kRowwiseChunk), min(position, chunk * kRowwiseChunk + kRowwiseChunk - 1));
#pragma unroll
        for (int g = 0; g < GW; ++g) {
            float new_max, keep, add;
            merge_scales(total_max[g], chunk_max[g], new_max, keep, add);
            total_sum[g] = merged(total_sum[g], keep, chunk_sum[g], add);
#pragma unroll
            for (int i = 0; i < DIMS; ++i) total[g][i] = merged(total[g][i], keep, acc[g][i], add);
            total_max[g] = new_max;
        }
    }
#pragma unroll
    for (int g = 0; g < GW; ++g) {
        if (g >= heads_here) break;
        T* out_row = out + (static_cast<int64_t>(token) * heads + first_head + g) * head_dim;
        const float inverse = 1.0f / total_sum[g];
#pragma unroll
        for (int i = 0; i < DIMS; ++i) {
            const int d = lane + i * kWave;
            if (d < head_dim) out_row[d] = from_float<T>(__fmul_rn(total[g][i], inverse));
        }
    }
}

// Register j of quarter q of the wave becomes register q of quarter j.
__device__ inline floatx4 transpose_quarters(floatx4 v) {
    auto swap32 = [](unsigned& low, unsigned& high) {
        const auto both = __builtin_amdgcn_permlane32_swap(low, high, false, false);
        low = both[0], high = both[1];
    };
    auto swap16 = [](unsigned& low, unsigned& high) {
        const auto both = __builtin_amdgcn_permlane16_swap(low, high, false, false);
        low = both[0], high = both[1];
    };
    const float e0 = v[0], e1 = v[1], e2 = v[2], e3 = v[3];
    unsigned r0 = __builtin_bit_cast(unsigned, e0), r1 = __builtin_bit_cast(unsigned, e1);
    unsigned r2 = __builtin_bit_cast(unsigned, e2), r3 = __builtin_bit_cast(unsigned, e3);
    swap32(r0, r2);
    swap32(r1, r3);
    swap16(r0, r1);
    swap16(r2, r3);
    return floatx4{__builtin_bit_cast(float, r0), __builtin_bit_cast(float, r1), __builtin_bit_cast(float, r2), __builtin_bit_cast(float, r3)};
}

// The value of the lane 32, or 16, away (xor), without LDS.
__device__ inline float from_32_away(float value) {
    const unsigned bits = __builtin_bit_cast(unsigned, value);
    const auto halves = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
    const unsigned low = halves[0], high = halves[1];       // every lane: the lower half's value, the upper half's
    return __builtin_bit_cast(float, threadIdx.x % kWave < 32 ? high : low);
}
__device__ inline float from_16_away(float value) {
    const unsigned bits = __builtin_bit_cast(unsigned, value);
    const auto rows = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
    const unsigned even = rows[0], odd = rows[1];
    return __builtin_bit_cast(float, threadIdx.x % 32 < 16 ? odd : even);
}

// A wave takes a stretch of one request's tokens (token_runs: up to `sides` waves a block of 16 tokens, one stretch each) and one head, and walks the
// chunks and tiles of 64 keys as the kernels above do for one token, on v_mfma_f32_16x16x4_f32: S^T = K . Q^T leaves in lane (token, quarter) the scores of keys 16 t + 4 quarter +
// i, whose sum over the tile meets in the order of wave_sum (32, 16 in the lane, 8 and 4 between lanes, 2, 1 in the
// lane); O^T = V^T . P^T adds the keys in ascending order. All three operands come from memory with 16 bytes a lane, four consecutive
// terms of the reduction, where the product wants one of every four consecutive ones a quarter: transpose_quarters. The four waves of
// a workgroup are neighbouring heads, which mostly read the same keys. The last tile's keys, which not every token sees, are
// multiplied with a weight of zero where a token does not see them, which changes nothing unless a value is not finite:
// then that tile's values are added one by one as above.
// Bound by the matrix units and, with one wave a SIMD (up to 477 registers), by the loads of a tile's keys and values, which
// fly over one tile's arithmetic. Prompts of 1003 tokens of 14 heads of 64: 292 -> 80 us against a wave a token and four heads, 300 of
// 28 heads of 128: 123 -> 55, 1500: 985 -> 330. A block's stretches one after the other in one wave made 32 requests of 10 tokens after 500
// slower than a wave a token (206 -> 236 us); side by side they take 169.
template <int HD_TILES>
__global__ __launch_bounds__(256) void paged_attention_rowwise_runs_kernel(
    const float* __restrict__ q, const float* __restrict__ k_cache, const float* __restrict__ v_cache,
    const int32_t* __restrict__ block_table, int table_width, const int32_t* __restrict__ seq_of_token,
    const int32_t* __restrict__ positions, float* __restrict__ out, float scale, int n_tokens, int heads, int kv_heads, int page_size, int sides) {
#pragma clang fp contract(off)      // a scaled score less the maximum is two roundings, as in the kernels above
    constexpr int HD = HD_TILES * 16;
    const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int col = lane % 16, quad = lane / 16;
    const int blocks = (n_tokens + kRunTokens - 1) / kRunTokens;
    const int unit = blockIdx.x * 4 + wave;
    if (unit >= blocks * sides * heads) return;
    // The last tokens see the most keys: they go first, and every block's first stretch before any block's second, which is mostly none.
    const int block = blocks - 1 - unit / heads % blocks, head = unit % heads;
    const TokenRuns runs = token_runs(seq_of_token, positions, block, n_tokens);
    if (!runs.taken()) return;
    const CacheLayout layout(kv_heads, page_size, HD);
    const int kv_head = head / (heads / kv_heads);
    int number = unit / heads / blocks;        // of the block's stretches the wave's own, then every sides-th after it
    for (int begin = 0, end; begin < kRunTokens; begin = end) {
    end = __builtin_amdgcn_readfirstlane(runs.end_of(begin));
    if (((runs.none >> begin) & 1) || number-- > 0) continue;
    number = sides - 1;
    const int first_token = block * kRunTokens + begin, count = end - begin;
    const int token = first_token + min(col, count - 1);         // lanes past the stretch repeat its last token and write nothing
    const int first_position = __builtin_amdgcn_readfirstlane(positions[first_token]);
    const int position = first_position + min(col, count - 1), last_position = first_position + count - 1;
    const int32_t* table = block_table + static_cast<int64_t>(__builtin_amdgcn_readfirstlane(seq_of_token[first_token])) * table_width;

    floatx4 q_piece[HD_TILES];      // the B operand: lane (token, quarter) holds dims 16 d + 4 j + quarter
#pragma unroll
    for (int d = 0; d < HD_TILES; ++d)
        q_piece[d] = transpose_quarters(*reinterpret_cast<const floatx4*>(q + (static_cast<int64_t>(token) * heads + head) * HD + 16 * d + 4 * quad));

    auto pages_of = [&](int tile, int64_t (&page)[4]) {
#pragma unroll
        for (int t = 0; t < 4; ++t) page[t] = max(table[min((tile + 16 * t) / page_size, table_width - 1)], 0);     // keys that nobody sees may have none
    };
    auto load_keys = [&](int tile, const int64_t (&page)[4], floatx4 (&k)[4][HD_TILES]) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const float* from = k_cache + layout.k_tile(page[t], kv_head, (tile + 16 * t) % page_size / 16) + (quad / 2) * 128 + col * 8 + (quad % 2) * 4;
#pragma unroll
            for (int d = 0; d < HD_TILES; ++d) k[t][d] = *reinterpret_cast<const floatx4*>(from + d * 256);
        }
    };
    auto load_values = [&](int tile, const int64_t (&page)[4], floatx4 (&v)[4][HD_TILES]) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const float* from = v_cache + layout.v_tile(page[t], kv_head, (tile + 16 * t) % page_size / 16);
#pragma unroll
            for (int d = 0; d < HD_TILES; ++d) {
                const int width = (HD_TILES % 2 == 1 && d == HD_TILES - 1) ? 16 : 32;      // dims of the block of 32 this tile of 16 lies in
                v[t][d] = *reinterpret_cast<const floatx4*>(from + (d / 2) * 512 + ((quad / 2) * width + (d % 2) * 16 + col) * 8 + (quad % 2) * 4);
            }
        }
    };

    floatx4 acc[HD_TILES], total[HD_TILES];
#pragma unroll
    for (int d = 0; d < HD_TILES; ++d) acc[d] = total[d] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    float chunk_max = -INFINITY, chunk_sum = 0.0f, total_max = -INFINITY, total_sum = 0.0f;
    floatx4 k[4][HD_TILES], v[4][HD_TILES];
    int64_t page[4];
    pages_of(0, page);
    load_keys(0, page, k);
    load_values(0, page, v);
    for (int tile = 0; tile <= last_position; tile += kWave) {
        float score[4][4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            floatx4 s = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int d = 0; d < HD_TILES; ++d) {
                const floatx4 piece = transpose_quarters(k[t][d]);
#pragma unroll
                for (int step = 0; step < 4; ++step) s = __builtin_amdgcn_mfma_f32_16x16x4f32(piece[step], q_piece[d][step], s, 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) score[t][i] = tile + 16 * t + 4 * quad + i <= position ? __fmul_rn(s[i], scale) : -INFINITY;
        }
        const int next = min(tile + kWave, last_position / kWave * kWave);      // after the last tile that one again, dropped
        int64_t next_page[4];
        pages_of(next, next_page);
        load_keys(next, next_page, k);

        float tile_max = score[0][0];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) tile_max = fmaxf(tile_max, score[t][i]);
        tile_max = fmaxf(tile_max, from_32_away(tile_max));
        tile_max = fmaxf(tile_max, from_16_away(tile_max));
        // A token before the tile has nothing in it: its numbers stay what they are.
        const bool here = tile <= position;
        const float new_max = here ? fmaxf(chunk_max, tile_max) : chunk_max;
        const float rescale = here ? expf(chunk_max - new_max) : 1.0f;
        float p[4][4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) p[t][i] = tile + 16 * t + 4 * quad + i <= position ? expf(score[t][i] - new_max) : 0.0f;
        float part[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            part[i] = (p[0][i] + p[2][i]) + (p[1][i] + p[3][i]);
            part[i] += from_32_away(part[i]);
            part[i] += from_16_away(part[i]);
        }
        const float tile_sum = (part[0] + part[2]) + (part[1] + part[3]);
        chunk_sum = here ? __fmaf_rn(chunk_sum, rescale, tile_sum) : chunk_sum;
        chunk_max = new_max;

        const bool whole = tile + kWave - 1 <= first_position;      // every token sees every key
        bool finite = true;
        if (!whole) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int d = 0; d < HD_TILES; ++d)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if (tile + 16 * t + 4 * quad + i > last_position) v[t][d][i] = 0.0f;       // what lies there may be stale
                        finite = finite && __builtin_isfinite(v[t][d][i]);
                    }
            finite = __all(finite);
        }
#pragma unroll
        for (int d = 0; d < HD_TILES; ++d)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[d][i] = __fmul_rn(acc[d][i], rescale);
        if (finite) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const floatx4 weights = transpose_quarters(floatx4{p[t][0], p[t][1], p[t][2], p[t][3]});
#pragma unroll
                for (int d = 0; d < HD_TILES; ++d) {
                    const floatx4 piece = transpose_quarters(v[t][d]);
#pragma unroll
                    for (int step = 0; step < 4; ++step) acc[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(piece[step], weights[step], acc[d], 0, 0, 0);
                }
            }
        } else {
            for (int key = tile; key <= min(last_position, tile + kWave - 1); ++key) {
                const int in_tile = key - tile;
                float weight = 0.0f;
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float there = __shfl(p[t][i], 16 * (in_tile % 16 / 4) + col, kWave);
                        if (in_tile == 16 * t + in_tile % 16 / 4 * 4 + i) weight = there;
                    }
                const float* from = v_cache + layout.v_tile(page[0], kv_head, 0);
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    if (in_tile / 16 == t) from = v_cache + layout.v_tile(page[t], kv_head, (tile + 16 * t) % page_size / 16);
#pragma unroll
                for (int d = 0; d < HD_TILES; ++d)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float value = from[layout.v_in_tile(key % 16, 16 * d + 4 * quad + i)];
                        if (key <= position) acc[d][i] = __fmaf_rn(weight, value, acc[d][i]);
                    }
            }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) page[t] = next_page[t];
        load_values(next, page, v);

        if (tile % kRowwiseChunk == kRowwiseChunk - kWave || tile + kWave > last_position) {       // the chunk's last tile
            const bool some = tile / kRowwiseChunk * kRowwiseChunk <= position;
            float merged_max, keep, add;
            merge_scales(total_max, chunk_max, merged_max, keep, add);
            total_sum = some ? merged(total_sum, keep, chunk_sum, add) : total_sum;
            total_max = some ? merged_max : total_max;
#pragma unroll
            for (int d = 0; d < HD_TILES; ++d)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    total[d][i] = some ? merged(total[d][i], keep, acc[d][i], add) : total[d][i];
                    acc[d][i] = 0.0f;
                }
            chunk_max = -INFINITY;
            chunk_sum = 0.0f;
        }
    }
    const float inverse = 1.0f / total_sum;
#pragma unroll
    for (int d = 0; d < HD_TILES; ++d) {
        floatx4 result;
#pragma unroll
        for (int i = 0; i < 4; ++i) result[i] = __fmul_rn(total[d][i], inverse);
        if (col < count) *reinterpret_cast<floatx4*>(out + (static_cast<int64_t>(token) * heads + head) * HD + 16 * d + 4 * quad) = result;
    }
    }
}

// MODE 1 for all query heads of a kv head (up to 16 a workgroup) on the matrix units, in float32: a workgroup of four waves takes a chunk of one
// token. S^T = K . Q^T with the heads as columns, 32 keys a wave; the waves' maxima and then the weights meet in LDS; O^T = V^T . P^T with the
// weights from there, every fourth 16 dims a wave. The operations of attend_chunk in their order (the products are ascending chains of fused
// multiply-adds, as in the kernel for runs above; the sums over a tile meet in the order of wave_sum), so the same bits; every key that counts
// counts for all heads, and what others hold is cleared. A wave asks for its keys and its values at once, so that a chunk waits for memory once,
// where a wave a head waits for every eight dims and every eight keys and reads every key again. With the merge, against a wave a head
// or several heads: 28 heads of 128 over 4, 8 requests of 2000 positions 57 -> 23.5 us (the reads alone 10), 64 of 1500 193 -> 92 (61), one of 2000
// 42 -> 13; 14 of 64 over 2, one of 2000 24 -> 10.
template <int HD_TILES>
__global__ __launch_bounds__(256) void paged_attention_rowwise_group_kernel(
    const float* __restrict__ q, const float* __restrict__ k_cache, const float* __restrict__ v_cache,
    const int32_t* __restrict__ block_table, int table_width, const int32_t* __restrict__ seq_of_token, const int32_t* __restrict__ positions,
    float* __restrict__ part_o, float* __restrict__ part_ml, int max_chunks, float scale, int window, int heads, int kv_heads, int page_size) {
#pragma clang fp contract(off)      // a scaled score less the maximum is two roundings, as in the kernels above
    constexpr int HD = HD_TILES * 16;
    constexpr int OWN = (HD_TILES + 3) / 4;         // tiles of 16 dims of a wave, in the second product
    constexpr int SUBTILES = kRowwiseChunk / 16;
    __shared__ float weights[kRowwiseChunk][16];    // [key][head]
    __shared__ float most[4][16];
    const CacheLayout layout(kv_heads, page_size, HD);
    const int token = blockIdx.x;
    const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int col = lane % 16, quad = lane / 16;
    const int seq = seq_of_token[token];
    if (seq < 0) return;
    const int position = positions[token];
    const int low = window > 0 ? max(0, position - window + 1) : 0;
    const int chunk = low / kRowwiseChunk + static_cast<int>(blockIdx.z), base = chunk * kRowwiseChunk;
    if (base > position) return;
    const int first = max(low, base), last = min(position, base + kRowwiseChunk - 1);      // the keys that count
    const int group = heads / kv_heads, parts = (group + 15) / 16;
    const int kv_head = static_cast<int>(blockIdx.y) / parts, in_group = static_cast<int>(blockIdx.y) % parts * 16 + col;
    const int64_t row = static_cast<int64_t>(token) * heads + kv_head * group + min(in_group, group - 1);       // columns past the group repeat its last head
    const int32_t* table = block_table + static_cast<int64_t>(seq) * table_width;
    auto subtile = [&](int s, int64_t& page, int& tile) {       // of 16 keys; those that nobody sees may have no page
        const int key = base + 16 * s;
        page = max(table[min(key / page_size, table_width - 1)], 0);
        tile = key % page_size / 16;
    };

    floatx4 k[2][HD_TILES], v[SUBTILES][OWN], q_piece[HD_TILES];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        int64_t page;
        int tile;
        subtile(2 * wave + u, page, tile);
        const float* from = k_cache + layout.k_tile(page, kv_head, tile) + (quad / 2) * 128 + col * 8 + (quad % 2) * 4;
#pragma unroll
        for (int d = 0; d < HD_TILES; ++d) k[u][d] = *reinterpret_cast<const floatx4*>(from + d * 256);
    }
#pragma unroll
    for (int d = 0; d < HD_TILES; ++d) q_piece[d] = *reinterpret_cast<const floatx4*>(q + row * HD + 16 * d + 4 * quad);
#pragma unroll
    for (int s = 0; s < SUBTILES; ++s) {
        int64_t page;
        int tile;
        subtile(s, page, tile);
        const float* from = v_cache + layout.v_tile(page, kv_head, tile);
#pragma unroll
        for (int n = 0; n < OWN; ++n) {
            const int d = min(wave + 4 * n, HD_TILES - 1);
            const int width = (HD_TILES % 2 == 1 && d == HD_TILES - 1) ? 16 : 32;      // dims of the block of 32 this tile of 16 lies in
            v[s][n] = *reinterpret_cast<const floatx4*>(from + (d / 2) * 512 + ((quad / 2) * width + (d % 2) * 16 + col) * 8 + (quad % 2) * 4);
        }
    }
    __builtin_amdgcn_sched_barrier(0);      // all on their way before the first is waited for

    floatx4 sums[2] = {floatx4{0.0f, 0.0f, 0.0f, 0.0f}, floatx4{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
    for (int d = 0; d < HD_TILES; ++d) {
        const floatx4 query = transpose_quarters(q_piece[d]);
        const floatx4 piece[2] = {transpose_quarters(k[0][d]), transpose_quarters(k[1][d])};
#pragma unroll
        for (int step = 0; step < 4; ++step)
#pragma unroll
            for (int u = 0; u < 2; ++u) sums[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(piece[u][step], query[step], sums[u], 0, 0, 0);
    }
    float score[2][4];      // of keys base + 16 (2 wave + u) + 4 quad + i
    bool counts[2][4];
    float own_most = -INFINITY;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int key = base + 16 * (2 * wave + u) + 4 * quad + i;
            counts[u][i] = key >= first && key <= last;
            score[u][i] = counts[u][i] ? __fmul_rn(sums[u][i], scale) : -INFINITY;
            own_most = fmaxf(own_most, score[u][i]);
        }
    own_most = fmaxf(own_most, from_32_away(own_most));
    own_most = fmaxf(own_most, from_16_away(own_most));
    if (quad == 0) most[wave][col] = own_most;
    __syncthreads();
    // The chunk's two tiles of 64 keys, of which one may have no key that counts and is passed over.
    const bool has[2] = {first < base + kWave, last >= base + kWave};
    float tile_max[2], rescale[2], so_far = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const float new_max = has[t] ? fmaxf(so_far, fmaxf(most[2 * t][col], most[2 * t + 1][col])) : so_far;
        rescale[t] = expf(so_far - new_max);
        so_far = tile_max[t] = new_max;
    }
    const float own_max = wave < 2 ? tile_max[0] : tile_max[1];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) weights[16 * (2 * wave + u) + 4 * quad + i][col] = counts[u][i] ? expf(score[u][i] - own_max) : 0.0f;
    __syncthreads();

    const bool writes = in_group < group;
    const int64_t slot = row * max_chunks + blockIdx.z;
    if (wave == 0) {
        float chunk_sum = 0.0f;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            float part[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float (*p)[16] = weights + 64 * t + 4 * quad + i;
                part[i] = (p[0][col] + p[32][col]) + (p[16][col] + p[48][col]);
                part[i] += from_32_away(part[i]);
                part[i] += from_16_away(part[i]);
            }
            const float sum = (part[0] + part[2]) + (part[1] + part[3]);
            chunk_sum = has[t] ? __fmaf_rn(chunk_sum, rescale[t], sum) : chunk_sum;
        }
        if (writes && quad == 0) {
            part_ml[slot * 2] = so_far;
            part_ml[slot * 2 + 1] = chunk_sum;
        }
    }
    floatx4 acc[OWN];
#pragma unroll
    for (int n = 0; n < OWN; ++n) acc[n] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        if (!has[t]) continue;
#pragma unroll
        for (int n = 0; n < OWN; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[n][i] = __fmul_rn(acc[n][i], rescale[t]);
#pragma unroll
        for (int s = 4 * t; s < 4 * t + 4; ++s) {
            float weight[4];        // of keys 16 s + 4 step + quad
#pragma unroll
            for (int step = 0; step < 4; ++step) weight[step] = weights[16 * s + 4 * step + quad][col];
#pragma unroll
            for (int n = 0; n < OWN; ++n) {
                floatx4 values = v[s][n];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int key = base + 16 * s + 4 * quad + i;
                    values[i] = key >= first && key <= last ? values[i] : 0.0f;        // what lies there may be stale
                }
                const floatx4 piece = transpose_quarters(values);
#pragma unroll
                for (int step = 0; step < 4; ++step) acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(piece[step], weight[step], acc[n], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int n = 0; n < OWN; ++n) {
        const int d = wave + 4 * n;
        if (writes && d < HD_TILES) *reinterpret_cast<floatx4*>(part_o + slot * HD + 16 * d + 4 * quad) = acc[n];
    }
}

// How many query heads of a kv head one wave of the kernel above takes in a step of `rows` (token, kv head, chunk)
// items: as many as leave the GPU its waves, of the counts that fill the group's waves evenly (7 heads: 7, or 4
// and 3, or 2, 2, 2 and 1; not 5 and 2). One: the kernel for one head a wave.
static int rowwise_heads_a_wave(int group, int64_t rows) {
    const int most = group < 8 ? group : 8;
    if (forced_heads_a_wave > 0) return forced_heads_a_wave < most ? forced_heads_a_wave : most;
    for (int count = most; count >= 2; --count) {
        const int waves = (group + count - 1) / count;
        if (waves * count - group > 1) continue;      // the group's last wave would have much less than the others
        if (rows * waves >= kRowwiseWavesWanted) return count;
    }
    return 1;
}

// Whether chunks go to the kernel for all heads of a kv head, by `work`, its workgroups. It takes about as long for a chunk of few keys as for a whole one,
// and 18 to 29 us for 1000 of heads of 128 where the chip is full; a wave a chunk and head takes 6.3 for 1000 of tokens that read the same keys
// (`portions`: more tokens than requests), so that with one or two heads a kv head many tokens of a portion are faster that way, but waits for memory 16
// (64 keys) to 40 us (128 and more) first. us on MI355X, waves and together, workgroups in brackets:
// few keys: 3 tokens 9.4 and 10.7, 160 single ones of 17, 28 heads of 128 over 4 (640), 17.0 and 21.5, 14 of 64 over 2 (320) 8.1 and 11.8, but 100 (200) 10.0 and 9.8;
// a head a kv head, single tokens: 8 heads of 128, 64 and 100 of 40 (512, 800) 20.3 and 16.1, 21.1 and 23.7; 16 of 64, 64 and 100 of 70 (1024, 1600) 23 and 19,
//   22.2 and 25.5; 12 of 48, 64 and 100 of 129 (1536, 2400) 24.2 and 21.9, 25.9 and 30.0; 8 of 128, 64 and 100 of 500 (2048, 3200) 72 and 63, 93 and 100;
// portions: 8 of 128, 60, 100, 128 from 0 (480, 800, 1024) 16.9 and 14.5, 32 and 24, 36 and 26, 100 after 60 and 200 from 0 (1600, 3200) 38 and 29, 39 and 47; 12 of 48, 80
//   from 0 (960) 13.9 and 15.3; 8 of 128, 32, 48 and 60 after 500 (1280, 1920, 2400) 40 and 29, 41 and 42, 41 and 49;
// two, portions: 16 heads of 128 over 8, two of 40 (640) 15.0 and 19.0, 64 after 200 (1536) 41 and 31, 64 after 500 (2560) 46 and 52, 100 after 3000 (20000) 219
//   and 339; single tokens: 64 of 1500 (6144) 166 and 158, one of 2000 beside 63 of 50 (8192, most of them empty) 57 and 84;
// three, 12 of 96 over 4: two of 40 14.5 and 17.0 (640), 64 and 150 after 3000 (6400, 15000) 123 and 100, 192 and 223.
static bool heads_together(int group, bool portions, int keys, int head_dim, int64_t work) {
    if (keys <= 24) return !portions && work < 320;
    if (group >= 4) return true;
    if (portions) {
        if (keys <= 64) return work < 320;
        if (group == 1) return work <= (keys <= 128 ? 8 * head_dim : keys <= 256 ? 16 * head_dim : 1536);
        return group == 3 || work < 2048;
    }
    if (group == 1) return work <= (keys <= 64 ? 640 : keys <= 128 ? 1280 : keys <= 256 ? 2048 : 2816);
    return group == 3 || work < 8192;
}

// Merges what MODE 1 left, in the order and with the arithmetic of MODE 0. One wave per (token, head).
template <typename T, int DIMS>
__global__ __launch_bounds__(kWave) void paged_attention_rowwise_merge_kernel(
    const float* __restrict__ part_o, const float* __restrict__ part_ml, const int32_t* __restrict__ seq_of_token,
    const int32_t* __restrict__ positions, T* __restrict__ out, int max_chunks, int window, int heads, int head_dim) {
    const int token = blockIdx.x;
    const int head = blockIdx.y;
    const int lane = threadIdx.x;
    if (seq_of_token[token] < 0) return;
    const int position = positions[token];
    const int low = window > 0 ? max(0, position - window + 1) : 0;
    const int chunks = position / kRowwiseChunk - low / kRowwiseChunk + 1;
    const int64_t first_slot = (static_cast<int64_t>(token) * heads + head) * max_chunks;
    float total[DIMS];
#pragma unroll
    for (int i = 0; i < DIMS; ++i) total[i] = 0.0f;
    float total_max = -INFINITY, total_sum = 0.0f;
    // Eight chunks' results are asked for at once and then merged one after the other: the loads of a chunk do not
    // wait for the merge of the chunk before.
    constexpr int kAtOnce = 8;
    for (int base = 0; base < chunks; base += kAtOnce) {
        float chunk_max[kAtOnce], chunk_sum[kAtOnce], chunk_o[kAtOnce][DIMS];
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
            const int64_t slot = first_slot + min(base + u, chunks - 1);
            chunk_max[u] = part_ml[slot * 2];
            chunk_sum[u] = part_ml[slot * 2 + 1];
#pragma unroll
            for (int i = 0; i < DIMS; ++i) {
                const int d = lane + i * kWave;
                chunk_o[u][i] = d < head_dim ? part_o[slot * head_dim + d] : 0.0f;
            }
        }
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
            if (base + u >= chunks) break;
            float new_max, keep, add;
            merge_scales(total_max, chunk_max[u], new_max, keep, add);
            total_sum = merged(total_sum, keep, chunk_sum[u], add);
#pragma unroll
            for (int i = 0; i < DIMS; ++i) total[i] = merged(total[i], keep, chunk_o[u][i], add);
            total_max = new_max;
        }
    }
    T* out_row = out + (static_cast<int64_t>(token) * heads + head) * head_dim;
    const float inverse = 1.0f / total_sum;
#pragma unroll
    for (int i = 0; i < DIMS; ++i) {
        const int d = lane + i * kWave;
        if (d < head_dim) out_row[d] = from_float<T>(__fmul_rn(total[i], inverse));
    }
}

template <typename T, int DIMS>
static int launch_rowwise_dims(const void* q, const void* k_cache, const void* v_cache, const int32_t* block_table, int requests,
                          int table_width, const int32_t* seq_of_token, const int32_t* positions, void* out,
                          float* part_o, float* part_ml, int max_chunks, int usual_chunks, float scale, int window, int reach, int n_tokens,
                          int heads, int kv_heads, int head_dim, int page_size, hipStream_t stream) {
    const int group = heads / kv_heads;
    const int64_t rows = static_cast<int64_t>(n_tokens) * kv_heads * (max_chunks > 0 ? (usual_chunks > 0 ? usual_chunks : max_chunks) : 1);
    const int gw = (std::is_same<T, float>::value && DIMS <= 2) ? rowwise_heads_a_wave(group, rows) : 1;
    const bool several_heads = gw >= 2;
    const int group_waves = kv_heads * ((group + gw - 1) / gw);
#define MLL_ROWWISE_HEADS(MODE, GW)                                                                                    \
    case GW:                                                                                                           \
        paged_attention_rowwise_heads_kernel<T, MODE, DIMS, GW><<<heads_grid, kWave, 0, stream>>>(                      \
            static_cast<const T*>(q), static_cast<const T*>(k_cache), static_cast<const T*>(v_cache), block_table,    \
            table_width, seq_of_token, positions, static_cast<T*>(out), part_o, part_ml, max_chunks, scale, window,   \
            heads, kv_heads, head_dim, page_size, runs_apart);                                                         \
        break;
#define MLL_ROWWISE_HEADS_ALL(MODE)                                                                                    \
    switch (gw) {                                                                                                      \
        MLL_ROWWISE_HEADS(MODE, 2) MLL_ROWWISE_HEADS(MODE, 3) MLL_ROWWISE_HEADS(MODE, 4) MLL_ROWWISE_HEADS(MODE, 5)    \
        MLL_ROWWISE_HEADS(MODE, 6) MLL_ROWWISE_HEADS(MODE, 7) MLL_ROWWISE_HEADS(MODE, 8)                               \
        default: break;                                                                                                \
    }
    int runs_apart = 0;
    if (max_chunks == 0) {
        if constexpr (std::is_same<T, float>::value && DIMS <= 2) {
            const int64_t keys = reach > 0 ? min(reach, table_width * page_size) : table_width * page_size;
            const int64_t work = static_cast<int64_t>(n_tokens) * heads * head_dim * keys;
            if (window == 0 && head_dim % 16 == 0 && n_tokens >= runs_from(keys) * requests && work >= kRunsWork) {
                runs_apart = 1;
                const int sides = requests > 1 ? kMostRuns : 1;
                const int64_t units = static_cast<int64_t>((n_tokens + kRunTokens - 1) / kRunTokens) * sides * heads;
                MLL_REQUIRE(units < (static_cast<int64_t>(1) << 31) - 4, "paged_attention: too many rows for one call");
                const dim3 run_grid((units + 3) / 4);
#define MLL_ROWWISE_RUNS(TILES)                                                                                        \
    case TILES:                                                                                                        \
        paged_attention_rowwise_runs_kernel<TILES><<<run_grid, 256, 0, stream>>>(                                      \
            static_cast<const T*>(q), static_cast<const T*>(k_cache), static_cast<const T*>(v_cache), block_table, table_width, seq_of_token, \
            positions, static_cast<T*>(out), scale, n_tokens, heads, kv_heads, page_size, sides);                     \
        break;
                switch (head_dim / 16) {
                    MLL_ROWWISE_RUNS(1) MLL_ROWWISE_RUNS(2) MLL_ROWWISE_RUNS(3) MLL_ROWWISE_RUNS(4)
                    MLL_ROWWISE_RUNS(5) MLL_ROWWISE_RUNS(6) MLL_ROWWISE_RUNS(7) MLL_ROWWISE_RUNS(8)
                    default: break;
                }
#undef MLL_ROWWISE_RUNS
                if (const int status = check_launch("paged_attention_rowwise")) return status;
            }
        }
        if constexpr (std::is_same<T, float>::value && DIMS <= 2) {
            if (several_heads) {
                const dim3 heads_grid(n_tokens, group_waves);
                MLL_ROWWISE_HEADS_ALL(0)
                return check_launch("paged_attention_rowwise");
            }
        }
        paged_attention_rowwise_kernel<T, 0, DIMS><<<dim3(n_tokens, heads), kWave, 0, stream>>>(
            static_cast<const T*>(q), static_cast<const T*>(k_cache), static_cast<const T*>(v_cache), block_table,
            table_width, seq_of_token, positions, static_cast<T*>(out), nullptr, nullptr, 0, scale, window, heads,
            kv_heads, head_dim, page_size, runs_apart);
        return check_launch("paged_attention_rowwise");
    }
    // Several query heads of a kv head in one wave where the step still has rows enough for the GPU that way
    // (float32, head sizes up to 128: the path of the 32-bit engine).
    bool grouped = false;
    if constexpr (std::is_same<T, float>::value && DIMS <= 2) {
        const bool aligned = (reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache) |
                              reinterpret_cast<uintptr_t>(part_o)) % 16 == 0;
        const int keys = reach > 0 ? min(reach, table_width * page_size) : table_width * page_size;
        if (head_dim % 16 == 0 && aligned && forced_heads_a_wave == 0 && heads_together(group, n_tokens > requests, keys, head_dim, rows)) {
            grouped = true;
            const dim3 group_grid(n_tokens, kv_heads * ((group + 15) / 16), max_chunks);
#define MLL_ROWWISE_GROUP(TILES)                                                                                       \
    case TILES:                                                                                                        \
        paged_attention_rowwise_group_kernel<TILES><<<group_grid, 256, 0, stream>>>(                                   \
            static_cast<const T*>(q), static_cast<const T*>(k_cache), static_cast<const T*>(v_cache), block_table, table_width, seq_of_token, \
            positions, part_o, part_ml, max_chunks, scale, window, heads, kv_heads, page_size);                        \
        break;
            switch (head_dim / 16) {
                MLL_ROWWISE_GROUP(1) MLL_ROWWISE_GROUP(2) MLL_ROWWISE_GROUP(3) MLL_ROWWISE_GROUP(4)
                MLL_ROWWISE_GROUP(5) MLL_ROWWISE_GROUP(6) MLL_ROWWISE_GROUP(7) MLL_ROWWISE_GROUP(8)
                default: break;
            }
#undef MLL_ROWWISE_GROUP
        } else if (several_heads) {
            grouped = true;
            const dim3 heads_grid(n_tokens, group_waves, max_chunks);
            MLL_ROWWISE_HEADS_ALL(1)
        }
    }
    if (!grouped)
        paged_attention_rowwise_kernel<T, 1, DIMS><<<dim3(n_tokens, heads, max_chunks), kWave, 0, stream>>>(
            static_cast<const T*>(q), static_cast<const T*>(k_cache), static_cast<const T*>(v_cache), block_table,
            table_width, seq_of_token, positions, static_cast<T*>(out), part_o, part_ml, max_chunks, scale, window, heads,
            kv_heads, head_dim, page_size, 0);
    if (const int status = check_launch("paged_attention_rowwise")) return status;
    paged_attention_rowwise_merge_kernel<T, DIMS><<<dim3(n_tokens, heads), kWave, 0, stream>>>(
        part_o, part_ml, seq_of_token, positions, static_cast<T*>(out), max_chunks, window, heads, head_dim);
    return check_launch("paged_attention_rowwise_merge");
#undef MLL_ROWWISE_HEADS_ALL
#undef MLL_ROWWISE_HEADS
}

template <typename T>
static int launch_rowwise(const void* q, const void* k_cache, const void* v_cache, const int32_t* block_table, int requests,
                          int table_width, const int32_t* seq_of_token, const int32_t* positions, void* out,
                          float* part_o, float* part_ml, int max_chunks, int usual_chunks, float scale, int window, int reach, int n_tokens,
                          int heads, int kv_heads, int head_dim, int page_size, hipStream_t stream) {
#define MLL_ROWWISE_DIMS(D)                                                                                            \
    return launch_rowwise_dims<T, D>(q, k_cache, v_cache, block_table, requests, table_width, seq_of_token, positions, out, part_o, \
                                     part_ml, max_chunks, usual_chunks, scale, window, reach, n_tokens, heads, kv_heads, head_dim, page_size, stream)
    if (head_dim <= kWave) MLL_ROWWISE_DIMS(1);
    if (head_dim <= 2 * kWave) MLL_ROWWISE_DIMS(2);
    if (head_dim <= 4 * kWave) MLL_ROWWISE_DIMS(4);
    MLL_ROWWISE_DIMS(8);
#undef MLL_ROWWISE_DIMS
}

}  // namespace mll

using namespace mll;

extern "C" int mll_paged_attention_rowwise_chunk() { return kRowwiseChunk; }

// Forces how many query heads of a kv head a wave of the float32 kernels takes (1 to 8; more than the group has:
// the group), or with 0 gives the choice back to the launch; returns the value before. Every count gives the same bits.
extern "C" int mll_rowwise_heads_a_wave(int count) {
    const int before = mll::forced_heads_a_wave;
    mll::forced_heads_a_wave = count < 0 ? 0 : count;
    return before;
}

// max_chunks 0: one wave per (token, head). Otherwise one wave per chunk, for rows whose keys span at most
// max_chunks chunks (the caller's promise: a row with more would lose its last ones), with part_o
// [n_tokens * heads * max_chunks * head_dim] and part_ml [n_tokens * heads * max_chunks * 2] floats as workspace.
// requests: rows of block_table, at least as many as the tokens' requests; reach: the step's longest request once it is done (0: what
// the table can hold). Only which kernel takes the tokens follows from them.
// usual_chunks (0: max_chunks): how many chunks the step's rows have now, where max_chunks leaves room for later
// steps of the same shape; only how many heads a wave takes follows from it.
extern "C" int mll_paged_attention_rowwise(const void* q, int dtype, const void* k_cache, const void* v_cache,
                                           const int32_t* block_table, int requests, int table_width,
                                           const int32_t* seq_of_token, const int32_t* positions, void* out,
                                           float* part_o, float* part_ml, int max_chunks, int usual_chunks, float scale,
                                           int window, int reach, int n_tokens, int heads, int kv_heads, int head_dim, int page_size,
                                           hipStream_t stream) {
    MLL_REQUIRE(heads > 0 && kv_heads > 0 && heads % kv_heads == 0, "paged_attention: heads must divide into kv_heads groups");
    MLL_REQUIRE(head_dim > 0 && head_dim <= kRowwiseMaxHeadDim, "paged_attention: head_dim must be in [1, 512]");
    MLL_REQUIRE(page_size > 0 && page_size % 16 == 0 && table_width > 0,
                "paged_attention: page_size must be a multiple of 16 and the table width positive");
    MLL_REQUIRE(heads <= 65535, "paged_attention: more than 65535 heads");
    MLL_REQUIRE(max_chunks >= 0 && max_chunks <= 65535, "paged_attention: bad number of chunks");
    MLL_REQUIRE(max_chunks == 0 || (part_o && part_ml), "paged_attention: chunks need the partial buffers");
    if (n_tokens == 0) return 0;
    if (dtype == kF32)
        return launch_rowwise<float>(q, k_cache, v_cache, block_table, requests, table_width, seq_of_token, positions, out, part_o,
                                     part_ml, max_chunks, usual_chunks, scale, window, reach, n_tokens, heads, kv_heads, head_dim, page_size, stream);
    if (dtype == kBF16)
        return launch_rowwise<bf16>(q, k_cache, v_cache, block_table, requests, table_width, seq_of_token, positions, out, part_o,
                                    part_ml, max_chunks, usual_chunks, scale, window, reach, n_tokens, heads, kv_heads, head_dim, page_size, stream);
    return fail("paged_attention: unknown dtype");
}
