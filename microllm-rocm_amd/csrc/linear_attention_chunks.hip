// Linear attention with one fixed decay a head for long portions, in chunks of 64 tokens:
//
//   S_t = a S_(t-1) + k_t v_t^T,   o_t = S_t^T q_t
//
// Within a chunk that begins with the state S (token t of the chunk, from 0)
//
//   o_t = a^(t+1) S^T q_t + sum_{j <= t} a^(t-j) (q_t . k_j) v_j,
//
// and a chunk of n tokens leaves a^n S + sum_j a^(n-1-j) k_j v_j^T. Three kernels: what every chunk adds to the state
// (all chunks at once), the states at the chunks' starts (a walk over a request's chunks, every element of the state on
// its own), and the results (all chunks at once). All products are float32 on the matrix units
// (v_mfma_f32_16x16x4_f32); state, powers of the decay and sums are float32. A chunk begins at every 64th token of a
// request's portion, so where a portion was cut changes a result by rounding alone.
//
// The kernels gla_channel_* do the same for a decay a key channel and token, a_t[d] = 2^(l_t[d]). With B_t[d] the sum of
// l over the chunk's tokens up to t,
//
//   o_t = (2^B_t q_t)^T S + sum_{j <= t} (sum_d q_t[d] k_j[d] 2^(B_t[d] - B_j[d])) v_j,
//
// and a chunk leaves 2^B_n S + sum_j (2^(B_n - B_j) k_j) v_j^T. No power has a positive exponent, so none overflows whatever
// the decays: 16 tokens among themselves take 2^(B_t - B_j) pair by pair, with those before them the query takes
// 2^(B_t - B_r) and the key 2^(B_r - B_j), r being the last token before the 16. Every exponent is the sum of the logarithms
// between its two tokens, never a difference of two sums: after a token that leaves nothing (-150) a difference would keep
// 1e-5 of the small logarithms that follow it.
#include "common.h"
#include "microllm_hip.h"

namespace mll {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kScanChunk = 64;          // tokens
constexpr int kScanThreads = 256;       // four waves: 16 rows (or 16 value channels) each
constexpr int kScanValues = 64;         // value channels a workgroup holds in LDS at a time

// Chunks are numbered so that every request's are consecutive and none are shared: request i's begin at
// cu[i] / 64 + i. Returns false for a number that no request uses.
__device__ inline bool find_chunk(const int32_t* cu_tokens, int n_seqs, int number, int* seq, int* first, int* count) {
    for (int i = 0; i < n_seqs; ++i) {
        const int begin = cu_tokens[i], end = cu_tokens[i + 1];
        const int base = begin / kScanChunk + i;
        const int chunks = (end - begin + kScanChunk - 1) / kScanChunk;
        if (number >= base && number < base + chunks) {
            *seq = i;
            *first = begin + (number - base) * kScanChunk;
            *count = min(kScanChunk, end - *first);
            return true;
        }
    }
    return false;
}

template <bool SILU>
__device__ inline float scan_input(float value) { return SILU ? activate(value, kActSilu) : value; }

// store(t, c, source[t][c]) for t < ROWS, c < COLUMNS; 0 beyond the first `count` rows and `channels` columns. Eight loads a
// thread are asked for before the first is used.
template <int ROWS, int COLUMNS, typename Store>
__device__ inline void load_tile(const float* source, int64_t row_stride, int count, int channels, Store store) {
    constexpr int kAtATime = 8;
    static_assert(ROWS * COLUMNS % (kScanThreads * kAtATime) == 0, "whole rounds of loads");
    for (int base = threadIdx.x; base < ROWS * COLUMNS; base += kScanThreads * kAtATime) {
        float value[kAtATime];
#pragma unroll
        for (int j = 0; j < kAtATime; ++j) {
            const int t = (base + j * kScanThreads) / COLUMNS, c = (base + j * kScanThreads) % COLUMNS;
            value[j] = t < count && c < channels ? source[t * row_stride + c] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < kAtATime; ++j) store((base + j * kScanThreads) / COLUMNS, (base + j * kScanThreads) % COLUMNS, value[j]);
    }
}

// powers[n] = decay^n for n <= 64.
__device__ inline void load_powers(float* powers, float decay) {
    if (threadIdx.x <= kScanChunk) powers[threadIdx.x] = threadIdx.x == 0 ? 1.0f : powf(decay, static_cast<float>(threadIdx.x));
}

// added[number][head][d][c] = sum_t decay^(n - 1 - t) k_t[d] v_t[c].
template <int KEYS, bool SILU>
__global__ void __launch_bounds__(kScanThreads)
gla_chunk_state_kernel(const float* __restrict__ proj, int64_t proj_stride, int k_offset, int v_offset, const float* __restrict__ decay,
                       const int32_t* __restrict__ cu_tokens, float* __restrict__ added, int n_seqs, int heads, int key_dim, int value_dim) {
    __shared__ float keys[kScanChunk][KEYS + 1];
    __shared__ float values[kScanChunk][kScanValues + 1];
    __shared__ float powers[kScanChunk + 1];
    const int number = blockIdx.x, head = blockIdx.y;
    int seq, first, count;
    if (!find_chunk(cu_tokens, n_seqs, number, &seq, &first, &count)) return;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int col = lane % 16, quad = lane / 16;
    const int key_tiles = (key_dim + 15) / 16;
    load_powers(powers, decay[head]);
    const float* row = proj + first * proj_stride;
    load_tile<kScanChunk, KEYS>(row + k_offset + head * key_dim, proj_stride, count, key_dim,
                                [&](int t, int c, float value) { keys[t][c] = scan_input<SILU>(value); });
    float* to = added + (static_cast<int64_t>(number) * heads + head) * key_dim * value_dim;
    for (int v0 = 0; v0 < value_dim; v0 += kScanValues) {
        __syncthreads();      // the tile before has been read (the first time: the powers are there)
        load_tile<kScanChunk, kScanValues>(row + v_offset + head * value_dim + v0, proj_stride, count, value_dim - v0, [&](int t, int c, float value) {
            values[t][c] = t < count ? powers[count - 1 - t] * scan_input<SILU>(value) : 0.0f;
        });
        __syncthreads();
        const int column = v0 + 16 * wave + col;
        for (int tile = 0; tile < key_tiles; ++tile) {
            floatx4 acc = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int t = 0; t < kScanChunk; t += 4)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(keys[t + quad][16 * tile + col], values[t + quad][16 * wave + col], acc, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int d = 16 * tile + 4 * quad + i;
                if (d < key_dim && column < value_dim) to[static_cast<int64_t>(d) * value_dim + column] = acc[i];
            }
        }
    }
}

// A request's chunks in order: what a chunk adds is replaced by the state it begins with; the state after the last one
// goes back to the request's slot.
__global__ void __launch_bounds__(256)
gla_chunk_carry_kernel(float* __restrict__ added, const float* __restrict__ decay, float* __restrict__ state,
                       const int32_t* __restrict__ cu_tokens, const int32_t* __restrict__ slots, int heads, int elements) {
    const int seq = blockIdx.x, head = blockIdx.y;
    const int element = blockIdx.z * blockDim.x + threadIdx.x;
    const int begin = cu_tokens[seq], tokens = cu_tokens[seq + 1] - begin;
    if (tokens <= 0 || element >= elements) return;
    const int chunks = (tokens + kScanChunk - 1) / kScanChunk;
    const int64_t step = static_cast<int64_t>(heads) * elements;
    float* place = added + (static_cast<int64_t>(begin / kScanChunk + seq) * heads + head) * elements + element;
    float* kept = state + (static_cast<int64_t>(slots[seq]) * heads + head) * elements + element;
    const float whole = powf(decay[head], static_cast<float>(kScanChunk));
    const int last = tokens - (chunks - 1) * kScanChunk;
    const float partly = powf(decay[head], static_cast<float>(last));
    float s = *kept;
    constexpr int kAtATime = 8;      // chunks asked for at a time, then walked in order
    for (int base = 0; base < chunks; base += kAtATime) {
        float more[kAtATime];
#pragma unroll
        for (int j = 0; j < kAtATime; ++j) more[j] = base + j < chunks ? place[(base + j) * step] : 0.0f;
#pragma unroll
        for (int j = 0; j < kAtATime; ++j)
            if (base + j < chunks) {
                place[(base + j) * step] = s;
                s = fmaf(base + j + 1 < chunks ? whole : partly, s, more[j]);
            }
    }
    *kept = s;
}

// The results of a chunk's tokens; wave w takes tokens 16 w .. 16 w + 15 of it.
template <int KEYS, bool SILU>
__global__ void __launch_bounds__(kScanThreads)
gla_chunk_out_kernel(const float* __restrict__ proj, int64_t proj_stride, int q_offset, int k_offset, int v_offset,
                     const float* __restrict__ decay, const int32_t* __restrict__ cu_tokens, const float* __restrict__ starts,
                     float* __restrict__ out, int n_seqs, int heads, int key_dim, int value_dim, float q_scale) {
    __shared__ float queries[kScanChunk][KEYS + 1];
    __shared__ float keys[kScanChunk][KEYS + 1];
    __shared__ float start[KEYS][kScanValues + 1];
    __shared__ float values[kScanChunk][kScanValues + 1];
    __shared__ float weights[kScanChunk][kScanChunk + 1];
    __shared__ float powers[kScanChunk + 1];
    const int number = blockIdx.x, head = blockIdx.y;
    int seq, first, count;
    if (!find_chunk(cu_tokens, n_seqs, number, &seq, &first, &count)) return;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int col = lane % 16, quad = lane / 16;
    const int padded = (key_dim + 15) / 16 * 16;
    load_powers(powers, decay[head]);
    const float* row = proj + first * proj_stride;
    load_tile<kScanChunk, KEYS>(row + q_offset + head * key_dim, proj_stride, count, key_dim,
                                [&](int t, int c, float value) { queries[t][c] = scan_input<SILU>(value); });
    load_tile<kScanChunk, KEYS>(row + k_offset + head * key_dim, proj_stride, count, key_dim,
                                [&](int t, int c, float value) { keys[t][c] = scan_input<SILU>(value); });
    __syncthreads();
    // weights[t][j] = decay^(t - j) q_t . k_j for j <= t
    for (int tile = 0; tile <= wave; ++tile) {
        floatx4 acc = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int d = 0; d < padded; d += 4)
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(queries[16 * wave + col][d + quad], keys[16 * tile + col][d + quad], acc, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = 16 * wave + 4 * quad + i, j = 16 * tile + col;
            weights[t][j] = j <= t ? acc[i] * powers[t - j] : 0.0f;
        }
    }
    const float* from = starts + (static_cast<int64_t>(number) * heads + head) * key_dim * value_dim;
    for (int v0 = 0; v0 < value_dim; v0 += kScanValues) {
        __syncthreads();      // the tile before has been read (the first time: the weights are there)
        load_tile<kScanChunk, kScanValues>(row + v_offset + head * value_dim + v0, proj_stride, count, value_dim - v0,
                                           [&](int t, int c, float value) { values[t][c] = scan_input<SILU>(value); });
        load_tile<KEYS, kScanValues>(from + v0, value_dim, key_dim, value_dim - v0, [&](int d, int c, float value) { start[d][c] = value; });
        __syncthreads();
        for (int tile = 0; tile < kScanValues / 16; ++tile) {
            const int column = v0 + 16 * tile + col;
            if (v0 + 16 * tile >= value_dim) break;
            floatx4 acc = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
            for (int d = 0; d < padded; d += 4)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(queries[16 * wave + col][d + quad], start[d + quad][16 * tile + col], acc, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] *= powers[16 * wave + 4 * quad + i + 1];
            for (int j = 0; j < 16 * (wave + 1); j += 4)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(weights[16 * wave + col][j + quad], values[j + quad][16 * tile + col], acc, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = 16 * wave + 4 * quad + i;
                if (t < count && column < value_dim)
                    out[(static_cast<int64_t>(first + t) * heads + head) * value_dim + column] = acc[i] * q_scale;
            }
        }
    }
}

// ---- a decay a key channel and token -------------------------------------------------------------------------------
// Two requests of 2000 and 1117 tokens, 8 heads of 64 x 128: 285 us by the walk, 78 here, bound by one workgroup's chain of LDS
// reads and products. Sums run in four chains, which both shortens the waits and keeps the error against float64 below the walk's
// for ordinary decays: 1.2e-7 (root mean square, of the results') against 1.65e-7 at 512 tokens; where strong and slow decays
// meet both err by 1e-7 (with exponents as differences of sums, 5 us faster, it was 1e-5 of the largest result).
constexpr int kChannelKeys = 64;        // the widest key heads here: queries, keys and decays of a chunk lie in LDS together

constexpr int kPart = 16;
constexpr int kParts = kScanChunk / kPart;

// A chunk's logarithms. Below 2^-149 a factor is zero in float32, and a sum of larger numbers would lose the others' digits.
__device__ inline float usable_log(float value) { return value < -150.0f ? -150.0f : value; }

// whole[part][c]: the sum of a part's logarithms `logs[t][c]`; with AFTER, logs[t][c] becomes the sum of those after it in its
// part. Called by every thread; the first and last things it does are barriers.
template <bool AFTER>
__device__ inline void sum_parts(float (*logs)[kChannelKeys + 1], float (*whole)[kChannelKeys]) {
    const int c = threadIdx.x % kChannelKeys, part = threadIdx.x / kChannelKeys;
    static_assert(kScanThreads == kParts * kChannelKeys, "a thread a channel and part");
    __syncthreads();
    float total = 0.0f;
#pragma unroll
    for (int t = kPart - 1; t >= 0; --t) {
        const float own = logs[kPart * part + t][c];
        if (AFTER) logs[kPart * part + t][c] = total;
        total += own;
    }
    whole[part][c] = total;
    __syncthreads();
}

// The value of the lane STEPS before, or after, within every 16 lanes; 0 where there is none.
template <int STEPS>
__device__ inline float lane_before(float value) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, value), 0x110 + STEPS, 0xf, 0xf, false));
}
template <int STEPS>
__device__ inline float lane_after(float value) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, value), 0x100 + STEPS, 0xf, 0xf, false));
}
// The sum of the lanes up to this one, or of those after it, within every 16 lanes (all lanes of the wave come here).
__device__ inline float sum_up_to(float value) {
    value += lane_before<1>(value);
    value += lane_before<2>(value);
    value += lane_before<4>(value);
    return value + lane_before<8>(value);
}
__device__ inline float sum_after(float value) {
    value = lane_after<1>(value);
    value += lane_after<1>(value);
    value += lane_after<2>(value);
    value += lane_after<4>(value);
    return value + lane_after<8>(value);
}

// whole[first] + .. + whole[last - 1] of channel c.
__device__ inline float sum_between(float (*whole)[kChannelKeys], int first, int last, int c) {
    float total = 0.0f;
    for (int part = first; part < last; ++part) total += whole[part][c];
    return total;
}

__device__ inline float power_of_two(float exponent) { return __builtin_amdgcn_exp2f(exponent); }

// added[number][head][d][c] = sum_t 2^(B_n - B_t)[d] k_t[d] v_t[c]; whole[number][head][d] = 2^B_n[d].
__global__ void __launch_bounds__(kScanThreads)
gla_channel_state_kernel(const float* __restrict__ proj, int64_t proj_stride, int k_offset, int v_offset, const float* __restrict__ log_decay,
                         const int32_t* __restrict__ cu_tokens, float* __restrict__ added, float* __restrict__ whole, int n_seqs, int heads,
                         int key_dim, int value_dim) {
    __shared__ float keys[kScanChunk][kChannelKeys + 1];
    __shared__ float sums[kScanChunk][kChannelKeys + 1];
    __shared__ float values[kScanChunk][kScanValues + 1];
    __shared__ float parts[kParts][kChannelKeys];
    const int number = blockIdx.x, head = blockIdx.y;
    int seq, first, count;
    if (!find_chunk(cu_tokens, n_seqs, number, &seq, &first, &count)) return;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int col = lane % 16, quad = lane / 16;
    const float* row = proj + first * proj_stride;
    load_tile<kScanChunk, kChannelKeys>(log_decay + (static_cast<int64_t>(first) * heads + head) * key_dim, static_cast<int64_t>(heads) * key_dim, count,
                                        key_dim, [&](int t, int c, float value) { sums[t][c] = usable_log(value); });
    load_tile<kScanChunk, kChannelKeys>(row + k_offset + head * key_dim, proj_stride, count, key_dim,
                                        [&](int t, int c, float value) { keys[t][c] = value; });
    sum_parts<true>(sums, parts);
    for (int index = threadIdx.x; index < kScanChunk * kChannelKeys; index += kScanThreads) {
        const int t = index / kChannelKeys, c = index % kChannelKeys, part = t / kPart;
        keys[t][c] *= power_of_two(sums[t][c] + sum_between(parts, part + 1, kParts, c));
    }
    if (threadIdx.x < key_dim)
        whole[(static_cast<int64_t>(number) * heads + head) * key_dim + threadIdx.x] = power_of_two(sum_between(parts, 0, kParts, threadIdx.x));
    float* to = added + (static_cast<int64_t>(number) * heads + head) * key_dim * value_dim;
    for (int v0 = 0; v0 < value_dim; v0 += kScanValues) {
        __syncthreads();      // the tile before has been read (the first time: the keys are there)
        load_tile<kScanChunk, kScanValues>(row + v_offset + head * value_dim + v0, proj_stride, count, value_dim - v0,
                                           [&](int t, int c, float value) { values[t][c] = value; });
        __syncthreads();
        const int column = v0 + 16 * wave + col;
        for (int tile = 0; tile < (key_dim + 15) / 16; ++tile) {
            floatx4 sum[kParts] = {};
#pragma unroll
            for (int t = 0; t < kPart; t += 4)
#pragma unroll
                for (int part = 0; part < kParts; ++part)
                    sum[part] = __builtin_amdgcn_mfma_f32_16x16x4f32(keys[kPart * part + t + quad][16 * tile + col],
                                                                     values[kPart * part + t + quad][16 * wave + col], sum[part], 0, 0, 0);
            const floatx4 acc = (sum[0] + sum[1]) + (sum[2] + sum[3]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int d = 16 * tile + 4 * quad + i;
                if (d < key_dim && column < value_dim) to[static_cast<int64_t>(d) * value_dim + column] = acc[i];
            }
        }
    }
}

// gla_chunk_carry_kernel with a factor a chunk and key channel.
__global__ void __launch_bounds__(256)
gla_channel_carry_kernel(float* __restrict__ added, const float* __restrict__ whole, float* __restrict__ state,
                         const int32_t* __restrict__ cu_tokens, const int32_t* __restrict__ slots, int heads, int key_dim, int value_dim) {
    const int seq = blockIdx.x, head = blockIdx.y;
    const int elements = key_dim * value_dim;
    const int element = blockIdx.z * blockDim.x + threadIdx.x;
    const int begin = cu_tokens[seq], tokens = cu_tokens[seq + 1] - begin;
    if (tokens <= 0 || element >= elements) return;
    const int chunks = (tokens + kScanChunk - 1) / kScanChunk;
    const int64_t step = static_cast<int64_t>(heads) * elements, factor_step = static_cast<int64_t>(heads) * key_dim;
    const int64_t base_number = begin / kScanChunk + seq;
    float* place = added + (base_number * heads + head) * elements + element;
    const float* factors = whole + (base_number * heads + head) * key_dim + element / value_dim;
    float* kept = state + (static_cast<int64_t>(slots[seq]) * heads + head) * elements + element;
    float s = *kept;
    constexpr int kAtATime = 8;      // chunks asked for at a time, then walked in order
    for (int base = 0; base < chunks; base += kAtATime) {
        float more[kAtATime], factor[kAtATime];
#pragma unroll
        for (int j = 0; j < kAtATime; ++j) {
            more[j] = base + j < chunks ? place[(base + j) * step] : 0.0f;
            factor[j] = base + j < chunks ? factors[(base + j) * factor_step] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < kAtATime; ++j)
            if (base + j < chunks) {
                place[(base + j) * step] = s;
                s = fmaf(factor[j], s, more[j]);
            }
    }
    *kept = s;
}

// The results of a chunk's tokens; wave w takes tokens 16 w .. 16 w + 15 of it.
__global__ void __launch_bounds__(kScanThreads)
gla_channel_out_kernel(const float* __restrict__ proj, int64_t proj_stride, int q_offset, int k_offset, int v_offset,
                       const float* __restrict__ log_decay, const int32_t* __restrict__ cu_tokens, const float* __restrict__ starts,
                       float* __restrict__ out, int n_seqs, int heads, int key_dim, int value_dim, float q_scale) {
    __shared__ float queries[kScanChunk][kChannelKeys + 1];
    __shared__ float keys[kScanChunk][kChannelKeys + 1];
    __shared__ float logs[kScanChunk][kChannelKeys + 1];
    __shared__ float weights[kScanChunk][kScanChunk + 1];
    __shared__ float parts[kParts][kChannelKeys];
    const int number = blockIdx.x, head = blockIdx.y;
    int seq, first, count;
    if (!find_chunk(cu_tokens, n_seqs, number, &seq, &first, &count)) return;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int col = lane % 16, quad = lane / 16;
    const float* row = proj + first * proj_stride;
    load_tile<kScanChunk, kChannelKeys>(log_decay + (static_cast<int64_t>(first) * heads + head) * key_dim, static_cast<int64_t>(heads) * key_dim, count,
                                        key_dim, [&](int t, int c, float value) { logs[t][c] = usable_log(value); });
    load_tile<kScanChunk, kChannelKeys>(row + q_offset + head * key_dim, proj_stride, count, key_dim,
                                        [&](int t, int c, float value) { queries[t][c] = value; });
    load_tile<kScanChunk, kChannelKeys>(row + k_offset + head * key_dim, proj_stride, count, key_dim,
                                        [&](int t, int c, float value) { keys[t][c] = value; });
    sum_parts<false>(logs, parts);
    const int own = kPart * wave + col;     // the token whose query this lane holds as a row of the first operand
    // weights[t][j] = sum_d q_t[d] k_j[d] 2^(B_t[d] - B_j[d]) for j <= t: the wave's tokens among themselves, four pairs a lane ...
    {
        float pair[4][4] = {};      // the sums over the channels, in four parts
        for (int d0 = 0; d0 < key_dim; d0 += 4)
#pragma unroll
            for (int d = 0; d < 4; ++d) {       // channels past the head are zero
                const float q = queries[own][d0 + d], log = logs[own][d0 + d];
                // the logarithms after the lane's four keys up to its token, then with those between the keys as well
                float exponent = sum_up_to(col > 4 * quad + 3 ? log : 0.0f);
#pragma unroll
                for (int i = 3; i >= 0; --i) {
                    const int j = kPart * wave + 4 * quad + i;
                    pair[d][i] = fmaf(q * keys[j][d0 + d], power_of_two(exponent), pair[d][i]);
                    exponent += 4 * quad + i <= col ? logs[j][d0 + d] : 0.0f;
                }
            }
#pragma unroll
        for (int i = 0; i < 4; ++i) weights[own][kPart * wave + 4 * quad + i] = 4 * quad + i <= col ? (pair[0][i] + pair[1][i]) + (pair[2][i] + pair[3][i]) : 0.0f;
    }
    // ... and with the parts before them
    float up_to[kChannelKeys / 4];          // B_t - B_r
    float reaching[kChannelKeys / 4];       // 2^(B_t - B_r) q_t
#pragma unroll
    for (int d = 0; d < kChannelKeys; d += 4) {
        up_to[d / 4] = sum_up_to(logs[own][d + quad]);
        reaching[d / 4] = queries[own][d + quad] * power_of_two(up_to[d / 4]);
    }
    for (int part = 0; part < wave; ++part) {
        floatx4 sum[4] = {};
#pragma unroll
        for (int d = 0; d < kChannelKeys; d += 4) {
            const int c = d + quad, j = kPart * part + col;
            const float k = keys[j][c] * power_of_two(sum_after(logs[j][c]) + sum_between(parts, part + 1, wave, c));
            sum[d / 4 % 4] = __builtin_amdgcn_mfma_f32_16x16x4f32(reaching[d / 4], k, sum[d / 4 % 4], 0, 0, 0);
        }
        const floatx4 acc = (sum[0] + sum[1]) + (sum[2] + sum[3]);
#pragma unroll
        for (int i = 0; i < 4; ++i) weights[kPart * wave + 4 * quad + i][kPart * part + col] = acc[i];
    }
    // What other lanes of the wave wrote to `weights` is read below: LDS takes a wave's accesses in order, the fence keeps the
    // compiler to it (it could tell a thread's own stores from the loads and move these up).
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const float* from = starts + (static_cast<int64_t>(number) * heads + head) * key_dim * value_dim;
    float decayed[kChannelKeys / 4];        // 2^B_t q_t: the operand that meets the state
#pragma unroll
    for (int d = 0; d < kChannelKeys; d += 4) decayed[d / 4] = queries[own][d + quad] * power_of_two(up_to[d / 4] + sum_between(parts, 0, wave, d + quad));
    float own_weight[kPart / 4];            // the weights of the wave's tokens among themselves
#pragma unroll
    for (int j = 0; j < kPart / 4; ++j) own_weight[j] = weights[own][kPart * wave + 4 * j + quad];
    float weight[kScanChunk / 4 - kPart / 4];       // and with those of the parts before them: rows that the wave wrote itself
#pragma unroll
    for (int j = 0; j < kScanChunk - kPart; j += 4) weight[j / 4] = j < kPart * wave ? weights[own][j + quad] : 0.0f;
    // Queries and keys are done with: the state and the values take their place.
    float (*start)[kScanValues + 1] = queries;
    float (*values)[kScanValues + 1] = keys;
    static_assert(kScanValues == kChannelKeys, "one shape");
    for (int v0 = 0; v0 < value_dim; v0 += kScanValues) {
        __syncthreads();      // the tile before has been read (the first time: queries and keys have, and the weights are there)
        load_tile<kScanChunk, kScanValues>(row + v_offset + head * value_dim + v0, proj_stride, count, value_dim - v0,
                                           [&](int t, int c, float value) { values[t][c] = value; });
        load_tile<kChannelKeys, kScanValues>(from + v0, value_dim, key_dim, value_dim - v0, [&](int d, int c, float value) { start[d][c] = value; });
        __syncthreads();
        for (int tile = 0; tile < kScanValues / 16; ++tile) {
            const int column = v0 + 16 * tile + col;
            if (v0 + 16 * tile >= value_dim) break;
            floatx4 sum[4] = {};
#pragma unroll
            for (int d = 0; d < kChannelKeys; d += 4)
                sum[d / 4 % 4] = __builtin_amdgcn_mfma_f32_16x16x4f32(decayed[d / 4], start[d + quad][16 * tile + col], sum[d / 4 % 4], 0, 0, 0);
            floatx4 acc = (sum[0] + sum[1]) + (sum[2] + sum[3]);
#pragma unroll
            for (int part = 0; part < kParts - 1; ++part) {
                if (part >= wave) break;
                floatx4 more = {};
#pragma unroll
                for (int j = kPart * part; j < kPart * (part + 1); j += 4)
                    more = __builtin_amdgcn_mfma_f32_16x16x4f32(weight[j / 4], values[j + quad][16 * tile + col], more, 0, 0, 0);
                acc += more;
            }
            // A value that is not finite must not reach the tokens before its own, as zero times it would.
            float own_values[kPart / 4];
            bool finite = true;
#pragma unroll
            for (int j = 0; j < kPart / 4; ++j) {
                own_values[j] = values[kPart * wave + 4 * j + quad][16 * tile + col];
                finite = finite && isfinite(own_values[j]);
            }
            if (__all(finite)) {
                floatx4 more = {};
#pragma unroll
                for (int j = 0; j < kPart / 4; ++j) more = __builtin_amdgcn_mfma_f32_16x16x4f32(own_weight[j], own_values[j], more, 0, 0, 0);
                acc += more;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    for (int j = kPart * wave; j <= kPart * wave + 4 * quad + i; ++j)
                        acc[i] = fmaf(weights[kPart * wave + 4 * quad + i][j], values[j][16 * tile + col], acc[i]);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = kPart * wave + 4 * quad + i;
                if (t < count && column < value_dim)
                    out[(static_cast<int64_t>(first + t) * heads + head) * value_dim + column] = acc[i] * q_scale;
            }
        }
    }
}

}  // namespace mll

using namespace mll;

extern "C" {

int64_t mll_gla_chunks_scratch(int n_tokens, int n_seqs, int heads, int key_dim, int value_dim) {
    return (static_cast<int64_t>(n_tokens) / kScanChunk + n_seqs) * heads * key_dim * value_dim;
}

int mll_gla_chunks(const float* proj, int64_t proj_stride, int q_offset, int k_offset, int v_offset, const float* decay, float* state,
                   const int32_t* cu_tokens, const int32_t* slots, float* out, float* scratch, int n_tokens, int n_seqs, int heads,
                   int key_dim, int value_dim, float q_scale, int silu_inputs, hipStream_t stream) {
    MLL_REQUIRE(n_tokens >= 0 && n_seqs >= 0 && heads > 0 && key_dim > 0 && value_dim > 0, "gla_chunks: sizes must be positive");
    MLL_REQUIRE(key_dim <= 128, "gla_chunks: key heads wider than 128 are not supported");
    MLL_REQUIRE(q_offset >= 0 && k_offset >= 0 && v_offset >= 0 && q_offset + heads * key_dim <= proj_stride &&
                    k_offset + heads * key_dim <= proj_stride && v_offset + heads * value_dim <= proj_stride,
                "gla_chunks: a projection lies outside its row");
    if (n_tokens == 0 || n_seqs == 0) return 0;
    const int64_t elements = static_cast<int64_t>(key_dim) * value_dim;
    MLL_REQUIRE(heads <= 65535 && elements <= 65535ll * 256, "gla_chunks: too many heads or a state too large for one launch");
    const dim3 chunks(n_tokens / kScanChunk + n_seqs, heads);
#define MLL_CHUNKS(KEYS, SILU)                                                                                                   \
    do {                                                                                                                         \
        gla_chunk_state_kernel<KEYS, SILU><<<chunks, kScanThreads, 0, stream>>>(proj, proj_stride, k_offset, v_offset, decay, cu_tokens, \
                                                                                scratch, n_seqs, heads, key_dim, value_dim);    \
        gla_chunk_carry_kernel<<<dim3(n_seqs, heads, static_cast<unsigned>((elements + 255) / 256)), 256, 0, stream>>>(         \
            scratch, decay, state, cu_tokens, slots, heads, static_cast<int>(elements));                                        \
        gla_chunk_out_kernel<KEYS, SILU><<<chunks, kScanThreads, 0, stream>>>(proj, proj_stride, q_offset, k_offset, v_offset, decay, \
                                                                              cu_tokens, scratch, out, n_seqs, heads, key_dim, value_dim, q_scale); \
    } while (0)
    if (key_dim <= 64 && silu_inputs) MLL_CHUNKS(64, true);
    else if (key_dim <= 64) MLL_CHUNKS(64, false);
    else if (silu_inputs) MLL_CHUNKS(128, true);
    else MLL_CHUNKS(128, false);
#undef MLL_CHUNKS
    return check_launch("gla_chunks");
}

int64_t mll_gla_channel_chunks_scratch(int n_tokens, int n_seqs, int heads, int key_dim, int value_dim) {
    return (static_cast<int64_t>(n_tokens) / kScanChunk + n_seqs) * heads * key_dim * (static_cast<int64_t>(value_dim) + 1);
}

int mll_gla_channel_chunks(const float* proj, int64_t proj_stride, int q_offset, int k_offset, int v_offset, const float* log_decay, float* state,
                           const int32_t* cu_tokens, const int32_t* slots, float* out, float* scratch, int n_tokens, int n_seqs, int heads,
                           int key_dim, int value_dim, float q_scale, hipStream_t stream) {
    MLL_REQUIRE(n_tokens >= 0 && n_seqs >= 0 && heads > 0 && key_dim > 0 && value_dim > 0, "gla_channel_chunks: sizes must be positive");
    MLL_REQUIRE(key_dim <= kChannelKeys, "gla_channel_chunks: key heads wider than 64 are not supported");
    MLL_REQUIRE(q_offset >= 0 && k_offset >= 0 && v_offset >= 0 && q_offset + heads * key_dim <= proj_stride &&
                    k_offset + heads * key_dim <= proj_stride && v_offset + heads * value_dim <= proj_stride,
                "gla_channel_chunks: a projection lies outside its row");
    if (n_tokens == 0 || n_seqs == 0) return 0;
    const int64_t elements = static_cast<int64_t>(key_dim) * value_dim;
    MLL_REQUIRE(heads <= 65535 && elements <= 65535ll * 256, "gla_channel_chunks: too many heads or a state too large for one launch");
    const dim3 chunks(n_tokens / kScanChunk + n_seqs, heads);
    float* whole = scratch + static_cast<int64_t>(chunks.x) * heads * elements;
    gla_channel_state_kernel<<<chunks, kScanThreads, 0, stream>>>(proj, proj_stride, k_offset, v_offset, log_decay, cu_tokens, scratch, whole, n_seqs,
                                                                  heads, key_dim, value_dim);
    gla_channel_carry_kernel<<<dim3(n_seqs, heads, static_cast<unsigned>((elements + 255) / 256)), 256, 0, stream>>>(
        scratch, whole, state, cu_tokens, slots, heads, key_dim, value_dim);
    gla_channel_out_kernel<<<chunks, kScanThreads, 0, stream>>>(proj, proj_stride, q_offset, k_offset, v_offset, log_decay, cu_tokens, scratch, out,
                                                                n_seqs, heads, key_dim, value_dim, q_scale);
    return check_launch("gla_channel_chunks");
}

}  // extern "C"
