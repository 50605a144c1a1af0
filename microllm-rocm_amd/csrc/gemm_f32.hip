// The float32 matrix product of the true 32-bit path: C = A * W^T (+ bias).
// Every output element is one chain of fused multiply-adds in ascending k, so a row's result is the same whatever
// other rows the call holds and whichever of the kernels here computes it. The chains run on the matrix units: the
// float32 MFMAs of gfx950 give, element by element, the bits of fmaf(a[k], b[k], c) applied in ascending k (checked on
// MI355X over normal, large, cancelling and denormal values), so they and the vector kernels may stand in for each other.
#include "common.h"
#include "microllm_hip.h"

namespace mll {

// The reduction may be cut into parts of k_split terms, one a blockIdx.z: part z sums k in [z * k_split, (z + 1) *
// k_split) in ascending order into C[z] (its own [m, n] array), the bias goes to part 0, and whoever reads the result
// adds the parts in order. The cut depends on the weight's shape alone (mll_gemm_f32_splits), never on the rows of the
// call, so a row's bits stay what they are under every batch. Inside a kernel `k` then is the part's end, and sums
// start at k_lo.
#define MLL_F32_SPLIT_RANGE                                                          \
    const int ld = k; /* elements from one row of A or W to the next */              \
    const int k_lo = blockIdx.z * k_split;                                           \
    k = min(k, k_lo + k_split);                                                      \
    c += static_cast<int64_t>(blockIdx.z) * m * n;                                   \
    if (blockIdx.z != 0) bias = nullptr;

typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

// Tiles for more than 16 rows: four waves of (32 TM) x (32 TN) elements on v_mfma_f32_32x32x2_f32, WAVES_M of them along
// the rows. Both operands come in chunks of kTileDepth of k with 16-byte loads (the next chunk is on its way while this
// one is multiplied) into one of two stages of LDS. An MFMA takes k from its lower 32 lanes and k + 1 from its upper 32, so a row
// of a chunk lies as [k % 2][k / 2]: a lane's 16-byte read holds its operands of four products in a row. Rows lie four
// banks apart, so that the eight rows of a 128-byte read fall on different banks. Bound by the matrix units (155 TFLOP/s of
// nothing but these products; the vector units' single multiply-adds, which the tiles ran on before, give half of that) and
// by filling the compute units: 2048 x 37888 x 3584 7190 -> 4500 us (124 TFLOP/s), 2048 x 3584 x 18944 3370 -> 2120, 1003 x 9728 x 896 257 ->
// 165, 64 x 37888 x 3584 323 -> 202.
constexpr int kTileDepth = 32;
constexpr int kNonTemporal = 2;
constexpr int kPast = 0x40000000;           // past the end of every descriptor here, and with any row's offset added to it
constexpr int kWidestVector = 1 << 20;      // k up to which the byte offsets of 128 rows stay below kPast

// The byte offset of element `at` of a row, past the end from element `end` on. Opaque to the compiler, which would
// otherwise branch around the loads that take it, and then wait for each of them.
__device__ inline int offset_below(int at, int end) {
    int offset = at < end ? at * 4 : kPast;
    asm("" : "+v"(offset));
    return offset;
}

template <int WAVES_M, int TM, int TN, bool VECTOR>
__global__ __launch_bounds__(256) void gemm_f32_tile_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                            const float* __restrict__ bias, float* __restrict__ c,
                                                            int m, int n, int k, int k_split) {
    MLL_F32_SPLIT_RANGE
    constexpr int WAVES_N = 4 / WAVES_M;
    constexpr int ROWS = WAVES_M * TM * 32, COLUMNS = WAVES_N * TN * 32;
    constexpr int QUADS = kTileDepth / 4;                  // float4 in a row of a chunk
    constexpr int LOADS_A = ROWS * QUADS / 256, LOADS_W = COLUMNS * QUADS / 256;
    constexpr int STRIDE = kTileDepth + 4;
    __shared__ __align__(16) float a_tile[2][ROWS][STRIDE];
    __shared__ __align__(16) float w_tile[2][COLUMNS][STRIDE];
    const int row0 = blockIdx.y * ROWS;
    const int col0 = blockIdx.x * COLUMNS;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int half = lane / 32;
    const int wave_row = wave / WAVES_N * TM * 32, wave_col = wave % WAVES_N * TN * 32;
    // VECTOR (k a multiple of 4, 16-byte aligned rows): through buffer descriptors of the tile's rows, whose loads give
    // zeros past the end, so that no branch (and with it a wait for every load before) stands between the loads.
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(a) + static_cast<int64_t>(row0) * ld, 0, VECTOR ? min(ROWS, m - row0) * ld * 4 : 0, kBufferFlags);
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(w) + static_cast<int64_t>(col0) * ld, 0, VECTOR ? min(COLUMNS, n - col0) * ld * 4 : 0, kBufferFlags);
    auto load4 = [&](const float* matrix, const __amdgpu_buffer_rsrc_t& rsrc, int rows, int first_row, int index, int k0) {
        const int r = index / QUADS, kk = k0 + (index % QUADS) * 4;
        if constexpr (VECTOR) {
            return __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, r * ld * 4 + offset_below(kk, k), 0, 0));
        } else {
            const bool live = first_row + r < rows;
            const float* source = matrix + static_cast<int64_t>(live ? first_row + r : 0) * ld + kk;
            floatx4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (live && kk + e < k) ? source[e] : 0.0f;
            return v;
        }
    };
    floatx4 a_next[LOADS_A], w_next[LOADS_W];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int j = 0; j < LOADS_A; ++j) a_next[j] = load4(a, a_rsrc, m, row0, threadIdx.x + j * 256, k0);
#pragma unroll
        for (int j = 0; j < LOADS_W; ++j) w_next[j] = load4(w, w_rsrc, n, col0, threadIdx.x + j * 256, k0);
    };
    auto put = [&](float (*tile)[STRIDE], int index, const floatx4& v) {
        float* row = &tile[index / QUADS][index % QUADS * 2];
        *reinterpret_cast<float2*>(row) = make_float2(v[0], v[2]);
        *reinterpret_cast<float2*>(row + kTileDepth / 2) = make_float2(v[1], v[3]);
    };
    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    fetch(k_lo);
    int stage = 0;
    for (int k0 = k_lo; k0 < k; k0 += kTileDepth, stage ^= 1) {
#pragma unroll
        for (int j = 0; j < LOADS_A; ++j) put(a_tile[stage], threadIdx.x + j * 256, a_next[j]);
#pragma unroll
        for (int j = 0; j < LOADS_W; ++j) put(w_tile[stage], threadIdx.x + j * 256, w_next[j]);
        __syncthreads();        // the stage written two chunks ago was read before the last barrier
        fetch(k0 + kTileDepth);     // zeros past the last chunk
        __builtin_amdgcn_sched_barrier(0);      // else the loads sink behind the products and are waited for at once
#pragma unroll
        for (int kk = 0; kk < kTileDepth / 2; kk += 4) {
            floatx4 av[TM], wv[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i)
                av[i] = *reinterpret_cast<const floatx4*>(&a_tile[stage][wave_row + 32 * i + lane % 32][half * (kTileDepth / 2) + kk]);
#pragma unroll
            for (int j = 0; j < TN; ++j)
                wv[j] = *reinterpret_cast<const floatx4*>(&w_tile[stage][wave_col + 32 * j + lane % 32][half * (kTileDepth / 2) + kk]);
#pragma unroll
            for (int step = 0; step < 4; ++step)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i][step], wv[j][step], acc[i][j], 0, 0, 0);
        }
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int col = col0 + wave_col + 32 * j + lane % 32;
        const float shift = (bias && col < n) ? bias[col] : 0.0f;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int r = row0 + wave_row + 32 * i + (e / 4) * 8 + half * 4 + e % 4;
                if (r < m && col < n) c[static_cast<int64_t>(r) * n + col] = acc[i][j][e] + shift;
            }
    }
}

// At most 16 rows (decoding), or 32 (SIXTEENS = 2) and groups of them (blockIdx.y), k a multiple of 4: a wave takes NT tiles of 16
// columns of C and its part of k, on v_mfma_f32_16x16x4_f32 with 16 rows of W as its A operand. A wave's load brings 256 bytes of each of four rows, without a
// branch between the loads, two blocks of 64 of k at a time; the wave then passes them through LDS of its own
// (no other wave reads it), where a row of 64 lies as [k % 4][k / 4]: of every four consecutive k the product wants one in
// each quarter of the wave, and a lane's 16-byte read holds its operands of four products in a row. GROUPS: how many
// times four rows of A there are. Bound by reading W; against the vector kernels below at 8 rows: 37888 x 3584 109 -> 101 us
// (5.4 TB/s), 3584 x 18944 63 -> 52, 3584 x 3584 18.4 -> 15.4, 152064 x 3584 420 -> 352 (with two tiles a wave at 9 to 16 rows 496
// -> 367); at 32 rows, against the matrix units' tiles, 168 -> 159, 84 -> 78, and 24 x 896 x 4864 19.0 -> 12.0. Two blocks of 128 instead of 64 of k in flight are slower (more is asked for past the ends: 52 -> 57).
constexpr int64_t kFewWaves = 384;      // waves from which this kernel is taken: 1152 x 896 in two parts, 144 waves, takes 5.6 us in the vector kernel and 7.7 here; 896 x 4864 in eight, 448 waves, 10.8 and 9.6
// 17 to 32 rows take it for parts of the reduction longer than this, or where the tiles would be a handful: 32 rows of 3584 x 3584 in parts
// of 448 19.4 us here and 17.2 in the tiles, of 37888 x 512 26.8 and 27.2, x 64 12.8 and 9.0, of 3584 x 18944 in parts of 2368 73.0 and
// 72.8 (17 rows 63.4 and 70.3), of 37888 x 2048 87 and 94.
constexpr int kFewLong = 600;
// Two tiles a wave, for 9 rows on, where one would read A too often: 16 rows of 152064 x 896 with one and two 100 and 93 us, 32 rows
// 141 and 123; of 37888 x 2048 66 and 80, of 16384 x 2048 28.5 and 35.4.
constexpr int kPairsFrom = 65536;
constexpr int kFewRow = 64 + 16;        // floats from one row in LDS to the next: the four rows of a load on different banks

template <int NT, int GROUPS, int SIXTEENS>
__global__ __launch_bounds__(256) void gemm_f32_few_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                           const float* __restrict__ bias, float* __restrict__ c,
                                                           int m, int n, int k, int k_split) {
    MLL_F32_SPLIT_RANGE
    __shared__ __align__(16) float shared[4][NT + SIXTEENS][16][kFewRow];
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int col = lane % 16, quad = lane / 16;
    const int first = (blockIdx.x * 4 + wave) * 16 * NT;        // the wave's first column of C, row of W
    if (first >= n) return;
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(w) + static_cast<int64_t>(first) * ld, 0,
                                                                            min(16 * NT, n - first) * ld * 4, kBufferFlags);
    const int row0 = blockIdx.y * 16 * SIXTEENS, rows = min(16 * SIXTEENS, m - row0);
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a) + static_cast<int64_t>(row0) * ld, 0, rows * ld * 4, kBufferFlags);
    floatx4 acc[NT][SIXTEENS];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int s = 0; s < SIXTEENS; ++s) acc[nt][s] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    struct Block {
        floatx4 w[NT][4], a[SIXTEENS * GROUPS];
    };
    auto load = [&](int k0, Block& block) {
        const int at = offset_below(k0 + col * 4, k);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                block.w[nt][g] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, (16 * nt + 4 * g + quad) * ld * 4 + at, 0, kNonTemporal));
#pragma unroll
        for (int g = 0; g < SIXTEENS * GROUPS; ++g)
            block.a[g] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, (4 * g + quad) * ld * 4 + at, 0, 0));
    };
    auto put = [&](float (*rows)[kFewRow], int g, const floatx4& v) {
#pragma unroll
        for (int e = 0; e < 4; ++e) rows[4 * g + quad][16 * e + col] = v[e];
    };
    auto multiply = [&](Block& block) {
        // LDS takes a wave's accesses in order; the fences keep the compiler to it.
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int g = 0; g < SIXTEENS * GROUPS; ++g) put(shared[wave][NT + g / GROUPS], g % GROUPS, block.a[g]);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int g = 0; g < 4; ++g) put(shared[wave][nt], g, block.w[nt][g]);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int part = 0; part < 4; ++part) {
            floatx4 av[SIXTEENS];
#pragma unroll
            for (int s = 0; s < SIXTEENS; ++s)
                av[s] = *reinterpret_cast<const floatx4*>(&shared[wave][NT + s][col % (4 * GROUPS)][16 * quad + 4 * part]);
            floatx4 wv[NT];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) wv[nt] = *reinterpret_cast<const floatx4*>(&shared[wave][nt][col][16 * quad + 4 * part]);
#pragma unroll
            for (int step = 0; step < 4; ++step)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                    for (int s = 0; s < SIXTEENS; ++s)
                        acc[nt][s] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[nt][step], av[s][step], acc[nt][s], 0, 0, 0);
        }
    };
    Block even, odd;
    constexpr int kBlock = 64;
    load(k_lo, even);
    load(k_lo + kBlock, odd);
    for (int k0 = k_lo + 2 * kBlock; k0 < k; k0 += 2 * kBlock) {
        multiply(even);
        load(k0, even);
        __builtin_amdgcn_sched_barrier(0);      // else the loads sink below the next products, behind their waits
        multiply(odd);
        load(k0 + kBlock, odd);
        __builtin_amdgcn_sched_barrier(0);
    }
    multiply(even);
    multiply(odd);
    // acc[nt][s][i] = C[row row0 + 16 s + col][column first + 16 nt + 4 quad + i]; columns of rows that are none hold other rows' sums
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int s = 0; s < SIXTEENS; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int column = first + 16 * nt + 4 * quad + i, row = 16 * s + col;
                if (row < rows && column < n) c[static_cast<int64_t>(row0 + row) * n + column] = acc[nt][s][i] + (bias ? bias[column] : 0.0f);
            }
}

template <int NT>
static void launch_few(const float* a, const float* w, const float* bias, float* c, int m, int n, int k, int k_split,
                       unsigned parts, hipStream_t stream) {
    const dim3 grid((n + 64 * NT - 1) / (64 * NT), m <= 16 ? 1 : (m + 31) / 32, parts);
    if (m <= 4) gemm_f32_few_kernel<NT, 1, 1><<<grid, 256, 0, stream>>>(a, w, bias, c, m, n, k, k_split);
    else if (m <= 8) gemm_f32_few_kernel<NT, 2, 1><<<grid, 256, 0, stream>>>(a, w, bias, c, m, n, k, k_split);
    else if (m <= 16) gemm_f32_few_kernel<NT, 4, 1><<<grid, 256, 0, stream>>>(a, w, bias, c, m, n, k, k_split);
    else gemm_f32_few_kernel<NT, 4, 2><<<grid, 256, 0, stream>>>(a, w, bias, c, m, n, k, k_split);
}

// Tiles of 16 x 32 for more than 16 rows of small weights, where tiles of the matrix units would be a handful of workgroups,
// each waiting for one chunk of k after the other: a thread takes 2 x 2 elements (rows r and r + 8, columns c and c + 16), each summed by
// that thread alone in ascending k. Chunks of 128 of k lie in LDS as [row][k] with rows four banks apart, so that a thread's
// four consecutive k are one read and the rows a wave reads at one k fall on different banks.
constexpr int64_t kFewBelow = 128;      // workgroups of the matrix units' tiles
// Small tiles up to this many: 200 x 1152 x 256, 468 of them, 11.2 us in the matrix units' tiles and 9.6 in these, 320 x 1152 x 256, 720, 11.2
// and 10.3, 33 x 2048 x 2048, 768, 16.8 and 15.4; 512 x 896 x 256, 896, 11.4 and 11.4, 2048 x 256 x 512, 1024, 17.1 and 18.7.
constexpr int64_t kGrainMost = 800;
template <bool VECTOR>
__global__ __launch_bounds__(128) void gemm_f32_grain_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                                const float* __restrict__ bias, float* __restrict__ c,
                                                                int m, int n, int k, int k_split) {
    MLL_F32_SPLIT_RANGE
    constexpr int THREADS = 128, TR = 2, TC = 2, DEPTH = 128;
    constexpr int ROW_STEP = THREADS / 16;
    constexpr int ROWS = ROW_STEP * TR;
    constexpr int COLUMNS = 16 * TC;
    constexpr int QUADS = DEPTH / 4;                       // float4 in a row of a chunk
    constexpr int LOADS_A = ROWS * QUADS / THREADS;
    constexpr int LOADS_W = COLUMNS * QUADS / THREADS;
    static_assert(ROWS * QUADS % THREADS == 0 && COLUMNS * QUADS % THREADS == 0, "a chunk is dealt evenly to the threads");
    __shared__ __align__(16) float a_tile[ROWS][DEPTH + 4];
    __shared__ __align__(16) float w_tile[COLUMNS][DEPTH + 4];
    const int row0 = blockIdx.y * ROWS;
    const int col0 = blockIdx.x * COLUMNS;
    const int column = threadIdx.x % 16;
    const int row = threadIdx.x / 16;
    auto load4 = [&](const float* matrix, int rows, int first_row, int index, int k0) {
        const int r = index / QUADS, kk = k0 + (index % QUADS) * 4;
        const bool live = first_row + r < rows;
        const float* source = matrix + static_cast<int64_t>(live ? first_row + r : 0) * ld + kk;
        if (VECTOR) return (live && kk < k) ? *reinterpret_cast<const float4*>(source) : make_float4(0.f, 0.f, 0.f, 0.f);
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (live && kk + e < k) ? source[e] : 0.0f;
        return make_float4(v[0], v[1], v[2], v[3]);
    };
    float4 a_next[LOADS_A], w_next[LOADS_W];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int j = 0; j < LOADS_A; ++j) a_next[j] = load4(a, m, row0, threadIdx.x + j * THREADS, k0);
#pragma unroll
        for (int j = 0; j < LOADS_W; ++j) w_next[j] = load4(w, n, col0, threadIdx.x + j * THREADS, k0);
    };
    float acc[TR][TC];
#pragma unroll
    for (int i = 0; i < TR; ++i)
#pragma unroll
        for (int j = 0; j < TC; ++j) acc[i][j] = 0.0f;
    fetch(k_lo);
    for (int k0 = k_lo; k0 < k; k0 += DEPTH) {
#pragma unroll
        for (int j = 0; j < LOADS_A; ++j) {
            const int index = threadIdx.x + j * THREADS;
            *reinterpret_cast<float4*>(&a_tile[index / QUADS][(index % QUADS) * 4]) = a_next[j];
        }
#pragma unroll
        for (int j = 0; j < LOADS_W; ++j) {
            const int index = threadIdx.x + j * THREADS;
            *reinterpret_cast<float4*>(&w_tile[index / QUADS][(index % QUADS) * 4]) = w_next[j];
        }
        __syncthreads();
        if (k0 + DEPTH < k) fetch(k0 + DEPTH);
#pragma unroll
        for (int kk = 0; kk < DEPTH; kk += 4) {
            float4 av[TR], wv[TC];
#pragma unroll
            for (int i = 0; i < TR; ++i) av[i] = *reinterpret_cast<const float4*>(&a_tile[row + ROW_STEP * i][kk]);
#pragma unroll
            for (int j = 0; j < TC; ++j) wv[j] = *reinterpret_cast<const float4*>(&w_tile[column + 16 * j][kk]);
#pragma unroll
            for (int i = 0; i < TR; ++i)
#pragma unroll
                for (int j = 0; j < TC; ++j) acc[i][j] = fmaf(av[i].x, wv[j].x, acc[i][j]);
#pragma unroll
            for (int i = 0; i < TR; ++i)
#pragma unroll
                for (int j = 0; j < TC; ++j) acc[i][j] = fmaf(av[i].y, wv[j].y, acc[i][j]);
#pragma unroll
            for (int i = 0; i < TR; ++i)
#pragma unroll
                for (int j = 0; j < TC; ++j) acc[i][j] = fmaf(av[i].z, wv[j].z, acc[i][j]);
#pragma unroll
            for (int i = 0; i < TR; ++i)
#pragma unroll
                for (int j = 0; j < TC; ++j) acc[i][j] = fmaf(av[i].w, wv[j].w, acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < TR; ++i)
#pragma unroll
        for (int j = 0; j < TC; ++j) {
            const int r = row0 + row + ROW_STEP * i, col = col0 + column + 16 * j;
            if (r < m && col < n) c[static_cast<int64_t>(r) * n + col] = acc[i][j] + (bias ? bias[col] : 0.0f);
        }
}

// The same product for at most 16 rows (decoding): a workgroup takes 16 columns of C, so that a weight of a few
// thousand rows fills the GPU where tiles of 64 would leave most of it idle, and one thread one output element.
// Each thread sums in ascending k with the same fused multiply-adds as the tiled kernel: the two give the same
// bits, so a token's result does not depend on how many rows the step had.
constexpr int kSmallColumns = 16;
constexpr int kSmallDepth = 256;      // of k in a chunk (128: 3 to 7 % slower)
constexpr int kSmallParts = kSmallDepth / 64;

// VECTOR: k is a multiple of 4 and both matrices are 16-byte aligned, so a thread's four consecutive elements are
// one load.
template <bool VECTOR>
__global__ __launch_bounds__(256) void gemm_f32_small_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                             const float* __restrict__ bias, float* __restrict__ c,
                                                             int m, int n, int k, int k_split) {
    MLL_F32_SPLIT_RANGE
    // Rows of kSmallDepth + 4 floats: 16-byte aligned, so that four consecutive k are one read, and four banks on
    // from row to row, so that the 16 rows (or columns) that a wave reads at one k fall on different banks.
    __shared__ __align__(16) float a_tile[16][kSmallDepth + 4];
    __shared__ __align__(16) float w_tile[kSmallColumns][kSmallDepth + 4];
    const int col0 = blockIdx.x * kSmallColumns;
    const int column = threadIdx.x % kSmallColumns;     // this thread's output: row `row`, column col0 + `column`
    const int row = threadIdx.x / kSmallColumns;
    // What a thread brings in of a chunk of kSmallDepth of k: of row load_row of A and of W, elements
    // load_k .. load_k + 3 of every 64.
    const int load_row = threadIdx.x / 16;
    const int load_k = (threadIdx.x % 16) * 4;
    const bool a_live = load_row < m, w_live = col0 + load_row < n;
    const float* a_row = a + static_cast<int64_t>(a_live ? load_row : 0) * ld;
    const float* w_row = w + static_cast<int64_t>(w_live ? col0 + load_row : 0) * ld;
    float4 a_next[kSmallParts], w_next[kSmallParts];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int part = 0; part < kSmallParts; ++part) {
            const int kk = k0 + 64 * part + load_k;
            if (VECTOR) {
                a_next[part] = (a_live && kk < k) ? *reinterpret_cast<const float4*>(a_row + kk) : make_float4(0.f, 0.f, 0.f, 0.f);
                w_next[part] = (w_live && kk < k) ? *reinterpret_cast<const float4*>(w_row + kk) : make_float4(0.f, 0.f, 0.f, 0.f);
            } else {
                float av[4], wv[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    av[e] = (a_live && kk + e < k) ? a_row[kk + e] : 0.0f;
                    wv[e] = (w_live && kk + e < k) ? w_row[kk + e] : 0.0f;
                }
                a_next[part] = make_float4(av[0], av[1], av[2], av[3]);
                w_next[part] = make_float4(wv[0], wv[1], wv[2], wv[3]);
            }
        }
    };
    float acc = 0.0f;
    fetch(k_lo);
    for (int k0 = k_lo; k0 < k; k0 += kSmallDepth) {
#pragma unroll
        for (int part = 0; part < kSmallParts; ++part) {
            const int at = 64 * part + load_k;
            *reinterpret_cast<float4*>(&a_tile[load_row][at]) = a_next[part];
            *reinterpret_cast<float4*>(&w_tile[load_row][at]) = w_next[part];
        }
        __syncthreads();
        if (k0 + kSmallDepth < k) fetch(k0 + kSmallDepth);      // the next chunk is on its way while this one is summed
        // Four k a read, summed one after the other in ascending k as before: the same bits.
#pragma unroll
        for (int kk = 0; kk < kSmallDepth; kk += 4) {
            const float4 av = *reinterpret_cast<const float4*>(&a_tile[row][kk]);
            const float4 wv = *reinterpret_cast<const float4*>(&w_tile[column][kk]);
            acc = fmaf(av.x, wv.x, acc);
            acc = fmaf(av.y, wv.y, acc);
            acc = fmaf(av.z, wv.z, acc);
            acc = fmaf(av.w, wv.w, acc);
        }
        __syncthreads();
    }
    const int col = col0 + column;
    if (row < m && col < n) c[static_cast<int64_t>(row) * n + col] = acc + (bias ? bias[col] : 0.0f);
}

// The same for weights with many rows, where the kernel above is bound by its reads from LDS (two a multiply-add). Of those,
// gemm_f32_few_kernel has what it can read 16 bytes at a time; this kernel has the others (reductions that are no multiple of 4,
// operands at no 16-byte boundary) and the weights whose rows lie a multiple of 32 KB apart (mll_gemm_f32). The figures here were
// measured before that kernel took gate/up and the head. A workgroup of 128 threads takes 32 columns of C and a thread 2 rows x 2 columns (rows r and r + 8,
// columns c and c + 16): half the reads a multiply-add, and four chains of additions a thread. Every element is still
// summed by one thread in ascending k: the same bits. Measured on MI355X at 7B sizes, 8 rows: gate/up 179 -> 140 us
// (3.9 TB/s), the head 602 -> 450 (4.8 TB/s); with few columns it has too few waves (q/k/v 37 -> 65 us, down 136 -> 330).
// Where W has few rows the kernel above stays at 1.8 to 2.0 TB/s: a wave an element's worth of lanes is all the
// parallelism there is, and its reads from LDS (512 KB for 16 KB of W) are what a compute unit can give; neither four
// sums an element instead of one, nor two chunks in flight instead of one, nor reading LDS a batch ahead changes that.
constexpr int kWideThreads = 128;
constexpr int kWideDepth = 128;                      // of k in a chunk
constexpr int kWideQuads = kWideDepth / 4;           // float4 in a row of a chunk
constexpr int kWideFrom = 16384;                     // columns of C from which the reduction is not cut, and this kernel taken before the one above

// TR x TC elements a thread: rows r (+ 8), columns c, c + 16, ... of the workgroup's 8 TR rows and 16 TC columns. Per
// four k a thread reads TR + TC times from LDS for 4 TR TC multiply-adds, and every element of W is read by 8 threads:
// with 2 x 2 that is 16 reads an element of W, which is what bounds the kernel (4.1 TB/s of W for gate/up at 8 rows,
// where half of the 16 rows are empty); 1 x 4 for at most 8 rows makes it 10 (4.8 TB/s; the head 4.95 -> 5.4).
template <bool VECTOR, int TR, int TC>
__global__ __launch_bounds__(kWideThreads) void gemm_f32_small_wide_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                                           const float* __restrict__ bias, float* __restrict__ c,
                                                                           int m, int n, int k, int k_split) {
    MLL_F32_SPLIT_RANGE
    constexpr int ROWS = 8 * TR, COLUMNS = 16 * TC;
    constexpr int LOADS_A = ROWS * kWideQuads / kWideThreads, LOADS_W = COLUMNS * kWideQuads / kWideThreads;
    __shared__ __align__(16) float a_tile[ROWS][kWideDepth + 4];
    __shared__ __align__(16) float w_tile[COLUMNS][kWideDepth + 4];
    const int col0 = blockIdx.x * COLUMNS;
    const int column = threadIdx.x % 16;      // this thread's outputs: rows `row` (+ 8); columns col0 + `column` + 16 j
    const int row = threadIdx.x / 16;
    // What a thread brings in of a chunk: float4 number threadIdx.x + j * 128 of the chunk's rows of A (ROWS rows of
    // kWideQuads) and of W (COLUMNS rows).
    auto load4 = [&](const float* matrix, int rows, int first_row, int index, int k0) {
        const int r = index / kWideQuads, kk = k0 + (index % kWideQuads) * 4;
        const bool live = first_row + r < rows;
        const float* source = matrix + static_cast<int64_t>(live ? first_row + r : 0) * ld + kk;
        if (VECTOR) return (live && kk < k) ? *reinterpret_cast<const float4*>(source) : make_float4(0.f, 0.f, 0.f, 0.f);
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (live && kk + e < k) ? source[e] : 0.0f;
        return make_float4(v[0], v[1], v[2], v[3]);
    };
    float4 a_next[LOADS_A], w_next[LOADS_W];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int j = 0; j < LOADS_A; ++j) a_next[j] = load4(a, m, 0, threadIdx.x + j * kWideThreads, k0);
#pragma unroll
        for (int j = 0; j < LOADS_W; ++j) w_next[j] = load4(w, n, col0, threadIdx.x + j * kWideThreads, k0);
    };
    float acc[TR][TC];
#pragma unroll
    for (int i = 0; i < TR; ++i)
#pragma unroll
        for (int j = 0; j < TC; ++j) acc[i][j] = 0.0f;
    fetch(k_lo);
    for (int k0 = k_lo; k0 < k; k0 += kWideDepth) {
#pragma unroll
        for (int j = 0; j < LOADS_A; ++j) {
            const int index = threadIdx.x + j * kWideThreads;
            *reinterpret_cast<float4*>(&a_tile[index / kWideQuads][(index % kWideQuads) * 4]) = a_next[j];
        }
#pragma unroll
        for (int j = 0; j < LOADS_W; ++j) {
            const int index = threadIdx.x + j * kWideThreads;
            *reinterpret_cast<float4*>(&w_tile[index / kWideQuads][(index % kWideQuads) * 4]) = w_next[j];
        }
        __syncthreads();
        if (k0 + kWideDepth < k) fetch(k0 + kWideDepth);      // the next chunk is on its way while this one is summed
        // Four k a read, added one after the other in ascending k.
#pragma unroll
        for (int kk = 0; kk < kWideDepth; kk += 4) {
            float4 av[TR], wv[TC];
#pragma unroll
            for (int i = 0; i < TR; ++i) av[i] = *reinterpret_cast<const float4*>(&a_tile[row + 8 * i][kk]);
#pragma unroll
            for (int j = 0; j < TC; ++j) wv[j] = *reinterpret_cast<const float4*>(&w_tile[column + 16 * j][kk]);
#pragma unroll
            for (int i = 0; i < TR; ++i)
#pragma unroll
                for (int j = 0; j < TC; ++j) acc[i][j] = fmaf(av[i].x, wv[j].x, acc[i][j]);
#pragma unroll
            for (int i = 0; i < TR; ++i)
#pragma unroll
                for (int j = 0; j < TC; ++j) acc[i][j] = fmaf(av[i].y, wv[j].y, acc[i][j]);
#pragma unroll
            for (int i = 0; i < TR; ++i)
#pragma unroll
                for (int j = 0; j < TC; ++j) acc[i][j] = fmaf(av[i].z, wv[j].z, acc[i][j]);
#pragma unroll
            for (int i = 0; i < TR; ++i)
#pragma unroll
                for (int j = 0; j < TC; ++j) acc[i][j] = fmaf(av[i].w, wv[j].w, acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < TR; ++i)
#pragma unroll
        for (int j = 0; j < TC; ++j) {
            const int r = row + 8 * i, col = col0 + column + 16 * j;
            if (r < m && col < n) c[static_cast<int64_t>(r) * n + col] = acc[i][j] + (bias ? bias[col] : 0.0f);
        }
}

template <int TR, int TC>
static void launch_small_wide(const float* a, const float* w, const float* bias, float* c, int m, int n, int k, int k_split,
                              unsigned parts, bool vector, hipStream_t stream) {
    const dim3 grid((n + 16 * TC - 1) / (16 * TC), 1, parts);
    if (vector) gemm_f32_small_wide_kernel<true, TR, TC><<<grid, kWideThreads, 0, stream>>>(a, w, bias, c, m, n, k, k_split);
    else gemm_f32_small_wide_kernel<false, TR, TC><<<grid, kWideThreads, 0, stream>>>(a, w, bias, c, m, n, k, k_split);
}

}  // namespace mll

using namespace mll;

// Which kernel takes a product of at most 16 rows: 0 the choice below; for measurements and tests 1 (an element a
// thread), 2 (2 x 2) or 4 (1 x 4, at most 8 rows). The same bits whichever.
static int f32_small_variant = 0;
extern "C" int mll_gemm_f32_small_variant(int variant) {
    const int before = f32_small_variant;
    f32_small_variant = (variant == 1 || variant == 2 || variant == 4) ? variant : 0;
    return before;
}

// Into how many parts the reduction over k is cut for a weight [n, k]: a function of the weight's shape alone. A
// weight with few rows of its own (q/k/v, o, down) gives the GPU too few tiles of C; its parts go to workgroups of
// their own. Parts are at least 448 terms long and at most 8.
extern "C" int mll_gemm_f32_splits(int n, int k) {
    if (n >= kWideFrom) return 1;
    int splits = 1;
    while (splits < 8 && (n / kSmallColumns) * splits < 2048 && k / (2 * splits) >= 448) splits *= 2;
    return splits;
}

// C[splits][m][n]; splits is 1 or mll_gemm_f32_splits(n, k).
extern "C" int mll_gemm_f32(const float* a, const float* w, const float* bias, float* c,
                            int m, int n, int k, int splits, hipStream_t stream) {
    MLL_REQUIRE(m >= 0 && n > 0 && k > 0, "gemm_f32: sizes must be positive");
    MLL_REQUIRE(splits == 1 || splits == mll_gemm_f32_splits(n, k), "gemm_f32: the reduction is cut as mll_gemm_f32_splits says, or not at all");
    if (m == 0) return 0;
    const int k_split = splits == 1 ? k : ((k + splits - 1) / splits + 3) / 4 * 4;
    MLL_REQUIRE(static_cast<int64_t>(k_split) * (splits - 1) < k, "gemm_f32: a part of the reduction would be empty");
    const unsigned parts = static_cast<unsigned>(splits);
    const bool vector = k % 4 == 0 && k <= kWidestVector && reinterpret_cast<uintptr_t>(a) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0;
    const int64_t waves = static_cast<int64_t>((n + 15) / 16) * splits;
    const int64_t thirty_twos = static_cast<int64_t>((n + 127) / 128) * splits;     // the matrix units' tiles for 17 to 32 rows
    // Rows of W a multiple of 32 KB apart fall on the same channels of the memory, of which a wave asks for 16 rows at a time; the vector
    // kernels ask for fewer: 4608 x 8192 in parts at 1, 8 and 16 rows 39, 42 and 45 us here, 33, 34 and 39 there, 9728 x 8192 70, 75
    // and 77, 65, 66 and 71, 3584 x 8192 29, 31 and 33, 29, 29 and 31; 2048 x 8192 16.8 and 25.1, whole 16384 x 8192 107 and 163.
    const bool same_channels = k % 8192 == 0 && splits > 1 && n >= 3584;
    if (vector && waves >= kFewWaves && (m <= 16 ? f32_small_variant == 0 && !same_channels : m <= 32 && (k_split > kFewLong || thirty_twos <= kFewBelow))) {
        if (n >= kPairsFrom && m > 8) launch_few<2>(a, w, bias, c, m, n, k, k_split, parts, stream);
        else launch_few<1>(a, w, bias, c, m, n, k, k_split, parts, stream);
        return check_launch("gemm_f32");
    }
    if (m <= 16) {
        // What the kernel of few rows does not take. Up to 8 rows: one row and four columns a thread where that still gives the GPU its workgroups (weights of
        // many rows; the others with their parts); else two rows and two columns where that does, else the kernel of
        // one element a thread. (Two rows and four columns for 9 to 16 rows are slower than two and two: gate/up at
        // 7B sizes 131 -> 156 us. A column a thread with all rows, which reads an element of W from LDS once, is
        // faster for one row alone (q/k/v 20 -> 16.5 us, down 60 -> 51) and 1 % in the step; from two rows on the
        // rows of A, read by all lanes at one address, cost more than is saved: 8 rows 115 -> 310 us.)
        const int64_t quads = static_cast<int64_t>((n + 63) / 64) * splits, pairs = static_cast<int64_t>((n + 31) / 32) * splits;
        int variant = f32_small_variant;
        if (variant == 4 && m > 8) variant = 2;
        if (variant == 0) {
            if (m <= 8 && (n >= kWideFrom || quads >= 384)) variant = 4;
            else if (n >= kWideFrom || pairs >= 512) variant = 2;
            else variant = 1;
        }
        if (variant == 4) {
            launch_small_wide<1, 4>(a, w, bias, c, m, n, k, k_split, parts, vector, stream);
            return check_launch("gemm_f32");
        }
        if (variant == 2) {
            launch_small_wide<2, 2>(a, w, bias, c, m, n, k, k_split, parts, vector, stream);
            return check_launch("gemm_f32");
        }
        const dim3 grid((n + kSmallColumns - 1) / kSmallColumns, 1, parts);
        if (vector) gemm_f32_small_kernel<true><<<grid, 256, 0, stream>>>(a, w, bias, c, m, n, k, k_split);
        else gemm_f32_small_kernel<false><<<grid, 256, 0, stream>>>(a, w, bias, c, m, n, k, k_split);
        return check_launch("gemm_f32");
    }
    // The tile that is done first: a tile's size, times what its elements take, times the rounds of 256 workgroups, of which the last counts by
    // four fifths of a whole one beside its share (workgroups that share a unit cover each other's ends). Where parts of the reduction are long the larger
    // tiles read LDS less for every product; where they are short the smaller ones' beginnings and ends overlap. Fitted to the four shapes' times at
    // 119 sizes (65 to 1500 rows of seven weights): 0.4 % above the fastest on the mean and 6 % at most, where rounds alone, whole below 4096 workgroups and
    // not above, were 2.8 and 44 % above it (1500 x 37888 x 3584 in tiles of 32 x 128 4746 us, of 128 x 128 3290; 512 rows of it 1308 and 1176; 600 1866 and
    // 1408; 512 x 896 x 4864 in eight parts 55 and, in tiles of 64 x 64, 49). The factors and the line at 1000 terms are that fit, no mechanism. At 221 sizes outside it
    // (17 to 4096 rows of weights of 300 to 152064 rows, reductions of 64 to 16000) 0.99 of the time of rounds alone, 0.77 at least; slower by more than
    // 2 %: 955 x 2048 x 8192 in eight parts 268 -> 283 us, 1468 x 16384 x 2048 798 -> 815. Up to 32 rows take tiles of 32 rows (32 x 9728 x 896 in tiles of 64 x 64 26.6 us, of 32 x 128 17.7).
    struct Shape { int rows, columns; double in_long, in_short; };
    const Shape shapes[4] = {{128, 128, 1.0, 1.0}, {128, 64, 1.06, 0.98}, {64, 64, 1.10, 0.92}, {32, 128, 1.30, 0.975}};
    constexpr int kLongParts = 1000;
    int best = 3;
    double least = 1e300;
    for (int index = m <= 32 ? 3 : 0; index < 4; ++index) {
        const Shape& shape = shapes[index];
        const int64_t groups = static_cast<int64_t>((n + shape.columns - 1) / shape.columns) * ((m + shape.rows - 1) / shape.rows) * splits;
        const double rounds = 0.8 * static_cast<double>((groups + 255) / 256) + 0.2 * groups / 256.0;
        const double cost = rounds * shape.rows * shape.columns * (k_split > kLongParts ? shape.in_long : shape.in_short);
        const bool fits = (m + shape.rows - 1) / shape.rows <= 65535;       // as the grid's second size
        if (fits && cost < least) least = cost, best = index;
    }
    const Shape& shape = shapes[best];
    const int64_t tiles = static_cast<int64_t>((n + shape.columns - 1) / shape.columns) * ((m + shape.rows - 1) / shape.rows) * splits;
    // Few tiles: 32 rows a wave and several groups of rows, each reading W from the caches: 64 x 896 x 4864 in eight parts, 112 tiles, 19.6 us
    // in them, 13.5 so; 64 x 896 x 9728, 152 tiles, 22.8 and 25.4; 48 x 896 x 1152 in two 11.4 in the small tiles below, 10.5 so.
    if (tiles < kFewBelow && m <= 128 && vector && waves * ((m + 31) / 32) >= kFewWaves / 2) {
        launch_few<1>(a, w, bias, c, m, n, k, k_split, parts, stream);
        return check_launch("gemm_f32");
    }
    if (static_cast<int64_t>((n + 31) / 32) * ((m + 15) / 16) * splits <= kGrainMost) {
        const dim3 grid((n + 31) / 32, (m + 15) / 16, parts);
        if (vector) gemm_f32_grain_kernel<true><<<grid, 128, 0, stream>>>(a, w, bias, c, m, n, k, k_split);
        else gemm_f32_grain_kernel<false><<<grid, 128, 0, stream>>>(a, w, bias, c, m, n, k, k_split);
        return check_launch("gemm_f32");
    }
    const dim3 grid((n + shape.columns - 1) / shape.columns, (m + shape.rows - 1) / shape.rows, parts);
    MLL_REQUIRE(grid.y <= 65535, "gemm_f32: too many rows for one call");
#define MLL_F32_TILE(WAVES_M, TM, TN)                                                                                  \
    if (vector) gemm_f32_tile_kernel<WAVES_M, TM, TN, true><<<grid, 256, 0, stream>>>(a, w, bias, c, m, n, k, k_split); \
    else gemm_f32_tile_kernel<WAVES_M, TM, TN, false><<<grid, 256, 0, stream>>>(a, w, bias, c, m, n, k, k_split)
    if (best == 0) { MLL_F32_TILE(2, 2, 2); }
    else if (best == 1) { MLL_F32_TILE(2, 2, 1); }
    else if (best == 2) { MLL_F32_TILE(2, 1, 1); }
    else { MLL_F32_TILE(1, 1, 1); }
#undef MLL_F32_TILE
    return check_launch("gemm_f32");
}
