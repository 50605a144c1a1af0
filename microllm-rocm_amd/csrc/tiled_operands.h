// What the products of large tiles (gemm_tiled.hip, moe_tiled.hip) share: the operands of a k step in registers, read from a stage in
// LDS between the products of the step before. A stage of 64 of k lies in a slot: up to 256 rows of A in pieces of 16 rows (2 KB), then 256
// rows of W in tiles of 16 (2 KB). Rows of 128 bytes have their eight 16-byte chunks at places exchanged by (row / 2).
#pragma once

#include <utility>

#include "common.h"

namespace mll {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) bf16 lds_bf16;

constexpr int kMaxWaveTilesM = 8;                         // a wave's part of C is at most 128 x 64
constexpr int kTiledWaves = 8;
constexpr int kTiledThreads = kTiledWaves * kWave;
constexpr int kWaveTilesN = 4;                            // a wave's 64 columns of C
constexpr int kSlotBytes = 65536;                         // a stage of 64 of k: up to 32 KB of A, then 32 KB of W
constexpr int kSlotElements = kSlotBytes / 2;
constexpr int kWBytes = 32768;                            // where W begins in a slot

__device__ inline unsigned lds_address(bf16* place) { return static_cast<unsigned>(reinterpret_cast<uintptr_t>((lds_bf16*)place)); }

template <int WM>
struct TiledOperands {       // of one k step: the wave's WM pieces of A and 4 of W, 16 bytes a lane each
    uintx4 a[WM];
    uintx4 w[kWaveTilesN];
};

#define MLL_DS_READ(TARGET, ADDRESS, BYTES) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(TARGET) : "v"(ADDRESS), "n"(BYTES))
#define MLL_MFMA(ACC, W, A) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(ACC) : "v"(W), "v"(A))

// The INDEX-th of the 4 + WM reads of k step STEP (0, 1) of a stage: pieces of A are 2 KB apart in a slot, tiles of W
// too, with the tile's second step W_STEP bytes after its first (0: the caller's address says which step). An INDEX beyond the reads is nothing.
template <int W_STEP, int WM, int INDEX, int STEP>
__device__ __attribute__((always_inline)) inline void read_operand(TiledOperands<WM>& f, unsigned a_address, unsigned w_address) {
    constexpr int W = kWBytes + STEP * W_STEP;
    if constexpr (INDEX == 0) MLL_DS_READ(f.w[0], w_address, W);
    if constexpr (INDEX == 1) MLL_DS_READ(f.w[1], w_address, W + 2048);
    if constexpr (INDEX == 2) MLL_DS_READ(f.a[0], a_address, 0);
    if constexpr (INDEX == 3) MLL_DS_READ(f.a[1], a_address, 2048);
    if constexpr (INDEX == 4) MLL_DS_READ(f.w[2], w_address, W + 4096);
    if constexpr (INDEX == 5) MLL_DS_READ(f.w[3], w_address, W + 6144);
    if constexpr (INDEX >= 6 && INDEX < 4 + WM) MLL_DS_READ(f.a[INDEX - 4], a_address, (INDEX - 4) * 2048);
}
template <int W_STEP, int WM, int STEP, int... INDEX>
__device__ __attribute__((always_inline)) inline void read_operands(TiledOperands<WM>& f, unsigned a_address, unsigned w_address,
                                                                    std::integer_sequence<int, INDEX...>) {
    (read_operand<W_STEP, WM, INDEX, STEP>(f, a_address, w_address), ...);
}

// The four products of row tile MT of a k step, and after every second of them a read of the next step's operands
// (the first 4 + WM of the 2 WM places take one).
template <int W_STEP, int WM, int NEXT_STEP, int MT>
__device__ __attribute__((always_inline)) inline void products_of_row_tile(floatx4 (&acc)[kWaveTilesN][WM], const TiledOperands<WM>& now,
                                                                           TiledOperands<WM>& next, unsigned a_address, unsigned w_address) {
    MLL_MFMA(acc[0][MT], now.w[0], now.a[MT]);
    MLL_MFMA(acc[1][MT], now.w[1], now.a[MT]);
    read_operand<W_STEP, WM, 2 * MT, NEXT_STEP>(next, a_address, w_address);
    MLL_MFMA(acc[2][MT], now.w[2], now.a[MT]);
    MLL_MFMA(acc[3][MT], now.w[3], now.a[MT]);
    read_operand<W_STEP, WM, 2 * MT + 1, NEXT_STEP>(next, a_address, w_address);
}
template <int W_STEP, int WM, int NEXT_STEP, int... MT>
__device__ __attribute__((always_inline)) inline void products(floatx4 (&acc)[kWaveTilesN][WM], const TiledOperands<WM>& now,
                                                               TiledOperands<WM>& next, unsigned a_address, unsigned w_address,
                                                               std::integer_sequence<int, MT...>) {
    (products_of_row_tile<W_STEP, WM, NEXT_STEP, MT>(acc, now, next, a_address, w_address), ...);
}

// The reads into `f` have arrived (and, LOADS, the wave's loads into LDS have landed). `f` passes through the
// statements, so that nothing that uses it is placed before.
template <bool LOADS, int WM>
__device__ __attribute__((always_inline)) inline void operands_arrived(TiledOperands<WM>& f) {
    if constexpr (LOADS)
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)"
                     : "+v"(f.a[0]), "+v"(f.a[1]), "+v"(f.a[2]), "+v"(f.a[3]), "+v"(f.w[0]), "+v"(f.w[1]), "+v"(f.w[2]), "+v"(f.w[3])
                     :: "memory");
    else
        asm volatile("s_waitcnt lgkmcnt(0)"
                     : "+v"(f.a[0]), "+v"(f.a[1]), "+v"(f.a[2]), "+v"(f.a[3]), "+v"(f.w[0]), "+v"(f.w[1]), "+v"(f.w[2]), "+v"(f.w[3])
                     :: "memory");
#pragma unroll
    for (int i = 4; i < WM; ++i) asm volatile("" : "+v"(f.a[i]));
}

}  // namespace mll
