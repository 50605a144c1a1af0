// What the products of large tiles (gemm_tiled.hip, moe_tiled.hip) share: the operands of a k step in registers, read from a stage in
// LDS between the products of the step before. A stage of 64 of k lies in slots: up to 256 rows of A in pieces of 16 rows (2 KB), 256
// rows of W in tiles of 16 (2 KB). Rows of 128 bytes have their eight 16-byte chunks at places exchanged by (row / 2).
#pragma once

#include <type_traits>
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
// A stage of 64 of k: two slots for up to 256 rows of A, then three for 256 rows of W, 32 KB each. W has one more, so that its loads may be on
// their way while the workgroup has not met since the slot before them was read.
constexpr int kSlotBytes = 32768;
constexpr int kSlotElements = kSlotBytes / 2;
constexpr int kASlots = 2, kWSlots = 3;
constexpr int kWTurns = 32 / kTiledWaves;                 // loads of W a wave and stage, 1 KB each
constexpr int kStageElements = (kASlots + kWSlots) * kSlotElements;

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
    constexpr int W = STEP * W_STEP;
    if constexpr (INDEX < kWaveTilesN) MLL_DS_READ(f.w[INDEX], w_address, W + INDEX * 2048);
    else if constexpr (INDEX < kWaveTilesN + WM) MLL_DS_READ(f.a[INDEX - kWaveTilesN], a_address, (INDEX - kWaveTilesN) * 2048);
}
template <int W_STEP, int WM, int STEP, int... INDEX>
__device__ __attribute__((always_inline)) inline void read_operands(TiledOperands<WM>& f, unsigned a_address, unsigned w_address,
                                                                    std::integer_sequence<int, INDEX...>) {
    (read_operand<W_STEP, WM, INDEX, STEP>(f, a_address, w_address), ...);
}

// The four products of row tile MT of a k step, and after every second of them a read of the next step's operands (the first 4 + WM of the
// 2 WM places take one) and what `between` does at that place: one load of a later stage here and there, so that the loads, which a compute
// unit takes one in 16 cycles, are not asked for in one go while no product is formed.
template <int W_STEP, int WM, int NEXT_STEP, int MT, typename Between>
__device__ __attribute__((always_inline)) inline void products_of_row_tile(floatx4 (&acc)[kWaveTilesN][WM], const TiledOperands<WM>& now,
                                                                           TiledOperands<WM>& next, unsigned a_address, unsigned w_address,
                                                                           const Between& between) {
    MLL_MFMA(acc[0][MT], now.w[0], now.a[MT]);
    MLL_MFMA(acc[1][MT], now.w[1], now.a[MT]);
    read_operand<W_STEP, WM, 2 * MT, NEXT_STEP>(next, a_address, w_address);
    between(std::integral_constant<int, 2 * MT>{});
    MLL_MFMA(acc[2][MT], now.w[2], now.a[MT]);
    MLL_MFMA(acc[3][MT], now.w[3], now.a[MT]);
    read_operand<W_STEP, WM, 2 * MT + 1, NEXT_STEP>(next, a_address, w_address);
    between(std::integral_constant<int, 2 * MT + 1>{});
}
template <int W_STEP, int WM, int NEXT_STEP, typename Between, int... MT>
__device__ __attribute__((always_inline)) inline void products(floatx4 (&acc)[kWaveTilesN][WM], const TiledOperands<WM>& now,
                                                               TiledOperands<WM>& next, unsigned a_address, unsigned w_address,
                                                               const Between& between, std::integer_sequence<int, MT...>) {
    (products_of_row_tile<W_STEP, WM, NEXT_STEP, MT>(acc, now, next, a_address, w_address, between), ...);
}

// The reads into `f` have arrived (and, LOADS >= 0, of the wave's loads into LDS all but the last LOADS have landed). `f` passes through the
// statements, so that nothing that uses it is placed before.
template <int LOADS, int WM>
__device__ __attribute__((always_inline)) inline void operands_arrived(TiledOperands<WM>& f) {
    if constexpr (LOADS >= 0)
        asm volatile("s_waitcnt vmcnt(%8) lgkmcnt(0)"
                     : "+v"(f.a[0]), "+v"(f.a[1]), "+v"(f.a[2]), "+v"(f.a[3]), "+v"(f.w[0]), "+v"(f.w[1]), "+v"(f.w[2]), "+v"(f.w[3])
                     : "n"(LOADS) : "memory");
    else
        asm volatile("s_waitcnt lgkmcnt(0)"
                     : "+v"(f.a[0]), "+v"(f.a[1]), "+v"(f.a[2]), "+v"(f.a[3]), "+v"(f.w[0]), "+v"(f.w[1]), "+v"(f.w[2]), "+v"(f.w[3])
                     :: "memory");
#pragma unroll
    for (int i = 4; i < WM; ++i) asm volatile("" : "+v"(f.a[i]));
}

// The loads of a tile's first two stages, from `first` to before `stages`, go out: copy_a(turn, stage, slot) and copy_w(turn, stage, slot) issue one of a
// wave's A_TURNS and kWTurns loads of a stage, every wave all of them. The slots are free: the workgroup has met since they were read. last_comes() is
// called once, before the loads of the last stage go out.
template <int A_TURNS, typename CopyA, typename CopyW, typename LastComes>
__device__ __attribute__((always_inline)) inline void begin_stages(int first, int stages, const CopyA& copy_a, const CopyW& copy_w, const LastComes& last_comes) {
    if (first + 1 == stages) last_comes();
#pragma unroll
    for (int t = 0; t < A_TURNS; ++t) copy_a(t, first, 0);
#pragma unroll
    for (int t = 0; t < kWTurns; ++t) copy_w(t, first, 0);
    if (first + 1 < stages) {
        if (first + 2 == stages) last_comes();
#pragma unroll
        for (int t = 0; t < A_TURNS; ++t) copy_a(t, first + 1, 1);
#pragma unroll
        for (int t = 0; t < kWTurns; ++t) copy_w(t, first + 1, 1);
    }
}

// The stages of a tile, from `first` to before `stages`, one at least, whose first two are on their way (begin_stages); acc is written, not added to.
// While a stage's first step is multiplied its second is read, and W's loads of the stage
// after next go out, into the slot that was read a stage ago; then the next stage has landed (the wave's loads before the barrier, everyone's after it) and this
// one has been read by all: A's loads of the stage after next go out while the second step is multiplied and the next stage's first is read. After the last
// stage nothing is copied, and what is read then is multiplied by nobody.
// STORES: how many stores to memory the wave has issued since begin_stages, at least, if `stored`: loads and stores are counted together as they
// were issued, and a wait that names the stores lets them go on while the first stages are multiplied.
template <int W_STEP, int WM, int A_TURNS, int STORES, typename CopyA, typename CopyW, typename LastComes>
__device__ __attribute__((always_inline)) inline void multiply_stages(floatx4 (&acc)[kWaveTilesN][WM], int first, int stages, bool stored, unsigned a_step0,
                                                                      unsigned a_step1, unsigned w_step0, unsigned w_step1, const CopyA& copy_a,
                                                                      const CopyW& copy_w, const LastComes& last_comes) {
    constexpr std::make_integer_sequence<int, WM> row_tiles{};
    constexpr int kStage = A_TURNS + kWTurns, kMostCounted = 63;
    constexpr int kStageAndStores = kStage + STORES < kMostCounted ? kStage + STORES : kMostCounted;
    constexpr int kTurnsAndStores = kWTurns + STORES < kMostCounted ? kWTurns + STORES : kMostCounted;
    TiledOperands<WM> even, odd;      // of a stage's first and second k step
#pragma unroll
    for (int nt = 0; nt < kWaveTilesN; ++nt)
#pragma unroll
        for (int mt = 0; mt < WM; ++mt) {
            acc[nt][mt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
            asm volatile("" : "+v"(acc[nt][mt]));      // once and here, while the loads are on their way: left to itself the compiler does it on every way to the loops
        }
    // The first stage's loads of this wave have landed when only what was issued after them is on its way.
    if (first + 1 == stages) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if (stored) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(kStageAndStores) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" :: "n"(kStage) : "memory");
    __builtin_amdgcn_s_barrier();
    read_operands<W_STEP, WM, 0>(even, a_step0, w_step0, std::make_integer_sequence<int, kWaveTilesN + WM>{});
    operands_arrived<-1>(even);
    unsigned a_now = 0, w_now = 0, w_next = 1, w_after = 2;        // slots
    // MORE: there is a stage after next. `wait`: how much of what was issued last may be on its way when the next stage has landed. Operands on their way never pass from one block to another (the compiler may copy a value there, and does
    // not know that it has not arrived): no branch stands in a stage, and a stage ends when the next one's first operands have arrived.
    auto multiply_stage = [&](int stage, auto more, auto wait) __attribute__((always_inline)) {
        constexpr bool MORE = decltype(more)::value;
        products<W_STEP, WM, 1>(acc, even, odd, a_step1 + a_now * kSlotBytes, w_step1 + w_now * kSlotBytes, [&](auto place) __attribute__((always_inline)) {
            constexpr int kPlace = decltype(place)::value, kApart = 2 * WM / kWTurns;
            if constexpr (MORE && kPlace % kApart == 0 && kPlace / kApart < kWTurns) copy_w(kPlace / kApart, stage + 2, w_after);
        }, row_tiles);
        operands_arrived<decltype(wait)::value>(odd);
        __builtin_amdgcn_s_barrier();
        products<W_STEP, WM, 0>(acc, odd, even, a_step0 + (1 - a_now) * kSlotBytes, w_step0 + w_next * kSlotBytes, [&](auto place) __attribute__((always_inline)) {
            constexpr int kPlace = decltype(place)::value;
            if constexpr (MORE && kPlace % 2 == 0 && kPlace / 2 < A_TURNS) copy_a(kPlace / 2, stage + 2, a_now);
        }, row_tiles);
        operands_arrived<-1>(even);
        a_now = 1 - a_now;
        const unsigned w = w_now;
        w_now = w_next, w_next = w_after, w_after = w;
    };
    int stage = first;
    if (STORES > 0 && stored && stage + 2 < stages) {
        if (stage + 3 == stages) last_comes();
        multiply_stage(stage++, std::true_type{}, std::integral_constant<int, kTurnsAndStores>{});
    }
#pragma clang loop unroll(disable)
    for (; stage + 2 < stages; ++stage) {
        if (stage + 3 == stages) last_comes();
        multiply_stage(stage, std::true_type{}, std::integral_constant<int, kWTurns>{});
    }
#pragma clang loop unroll(disable)
    for (; stage < stages; ++stage) multiply_stage(stage, std::false_type{}, std::integral_constant<int, 0>{});
    // No load is on its way into LDS now and no read into registers; the last products must have written their results before these are read (the
    // compiler does not know that the asm statements are products).
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
}

// Every wave's reads and writes of the slots before this are done: the slots may hold something else after it.
__device__ __attribute__((always_inline)) inline void workgroup_meets() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// A tile's results of 128 columns in bfloat16, 32 of them a wave's, go through the last slot of W, so that they leave as rows of 64 bytes (a lane has 4
// or 8 bytes of a row, which would touch every line of memory 8 to 32 times: 9728 columns of 1280 rows, reduction 896: 34 -> 30 us). A wave has 64 rows
// of 64 bytes there, for itself: nobody waits for another wave, and the next tile's loads into the other slots are on their way meanwhile. By asm: the
// compiler, which does not know which slots those fill, would wait for them. A row's 16-byte chunks lie at places exchanged by (row / 4): 16 rows' words meet
// no bank twice.
constexpr int kResultColumns = 128;      // of a tile
constexpr int kResultRows = 64;          // of a wave at a time, 16 a store
constexpr int kResultBytes = 64;         // of a wave's row
// The kernels exchange a row's chunks in the LDS address itself, whose lower bits must be the place in the row's alone wherever the compiler puts the slots.
constexpr int kSlotsAlign = 128;
static_assert(kSlotsAlign % kResultBytes == 0 && kSlotBytes % kResultBytes == 0, "a wave's rows of results begin at multiples of their length");
template <int OFFSET> __device__ __attribute__((always_inline)) inline void put_result(unsigned address, unsigned word) {
    asm volatile("ds_write_b32 %0, %1 offset:%2" ::"v"(address), "v"(word), "n"(OFFSET) : "memory");
}
template <int OFFSET> __device__ __attribute__((always_inline)) inline void put_result(unsigned address, uint64_t words) {
    asm volatile("ds_write_b64 %0, %1 offset:%2" ::"v"(address), "v"(words), "n"(OFFSET) : "memory");
}
// The wave's rows 16 i + lane / 4, chunk lane % 4.
__device__ __attribute__((always_inline)) inline void get_results(uintx4 (&piece)[4], unsigned place, int lane) {
    const unsigned at = place + (lane / 4) * kResultBytes + (((lane % 4) ^ (lane / 16)) * 16);
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:1024\n\tds_read_b128 %2, %4 offset:2048\n\tds_read_b128 %3, %4 offset:3072\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(piece[0]), "=&v"(piece[1]), "=&v"(piece[2]), "=&v"(piece[3]) : "v"(at) : "memory");
}

}  // namespace mll
