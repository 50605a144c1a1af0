// Shared device helpers for the gfx950 kernels: element types, wave reductions, error reporting.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>
#include <cstdio>
#include <string>

namespace mll {

constexpr int kWave = 64;  // CDNA wavefront width

// Element type tags shared with the Python bindings.
enum DType : int { kF32 = 0, kBF16 = 1 };

// bfloat16 as raw bits: widening is a shift, narrowing rounds to nearest even.
struct bf16 {
    uint16_t bits;
};

__host__ __device__ inline float to_float(float value) { return value; }
__host__ __device__ inline float to_float(bf16 value) {
    union { uint32_t u; float f; } caster;
    caster.u = static_cast<uint32_t>(value.bits) << 16;
    return caster.f;
}

// A rotation by (cos, sin) with its roundings spelled out (one product rounded, then one fused multiply-add), so
// that every kernel that rotates gives the same bits whatever the compiler would contract.
__device__ inline float rotate_first(float x1, float x2, float c, float s) { return fmaf(x1, c, -(x2 * s)); }
__device__ inline float rotate_second(float x1, float x2, float c, float s) { return fmaf(x1, s, x2 * c); }

// Waits until every load this wave has issued has arrived. The compiler waits by itself for loads into registers;
// loads from memory straight into LDS return nothing to wait for, so whoever reads that LDS calls this first (and
// then a barrier, if another wave's loads are read).
__device__ inline void wait_for_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// op over the two lanes {l, l ^ 32}, or {l, l ^ 16}, of a wave, both of which get the result: an exchange on the vector unit
// (v_permlane32_swap, v_permlane16_swap of gfx950). op must be commutative. (The elements of the builtins' result are copied to scalars before they
// are reinterpreted: a reinterpretation of the element expression itself reads element 0 twice with this compiler.)
template <typename Op>
__device__ inline float reduce_lanes_32_apart(float value, Op op) {
    const unsigned bits = __builtin_bit_cast(unsigned, value);
    const auto halves = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
    const unsigned low = halves[0], high = halves[1];
    return op(__builtin_bit_cast(float, low), __builtin_bit_cast(float, high));
}
template <typename Op>
__device__ inline float reduce_rows_apart(float value, Op op) {
    const unsigned bits = __builtin_bit_cast(unsigned, value);
    const auto rows = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
    const unsigned even = rows[0], odd = rows[1];
    return op(__builtin_bit_cast(float, even), __builtin_bit_cast(float, odd));
}

// op over the four lanes {l, l ^ 16, l ^ 32, l ^ 48} of a wave, every one of which gets the result, instead of four trips through LDS.
template <typename Op>
__device__ inline float reduce_lanes_16_apart(float value, Op op) { return reduce_lanes_32_apart(reduce_rows_apart(value, op), op); }
__device__ inline float max_lanes_16_apart(float value) {
    return reduce_lanes_16_apart(value, [](float a, float b) { return fmaxf(a, b); });
}
__device__ inline float sum_lanes_16_apart(float value) {
    return reduce_lanes_16_apart(value, [](float a, float b) { return a + b; });
}

// BYTES (4 or 16) a lane from `base` (the same for the whole wave) and the lane's `offset` in bytes, straight into LDS at `place` and what follows it.
// Buffer loads: a global load into LDS is encoded as a flat one, and while one is under way the compiler waits for every load and for every read
// from LDS, not for those it needs. Nothing is checked: the caller's offsets lie within what `base` holds. (A macro: as a function's arguments
// the places lose their address space.)
constexpr int kBufferFlags = 0x00027000;    // a raw buffer of 32-bit words
#define MLL_LOAD_INTO_LDS(BYTES, base, offset, place)                                                                    \
    __builtin_amdgcn_raw_ptr_buffer_load_lds(                                                                            \
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, 0x7fffffff, kBufferFlags), place, BYTES, offset, 0, 0, 0)

template <typename T> __host__ __device__ inline T from_float(float value);
template <> __host__ __device__ inline float from_float<float>(float value) { return value; }
template <> __host__ __device__ inline bf16 from_float<bf16>(float value) {
    bf16 out;
#if defined(__HIP_DEVICE_COMPILE__)
    // Round to nearest even in one instruction (v_cvt_pk_bf16_f32 of gfx950); a NaN stays a NaN.
    out.bits = __builtin_bit_cast(uint16_t, static_cast<__bf16>(value));
#else
    union { uint32_t u; float f; } caster;
    caster.f = value;
    if ((caster.u & 0x7fffffffu) > 0x7f800000u) {  // NaN stays NaN
        out.bits = static_cast<uint16_t>((caster.u >> 16) | 0x0040u);
        return out;
    }
    const uint32_t rounding = 0x7fffu + ((caster.u >> 16) & 1u);
    out.bits = static_cast<uint16_t>((caster.u + rounding) >> 16);
#endif
    return out;
}

// The activations a kernel may be asked for by number: 0 SiLU, 1 the exact gelu, 2 the tanh form of gelu.
constexpr int kActSilu = 0, kActGeluErf = 1, kActGeluTanh = 2;
__device__ inline float activate(float z, int act) {
    if (act == kActGeluErf) return 0.5f * z * (1.0f + erff(z * 0.70710678118654752440f));
    if (act == kActGeluTanh) return 0.5f * z * (1.0f + tanhf(0.79788456080286535588f * (z + 0.044715f * z * z * z)));
    return z / (1.0f + expf(-z));
}

// The fourth kind is for a gated pair alone: both inputs clamped, a sigmoid of steeper argument, one added to the second.
constexpr int kActClampedGlu = 3;
__device__ inline float gated_value(float g, float u, int act, float limit, float slope) {
    if (act != kActClampedGlu) return activate(g, act) * u;
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return g / (1.0f + expf(-slope * g)) * (u + 1.0f);
}

// n / (1 + exp(-t)) to about an ulp, in fewer instructions than expf and a division: exp by the hardware's exp2 with what the product with
// log2(e) loses put back, and a reciprocal refined once, for t up to 87 in size, where neither leaves the numbers. Beyond 87 the quotient is n; below -87,
// where it is n exp(t), it goes on to nothing by a factor of its own, which is one otherwise: n has no bound, so a quotient that stayed at
// exp(-87) would leave 5.6 of the lowest bfloat16. (The factor is free in rows that wait for memory; it holds up tiles of
// gated products, 413 -> 419 us and 38.4 -> 39.9, of which a look at a wave's gates that leaves it out gave back a half, and made experts' tiles slower.)
__device__ inline float over_one_plus_exp(float n, float t) {
    constexpr float kLog2e = 1.44269502162933349609f, kLog2eRest = 1.92596299112661746887e-8f, kLn2 = 0.69314718055994530942f;
    constexpr float k87Log2e = 125.514473f;     // not less than 87 kLog2e
    const float within = __builtin_amdgcn_fmed3f(t, -87.0f, 87.0f);
    const float high = -within * kLog2e, low = fmaf(-within, kLog2eRest, fmaf(-within, kLog2e, -high));
    const float power = __builtin_amdgcn_exp2f(high), d = 1.0f + fmaf(power, low * kLn2, power);
    const float r = __builtin_amdgcn_rcpf(d);
    return n * fmaf(fmaf(-d, r, 1.0f), r, r) * __builtin_amdgcn_exp2f(fminf(fmaf(t, kLog2e, k87Log2e), 0.0f));
}

// The gate of a gated product's epilogue: silu(z), or the tanh form of gelu, which is z sigmoid(2 sqrt(2 / pi) (z + 0.044715 z^3)).
template <bool GELU>
__device__ inline float gate_fast(float z) {
    return over_one_plus_exp(z, GELU ? 1.59576912160573071176f * (z + 0.044715f * z * z * z) : z);
}

// gated_value in the epilogue of a product whose result is rounded to bfloat16.
__device__ inline float gated_value_fast(float g, float u, int act, float limit, float slope) {
    if (act == kActSilu) return gate_fast<false>(g) * u;
    if (act != kActClampedGlu) return activate(g, act) * u;
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return over_one_plus_exp(g, slope * g) * (u + 1.0f);
}

// cap * tanh(value / cap) as cap - 2 cap / (1 + exp(2 value / cap)), with the fast exponential and reciprocal (absolute
// error about 1e-7 of cap).
__device__ inline float softcap_fast(float value, float cap, float inverse_cap) {
    return fmaf(-2.0f * cap, __builtin_amdgcn_rcpf(1.0f + __expf(2.0f * value * inverse_cap)), cap);
}

// `value` of lane l ^ DISTANCE, for every lane (of a whole wave), DISTANCE within a row of 16: by DPP, without a way through LDS.
template <int CONTROL>
__device__ inline int dpp(int value) { return __builtin_amdgcn_update_dpp(0, value, CONTROL, 0xf, 0xf, false); }
template <int DISTANCE>
__device__ inline float lane_across(float value) {
    const int bits = __builtin_bit_cast(int, value);
    static_assert(DISTANCE == 1 || DISTANCE == 2 || DISTANCE == 4 || DISTANCE == 8, "within a row of 16 lanes");
    constexpr int kEveryFourMirrored = 0x1B, kEveryEightMirrored = 0x141;
    const int there = DISTANCE == 1   ? dpp<0xB1>(bits)      // lanes 1, 0, 3, 2 of every four
                      : DISTANCE == 2 ? dpp<0x4E>(bits)      // lanes 2, 3, 0, 1 of every four
                      : DISTANCE == 4 ? dpp<kEveryFourMirrored>(dpp<kEveryEightMirrored>(bits))
                                      : dpp<0x128>(bits);    // a row turned by eight
    return __builtin_bit_cast(float, there);
}

// op over a wave, every lane of which gets the result: pairs of lanes 32 apart, then 16, 8, 4, 2, 1. Six exchanges in registers: through LDS
// (__shfl_xor) each of them is a trip of its own for the wave, which kernels of few waves wait for.
template <typename Op>
__device__ inline float reduce_wave(float value, Op op) {
    value = reduce_rows_apart(reduce_lanes_32_apart(value, op), op);
    value = op(value, lane_across<8>(value));
    value = op(value, lane_across<4>(value));
    value = op(value, lane_across<2>(value));
    return op(value, lane_across<1>(value));
}

__device__ inline float wave_sum(float value) {
    return reduce_wave(value, [](float a, float b) { return a + b; });
}

__device__ inline float wave_max(float value) {
    return reduce_wave(value, [](float a, float b) { return fmaxf(a, b); });
}

// Sum over a block of up to 1024 threads; every thread gets the total. `scratch` holds 16 floats.
// The order of additions depends only on the block size, never on the data's place in a batch.
__device__ inline float block_sum(float value, float* scratch) {
    const int lane = threadIdx.x % kWave;
    const int wave = threadIdx.x / kWave;
    const int waves = (blockDim.x + kWave - 1) / kWave;
    value = wave_sum(value);
    __syncthreads();  // scratch may still be read from an earlier call
    if (lane == 0) scratch[wave] = value;
    __syncthreads();
    float total = 0.0f;
    if (waves <= 4) {
        for (int index = 0; index < waves; ++index) total += scratch[index];
        return total;
    }
    float sums[16];     // all read at once: in a loop of unknown length every addition waits for its own read
#pragma unroll
    for (int index = 0; index < 16; ++index) sums[index] = scratch[index];
#pragma unroll
    for (int index = 0; index < 16; ++index) total = index < waves ? total + sums[index] : total;
    return total;
}

// Host-side error text, one per thread, read through mll_last_error().
void set_error(const std::string& text);
int fail(const std::string& text);

inline int check_launch(const char* what) {
    const hipError_t status = hipGetLastError();
    if (status != hipSuccess) return fail(std::string(what) + ": " + hipGetErrorString(status));
    return 0;
}

}  // namespace mll

#define MLL_REQUIRE(condition, text)                         \
    do {                                                     \
        if (!(condition)) return ::mll::fail(text);          \
    } while (0)
