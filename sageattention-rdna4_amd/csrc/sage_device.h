// Device helpers shared by the prologue and the main loop (gfx950 / CDNA4, wave64).
//
// Numerics rules that every quantizer in this library follows, because the quantized tensors must
// be bit-exact with the reference scheme:
//   * fp32 division is correctly rounded (`__fdiv_rn`); the library is never built with fast-math;
//   * rounding to an integer is round-half-to-even, of values clamped to its range (i8x4);
//   * fp32 -> e4m3 goes through v_cvt_pk_fp8_f32 (OCP e4m3fn, round-to-nearest-even on gfx950);
//   * no fused multiply-add is formed where the scheme has two roundings: every such expression has
//     no addition (a*b*c), so contraction cannot apply.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace sage {

typedef uint8_t u8;
typedef uint32_t u32;
typedef uint64_t u64;
typedef _Float16 f16;
typedef __bf16 bf16;

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int HD = 128;          // the largest head_dim served (64 is the other)
constexpr int NPAD = 64;         // N_pad granule
constexpr float P_SCALE = 448.0f;
constexpr float I8_MAX = 127.0f;
constexpr float SCALE_FLOOR = 1e-12f;
constexpr float LOG2E_F = 1.4426950408889634f;

// 16-bit element widen. bf16 -> fp32 and fp16 -> fp32 are exact.
__device__ __forceinline__ float widen(f16 x) { return (float)x; }
__device__ __forceinline__ float widen(bf16 x) { return (float)x; }

// Unpack 8 16-bit elements held in a 16-byte vector.
template <typename T>
__device__ __forceinline__ void unpack8(const u32x4 w, float* out) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t x = w[i];
    const uint16_t lo = (uint16_t)(x & 0xffffu), hi = (uint16_t)(x >> 16);
    T a, b;
    __builtin_memcpy(&a, &lo, 2);
    __builtin_memcpy(&b, &hi, 2);
    out[2 * i] = widen(a);
    out[2 * i + 1] = widen(b);
  }
}

// Four fp32 -> four e4m3 bytes, memory order a, b, c, d.
__device__ __forceinline__ uint32_t fp8x4(float a, float b, float c, float d) {
  // The first convert writes the low half-word and keeps the high half of its "old" operand,
  // which the second convert overwrites, so any value does: passing a's own bits lets the
  // convert write over a's register instead of a zeroed copy.
  int r = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, __float_as_int(a), false);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(c, d, r, true);
}

// Four fp32, each rounded half to even and clamped to [-128, 127], as four int8 bytes (memory order
// a, b, c, d). Adding 1.5 * 2^23 rounds the clamped value to an integer in the low mantissa bits,
// whose low byte is the two's complement byte: per value a clamp and an add (about 4.3 and 2.3
// cycles), where rounding, clamping, converting and masking take 19 cycles with their packing.
__device__ __forceinline__ uint32_t i8x4(float a, float b, float c, float d) {
  auto bits = [](float x) {
    return __float_as_uint(__builtin_amdgcn_fmed3f(x, -128.0f, 127.0f) + 12582912.0f);
  };
  // v_perm_b32: selector bytes 0-3 take the second operand's bytes, 4-7 the first's, 12 is zero
  return __builtin_amdgcn_perm(bits(b), bits(a), 0x0c0c0400u) |
         __builtin_amdgcn_perm(bits(d), bits(c), 0x04000c0cu);
}

// RN(x / s) from y = RN(1 / s), in three operations instead of a full division: q = RN(x*y) is
// within an ulp of x/s, e = RN(q*s - x) is then exact (one fma), and RN(q - e*y) is the correctly
// rounded quotient (Markstein's theorem for round-to-nearest with a correctly rounded reciprocal).
// The bits equal __fdiv_rn(x, s) for normal quotients; signed zeros pass through (-0 / s = -0).
// The quantizers call it with one reciprocal per row (or a constant divisor), so a row of D
// quotients costs one full division.
__device__ __forceinline__ float div_by(float x, float s, float y) {
  const float q = x * y;
  const float e = __builtin_fmaf(q, s, -x);
  return __builtin_fmaf(-e, y, q);
}
constexpr float RCP_P_SCALE = 1.0f / 448.0f;   // RN(1/448)
constexpr float RCP_I8_MAX = 1.0f / 127.0f;    // RN(1/127)

// One DPP lane move within each 16-lane row (ctrl: quad_perm / row_mirror / row_half_mirror).
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
// Max over the lanes of each 16-lane row, as DPP moves folded into v_max_f32: xor 1 and xor 2
// (quad_perm), then the mirrored lane of the 8-lane half-row (the other quad) and of the 16-lane
// row (the other half).
__device__ __forceinline__ float max_row16(float x) {
  x = fmaxf(x, dpp_mov<0xB1>(x));    // quad_perm [1,0,3,2]
  x = fmaxf(x, dpp_mov<0x4E>(x));    // quad_perm [2,3,0,1]
  x = fmaxf(x, dpp_mov<0x141>(x));   // row_half_mirror
  x = fmaxf(x, dpp_mov<0x140>(x));   // row_mirror
  return x;
}

// max(m, |a|, |b|) in one instruction (a plain fmaxf of inputs the compiler cannot prove quiet costs
// a canonicalizing max per input). Quiet NaNs are ignored, as by fmaxf; for a signalling one the
// result is a NaN, and the maximum before it is lost with the next pair.
__device__ __forceinline__ float max3abs(float m, float a, float b) {
  float r;
  asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b));
  return r;
}
// The same, but NaN if one of them is a NaN of either kind.
__device__ __forceinline__ float maximum3abs(float m, float a, float b) {
  float r;
  asm("v_maximum3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b));
  return r;
}
template <bool QUIET>
__device__ __forceinline__ float absmax8(const float* f) {
  float m = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; e += 2)
    m = QUIET ? max3abs(m, f[e], f[e + 1]) : maximum3abs(m, f[e], f[e + 1]);
  return m;
}
// Over the values that are no NaN: each is quieted first, and v_max_f32 ignores quiet NaNs.
__device__ __forceinline__ float absmax8_no_nan(const float* f) {
  float m = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e)
    asm("v_max_f32 %0, %1, %1\n\tv_max_f32 %0, %2, |%0|" : "=&v"(m) : "v"(f[e]), "v"(m));
  return m;
}
// Non-negative floats order as their bits.
__device__ __forceinline__ u32 umax(u32 a, u32 b) { return a > b ? a : b; }

template <int CTRL>
__device__ __forceinline__ u32 dpp_u32(u32 v) {
  return (u32)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
}

// Calls f(integral_constant<int, i>) for i = I .. N-1, unrolled (compile-time lane selectors).
template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

// Eight values per lane, reduced over the aligned group of CG = 8 or 16 lanes that share the
// rows: lane l of the group returns the group's maximum of value l & 7. Three exchange steps, each
// of which hands over half of the values that are left (lanes 7 - l, l ^ 1, l ^ 2; and l ^ 8 for
// 16 lanes): 22 operations, where a full reduction of each value takes 8 x 4 moves and maxima.
template <int CG>
__device__ __forceinline__ float row_max(const float (&m)[8], int lane) {
  const bool b0 = lane & 1, b1 = lane & 2, b2 = lane & 4;
  u32 a[4], c[2];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const u32 lo = __float_as_uint(m[j]), hi = __float_as_uint(m[j + 4]);
    a[j] = umax(b2 ? hi : lo, dpp_u32<0x141>(b2 ? lo : hi));       // row_half_mirror
  }
#pragma unroll
  for (int j = 0; j < 2; ++j)                                       // rows 2j, 2j + 1 (by b0)
    c[j] = umax(b0 ? a[2 * j + 1] : a[2 * j], dpp_u32<0xB1>(b0 ? a[2 * j] : a[2 * j + 1]));
  u32 r = umax(b1 ? c[1] : c[0], dpp_u32<0x4E>(b1 ? c[0] : c[1]));
  if (CG == 16) r = umax(r, dpp_u32<0x128>(r));                     // row_ror:8
  return __uint_as_float(r);
}

// The same for four values per lane over a group of 8 lanes: lane l returns the maximum of value
// l & 3 (lanes l ^ 1 and l ^ 2 exchange, then both quads).
__device__ __forceinline__ float row_max(const float (&m)[4], int lane) {
  const bool b0 = lane & 1, b1 = lane & 2;
  u32 c[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const u32 lo = __float_as_uint(m[2 * j]), hi = __float_as_uint(m[2 * j + 1]);
    c[j] = umax(b0 ? hi : lo, dpp_u32<0xB1>(b0 ? lo : hi));
  }
  const u32 r = umax(b1 ? c[1] : c[0], dpp_u32<0x4E>(b1 ? c[0] : c[1]));
  // lane l ^ 4: row_shl:4 for the even quads, row_shr:4 for the odd ones
  u32 o = (u32)__builtin_amdgcn_update_dpp(0, (int)r, 0x104, 0xF, 0x5, false);
  o = (u32)__builtin_amdgcn_update_dpp((int)o, (int)r, 0x114, 0xF, 0xA, false);
  return __uint_as_float(umax(r, o));
}

// The row absmax of the rows f[0 .. NR-1] (8 columns of each per lane), over the group of CG lanes
// that share them, NaNs ignored: lane l of the group returns row l % NR's.
// QUIET: the values hold no signalling NaN (the result of an operation or of an fp16 -> fp32
// conversion; a bf16 widened by a shift may be one). Otherwise the maxima keep NaNs: one in any
// lane's columns is the largest of the row's bit patterns, so it shows in the result, and a wave
// that holds one (all its lanes then, the exchange moves data between lanes) works its maxima out
// again without them.
template <int CG, bool QUIET, int NR>
__device__ __forceinline__ float row_absmax(const float (&f)[NR][8], int lane) {
  float m[NR];
  auto reduce = [&]() {
    if constexpr (NR == 8)
      return row_max<CG>(m, lane);
    else
      return row_max(m, lane);
  };
#pragma unroll
  for (int i = 0; i < NR; ++i) m[i] = absmax8<QUIET>(f[i]);
  float r = reduce();
  if (!QUIET && __builtin_expect(__builtin_amdgcn_ballot_w64(__float_as_uint(r) > 0x7f800000u) != 0, 0)) {
#pragma unroll
    for (int i = 0; i < NR; ++i) m[i] = absmax8_no_nan(f[i]);
    r = reduce();
  }
  return r;
}

// Every lane of a CG-lane group receives lane I (0 .. 7) of its own group.
template <int CG, int I>
__device__ __forceinline__ float group_bcast(float v) {
  int r = __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + I, 0xF, 0xF, true);
  if (CG == 8)   // two groups per 16-lane row: the second one's banks take its own lane
    r = __builtin_amdgcn_update_dpp(r, __float_as_int(v), 0x158 + I, 0xF, 0xC, false);
  return __int_as_float(r);
}

}  // namespace sage
