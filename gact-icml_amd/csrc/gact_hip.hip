// GACT saved-activation compression for MI355X (gfx950): per-group min/max, scale, stochastic
// rounding, bit packing, and the inverse, as hand-written HIP kernels behind a C ABI.
//
// Quantize: a DPP row of 16 lanes owns one "super-group", the 8/bits consecutive groups of 256
// elements whose codes share output bytes.  Inside a group lane i of the row owns 16 columns in chunks
// of one 16-byte load each - float: 4 chunks of 4 columns at 4i + 64m, half: 2 chunks of 8 columns at
// 8i + 128m - so every load instruction of a row reads 256 contiguous bytes.  Per-group reductions are
// four row_ror DPP steps that never leave the row, and - because the reference packs the SAME column of
// 8/bits consecutive groups into one byte - the lane that owns a column owns every code of that byte:
// packing needs no cross-lane traffic at all.  One Philox block feeds 8 consecutive columns of two consecutive
// groups - a half chunk, or the float chunks of a pair of neighbouring lanes (which swap the words they need) -
// and, mirrored, the 8 columns half a group further on, which the same lane owns.
//
// Dequantize has no reduction, so a unit of 4 or 8 consecutive groups goes to a whole wave (float: lane l owns
// columns 4l .. 4l+3) or half a wave (half: 8l .. 8l+7): one 16-byte store per lane and group, every store
// instruction writing whole groups contiguously.  At 1, 2 and 4 bit the possible values of a unit (2^bits per
// group) are tabulated once across its lanes and fetched with ds_bpermute.  The stores are buffer stores whose
// cache policy the kernel chooses (nontemporal, written through at system scope).
//
// Element types: float and half as in the reference; bfloat16 (an addition) is quantized as the float
// values it holds, in the half layout.
//
// Workgroups are dealt to the 8 XCDs round-robin; xcd_tile() reorders the tiles so that each XCD's L2
// streams runs of consecutive tiles.
//
// Floating-point contract: this file is compiled with -ffp-contract=off, so every operation below is
// the IEEE operation it spells; the fused multiply-adds of the path are written __builtin_fmaf.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>
#include <queue>
#include <type_traits>
#include <utility>
#include <vector>

#include "gact_hip.h"

typedef _Float16 f16;
typedef __bf16 bf16;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

#define GROUP 256
#define ROW_GROUPS 8 /* groups of a dequantize unit and of a minimax row */

// ------------------------------------------------------------------------------------------------
// DPP row reductions (16 lanes).  Rotating by 8, 4, 2, 1 leaves the row-wide result in every lane.
// ------------------------------------------------------------------------------------------------
// Row-wide min of lo and max of hi, left in every lane of the row, with the rotated operand folded into the
// min / max instruction itself (VOP2 DPP).  lo and hi must not be NaN (they are per-lane results that
// started from a finite or infinite initial value).  A DPP operand has to be written two wait states before
// it is read, five after a vector write of EXEC; the compiler's hazard pass does not look inside an asm
// block, so the block keeps those distances itself, at both ends as well.
#define GACT_DPP_STEP(MIN, MAX, N)                                         \
  MIN " %0, %0, %0 row_ror:" #N " row_mask:0xf bank_mask:0xf\n\t"          \
  MAX " %1, %1, %1 row_ror:" #N " row_mask:0xf bank_mask:0xf\n\t"
#define GACT_DPP_ALL(MIN, MAX)                                             \
  "s_nop 4\n\t" GACT_DPP_STEP(MIN, MAX, 8) "s_nop 0\n\t" GACT_DPP_STEP(MIN, MAX, 4) "s_nop 0\n\t" \
  GACT_DPP_STEP(MIN, MAX, 2) "s_nop 0\n\t" GACT_DPP_STEP(MIN, MAX, 1) "s_nop 1"
__device__ __forceinline__ void row_all_minmax(float& lo, float& hi) {
  asm(GACT_DPP_ALL("v_min_f32_dpp", "v_max_f32_dpp") : "+v"(lo), "+v"(hi));
}
__device__ __forceinline__ void row_all_minmax(f16& lo, f16& hi) {
  asm(GACT_DPP_ALL("v_min_f16_dpp", "v_max_f16_dpp") : "+v"(lo), "+v"(hi));
}
// The same over each half of the row (8 lanes): the half mirrored, then the lanes of a quad exchanged twice.
#define GACT_DPP_HALF_STEP(MIN, MAX, CTRL)                                 \
  MIN " %0, %0, %0 " CTRL " row_mask:0xf bank_mask:0xf\n\t"                \
  MAX " %1, %1, %1 " CTRL " row_mask:0xf bank_mask:0xf\n\t"
__device__ __forceinline__ void half_row_all_minmax(f16& lo, f16& hi) {
  asm("s_nop 4\n\t" GACT_DPP_HALF_STEP("v_min_f16_dpp", "v_max_f16_dpp", "row_half_mirror") "s_nop 0\n\t"
      GACT_DPP_HALF_STEP("v_min_f16_dpp", "v_max_f16_dpp", "quad_perm:[1,0,3,2]") "s_nop 0\n\t"
      GACT_DPP_HALF_STEP("v_min_f16_dpp", "v_max_f16_dpp", "quad_perm:[2,3,0,1]") "s_nop 1"
      : "+v"(lo), "+v"(hi));
}
// ------------------------------------------------------------------------------------------------
// Philox4x32.  The key schedule only depends on the seed, so it stays on the scalar unit; each
// round is two 32x32->64 multiplies and two three-input XORs (v_bitop3_b32, truth table 0x96).
// Ten rounds for the reference's stream (cuRAND's generator); seven for the fast stream - the fewest
// for which the generator's authors report that it passes BigCrush (Salmon et al., SC'11, table 2).
// ------------------------------------------------------------------------------------------------
#define PHILOX_REF_ROUNDS 10
#define PHILOX_FAST_ROUNDS 7
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
  return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}
template <int ROUNDS>
__device__ __forceinline__ void philox4x32(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0,
                                           uint32_t k1, uint32_t (&out)[4]) {
#pragma unroll
  for (int r = 0; r < ROUNDS; r++) {
    uint64_t p0 = (uint64_t)0xD2511F53u * c0;
    uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
    uint32_t n0 = xor3((uint32_t)(p1 >> 32), c1, k0);
    uint32_t n2 = xor3((uint32_t)(p0 >> 32), c3, k1);
    c1 = (uint32_t)p1;
    c3 = (uint32_t)p0;
    c0 = n0;
    c2 = n2;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  out[0] = c0; out[1] = c1; out[2] = c2; out[3] = c3;
}

// cuRAND's uniform map: float(x) * 2^-32 + 2^-33, in (0, 1].  The product is exact, so the fused form
// rounds once exactly like the separate multiply and add.
__device__ __forceinline__ float curand_uniform_map(uint32_t x) {
  return __builtin_fmaf((float)x, 0x1p-32f, 0x1p-33f);
}
// The same with the addend held in a register by the caller (uniform_addend(), once per kernel): left to itself the
// compiler builds the addend anew in front of every multiply-add, one instruction in nine of a kernel that is bound by
// its instruction count.
__device__ __forceinline__ float uniform_addend() {
  float c;
  asm volatile("v_mov_b32 %0, 0x2f000000" : "=v"(c));
  return c;
}
__device__ __forceinline__ float curand_uniform_map(uint32_t x, float addend) {
  float u;
  asm("v_fmamk_f32 %0, %1, 0x2f800000, %2" : "=v"(u) : "v"((float)x), "v"(addend));
  return u;
}
// 8-bit centred noise of the fast stream from byte B of a Philox word: (2h - 255) / 512 = (h + 0.5) / 256 - 1/2,
// exact in float (v_cvt_f32_ubyteB and one fma).
template <int B>
__device__ __forceinline__ float fast_centred_map(uint32_t w) {
  return __builtin_fmaf((float)((w >> (8 * B)) & 0xffu), 0x1p-8f, -255.0f / 512.0f);
}
__device__ __forceinline__ float fast_centred_map(uint32_t w, int b) {
  return (b & 2) ? ((b & 1) ? fast_centred_map<3>(w) : fast_centred_map<2>(w))
                 : ((b & 1) ? fast_centred_map<1>(w) : fast_centred_map<0>(w));
}

// Activations and codes are touched exactly once per kernel: load and store them with the streaming
// (nontemporal) hint so that they do not displace each other in L2 / Infinity Cache.
#ifndef GACT_STREAMING
#define GACT_STREAMING 1
#endif
template <typename V>
__device__ __forceinline__ V stream_load(const V* p) {
#if GACT_STREAMING
  return __builtin_nontemporal_load(p);
#else
  return *p;
#endif
}
template <typename V>
__device__ __forceinline__ void stream_store(V v, V* p) {
#if GACT_STREAMING
  __builtin_nontemporal_store(v, p);
#else
  *p = v;
#endif
}

// The dequantized tensor leaves through buffer stores whose cache policy the kernel chooses: nontemporal, and for
// every type and width but float at 1 bit also written through at system scope (sc0 sc1 nt).  The plain nontemporal
// store the compiler emits for __builtin_nontemporal_store lets the L2 collect the lines first, which costs a float
// write stream up to 6 % (dequantize alone, buffers cold in every cache: 4 bit 103 M elements 75.5 -> 71.3 us, 256 M
// 183.4 -> 172.4; 8 bit 1 %; 2 bit equal; 17 M elements 1-3 % at every width; half 0-2 %), while float at 1 bit,
// whose stream has the smallest share of reads, loses 3-4 % by it from 50 M elements on (66.3 -> 68.5 us at 103 M)
// and keeps the plain nontemporal store on large tensors.
// A window is a buffer resource over the bytes from a wave-uniform base to the end of the tensor (at most 4 GB of
// them: offsets inside a window are 32 bit), so a store past the end of the tensor is dropped by the hardware.
#define GACT_STORE_NT 2          /* cache-policy bits of a buffer store: 1 sc0, 2 nt, 16 sc1 */
#define GACT_STORE_NT_SYSTEM 19
struct OutWindow {
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ OutWindow(void* base, int64_t bytes) {
    const uint32_t n = bytes <= 0 ? 0u : bytes > 0xffffffffLL ? 0xffffffffu : (uint32_t)bytes;
    rsrc = __builtin_amdgcn_make_buffer_rsrc(base, 0, (int)n, 0x00020000);
  }
  template <int POLICY>
  __device__ __forceinline__ void store16(u32x4 v, uint32_t byte_offset) const {
    __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, (int)byte_offset, 0, POLICY);
  }
};
__device__ __forceinline__ int64_t wave_first(int64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// round-to-nearest-even integer of z clamped below at 0: rint(max(z, 0)) of the reference's
// __float2int_rn(fmax(z, 0)).  v_cvt_u32_f32 clamps negative inputs and NaN to 0, so no separate max is
// needed.  From 2^31 on the reference's signed conversion saturates to 0x7fffffff: SAT = true reproduces
// that (only min / max handed in by the caller can push a float code that far; with the group's own min
// and max a code stays below 2^bits + 1), SAT = false leaves it out.
template <bool SAT>
__device__ __forceinline__ uint32_t rint_clamp0(float z) {
  float r = __builtin_rintf(z);
  uint32_t c;
  asm("v_cvt_u32_f32_e32 %0, %1" : "=v"(c) : "v"(r));
  if (SAT) c = c < 0x7fffffffu ? c : 0x7fffffffu;
  return c;
}

// The same code read off the float.  For 0.5 <= y < 2^22, y - 0.5 is exact and adding 1.5 * 2^23 rounds it to
// 1.5 * 2^23 + rint(y - 0.5): in that binade a float's unit in the last place is 1, the constant is even, so
// ties go to even exactly as rint's do, and the integer sits in the low mantissa bits.  For 0 <= y < 0.5 the
// difference lies in [-0.5, 0) (possibly rounded, which cannot take it out of that interval) and the sum rounds
// to the constant itself: code 0, the reference's fmax.  NaN stays NaN with its payload: code 0 only where the
// payload's low byte is 0 - true of every NaN widened from half or bfloat16 and of the NaN arithmetic generates,
// not of any float NaN (the float path takes code_bits_of_any).
// Two additions; the bits above the code (0x4B4...) never reach the low 8 bits a byte keeps of a code shifted
// left by at most 7.  NOT valid for negative y (the callers' y is a sum of non-negative terms: with the group's own
// minimum no element lies below it) and for +inf, whose bits have a zero low byte where the reference's saturated
// conversion has 0xff: the one caller that can meet +inf (a half scale that overflowed) repairs those groups
// afterwards (quantize_supergroup).
__device__ __forceinline__ uint32_t code_bits_of(float y) {
  const float z = y - 0.5f;
  return __builtin_bit_cast(uint32_t, z + 12582912.0f);
}
// The same for any y: y + (2^23 - 0.5) rounds to 2^23 + rint(y - 0.5) in one step, and the median clamps to
// [2^23, 2^23 + 0x3fffff]: everything below 0.5, negative or NaN gives 0, +inf gives low bits of all ones.
__device__ __forceinline__ uint32_t clamp_code_bits(float w) {
  float c;
  asm("v_med3_f32 %0, %1, %2, %3" : "=v"(c) : "v"(w), "v"(8388608.0f), "v"(12582911.0f));
  return __builtin_bit_cast(uint32_t, c);
}
__device__ __forceinline__ uint32_t code_bits_of_any(float y) { return clamp_code_bits(y + 8388607.5f); }
// The fast stream adds a centred draw, so its sum z already is the reference's y - 0.5 and the code is rint(max(z, 0)):
// one addition (z > -0.5 with the group's own minimum, so z + 1.5 * 2^23 rounds to 1.5 * 2^23 + rint(z), -0 included),
// or the clamping form for any z.
__device__ __forceinline__ uint32_t centred_code_bits_of(float z) { return __builtin_bit_cast(uint32_t, z + 12582912.0f); }
__device__ __forceinline__ uint32_t centred_code_bits_of_any(float z) { return clamp_code_bits(z + 8388608.0f); }

// Codes as packed bytes: v_cvt_pk_u8_f32 rounds z to the nearest integer, ties to even, clamps it to [0, 255] (NaN: 0) and puts it into
// a byte of a word - rint(max(z, 0)) of the reference and the packing of four columns in four instructions, where a code read off the
// float's mantissa takes an addition (and a median) of its own, a shift-or into its byte's register and the joining of four registers.
// Fields of one to four bits then join word by word.  It differs from the reference from 256 on, which truncates to the byte: the
// 8-bit code of a half tensor (whose scale, rounded to half, can put the largest element at 256), injected noise and a caller's min and
// max stay with the forms above - and so do half kernels that the registers saved let hold more waves than HBM bears (2 bit from 2^17 groups
// on, batches by batch_packs, deterministic 1 bit in long tensors of groups of 512), and float under the reference stream, which a Philox block per byte bounds: 1 % faster to 4 %
// slower with packed bytes (103 M elements, 2 bit 74.2 -> 76.9 us) where half is 2-4 % faster (134 M, 4 bit 105.5 -> 101.0).
// Quantize alone, before -> after: 4 M elements float 1 bit 5.73 -> 5.45 us, 2 bit 5.40 -> 5.21, bfloat16 4 bit 4.11 -> 4.02; half in groups of 128
// [16384,1024] 4 bit 9.57 -> 9.28; large contiguous tensors are bound by HBM and gain 0-3 %.  A half scale that overflowed to +inf makes
// products of +inf: 255, every bit of the field and above it, as the reference's saturated conversion leaves in the byte.
template <typename T, int BITS, int NOISE, bool GIVEN>
constexpr bool packs_bytes() {
  constexpr bool HALF = std::is_same<T, f16>::value;
  return !GIVEN && NOISE != GACT_NOISE_INJECT && !(HALF && BITS == 8) && (HALF || NOISE != GACT_NOISE_REF);
}
template <int W>
__device__ __forceinline__ void pack_bytes(const float (&z)[W], uint32_t (&w)[W / 4]) {
#pragma unroll
  for (int d = 0; d < W / 4; d++) {
    uint32_t v = 0u;
    v = __builtin_amdgcn_cvt_pk_u8_f32(z[4 * d], 0, v);
    v = __builtin_amdgcn_cvt_pk_u8_f32(z[4 * d + 1], 1, v);
    v = __builtin_amdgcn_cvt_pk_u8_f32(z[4 * d + 2], 2, v);
    w[d] = __builtin_amdgcn_cvt_pk_u8_f32(z[4 * d + 3], 3, v);
  }
}
// Four bytes' codes moved up to their field.  EXACT: a code has at most its field's bits (float and bfloat16: the largest element's sum
// stays within half a step of 2^bits - 1); else one more, which stays within its byte.
template <bool EXACT>
__device__ __forceinline__ uint32_t field_of(uint32_t w, uint32_t shift) {
  return EXACT ? w << shift : (w << shift) & (0x01010101u * ((0xffu << shift) & 0xffu));
}

// Correctly rounded c / s from the correctly rounded reciprocal r = RN(1/s) (Markstein): q = RN(c*r),
// e = c - s*q exactly (one FMA), result RN(q + e*r).  Valid for finite nonzero s with a normal quotient;
// the callers fall back to the division otherwise.
__device__ __forceinline__ float div_by_reciprocal(float c, float s, float r) {
  float q = c * r;
  float e = __builtin_fmaf(-q, s, c);
  return __builtin_fmaf(e, r, q);
}
// s is a scale the quotient c/s (0 <= c <= 255) can be taken through the reciprocal for: finite, and
// far enough from the ends of the exponent range that neither 1/s nor c/s is subnormal or overflows
__device__ __forceinline__ bool reciprocal_safe(float s) {
  float a = __builtin_fabsf(s);
  return a > 0x1p-100f && a < 0x1p100f;
}

// ------------------------------------------------------------------------------------------------
// Per-type pieces.  Store holds the 16 elements of one group a quantize lane owns (float: 4 chunks of 4,
// half and bfloat16: 2 chunks of 8).
// ------------------------------------------------------------------------------------------------
template <typename T> struct Elem;

template <> struct Elem<float> {
  // quantize layout: 4 chunks of 4 columns, 4i + 64m: one 16-byte load per chunk, 256 contiguous
  // bytes per row and load instruction
  static constexpr int kQChunks = 4, kQWidth = 4;
  static constexpr int kDtype = GACT_F32;
  typedef float Stat;   // type min, max and scale are computed and stored in (scale: always; min: as T)
  __device__ static __forceinline__ float stat_of(float x) { return x; }
  __device__ static __forceinline__ float elem_of(float x) { return x; }
  struct Store { float v[4][4]; };
  __device__ static __forceinline__ void load_noise(const float* p, float (&u)[4]) {
    f32x4 a = stream_load(reinterpret_cast<const f32x4*>(p));
    u[0] = a.x; u[1] = a.y; u[2] = a.z; u[3] = a.w;
  }
  __device__ static __forceinline__ void load_chunk(const float* p, Store& st, int k) { load_noise(p, st.v[k]); }
  __device__ static __forceinline__ void set(Store& st, int k, int e, float x) { st.v[k][e] = x; }
  __device__ static __forceinline__ float init_lo() { return 1e30f; }
  __device__ static __forceinline__ float init_hi() { return -1e30f; }
  __device__ static __forceinline__ float from_float(float v) { return v; }
  // min and max of the lane's chunks K0 .. K1 - 1
  template <int K0, int K1>
  __device__ static __forceinline__ void lane_minmax(const Store& st, float& lo_out, float& hi_out) {
    float lo = init_lo(), hi = init_hi();
#pragma unroll
    for (int k = K0; k < K1; k++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        lo = __builtin_fminf(lo, st.v[k][e]);
        hi = __builtin_fmaxf(hi, st.v[k][e]);
      }
    lo_out = lo;
    hi_out = hi;
  }
  // the same, NaN apart: nan says that the lane's elements have to go through lane_minmax instead (see Elem<f16>)
  template <int K0, int K1>
  __device__ static __forceinline__ void lane_ordered(const Store& st, float& lo_out, float& hi_out, bool&) { lane_minmax<K0, K1>(st, lo_out, hi_out); }
  // min and max of the first `there` of G whole groups, in every lane of the row; of the others 0
  template <int G, bool ORDERED = true>
  __device__ static __forceinline__ void groups_minmax(const Store* st, float* lo_out, float* hi_out, int64_t there = G) {
#pragma unroll
    for (int g = 0; g < G; g++) {
      lo_out[g] = hi_out[g] = 0.0f;
      if (g < there) {
        lane_minmax<0, kQChunks>(st[g], lo_out[g], hi_out[g]);
        row_all_minmax(lo_out[g], hi_out[g]);
      }
    }
  }
  __device__ static __forceinline__ void store_codes(uint8_t* p, const uint32_t (&b)[4]) {
    // the reference accumulates in a uint8_t: keep the low 8 bits of every byte
    uint32_t w = (b[0] & 0xffu) | ((b[1] & 0xffu) << 8) | ((b[2] & 0xffu) << 16) | (b[3] << 24);
    stream_store(w, reinterpret_cast<uint32_t*>(p));
  }
  // scale = float( double(float(qmax)) / (double(max - min) + 2e-6) )
  __device__ static __forceinline__ float make_scale(float lo, float hi, int qmax) {
    float range = hi - lo;
    return (float)((double)(float)qmax / ((double)range + 2e-6));
  }
  // code = rint(max(fma(x - mn, s, u) - 0.5, 0)).  ANY = true: min and scale may be anything (the pack entry
  // point), the code is converted as the reference converts it; ANY = false: they are the group's own, the
  // sum stays below 2^bits + 1 and the code is read off the float (code_bits_of: its low 8 bits count)
  // CENTRED: u is a centred draw of the fast stream (the - 0.5 is in it)
  template <bool ANY, bool CENTRED = false>
  __device__ static __forceinline__ uint32_t code1(const Store& st, int k, int e, float mn, float s, float u) {
    float t = st.v[k][e] - mn;
    float y = __builtin_fmaf(t, s, u);
    // a NaN element keeps its payload through the subtraction and the fma, and a payload may have anything in its
    // low byte: the clamping form (code 0 for every NaN, like the reference's fmax) rather than code_bits_of
    if (CENTRED) return ANY ? rint_clamp0<true>(y) : centred_code_bits_of_any(y);
    return ANY ? rint_clamp0<true>(y - 0.5f) : code_bits_of_any(y);
  }
  // elements e (even) and e + 1 of chunk k
  template <bool ANY>
  __device__ static __forceinline__ void code2(const Store& st, int k, int e, float mn, float s, float ua, float ub,
                                               uint32_t& ca, uint32_t& cb) {
    ca = code1<ANY>(st, k, e, mn, s, ua);
    cb = code1<ANY>(st, k, e + 1, mn, s, ub);
  }
  // NEG (with CENTRED): the chunk takes the mirrored draws, -u (the negation folds into the fma)
  template <bool CONST_NOISE, bool ANY, bool CENTRED = false, bool NEG = false>
  __device__ static __forceinline__ void codes(const Store& st, int k, float mn, float s, const float (&u)[4],
                                               uint32_t (&c)[4]) {
#pragma unroll
    for (int e = 0; e < 4; e++) c[e] = code1<ANY, CENTRED>(st, k, e, mn, s, NEG ? -u[e] : u[e]);
  }
  // what pack_bytes takes: the sums whose rint, clamped at 0, are the codes (of the fast stream: CENTRED, of the deterministic one: u 0.5)
  template <bool CENTRED, bool NEG>
  __device__ static __forceinline__ void sums(const Store& st, int k, float mn, float s, const float (&u)[4], float (&z)[4]) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const float y = __builtin_fmaf(st.v[k][e] - mn, s, NEG ? -u[e] : u[e]);
      z[e] = CENTRED ? y : y - 0.5f;   // exact from 0.5 on, and below it the code is 0 either way
    }
  }
  static constexpr bool kExactField = true;
  __device__ static __forceinline__ void store_words(uint8_t* p, const uint32_t (&w)[1]) { stream_store(w[0], reinterpret_cast<uint32_t*>(p)); }
  // a float scale is never infinite (the denominator is at least 2e-6) and with the group's own min and max the
  // sum stays finite: nothing to repair
  static constexpr bool kRepairsInfiniteScale = false;
  __device__ static __forceinline__ bool scale_is_inf(float) { return false; }
  __device__ static __forceinline__ bool above(const Store&, int, int, float) { return false; }

  // ---- dequantize: out = float(code) / scale + min ----
  struct Dq { float s, r, mn; bool fast; };
  __device__ static __forceinline__ Dq dq_prepare(float s, float mn) {
    Dq d;
    d.s = s; d.mn = mn;
    d.fast = reciprocal_safe(s);
    d.r = 1.0f / s;
    return d;
  }
  __device__ static __forceinline__ float decode(int c, const Dq& d) {
    float q = d.fast ? div_by_reciprocal((float)c, d.s, d.r) : (float)c / d.s;
    return q + d.mn;
  }
  // quotient -> output; one table entry T(c)/scale + min; 32 bits fetched from another lane -> value
  __device__ static __forceinline__ float finish(float q, float mn) { return q + mn; }
  __device__ static __forceinline__ uint32_t table_entry(float c, float s, float mn) {
    return __builtin_bit_cast(uint32_t, c / s + mn);
  }
  __device__ static __forceinline__ float from_bits(uint32_t b) { return __builtin_bit_cast(float, b); }
  static constexpr int kDqWidth = 4;  // columns per dequantize lane: one 16-byte store
  template <int POLICY>
  __device__ static __forceinline__ void store_dq(const OutWindow& w, uint32_t byte_offset, const float (&v)[4]) {
    f32x4 a = {v[0], v[1], v[2], v[3]};
    w.template store16<POLICY>(__builtin_bit_cast(u32x4, a), byte_offset);
  }
};

template <> struct Elem<f16> {
  // quantize layout: 2 chunks of 8 columns, 8i + 128m: one 16-byte load per chunk
  static constexpr int kQChunks = 2, kQWidth = 8;
  static constexpr int kDtype = GACT_F16;
  typedef f16 Stat;
  __device__ static __forceinline__ f16 stat_of(f16 x) { return x; }
  __device__ static __forceinline__ f16 elem_of(f16 x) { return x; }
  struct Store { f16x2 v[2][4]; };   // pairs, so that subtraction and product run as packed ops
  __device__ static __forceinline__ void store_codes(uint8_t* p, const uint32_t (&b)[8]) {
    u32x2 w;
    w.x = (b[0] & 0xffu) | ((b[1] & 0xffu) << 8) | ((b[2] & 0xffu) << 16) | (b[3] << 24);
    w.y = (b[4] & 0xffu) | ((b[5] & 0xffu) << 8) | ((b[6] & 0xffu) << 16) | (b[7] << 24);
    stream_store(w, reinterpret_cast<u32x2*>(p));
  }
  __device__ static __forceinline__ void load_noise(const float* p, float (&u)[8]) {
    f32x4 a = stream_load(reinterpret_cast<const f32x4*>(p));
    f32x4 b = stream_load(reinterpret_cast<const f32x4*>(p + 4));
    u[0] = a.x; u[1] = a.y; u[2] = a.z; u[3] = a.w;
    u[4] = b.x; u[5] = b.y; u[6] = b.z; u[7] = b.w;
  }
  __device__ static __forceinline__ void load_chunk(const f16* p, Store& st, int k) {
    f16x8 a = stream_load(reinterpret_cast<const f16x8*>(p));
#pragma unroll
    for (int j = 0; j < 4; j++) st.v[k][j] = f16x2{a[2 * j], a[2 * j + 1]};
  }
  __device__ static __forceinline__ void set(Store& st, int k, int e, f16 x) { st.v[k][e >> 1][e & 1] = x; }
  __device__ static __forceinline__ float init_lo() { return __builtin_inff(); }  // half(1e30) is +inf
  __device__ static __forceinline__ float init_hi() { return -__builtin_inff(); }
  __device__ static __forceinline__ f16 from_float(float v) { return (f16)v; }
  // Packed min / max in assembly, without the canonicalising copy the compiler puts in front of every minnum / maxnum
  // operand: a quiet NaN operand loses against the other one, which is the reference's "NaN is ignored".
  // (A signalling NaN, which arithmetic never produces, would be returned quieted instead.)
  // Min and max of the lane's chunks K0 .. K1 - 1: packed min / max from +-inf (the start values only survive in a lane
  // whose elements are all NaN), then the two halves against each other
  template <int K0, int K1>
  __device__ static __forceinline__ void lane_minmax(const Store& st, f16& lo_out, f16& hi_out) {
    const f16 inf = (f16)__builtin_inff();
    f16x2 l = {inf, inf}, h = {(f16)-inf, (f16)-inf};
    // a chunk's eight instructions in one block: the compiler puts a wait state behind every block it cannot look into
#pragma unroll
    for (int k = K0; k < K1; k++)
      asm("v_pk_min_f16 %0, %0, %2\n\tv_pk_max_f16 %1, %1, %2\n\tv_pk_min_f16 %0, %0, %3\n\tv_pk_max_f16 %1, %1, %3\n\t"
          "v_pk_min_f16 %0, %0, %4\n\tv_pk_max_f16 %1, %1, %4\n\tv_pk_min_f16 %0, %0, %5\n\tv_pk_max_f16 %1, %1, %5"
          : "+&v"(l), "+&v"(h) : "v"(st.v[k][0]), "v"(st.v[k][1]), "v"(st.v[k][2]), "v"(st.v[k][3]));
    f16 lo, hi;
    asm("v_min_f16_sdwa %0, %1, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:WORD_0 src1_sel:WORD_1"
        : "=v"(lo) : "v"(l));
    asm("v_max_f16_sdwa %0, %1, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:WORD_0 src1_sel:WORD_1"
        : "=v"(hi) : "v"(h));
    lo_out = lo;
    hi_out = hi;
  }
  // The same from the packed three-operand minimum and maximum, half the instructions.  These hand a NaN on where the others ignore it, so
  // a lane that holds one ends up with NaN, which the callers look for: they then take lane_minmax.  Anything else comes out bit
  // for bit alike (subnormals, infinities, zeros of either sign: -0 below +0).
  template <int K0, int K1>
  __device__ static __forceinline__ void lane_ordered(const Store& st, f16& lo_out, f16& hi_out, bool& nan) {
    f16x2 l, h;
    ordered8<K1 - K0 == 2>(st.v[K0], st.v[K1 - 1], l, h);
    lo_out = l[0];
    hi_out = h[0];
    nan |= lo_out != lo_out;
  }
  // Over eight or (BOTH) sixteen elements in pairs; the low half of l and h holds the result.  The last but one step takes the last
  // pair and the two halves of what came before, the last one its own halves.
  template <bool BOTH, typename V>
  __device__ static __forceinline__ void ordered8(const V (&a)[4], const V (&b)[4], f16x2& l, f16x2& h) {
    if constexpr (BOTH)
      asm("v_pk_minimum3_f16 %0, %2, %3, %4\n\tv_pk_maximum3_f16 %1, %2, %3, %4\n\t"
          "v_pk_minimum3_f16 %0, %0, %5, %6\n\tv_pk_maximum3_f16 %1, %1, %5, %6\n\t"
          "v_pk_minimum3_f16 %0, %0, %7, %8\n\tv_pk_maximum3_f16 %1, %1, %7, %8\n\t"
          "v_pk_minimum3_f16 %0, %0, %9, %0 op_sel:[0,0,1] op_sel_hi:[1,1,0]\n\tv_pk_maximum3_f16 %1, %1, %9, %1 op_sel:[0,0,1] op_sel_hi:[1,1,0]\n\t"
          "v_pk_minimum3_f16 %0, %0, %0, %0 op_sel:[0,1,1] op_sel_hi:[1,0,0]\n\tv_pk_maximum3_f16 %1, %1, %1, %1 op_sel:[0,1,1] op_sel_hi:[1,0,0]"
          : "=&v"(l), "=&v"(h) : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]));
    else
      asm("v_pk_minimum3_f16 %0, %2, %3, %4\n\tv_pk_maximum3_f16 %1, %2, %3, %4\n\t"
          "v_pk_minimum3_f16 %0, %0, %5, %0 op_sel:[0,0,1] op_sel_hi:[1,1,0]\n\tv_pk_maximum3_f16 %1, %1, %5, %1 op_sel:[0,0,1] op_sel_hi:[1,1,0]\n\t"
          "v_pk_minimum3_f16 %0, %0, %0, %0 op_sel:[0,1,1] op_sel_hi:[1,0,0]\n\tv_pk_maximum3_f16 %1, %1, %1, %1 op_sel:[0,1,1] op_sel_hi:[1,0,0]"
          : "=&v"(l), "=&v"(h) : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]));
  }
  // min and max of the first `there` of G whole groups, in every lane of the row; of the others 0
  template <int G, bool ORDERED = true>
  __device__ static __forceinline__ void groups_minmax(const Store* st, f16* lo_out, f16* hi_out, int64_t there = G) {
    bool nan = false;
#pragma unroll
    for (int g = 0; g < G; g++) {
      lo_out[g] = hi_out[g] = (f16)0.0f;
      if (g < there) lane_ordered<0, kQChunks>(st[g], lo_out[g], hi_out[g], nan);
    }
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(nan) != 0, 0)) {
#pragma unroll
      for (int g = 0; g < G; g++)
        if (g < there) lane_minmax<0, kQChunks>(st[g], lo_out[g], hi_out[g]);
    }
#pragma unroll
    for (int g = 0; g < G; g++) row_all_minmax(lo_out[g], hi_out[g]);   // a group is there for the whole row or for none of it
  }
  // range is a half operation; the quotient is a double narrowed to float and then to half
  __device__ static __forceinline__ f16 make_scale(f16 lo, f16 hi, int qmax) {
    f16 range = hi - lo;
    return (f16)(float)((double)(float)qmax / ((double)(float)range + 2e-6));
  }
  // float(p) + u with p taken from the low / high half of a pair: one v_fma_mix_f32 (p * 1.0 + u)
  __device__ static __forceinline__ float widen_add_lo(f16x2 p, float u) {
    float y;
    asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(y) : "v"(p), "v"(u));
    return y;
  }
  __device__ static __forceinline__ float widen_add_hi(f16x2 p, float u) {
    float y;
    asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(y) : "v"(p), "v"(u));
    return y;
  }
  // float(p) - u: the same instruction with the addend's sign flipped
  __device__ static __forceinline__ float widen_sub_lo(f16x2 p, float u) {
    float y;
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(y) : "v"(p), "v"(u));
    return y;
  }
  __device__ static __forceinline__ float widen_sub_hi(f16x2 p, float u) {
    float y;
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(y) : "v"(p), "v"(u));
    return y;
  }
  // half subtraction and half product (each rounded to half), then float: y = float(p) + u,
  // code = rint(max(y - 0.5, 0)).  |y| <= 65505 or y is infinite or NaN whatever min and scale are, so the
  // code is always read off the float.  ANY = true (min and scale from the caller): y may be negative or +inf,
  // the clamping form takes both.  ANY = false: y >= 0, and where it is +inf (the scale overflowed to inf)
  // the caller repairs the group afterwards.
  template <bool ANY, bool CENTRED = false>
  __device__ static __forceinline__ uint32_t code1(const Store& st, int k, int e, f16 mn, f16 s, float u) {
    f16 t = st.v[k][e >> 1][e & 1] - mn;
    f16 p = t * s;
    float y = (float)p + u;
    if (CENTRED) return ANY ? centred_code_bits_of_any(y) : centred_code_bits_of(y);
    return ANY ? code_bits_of_any(y) : code_bits_of(y);
  }
  // elements e (even) and e + 1 of chunk k, one pair: packed subtraction and product, the sum with the widening folded in
  template <bool ANY>
  __device__ static __forceinline__ void code2(const Store& st, int k, int e, f16 mn, f16 s, float ua, float ub,
                                               uint32_t& ca, uint32_t& cb) {
    const f16x2 mn2 = {mn, mn}, s2 = {s, s};
    const f16x2 p = (st.v[k][e >> 1] - mn2) * s2;
    const float ya = widen_add_lo(p, ua), yb = widen_add_hi(p, ub);
    ca = ANY ? code_bits_of_any(ya) : code_bits_of(ya);
    cb = ANY ? code_bits_of_any(yb) : code_bits_of(yb);
  }
  // elements e (even) and e + 1 of chunk k under the reference stream, for pack_bytes
  __device__ static __forceinline__ void sum2(const Store& st, int k, int e, f16 mn, f16 s, float ua, float ub, float& za, float& zb) {
    const f16x2 mn2 = {mn, mn}, s2 = {s, s};
    const f16x2 p = (st.v[k][e >> 1] - mn2) * s2;
    za = widen_add_lo(p, ua) - 0.5f;
    zb = widen_add_hi(p, ub) - 0.5f;
  }
  template <bool CONST_NOISE, bool ANY, bool CENTRED = false, bool NEG = false>
  __device__ static __forceinline__ void codes(const Store& st, int k, f16 mn, f16 s, const float (&u)[8],
                                               uint32_t (&c)[8]) {
    const f16x2 mn2 = {mn, mn}, s2 = {s, s};
#pragma unroll
    for (int j = 0; j < 4; j++) {
      f16x2 t = st.v[k][j] - mn2;
      f16x2 p = t * s2;
      if (CENTRED) {
        // the fast stream: float(p) +- c in one v_fma_mix_f32, then the code off the float
        const float zl = NEG ? widen_sub_lo(p, u[2 * j]) : widen_add_lo(p, u[2 * j]);
        const float zh = NEG ? widen_sub_hi(p, u[2 * j + 1]) : widen_add_hi(p, u[2 * j + 1]);
        c[2 * j] = ANY ? centred_code_bits_of_any(zl) : centred_code_bits_of(zl);
        c[2 * j + 1] = ANY ? centred_code_bits_of_any(zh) : centred_code_bits_of(zh);
      } else if (CONST_NOISE) {
        // u = 0.5: float(p) + 0.5 and the following - 0.5 are both exact for every half p (at most 24
        // significant bits between 2^-1 and p's last bit), so y - 0.5 == float(p) and the code is
        // rint(float(p)): float(p) plus the constant rounds to the constant + rint(float(p))
        if (ANY) {
          c[2 * j] = clamp_code_bits(widen_add_lo(p, 8388608.0f));
          c[2 * j + 1] = clamp_code_bits(widen_add_hi(p, 8388608.0f));
        } else {
          c[2 * j] = __builtin_bit_cast(uint32_t, widen_add_lo(p, 12582912.0f));
          c[2 * j + 1] = __builtin_bit_cast(uint32_t, widen_add_hi(p, 12582912.0f));
        }
      } else if (ANY) {
        c[2 * j] = code_bits_of_any(widen_add_lo(p, u[2 * j]));
        c[2 * j + 1] = code_bits_of_any(widen_add_hi(p, u[2 * j + 1]));
      } else {
        c[2 * j] = code_bits_of(widen_add_lo(p, u[2 * j]));
        c[2 * j + 1] = code_bits_of(widen_add_hi(p, u[2 * j + 1]));
      }
    }
  }
  // what pack_bytes takes (the deterministic stream: float(p), see codes)
  template <bool CENTRED, bool NEG>
  __device__ static __forceinline__ void sums(const Store& st, int k, f16 mn, f16 s, const float (&u)[8], float (&z)[8]) {
    const f16x2 mn2 = {mn, mn}, s2 = {s, s};
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const f16x2 p = (st.v[k][j] - mn2) * s2;
      if (!CENTRED) {
        z[2 * j] = (float)p[0];
        z[2 * j + 1] = (float)p[1];
      } else if (NEG) {
        asm("v_fma_mix_f32 %0, %2, 1.0, -%3 op_sel:[0,0,0] op_sel_hi:[1,0,0]\n\tv_fma_mix_f32 %1, %2, 1.0, -%4 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
            : "=&v"(z[2 * j]), "=v"(z[2 * j + 1]) : "v"(p), "v"(u[2 * j]), "v"(u[2 * j + 1]));
      } else {
        asm("v_fma_mix_f32 %0, %2, 1.0, %3 op_sel:[0,0,0] op_sel_hi:[1,0,0]\n\tv_fma_mix_f32 %1, %2, 1.0, %4 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
            : "=&v"(z[2 * j]), "=v"(z[2 * j + 1]) : "v"(p), "v"(u[2 * j]), "v"(u[2 * j + 1]));
      }
    }
  }
  static constexpr bool kExactField = false;
  __device__ static __forceinline__ void store_words(uint8_t* p, const uint32_t (&w)[2]) { stream_store(u32x2{w[0], w[1]}, reinterpret_cast<u32x2*>(p)); }
  // Where the scale is +inf every element above the minimum has an infinite product, whose code the reference
  // saturates to 0x7fffffff: all ones from the element's field upwards.  (An element equal to the minimum gives
  // 0 * inf = NaN: code 0.)  code_bits_of leaves 0 in both cases; this adds the ones.
  static constexpr bool kRepairsInfiniteScale = true;
  __device__ static __forceinline__ bool scale_is_inf(f16 s) { return __builtin_isinf((float)s); }
  __device__ static __forceinline__ bool above(const Store& st, int k, int e, f16 mn) { return st.v[k][e >> 1][e & 1] > mn; }

  // ---- dequantize: half(code) / scale is a float division rounded to half; the sum is rounded to half ----
  struct Dq { float s, r; f16 mn; bool fast; };
  __device__ static __forceinline__ Dq dq_prepare(f16 s, f16 mn) {
    Dq d;
    d.s = (float)s; d.mn = mn;
    d.fast = reciprocal_safe(d.s);
    d.r = 1.0f / d.s;
    return d;
  }
  __device__ static __forceinline__ f16 decode(int c, const Dq& d) {
    float q = d.fast ? div_by_reciprocal((float)c, d.s, d.r) : (float)c / d.s;
    return (f16)q + d.mn;
  }
  __device__ static __forceinline__ f16 finish(float q, f16 mn) { return (f16)q + mn; }
  __device__ static __forceinline__ uint32_t table_entry(float c, f16 s, f16 mn) {
    return (uint32_t)__builtin_bit_cast(uint16_t, (f16)((f16)(c / (float)s) + mn));
  }
  __device__ static __forceinline__ f16 from_bits(uint32_t b) { return __builtin_bit_cast(f16, (uint16_t)b); }
  static constexpr int kDqWidth = 8;  // columns per dequantize lane: one 16-byte store
  template <int POLICY>
  __device__ static __forceinline__ void store_dq(const OutWindow& w, uint32_t byte_offset, const f16 (&v)[8]) {
    f16x8 a;
#pragma unroll
    for (int e = 0; e < 8; e++) a[e] = v[e];
    w.template store16<POLICY>(__builtin_bit_cast(u32x4, a), byte_offset);
  }
};

// bfloat16 (not in the reference, which knows float and half): every bfloat16 is a float, so the group is
// widened on load and quantized exactly as the float path quantizes those floats - same min, same float
// scale, same codes - with the half layout (8-column chunks, one 16-byte load each).  The scale is kept in
// float (8 significant bits would not do), the minimum is one of the inputs and goes back to bfloat16
// unchanged, and dequantize rounds float(code) / scale + min to bfloat16 once, to nearest even.
template <> struct Elem<bf16> {
  static constexpr int kQChunks = 2, kQWidth = 8;
  static constexpr int kDtype = GACT_BF16;
  typedef float Stat;
  __device__ static __forceinline__ float stat_of(bf16 x) { return (float)x; }
  __device__ static __forceinline__ bf16 elem_of(float x) { return (bf16)x; }
  // the group stays in registers as loaded (pairs of bfloat16) and is widened where it is used - once for
  // min / max, once for the codes: half the registers of a widened copy (1 bit: 8 groups per lane)
  struct Store { uint32_t w[2][4]; };
  __device__ static __forceinline__ float widen(const Store& st, int k, int e) {
    const uint32_t w = st.w[k][e >> 1];
    return __builtin_bit_cast(float, (e & 1) ? (w & 0xffff0000u) : (w << 16));
  }
  __device__ static __forceinline__ void store_codes(uint8_t* p, const uint32_t (&b)[8]) { Elem<f16>::store_codes(p, b); }
  __device__ static __forceinline__ void load_noise(const float* p, float (&u)[8]) { Elem<f16>::load_noise(p, u); }
  __device__ static __forceinline__ void load_chunk(const bf16* p, Store& st, int k) {
    const u32x4 a = stream_load(reinterpret_cast<const u32x4*>(p));
    st.w[k][0] = a.x; st.w[k][1] = a.y; st.w[k][2] = a.z; st.w[k][3] = a.w;
  }
  __device__ static __forceinline__ void set(Store& st, int k, int e, bf16 x) {
    const uint32_t h = (uint32_t)__builtin_bit_cast(uint16_t, x);
    if (e & 1) st.w[k][e >> 1] |= h << 16;   // the callers set a chunk's elements in order: the even one starts the pair
    else st.w[k][e >> 1] = h;
  }
  // Min and max of the first `there` of G whole groups, in every lane of the row, of the others 0.
  // ORDERED: two bfloat16 of magnitude up to 2^121 (bits 0x7c00) are ordered as the halves with their bits are, so they take half's packed
  // instructions, a quarter of what widening every element takes; a larger one, an infinity or a NaN is a half NaN, and then
  // every element of the wave is widened.  The float path's start values bound the results either way.
  template <int G, bool ORDERED = true>
  __device__ static __forceinline__ void groups_minmax(const Store* st, float* lo_out, float* hi_out, int64_t there = G) {
    f16 lo16[G], hi16[G];
    bool nan = !ORDERED;
    if constexpr (ORDERED) {
#pragma unroll
      for (int g = 0; g < G; g++) {
        lo16[g] = hi16[g] = (f16)0.0f;
        if (g < there) {
          f16x2 l, h;
          Elem<f16>::template ordered8<true>(st[g].w[0], st[g].w[1], l, h);
          lo16[g] = l[0];
          hi16[g] = h[0];
          nan |= lo16[g] != lo16[g];
        }
      }
    }
    if (!ORDERED || __builtin_expect(__builtin_amdgcn_ballot_w64(nan) != 0, 0)) {
#pragma unroll
      for (int g = 0; g < G; g++) {
        lo_out[g] = hi_out[g] = 0.0f;
        if (g < there) {
          float lo = Elem<float>::init_lo(), hi = Elem<float>::init_hi();
#pragma unroll
          for (int k = 0; k < kQChunks; k++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
              lo = __builtin_fminf(lo, widen(st[g], k, e));
              hi = __builtin_fmaxf(hi, widen(st[g], k, e));
            }
          row_all_minmax(lo, hi);
          lo_out[g] = lo;
          hi_out[g] = hi;
        }
      }
    } else {
#pragma unroll
      for (int g = 0; g < G; g++) {
        row_all_minmax(lo16[g], hi16[g]);
        lo_out[g] = __builtin_fminf(Elem<float>::init_lo(), __builtin_bit_cast(float, (uint32_t)__builtin_bit_cast(uint16_t, lo16[g]) << 16));
        hi_out[g] = __builtin_fmaxf(Elem<float>::init_hi(), __builtin_bit_cast(float, (uint32_t)__builtin_bit_cast(uint16_t, hi16[g]) << 16));
      }
    }
  }
  __device__ static __forceinline__ float make_scale(float lo, float hi, int qmax) {
    return Elem<float>::make_scale(lo, hi, qmax);
  }
  template <bool ANY, bool CENTRED = false>
  __device__ static __forceinline__ uint32_t code1(const Store& st, int k, int e, float mn, float s, float u) {
    float t = widen(st, k, e) - mn;
    float y = __builtin_fmaf(t, s, u);
    if (CENTRED) return ANY ? rint_clamp0<true>(y) : centred_code_bits_of(y);
    return ANY ? rint_clamp0<true>(y - 0.5f) : code_bits_of(y);
  }
  template <bool ANY>
  __device__ static __forceinline__ void code2(const Store& st, int k, int e, float mn, float s, float ua, float ub,
                                               uint32_t& ca, uint32_t& cb) {
    ca = code1<ANY>(st, k, e, mn, s, ua);
    cb = code1<ANY>(st, k, e + 1, mn, s, ub);
  }
  template <bool CONST_NOISE, bool ANY, bool CENTRED = false, bool NEG = false>
  __device__ static __forceinline__ void codes(const Store& st, int k, float mn, float s, const float (&u)[8],
                                               uint32_t (&c)[8]) {
#pragma unroll
    for (int e = 0; e < 8; e++) c[e] = code1<ANY, CENTRED>(st, k, e, mn, s, NEG ? -u[e] : u[e]);
  }
  template <bool CENTRED, bool NEG>
  __device__ static __forceinline__ void sums(const Store& st, int k, float mn, float s, const float (&u)[8], float (&z)[8]) {
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float y = __builtin_fmaf(widen(st, k, e) - mn, s, NEG ? -u[e] : u[e]);
      z[e] = CENTRED ? y : y - 0.5f;
    }
  }
  static constexpr bool kExactField = true;
  __device__ static __forceinline__ void store_words(uint8_t* p, const uint32_t (&w)[2]) { Elem<f16>::store_words(p, w); }
  static constexpr bool kRepairsInfiniteScale = false;
  __device__ static __forceinline__ bool scale_is_inf(float) { return false; }
  __device__ static __forceinline__ bool above(const Store&, int, int, float) { return false; }
  __device__ static __forceinline__ bf16 finish(float q, float mn) { return (bf16)(q + mn); }
  __device__ static __forceinline__ uint32_t table_entry(float c, float s, float mn) {
    return (uint32_t)__builtin_bit_cast(uint16_t, (bf16)(c / s + mn));
  }
  __device__ static __forceinline__ bf16 from_bits(uint32_t b) { return __builtin_bit_cast(bf16, (uint16_t)b); }
  static constexpr int kDqWidth = 8;
  template <int POLICY>
  __device__ static __forceinline__ void store_dq(const OutWindow& w, uint32_t byte_offset, const bf16 (&v)[8]) {
    typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
    bf16x8 a;
#pragma unroll
    for (int e = 0; e < 8; e++) a[e] = v[e];
    w.template store16<POLICY>(__builtin_bit_cast(u32x4, a), byte_offset);
  }
};

// Column of the first element of chunk k for row lane i: chunks are W columns wide and 16*W apart.
template <typename T>
__device__ __forceinline__ int chunk_col(int k, int i) { return Elem<T>::kQWidth * (16 * k + i); }

// Load the 16 elements lane i owns of group n; elements at or beyond numel read as zero (the zero
// padding of gact/gact/ops.py:12-17 without the copy).
template <typename T>
__device__ __forceinline__ void load_group(const T* __restrict__ x, int64_t numel, int64_t n, int i,
                                           typename Elem<T>::Store& st) {
  constexpr int CH = Elem<T>::kQChunks, W = Elem<T>::kQWidth;
  const int64_t base = n * GROUP;
  if (base + GROUP <= numel) {
#pragma unroll
    for (int k = 0; k < CH; k++) Elem<T>::load_chunk(x + base + chunk_col<T>(k, i), st, k);
  } else {
#pragma unroll
    for (int k = 0; k < CH; k++)
#pragma unroll
      for (int e = 0; e < W; e++) {
        int64_t idx = base + chunk_col<T>(k, i) + e;
        Elem<T>::set(st, k, e, idx < numel ? x[idx] : (T)0.0f);
      }
  }
}

// Where a quantize row takes its groups from: load() fills the lane's 16 elements of group n (elements past the end are
// zero), and a contiguous source also has its elements side by side (x).
template <typename T>
struct ContiguousSource {
  static constexpr bool kContiguous = true;
  const T* x;
  int64_t numel;
  __device__ __forceinline__ void load(int64_t n, int i, typename Elem<T>::Store& st) const { load_group<T>(x, numel, n, i, st); }
};
// q = x / d for x < 2^31, as a multiplication (multiplier 0: d is 1)
struct Divisor {
  uint32_t d, m, s;
  __device__ __forceinline__ uint32_t quotient(uint32_t x) const { return m ? __umulhi(x, m) >> s : x; }
};
// A tensor of up to four dimensions whose innermost runs are contiguous and whole 16-byte pieces (attention heads: [batch,
// seq, heads, width] seen as [batch, heads, seq, width]): every 16-byte piece has an address of its own.  Counts and
// strides are in pieces.
struct GatherShape {
  Divisor run, n2, n1;
  int64_t s0, s1, s2;
};
template <typename T>
struct GatherSource {
  static constexpr bool kContiguous = false;
  const T* x;
  int64_t numel;
  GatherShape g;
  __device__ __forceinline__ void load(int64_t n, int i, typename Elem<T>::Store& st) const {
    constexpr int CH = Elem<T>::kQChunks, W = Elem<T>::kQWidth;
#pragma unroll
    for (int k = 0; k < CH; k++) {
      const uint32_t piece = (uint32_t)(n * (GROUP / W)) + (uint32_t)(16 * k + i);
      if ((int64_t)piece * W < numel) {
        const uint32_t i2 = g.run.quotient(piece), i1 = g.n2.quotient(i2), i0 = g.n1.quotient(i1);
        const int64_t at = (int64_t)i0 * g.s0 + (int64_t)(i1 - i0 * g.n1.d) * g.s1 + (int64_t)(i2 - i1 * g.n2.d) * g.s2 + (piece - i2 * g.run.d);
        Elem<T>::load_chunk(x + at * W, st, k);
      } else {
#pragma unroll
        for (int e = 0; e < W; e++) Elem<T>::set(st, k, e, (T)0.0f);
      }
    }
  }
};

// value of lane LANE of the row, in every lane of the row (DPP row_newbcast)
template <int LANE>
__device__ __forceinline__ uint32_t row_bcast_u32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x150 + LANE, 0xf, 0xf, false);
}
template <int LANE> __device__ __forceinline__ float row_bcast(float v) {
  return __builtin_bit_cast(float, row_bcast_u32<LANE>(__builtin_bit_cast(uint32_t, v)));
}
template <int LANE> __device__ __forceinline__ f16 row_bcast(f16 v) {
  return __builtin_bit_cast(f16, (uint16_t)row_bcast_u32<LANE>((uint32_t)__builtin_bit_cast(uint16_t, v)));
}

// swap with the neighbouring lane (lane ^ 1): DPP quad_perm [1,0,3,2]
__device__ __forceinline__ uint32_t swap_with_neighbour(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0xB1, 0xf, 0xf, false);
}

// The fast stream.  Two consecutive groups (512 elements) draw 16 Philox blocks; block j serves columns 8j .. 8j+7 of
// both: its bytes 0..7 (word by word, low byte first) the first group's, bytes 8..15 the second's, one byte h per
// element, taken as the centred draw c = (2h - 255) / 512.  The column 128 further on takes -c, the same draw
// mirrored: every element's noise is uniform on the same 256-point grid, symmetric about 0 and strictly inside
// (-1/2, 1/2), and the two elements of a pair (which sit half a group apart) round in opposite directions more
// often than not (their rounding errors have covariance <= 0).  One block per 32 elements, one conversion and one
// fma per two elements (the mirrored draw is a sign flip that folds into the instruction that adds it).
// In terms of the flat element index E: block (E / 512) * 16 + (E % 128) / 8, byte ((E / 256) % 2) * 8 + E % 8,
// mirrored if E % 256 >= 128.
__device__ __forceinline__ uint64_t fast_block_of(uint64_t E) { return (E >> 9) * 16 + ((E & 127) >> 3); }
// the centred draw of element E from the words of its block
__device__ __forceinline__ float fast_centred_of(const uint32_t (&r)[4], uint64_t E) {
  const int b = (int)(((E >> 8) & 1) * 8 + (E & 7));
  const uint32_t w = (b & 8) ? ((b & 4) ? r[3] : r[2]) : ((b & 4) ? r[1] : r[0]);
  const float c = fast_centred_map(w, b & 3);
  return (E & 128) ? -c : c;
}

// The two words of each group of the pair `pair` that row lane i needs: w[g][0..1] hold the 8 draws of the lane's
// unmirrored columns of group 2 * pair + g, in column order.  With 8-column chunks (8i + 128m) that is the lane's
// own block.  With 4-column chunks (4i + 64m) chunks 0 and 1 are halves of blocks i/2 and 8 + i/2, which two
// neighbouring lanes share: the even lane computes the first, the odd lane the second, and they exchange the words
// the other one needs (the even lane owns words 0 and 2 of a block, the odd lane words 1 and 3).
template <typename T>
__device__ __forceinline__ void fast_pair_words(int64_t pair, int i, uint32_t k0, uint32_t k1, uint32_t (&w)[2][2]) {
  constexpr int CH = Elem<T>::kQChunks, W = Elem<T>::kQWidth;
  uint32_t r[4];
  if (W == 8) {
    static_assert(W != 8 || CH == 2, "two chunks of 8 columns, 128 apart");
    const uint64_t blk = (uint64_t)pair * 16 + i;
    philox4x32<PHILOX_FAST_ROUNDS>(0u, 0u, (uint32_t)blk, (uint32_t)(blk >> 32), k0, k1, r);
    w[0][0] = r[0]; w[0][1] = r[1]; w[1][0] = r[2]; w[1][1] = r[3];
  } else {
    static_assert(W == 8 || CH == 4, "four chunks of 4 columns, 64 apart");
    const bool odd = i & 1;
    const uint64_t blk = (uint64_t)pair * 16 + (odd ? 8 : 0) + (i >> 1);
    philox4x32<PHILOX_FAST_ROUNDS>(0u, 0u, (uint32_t)blk, (uint32_t)(blk >> 32), k0, k1, r);
    const uint32_t g0 = swap_with_neighbour(odd ? r[0] : r[1]);
    const uint32_t g1 = swap_with_neighbour(odd ? r[2] : r[3]);
    w[0][0] = odd ? g0 : r[0];   // chunk 0: block i/2
    w[0][1] = odd ? r[1] : g0;   // chunk 1: block 8 + i/2
    w[1][0] = odd ? g1 : r[2];
    w[1][1] = odd ? r[3] : g1;
  }
}
// The centred draws of the lane's unmirrored chunks (the first half of its chunks) from the group's two words: draw
// k * W + e belongs to element e of chunk k; chunk k + CH/2 takes the same draws negated.
template <typename T>
__device__ __forceinline__ void fast_centred_draws(const uint32_t (&w)[2], float (&c)[Elem<T>::kQChunks / 2][Elem<T>::kQWidth]) {
  constexpr int CH = Elem<T>::kQChunks, W = Elem<T>::kQWidth;
#pragma unroll
  for (int k = 0; k < CH / 2; k++)
#pragma unroll
    for (int e = 0; e < W; e++) {
      const int f = k * W + e;
      c[k][e] = (f & 2) ? ((f & 1) ? fast_centred_map<3>(w[f >> 2]) : fast_centred_map<2>(w[f >> 2]))
                        : ((f & 1) ? fast_centred_map<1>(w[f >> 2]) : fast_centred_map<0>(w[f >> 2]));
    }
}
// The state of the fast stream along a row's groups: group g of the row (first group n0) draws from the words of its
// pair, which are computed when the row enters the pair.  Rows of two or more groups start on an even group, so that
// happens at every even g; a row of one group computes its pair's block and takes its half.
template <typename T, int GPR>
struct FastRow {
  uint32_t w[2][2];
  __device__ __forceinline__ void draws(int g, int64_t n0, int i, uint32_t k0, uint32_t k1,
                                        float (&c)[Elem<T>::kQChunks / 2][Elem<T>::kQWidth]) {
    if (GPR == 1) {
      const int64_t n = n0 + g;
      fast_pair_words<T>(n >> 1, i, k0, k1, w);
      const uint32_t mine[2] = {(n & 1) ? w[1][0] : w[0][0], (n & 1) ? w[1][1] : w[0][1]};
      fast_centred_draws<T>(mine, c);
    } else {
      if ((g & 1) == 0) fast_pair_words<T>((n0 + g) >> 1, i, k0, k1, w);
      fast_centred_draws<T>(w[g & 1], c);
    }
  }
};

// Chunk k of a group as packed bytes (packs_bytes), with the group's centred draws where the stream is the fast one
template <typename T, int NOISE>
__device__ __forceinline__ void chunk_words(const typename Elem<T>::Store& st, int k, typename Elem<T>::Stat mn, typename Elem<T>::Stat s,
                                            const float (&cd)[Elem<T>::kQChunks / 2][Elem<T>::kQWidth], uint32_t (&w)[Elem<T>::kQWidth / 4]) {
  constexpr int CH = Elem<T>::kQChunks, W = Elem<T>::kQWidth;
  float z[W];
  if (NOISE == GACT_NOISE_FAST) {
    if (k < CH / 2) Elem<T>::template sums<true, false>(st, k, mn, s, cd[k % (CH / 2)], z);
    else Elem<T>::template sums<true, true>(st, k, mn, s, cd[k % (CH / 2)], z);
  } else {
    float u[W];
#pragma unroll
    for (int e = 0; e < W; e++) u[e] = 0.5f;
    Elem<T>::template sums<false, false>(st, k, mn, s, u, z);
  }
  pack_bytes(z, w);
}

// ------------------------------------------------------------------------------------------------
// Quantize SGR consecutive super-groups (one 16-lane row): all their groups are loaded first, reduced, and share
// one scale division per lane; the codes then go out super-group by super-group.
//   STAGE > 0 (rows of whole groups): STAGE groups at a time instead, see below; LAZY: each stage issues its own loads.
//   GIVEN = false: min/max are reduced here (fused minimax + scale + pack, one read of x).
//   GIVEN = true : min/max are read from mn_io / mx_io (the pack entry point's contract).
// Codes follow quantization_cuda_kernel.cu:38-71; see Elem<T>::code1 for the arithmetic.
// ------------------------------------------------------------------------------------------------
template <typename T, int BITS, int NOISE, bool GIVEN, int SGR = 1, int STAGE = 0, bool LAZY = false, bool PACKS = true, bool ORDERED = true, typename SRC>
__device__ __forceinline__ void quantize_supergroup(const SRC& src, int64_t N, int64_t sg0,
                                                    int i, uint8_t* __restrict__ packed,
                                                    typename Elem<T>::Stat* __restrict__ scale_out,
                                                    T* mn_io, T* mx_io, uint32_t k0, uint32_t k1,
                                                    const float* __restrict__ noise) {
  constexpr int WPT = 8 / BITS;
  constexpr int GPR = SGR * WPT;   // groups of the row
  static_assert(GPR == 1 || GPR == 2 || GPR == 4 || GPR == 8, "a row holds 1, 2, 4 or 8 groups");
  constexpr int QMAX = (1 << BITS) - 1;
  constexpr int CH = Elem<T>::kQChunks, W = Elem<T>::kQWidth;
  constexpr bool PK = PACKS && packs_bytes<T, BITS, NOISE, GIVEN>();
  const int64_t n0 = sg0 * WPT;

  typename Elem<T>::Store v[GPR];
  typedef typename Elem<T>::Stat Stat;
  Stat lo_t[GPR], hi_t[GPR], s_t[GPR];
  // The staged path is for rows of whole groups.  The choice is made for the wave, not for the row: a wave in which
  // one row is ragged (the tensor's last) would otherwise run both paths one after the other, each with its own
  // round trip to memory - and being the tensor's last wave it would hold up the end of the kernel.
  if constexpr (STAGE > 0 && STAGE < GPR && !GIVEN && NOISE != GACT_NOISE_REF && SRC::kContiguous) {
  const T* __restrict__ x = src.x;
  const bool whole_row = (n0 + GPR) * GROUP <= src.numel;
  if (__builtin_amdgcn_ballot_w64(!whole_row) == 0) {
    // All groups whole: the loads in one straight line, then STAGE groups at a time as they arrive: reduce, divide
    // (lane j for group j % STAGE of the stage), encode; a super-group goes out when its last group is done.  The
    // work on the first groups overlaps the loads of the later ones within the wave, which pays where few waves
    // share a SIMD (small tensors) and costs the extra divisions elsewhere.  LAZY: a stage's loads are issued when
    // the stage begins (the compiler still hoists what its register budget allows), which suits the
    // instruction-heavy half kernels once several waves share a SIMD.
    static_assert(STAGE <= 0 || (GPR % (STAGE > 0 ? STAGE : 1) == 0 && (STAGE & (STAGE - 1)) == 0), "stages divide the row");
    constexpr int ST = STAGE > 0 ? STAGE : 1;
    if (!LAZY) {
#pragma unroll
      for (int g = 0; g < GPR; g++)
#pragma unroll
        for (int k = 0; k < CH; k++) Elem<T>::load_chunk(x + (n0 + g) * GROUP + chunk_col<T>(k, i), v[g], k);
    }
    uint32_t bytes[CH][W];
    uint32_t words[CH][W / 4];   // PK
    FastRow<T, GPR> fast;
#pragma unroll
    for (int g0 = 0; g0 < GPR; g0 += ST) {
      if (LAZY) {
#pragma unroll
        for (int j = 0; j < ST; j++)
#pragma unroll
          for (int k = 0; k < CH; k++) Elem<T>::load_chunk(x + (n0 + g0 + j) * GROUP + chunk_col<T>(k, i), v[g0 + j], k);
      }
      Stat lo_s[ST], hi_s[ST], sc_s[ST];
      Elem<T>::template groups_minmax<ST, ORDERED>(v + g0, lo_s, hi_s);
      {
        const int mine = i & (ST - 1);
        Stat lo_m = lo_s[0], hi_m = hi_s[0];
#pragma unroll
        for (int j = 1; j < ST; j++) {
          lo_m = (mine == j) ? lo_s[j] : lo_m;
          hi_m = (mine == j) ? hi_s[j] : hi_m;
        }
        const Stat s_m = Elem<T>::make_scale(lo_m, hi_m, QMAX);
        if (i < ST) {
          scale_out[n0 + g0 + i] = s_m;
          mn_io[n0 + g0 + i] = Elem<T>::elem_of(lo_m);
          if (mx_io) mx_io[n0 + g0 + i] = Elem<T>::elem_of(hi_m);
        }
        if (ST == 1) {
          sc_s[0] = s_m;
        } else {
          sc_s[0] = row_bcast<0>(s_m);
          sc_s[1 % ST] = row_bcast<1>(s_m);
          if (ST > 2) { sc_s[2 % ST] = row_bcast<2>(s_m); sc_s[3 % ST] = row_bcast<3>(s_m); }
        }
      }
#pragma unroll
      for (int j = 0; j < ST; j++) {
        const int g = g0 + j;
        const int64_t n = n0 + g;
        const int ni = g % WPT;
        if constexpr (PK) {
          float cd[CH / 2][W];
          if (NOISE == GACT_NOISE_FAST) fast.draws(g, n0, i, k0, k1, cd);
#pragma unroll
          for (int k = 0; k < CH; k++) {
            uint32_t w[W / 4];
            chunk_words<T, NOISE>(v[g], k, lo_s[j], sc_s[j], cd, w);
#pragma unroll
            for (int d = 0; d < W / 4; d++) words[k][d] = ni == 0 ? w[d] : words[k][d] | field_of<Elem<T>::kExactField>(w[d], ni * BITS);
            if (ni == WPT - 1) Elem<T>::store_words(packed + (sg0 + g / WPT) * GROUP + chunk_col<T>(k, i), words[k]);
          }
          continue;
        }
        if (ni == 0) {
#pragma unroll
          for (int k = 0; k < CH; k++)
#pragma unroll
            for (int e = 0; e < W; e++) bytes[k][e] = 0;
        }
        if (NOISE == GACT_NOISE_FAST) {
          float cd[CH / 2][W];
          fast.draws(g, n0, i, k0, k1, cd);
#pragma unroll
          for (int k = 0; k < CH; k++) {
            uint32_t c[W];
            if (k < CH / 2) Elem<T>::template codes<false, GIVEN, true, false>(v[g], k, lo_s[j], sc_s[j], cd[k % (CH / 2)], c);
            else Elem<T>::template codes<false, GIVEN, true, true>(v[g], k, lo_s[j], sc_s[j], cd[k % (CH / 2)], c);
#pragma unroll
            for (int e = 0; e < W; e++) bytes[k][e] |= c[e] << (ni * BITS);
          }
        } else {
          float u[CH][W];
#pragma unroll
          for (int k = 0; k < CH; k++) {
            if (NOISE == GACT_NOISE_INJECT) {
              Elem<T>::load_noise(noise + n * GROUP + chunk_col<T>(k, i), u[k]);
            } else {
#pragma unroll
              for (int e = 0; e < W; e++) u[k][e] = 0.5f;
            }
          }
#pragma unroll
          for (int k = 0; k < CH; k++) {
            uint32_t c[W];
            Elem<T>::template codes<NOISE == GACT_NOISE_CONST, GIVEN>(v[g], k, lo_s[j], sc_s[j], u[k], c);
#pragma unroll
            for (int e = 0; e < W; e++) bytes[k][e] |= c[e] << (ni * BITS);
          }
        }
        if (Elem<T>::kRepairsInfiniteScale && __builtin_amdgcn_ballot_w64(Elem<T>::scale_is_inf(sc_s[j])) != 0) {
          if (Elem<T>::scale_is_inf(sc_s[j])) {
#pragma unroll
            for (int k = 0; k < CH; k++)
#pragma unroll
              for (int e = 0; e < W; e++)
                if (Elem<T>::above(v[g], k, e, lo_s[j])) bytes[k][e] |= 0xffffffffu << (ni * BITS);
          }
        }
        if (ni == WPT - 1) {
#pragma unroll
          for (int k = 0; k < CH; k++)
            Elem<T>::store_codes(packed + (sg0 + g / WPT) * GROUP + chunk_col<T>(k, i), bytes[k]);
        }
      }
      if ((g0 + ST) % WPT != 0) {
        // the codes of this stage exist before the next stage's loads are waited for
#pragma unroll
        for (int k = 0; k < CH; k++) {
          if constexpr (PK) {
#pragma unroll
            for (int d = 0; d < W / 4; d++) asm volatile("" : "+v"(words[k][d]));
          } else {
#pragma unroll
            for (int e = 0; e < W; e++) asm volatile("" : "+v"(bytes[k][e]));
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    return;
  }
  }
#pragma unroll
  for (int g = 0; g < GPR; g++) {
    if (n0 + g < N) src.load(n0 + g, i, v[g]);
  }
  if constexpr (GIVEN) {
#pragma unroll
    for (int g = 0; g < GPR; g++) {
      const int64_t n = n0 + g;
      lo_t[g] = hi_t[g] = (Stat)0.0f;
      if (n < N) {
        lo_t[g] = Elem<T>::stat_of(mn_io[n]);
        hi_t[g] = Elem<T>::stat_of(mx_io[n]);
      }
    }
  } else {
    Elem<T>::template groups_minmax<GPR, ORDERED>(v, lo_t, hi_t, N - n0);
  }
  // one scale division per lane: lane j of the row takes group j % GPR, then the row shares the results
  {
    const int mine = i & (GPR - 1);
    Stat lo_m = lo_t[0], hi_m = hi_t[0];
#pragma unroll
    for (int g = 1; g < GPR; g++) {
      lo_m = (mine == g) ? lo_t[g] : lo_m;
      hi_m = (mine == g) ? hi_t[g] : hi_m;
    }
    const Stat s_m = Elem<T>::make_scale(lo_m, hi_m, QMAX);
    if (i < GPR && n0 + i < N) {
      scale_out[n0 + i] = s_m;
      if (!GIVEN) {
        mn_io[n0 + i] = Elem<T>::elem_of(lo_m);
        if (mx_io) mx_io[n0 + i] = Elem<T>::elem_of(hi_m);
      }
    }
    if (GPR == 1) {
      s_t[0] = s_m;
    } else {
      s_t[0] = row_bcast<0>(s_m);
      if (GPR > 1) s_t[1 % GPR] = row_bcast<1>(s_m);
      if (GPR > 2) { s_t[2 % GPR] = row_bcast<2>(s_m); s_t[3 % GPR] = row_bcast<3>(s_m); }
      if (GPR > 4) {
        s_t[4 % GPR] = row_bcast<4>(s_m); s_t[5 % GPR] = row_bcast<5>(s_m);
        s_t[6 % GPR] = row_bcast<6>(s_m); s_t[7 % GPR] = row_bcast<7>(s_m);
      }
    }
  }

  FastRow<T, GPR> fast;
#pragma unroll
  for (int q = 0; q < SGR; q++) {
    const int64_t sg = sg0 + q;
    if (q == 0 || sg * WPT < N) {
    if constexpr (PK && NOISE == GACT_NOISE_REF) {
      // four neighbouring bytes at a time: one Philox state per output byte j, key = seed, counter = (draw/4, 0, j lo, j hi), two of
      // them side by side so that the half path can take its elements in pairs
      const float addend = uniform_addend();
#pragma unroll
      for (int k = 0; k < CH; k++) {
        uint32_t words[W / 4];
#pragma unroll
        for (int d = 0; d < W / 4; d++) {
          uint32_t w[WPT];
#pragma unroll
          for (int ni = 0; ni < WPT; ni++) w[ni] = 0u;
#pragma unroll
          for (int e = 0; e < 4; e += 2) {
            const uint64_t j = (uint64_t)sg * GROUP + chunk_col<T>(k, i) + 4 * d + e;
            uint32_t ra[4], rb[4];
#pragma unroll
            for (int ni = 0; ni < WPT; ni++) {
              const int g = q * WPT + ni;
              if ((ni & 3) == 0) {
                philox4x32<PHILOX_REF_ROUNDS>(ni >> 2, 0u, (uint32_t)j, (uint32_t)(j >> 32), k0, k1, ra);
                philox4x32<PHILOX_REF_ROUNDS>(ni >> 2, 0u, (uint32_t)(j + 1), (uint32_t)((j + 1) >> 32), k0, k1, rb);
              }
              if (n0 + g < N) {
                float za, zb;
                Elem<T>::sum2(v[g], k, 4 * d + e, lo_t[g], s_t[g], curand_uniform_map(ra[ni & 3], addend),
                              curand_uniform_map(rb[ni & 3], addend), za, zb);
                w[ni] = __builtin_amdgcn_cvt_pk_u8_f32(za, e, w[ni]);
                w[ni] = __builtin_amdgcn_cvt_pk_u8_f32(zb, e + 1, w[ni]);
              }
            }
          }
          words[d] = w[0];
#pragma unroll
          for (int ni = 1; ni < WPT; ni++) words[d] |= field_of<false>(w[ni], ni * BITS);
        }
        Elem<T>::store_words(packed + sg * GROUP + chunk_col<T>(k, i), words);
      }
      continue;
    } else if constexpr (PK) {
      uint32_t words[CH][W / 4];
#pragma unroll
      for (int k = 0; k < CH; k++)
#pragma unroll
        for (int d = 0; d < W / 4; d++) words[k][d] = 0;
#pragma unroll
      for (int ni = 0; ni < WPT; ni++) {
        const int g = q * WPT + ni;
        if (n0 + g < N) {
          float cd[CH / 2][W];
          if (NOISE == GACT_NOISE_FAST) fast.draws(g, n0, i, k0, k1, cd);
#pragma unroll
          for (int k = 0; k < CH; k++) {
            uint32_t w[W / 4];
            chunk_words<T, NOISE>(v[g], k, lo_t[g], s_t[g], cd, w);
#pragma unroll
            for (int d = 0; d < W / 4; d++) words[k][d] |= field_of<Elem<T>::kExactField>(w[d], ni * BITS);
          }
        }
      }
#pragma unroll
      for (int k = 0; k < CH; k++) Elem<T>::store_words(packed + sg * GROUP + chunk_col<T>(k, i), words[k]);
      continue;
    }
    uint32_t bytes[CH][W];
#pragma unroll
    for (int k = 0; k < CH; k++)
#pragma unroll
      for (int e = 0; e < W; e++) bytes[k][e] = 0;

    if (NOISE == GACT_NOISE_REF) {
      // one Philox state per output byte j: key = seed, counter = (draw/4, 0, j lo, j hi); two neighbouring bytes at
      // a time, so that the half path can take its elements in pairs
      const float addend = uniform_addend();
#pragma unroll
      for (int k = 0; k < CH; k++)
#pragma unroll
        for (int e = 0; e < W; e += 2) {
          const uint64_t j = (uint64_t)sg * GROUP + chunk_col<T>(k, i) + e;
          uint32_t ra[4], rb[4];
#pragma unroll
          for (int ni = 0; ni < WPT; ni++) {
            const int g = q * WPT + ni;
            if ((ni & 3) == 0) {
              philox4x32<PHILOX_REF_ROUNDS>(ni >> 2, 0u, (uint32_t)j, (uint32_t)(j >> 32), k0, k1, ra);
              philox4x32<PHILOX_REF_ROUNDS>(ni >> 2, 0u, (uint32_t)(j + 1), (uint32_t)((j + 1) >> 32), k0, k1, rb);
            }
            if (n0 + g < N) {
              uint32_t ca, cb;
              Elem<T>::template code2<GIVEN>(v[g], k, e, lo_t[g], s_t[g], curand_uniform_map(ra[ni & 3], addend),
                                             curand_uniform_map(rb[ni & 3], addend), ca, cb);
              bytes[k][e] |= ca << (ni * BITS);
              bytes[k][e + 1] |= cb << (ni * BITS);
            }
          }
        }
    } else {
#pragma unroll
      for (int ni = 0; ni < WPT; ni++) {
        const int g = q * WPT + ni;
        const int64_t n = n0 + g;
        if (n < N) {
          if (NOISE == GACT_NOISE_FAST) {
            float cd[CH / 2][W];
            fast.draws(g, n0, i, k0, k1, cd);
#pragma unroll
            for (int k = 0; k < CH; k++) {
              uint32_t c[W];
              if (k < CH / 2) Elem<T>::template codes<false, GIVEN, true, false>(v[g], k, lo_t[g], s_t[g], cd[k % (CH / 2)], c);
              else Elem<T>::template codes<false, GIVEN, true, true>(v[g], k, lo_t[g], s_t[g], cd[k % (CH / 2)], c);
#pragma unroll
              for (int e = 0; e < W; e++) bytes[k][e] |= c[e] << (ni * BITS);
            }
          } else {
            float u[CH][W];
#pragma unroll
            for (int k = 0; k < CH; k++) {
              if (NOISE == GACT_NOISE_INJECT) {
                Elem<T>::load_noise(noise + n * GROUP + chunk_col<T>(k, i), u[k]);
              } else {
#pragma unroll
                for (int e = 0; e < W; e++) u[k][e] = 0.5f;
              }
            }
#pragma unroll
            for (int k = 0; k < CH; k++) {
              uint32_t c[W];
              Elem<T>::template codes<NOISE == GACT_NOISE_CONST, GIVEN>(v[g], k, lo_t[g], s_t[g], u[k], c);
#pragma unroll
              for (int e = 0; e < W; e++) bytes[k][e] |= c[e] << (ni * BITS);
            }
          }
        }
      }
    }

    if (Elem<T>::kRepairsInfiniteScale && !GIVEN) {
      // rare: a scale of the super-group overflowed to +inf (see Elem<T>::kRepairsInfiniteScale)
      bool any_inf = false;
#pragma unroll
      for (int ni = 0; ni < WPT; ni++) any_inf |= Elem<T>::scale_is_inf(s_t[q * WPT + ni]);
      if (__builtin_amdgcn_ballot_w64(any_inf) != 0) {
#pragma unroll
        for (int ni = 0; ni < WPT; ni++) {
          const int g = q * WPT + ni;
          if (n0 + g < N && Elem<T>::scale_is_inf(s_t[g])) {
#pragma unroll
            for (int k = 0; k < CH; k++)
#pragma unroll
              for (int e = 0; e < W; e++)
                if (Elem<T>::above(v[g], k, e, lo_t[g])) bytes[k][e] |= 0xffffffffu << (ni * BITS);
          }
        }
      }
    }
#pragma unroll
    for (int k = 0; k < CH; k++) Elem<T>::store_codes(packed + sg * GROUP + chunk_col<T>(k, i), bytes[k]);
    }
  }
}

// ------------------------------------------------------------------------------------------------
// Dequantize a unit: G = SGS * (8/BITS) / PARTS consecutive groups - SGS whole super-groups, or (PARTS > 1, SGS = 1)
// one of PARTS equal parts of a super-group, the code words of which its other units load as well.  A lane owns the
// W = 16/sizeof(T) columns W*l .. W*l+W-1 of every group (one 16-byte store per group), so 256/W lanes cover a
// group: a whole wave per unit for float, half a wave for half.  All code words are loaded first, then the
// groups are written, each store instruction covering whole groups contiguously.
// The values follow quantization_cuda_kernel.cu:149-177: T(code) / scale with a real division, + min.
// 1, 2 and 4 bit tabulate the 2^BITS values of a group once and look them up; 8 bit computes
// them per element from one correctly rounded reciprocal per group.
// ------------------------------------------------------------------------------------------------
// value of lane g (0..7) of the row in every lane of the row; g is a constant once the caller's loop is unrolled
__device__ __forceinline__ float row_bcast_at(float v, int g) {
  switch (g) {
    case 0: return row_bcast<0>(v);
    case 1: return row_bcast<1>(v);
    case 2: return row_bcast<2>(v);
    case 3: return row_bcast<3>(v);
    case 4: return row_bcast<4>(v);
    case 5: return row_bcast<5>(v);
    case 6: return row_bcast<6>(v);
    default: return row_bcast<7>(v);
  }
}

template <typename T, int BITS, int SGS, int PARTS = 1, bool LARGE = true, bool SHARE_STATS = true>
__device__ __forceinline__ void dequantize_unit(const uint8_t* __restrict__ packed,
                                                const typename Elem<T>::Stat* __restrict__ scale,
                                                const T* __restrict__ mn, int64_t numel, int64_t N, int64_t unit,
                                                int l, T* __restrict__ out) {
  typedef typename Elem<T>::Stat Stat;
  constexpr int WPT = 8 / BITS;
  constexpr int W = Elem<T>::kDqWidth;
  constexpr int NI = WPT / PARTS;   // groups of a super-group that this unit writes
  constexpr int G = SGS * NI;
  static_assert(PARTS >= 1 && WPT % PARTS == 0 && (PARTS == 1 || SGS == 1), "parts divide one super-group");
  static_assert(G >= 1 && G <= ROW_GROUPS && (G & (G - 1)) == 0, "a dequantize unit is 1, 2, 4 or 8 groups");
  const int64_t sg0 = unit / PARTS * SGS;
  const int part = (int)(unit % PARTS);
  const int64_t n_sg = (N + WPT - 1) / WPT;
  const int64_t g0 = sg0 * WPT + part * NI;   // first group of the unit
  const int rl = l & 15;  // lane within its 16-lane row
  // float at 1 bit keeps the plain nontemporal store on large tensors (and in the batched launch)
  constexpr int POLICY = (sizeof(T) == 4 && BITS == 1 && LARGE) ? GACT_STORE_NT : GACT_STORE_NT_SYSTEM;
  // the wave's output window starts at the first group of its first unit (a wave holds one or two units, in order)
  const int64_t window_first = wave_first(g0) * GROUP;
  const OutWindow window(out + window_first, (numel - window_first) * (int64_t)sizeof(T));
  uint32_t w[SGS][W / 4];
#pragma unroll
  for (int it = 0; it < SGS; it++) {
    const uint8_t* p = packed + (sg0 + it) * GROUP + W * l;
    const bool live = sg0 + it < n_sg;
    if (W == 4) {
      w[it][0] = live ? stream_load(reinterpret_cast<const uint32_t*>(p)) : 0u;
    } else {
      u32x2 t = {0u, 0u};
      if (live) t = stream_load(reinterpret_cast<const u32x2*>(p));
      w[it][0] = t.x;
      w[it][W / 4 - 1] = t.y;
    }
    if (PARTS > 1) {   // this part's fields down to where part 0 has them (the shift is less than a byte)
#pragma unroll
      for (int k = 0; k < W / 4; k++) w[it][k] >>= part * NI * BITS;
    }
  }

  if constexpr (BITS <= 4) {
    // A group has only 2^BITS distinct outputs T(c)/scale + min: 8 * 2^BITS values for the unit.  Its lanes
    // tabulate them - entry e = group * 2^BITS + code in lane e % LPU, pass e / LPU, each with the real
    // division and the real sum - and every element then fetches its value from the lane that holds it
    // (ds_bpermute: the LDS crossbar, no LDS memory).  2 vector instructions per element instead of 6, and
    // one or two divisions per lane (four for half at 4 bit) instead of one per element.
    constexpr int LPU = GROUP / W;
    constexpr int ENT = 1 << BITS, TOT = G * ENT, PASSES = (TOT + LPU - 1) / LPU;
    // Scale and min of the unit's groups.  SHARE_STATS: lane j < G of the unit loads those of group g0 + j - one load
    // instruction each, a handful of lanes active - and the table entries fetch theirs across the unit.  Letting every
    // entry load its own (2 * PASSES instructions, all lanes active, for a fraction of a percent of the bytes) cost the
    // single-tensor kernel 7 % at half 4 bit (67 M elements 30.3 -> 28.2 us) and 4 % at half 2 bit (134 M: 50.5 -> 48.5);
    // with half units of 8 groups sharing loses instead (the batched launch when it had such units: 2 bit 683 -> 705 us,
    // 4 bit 757 -> 812 for 1.83 G elements), and float units, a whole wave each, are within 1 % either way.
    const uint32_t unitbase = (threadIdx.x & 63u) & ~(uint32_t)(LPU - 1);  // first lane of the unit within its wave
    uint32_t tab[PASSES];
    if constexpr (SHARE_STATS) {
      Stat s_mine = (Stat)1.0f, m_mine = (Stat)0.0f;
      if (l < G && g0 + l < N) {
        s_mine = scale[g0 + l];
        m_mine = Elem<T>::stat_of(mn[g0 + l]);
      }
      uint32_t s_bits, m_bits;
      if constexpr (sizeof(Stat) == 4) {
        s_bits = __builtin_bit_cast(uint32_t, s_mine);
        m_bits = __builtin_bit_cast(uint32_t, m_mine);
      } else {
        s_bits = (uint32_t)__builtin_bit_cast(uint16_t, s_mine);
        m_bits = (uint32_t)__builtin_bit_cast(uint16_t, m_mine);
      }
#pragma unroll
      for (int p = 0; p < PASSES; p++) {
        const int e = p * LPU + l;   // entries past the table (e >= TOT) wrap onto a lane of the unit and are never fetched
        const uint32_t src = (unitbase + (uint32_t)((e / ENT) & (G - 1))) << 2;
        const uint32_t sb = (uint32_t)__builtin_amdgcn_ds_bpermute((int)src, (int)s_bits);
        const uint32_t mb = (uint32_t)__builtin_amdgcn_ds_bpermute((int)src, (int)m_bits);
        Stat sv, mv;
        if constexpr (sizeof(Stat) == 4) {
          sv = __builtin_bit_cast(Stat, sb);
          mv = __builtin_bit_cast(Stat, mb);
        } else {
          sv = __builtin_bit_cast(Stat, (uint16_t)sb);
          mv = __builtin_bit_cast(Stat, (uint16_t)mb);
        }
        tab[p] = Elem<T>::table_entry((float)(e & (ENT - 1)), sv, mv);
      }
    } else {
#pragma unroll
      for (int p = 0; p < PASSES; p++) {
        const int e = p * LPU + l;
        const int64_t g = g0 + e / ENT;
        const bool live = e < TOT && g < N;
        tab[p] = Elem<T>::table_entry((float)(e & (ENT - 1)), live ? scale[g] : (Stat)1.0f,
                                      live ? Elem<T>::stat_of(mn[g]) : (Stat)0.0f);
      }
    }
#pragma unroll
    for (int it = 0; it < SGS; it++) {
#pragma unroll
      for (int ni = 0; ni < NI; ni++) {
        const int64_t n = g0 + it * WPT + ni;
        if (n < N) {
          const int g = it * NI + ni;
          const uint32_t base4 = (unitbase + (uint32_t)((g * ENT) % LPU)) << 2;
          T v[W];
#pragma unroll
          for (int e = 0; e < W; e++) {
            const uint32_t c = __builtin_amdgcn_ubfe(w[it][e >> 2], 8 * (e & 3) + ni * BITS, BITS);
            v[e] = Elem<T>::from_bits((uint32_t)__builtin_amdgcn_ds_bpermute((int)((c << 2) + base4), (int)tab[(g * ENT) / LPU]));
          }
          const int64_t at = n * GROUP + W * l;
          if (n * GROUP + GROUP <= numel) {
            Elem<T>::template store_dq<POLICY>(window, (uint32_t)((at - window_first) * (int64_t)sizeof(T)), v);
          } else {
#pragma unroll
            for (int e = 0; e < W; e++)
              if (at + e < numel) out[at + e] = v[e];
          }
        }
      }
    }
    return;
  } else {
  // 8 bit.  scale and min of the unit's groups: 16-byte loads when the whole unit exists and the arrays allow it
  constexpr int PERS = 16 / (int)sizeof(Stat), PERM = 16 / (int)sizeof(T);
  Stat sv[G], mv[G];
  if (G % PERS == 0 && G % PERM == 0 && g0 + G <= N &&
      ((reinterpret_cast<uintptr_t>(scale + g0) | reinterpret_cast<uintptr_t>(mn + g0)) & 15u) == 0) {
    typedef Stat svec __attribute__((ext_vector_type(PERS)));
    typedef T mvec __attribute__((ext_vector_type(PERM)));
#pragma unroll
    for (int c = 0; c < G / PERS; c++) {
      const svec a = *reinterpret_cast<const svec*>(scale + g0 + c * PERS);
#pragma unroll
      for (int e = 0; e < PERS; e++) sv[c * PERS + e] = a[e];
    }
#pragma unroll
    for (int c = 0; c < G / PERM; c++) {
      const mvec m = *reinterpret_cast<const mvec*>(mn + g0 + c * PERM);
#pragma unroll
      for (int e = 0; e < PERM; e++) mv[c * PERM + e] = Elem<T>::stat_of(m[e]);
    }
  } else {
#pragma unroll
    for (int g = 0; g < G; g++) {
      sv[g] = g0 + g < N ? scale[g0 + g] : (Stat)1.0f;
      mv[g] = g0 + g < N ? Elem<T>::stat_of(mn[g0 + g]) : (Stat)0.0f;
    }
  }
  // one correctly rounded reciprocal per group and row instead of one per group and lane: row lane j takes
  // group j % G and the row shares the results; when any scale of the wave is outside the range the
  // reciprocal form is valid for, the wave takes the plain division instead
  const int64_t gm = g0 + (rl & (G - 1));
  const float s_mine = gm < N ? (float)scale[gm] : 1.0f;
  const float r_mine = 1.0f / s_mine;
  const bool by_reciprocal = __builtin_amdgcn_ballot_w64(!reciprocal_safe(s_mine)) == 0;
#pragma unroll
  for (int it = 0; it < SGS; it++) {
    const int64_t n = sg0 + it;
    if (n < N) {
      T v[W];
      if (by_reciprocal) {
        const float sf = (float)sv[it], r = row_bcast_at(r_mine, it);
#pragma unroll
        for (int e = 0; e < W; e++) {
          const int c = (int)__builtin_amdgcn_ubfe(w[it][e >> 2], 8 * (e & 3), 8);
          v[e] = Elem<T>::finish(div_by_reciprocal((float)c, sf, r), mv[it]);
        }
      } else {
#pragma unroll
        for (int e = 0; e < W; e++) {
          const int c = (int)__builtin_amdgcn_ubfe(w[it][e >> 2], 8 * (e & 3), 8);
          v[e] = Elem<T>::finish((float)c / (float)sv[it], mv[it]);
        }
      }
      const int64_t at = n * GROUP + W * l;
      if (n * GROUP + GROUP <= numel) {
        Elem<T>::template store_dq<POLICY>(window, (uint32_t)((at - window_first) * (int64_t)sizeof(T)), v);
      } else {
#pragma unroll
        for (int e = 0; e < W; e++)
          if (at + e < numel) out[at + e] = v[e];
      }
    }
  }
  }
}

// Batched launch: a block owns 128 consecutive groups of one tensor whatever the width, so the grid does
// not depend on the widths.  Quantize: each of the workgroup's 16 rows takes 8 consecutive groups - BITS
// super-groups - in one go: no loop, 16 KB (half) in flight per wave at every width, one scale division per
// lane and 8 groups.
#ifndef GACT_QB_STAGE
#define GACT_QB_STAGE 0 /* groups at a time in the batched quantize rows (0: all 8 at once) */
#endif
template <typename T, int BITS, int NOISE, bool PACKS = true>
__device__ __forceinline__ void quantize_block128(const T* __restrict__ x, int64_t numel, int64_t N, int64_t lb,
                                                  uint8_t* __restrict__ packed,
                                                  typename Elem<T>::Stat* __restrict__ scale_out,
                                                  T* __restrict__ mn_out, uint64_t seed) {
  constexpr int WPT = 8 / BITS;
  const int row = threadIdx.x >> 4, i = threadIdx.x & 15;
  const int64_t sg0 = (lb * 16 + row) * BITS;
  if (NOISE == GACT_NOISE_REF) {
    // one Philox block per output byte: far too much code to lay out for 8 groups at once; super-group by super-group
#pragma unroll 1
    for (int q = 0; q < BITS; q++)
      if ((sg0 + q) * WPT < N)
        quantize_supergroup<T, BITS, NOISE, false, 1>(ContiguousSource<T>{x, numel}, N, sg0 + q, i, packed, scale_out, mn_out, (T*)nullptr,
                                                      (uint32_t)seed, (uint32_t)(seed >> 32), nullptr);
  } else if (sg0 * WPT < N) {
    quantize_supergroup<T, BITS, NOISE, false, BITS, GACT_QB_STAGE, false, PACKS>(ContiguousSource<T>{x, numel}, N, sg0, i, packed, scale_out, mn_out,
                                                                                  (T*)nullptr, (uint32_t)seed, (uint32_t)(seed >> 32), nullptr);
  }
}
// Dequantize: four workgroups share a block of 128 groups, 32 groups each - 4 units of 8 groups for float (a wave
// each), 8 units of 4 groups for half and bfloat16 (half a wave each; at 1 bit a unit is half a super-group and two
// units load the same code words): one unit per slot, several in a row per wave cost 10-20 %.  Half units of 4 groups
// with their scale and min shared across the unit are what the single-tensor kernel prefers on tensors of this size;
// against two workgroups per block and half units of 8 groups (120 half tensors, 1.83 G elements, all at one width):
// 2 bit 696 -> 677 us, 4 bit 758 -> 732, 8 bit 937 -> 929, 1 bit 651 -> 683; a mix of widths 719 -> 687.
template <typename T, int BITS>
__device__ __forceinline__ void dequantize_block128(const uint8_t* __restrict__ packed,
                                                    const typename Elem<T>::Stat* __restrict__ scale,
                                                    const T* __restrict__ mn, int64_t numel, int64_t N, int64_t lb,
                                                    int quarter, T* __restrict__ out) {
  constexpr int LPU = GROUP / Elem<T>::kDqWidth;  // lanes per unit
  constexpr int SLOTS = 256 / LPU;                // units of the workgroup
  const int slot = threadIdx.x / LPU, l = threadIdx.x % LPU;
  if constexpr (LPU == 64) {
    const int64_t unit = lb * 16 + quarter * SLOTS + slot;   // units of 8 groups
    if (unit * 8 < N) dequantize_unit<T, BITS, BITS, 1, true, false>(packed, scale, mn, numel, N, unit, l, out);
  } else {
    const int64_t unit = lb * 32 + quarter * SLOTS + slot;   // units of 4 groups
    constexpr int SGS = BITS == 1 ? 1 : BITS / 2, PARTS = BITS == 1 ? 2 : 1;
    if (unit * 4 < N) dequantize_unit<T, BITS, SGS, PARTS, true, true>(packed, scale, mn, numel, N, unit, l, out);
  }
}

// Row min/max only (the minimax entry point at D = 256): a 16-lane row takes MINIMAX_ROW_GROUPS consecutive
// groups, issues all their loads, reduces them one after the other and lets lane g store the results of group g.
// One group per row in one-wave workgroups (4 KB per float wave) reads fastest.  float, buffers cold in every cache,
// 1 group per row in 64-thread workgroups / 2 in 256 / 4 in 256 / 8 in 256: 4 M elements 4.68 / 4.81 / 5.44 / 5.94 us,
// 43 M 26.6 / 26.9 / 29.0 / 31.9, 103 M 60.3 / 61.6 / 61.8 / 65.6, 256 M 148.9 / 155.1 / 155.6 / 159; half 17 M
// 6.81 / 7.16 / 7.30 / 8.39, 256 M 72.3 / 74.8 / 75.7 / 77.7.
#define MINIMAX_ROW_GROUPS 1
#define MINIMAX_THREADS 64
template <typename T>
__device__ __forceinline__ void minimax_row(const T* __restrict__ x, int64_t N, int64_t row, int i,
                                            T* __restrict__ mn, T* __restrict__ mx) {
  const int64_t n0 = row * MINIMAX_ROW_GROUPS;
  typename Elem<T>::Store v[MINIMAX_ROW_GROUPS];
#pragma unroll
  for (int g = 0; g < MINIMAX_ROW_GROUPS; g++)
    if (n0 + g < N) load_group<T>(x, N * GROUP, n0 + g, i, v[g]);
  T lo_m = (T)0.0f, hi_m = (T)0.0f;
#pragma unroll
  for (int g = 0; g < MINIMAX_ROW_GROUPS; g++) {
    if (n0 + g < N) {
      T lo, hi;
      Elem<T>::template groups_minmax<1>(v + g, &lo, &hi);
      lo_m = i == g ? lo : lo_m;
      hi_m = i == g ? hi : hi_m;
    }
  }
  if (i < MINIMAX_ROW_GROUPS && n0 + i < N) {
    mn[n0 + i] = lo_m;
    mx[n0 + i] = hi_m;
  }
}

// ------------------------------------------------------------------------------------------------
// Single-tensor kernels.
// ------------------------------------------------------------------------------------------------

// Workgroups go to the 8 XCDs round-robin (workgroup b runs on XCD b % 8) and every XCD streams through its
// own L2.  With the plain mapping an XCD sees every 8th tile, i.e. addresses in which three bits never
// change; handing each XCD runs of RUN consecutive tiles instead lets its writes leave as contiguous
// stretches (pure-write kernels with 8 KB per wave: 5.4 -> 6.2 TB/s).  The tail that does not fill a
// round of 8 * RUN tiles keeps the plain mapping.  RUN = 0 switches the remapping off.
#ifndef GACT_XCD_RUN_DQ
#define GACT_XCD_RUN_DQ 16
#endif
#ifndef GACT_XCD_RUN_DQB
#define GACT_XCD_RUN_DQB 16 /* batched dequantize */
#endif
#ifndef GACT_XCD_RUN_QB
#define GACT_XCD_RUN_QB 16 /* batched quantize: 4-6 % over the plain order at every width (120 half tensors, 1.83 G elements) */
#endif
#ifndef GACT_XCD_RUN_Q_LOW
#define GACT_XCD_RUN_Q_LOW 0 /* quantize, 1 bit: the long one-wave workgroups gain nothing or lose (mid-sized tensors 3 %) */
#endif
#ifndef GACT_XCD_RUN_Q
#define GACT_XCD_RUN_Q 128 /* quantize, 2, 4 and 8 bit: 2-6 % (half 2 bit 52.7 -> 50.2 us, float 2 bit 70.1 -> 68.8 us at 134 / 103 M elements) */
#endif
#ifndef GACT_XCD_RUN_TR
#define GACT_XCD_RUN_TR 16 /* quantize of transposed tensors */
#endif
template <uint32_t RUN>
__device__ __forceinline__ uint32_t xcd_tile(uint32_t b, uint32_t nb) {
  if (RUN == 0) return b;
  constexpr uint32_t XCDS = 8, ROUND = XCDS * (RUN ? RUN : 1);
  if (b >= nb / ROUND * ROUND) return b;
  const uint32_t q = b / XCDS, x = b % XCDS;
  return ((q / (RUN ? RUN : 1)) * XCDS + x) * (RUN ? RUN : 1) + q % (RUN ? RUN : 1);
}

// The seed of a launch: a host value plus, optionally, a value read from device memory when the kernel runs -
// so that a launch recorded in a HIP graph draws fresh noise on every replay (the host updates the device word
// between replays).
struct SeedArg {
  uint64_t seed;
  const uint64_t* add;  // device pointer or null
  __device__ __forceinline__ uint64_t value() const { return add ? seed + *add : seed; }
};

// Geometry of the single-tensor quantize launch for an element type and width (1, 2, 4, 8 bit): super-groups per
// row (a row always issues the loads of all its groups first), threads per workgroup, the XCD-aware run of tiles,
// and how many groups at a time a row of whole groups is worked through (0: all at once) - `stage` in general,
// `stage_small` for tensors of fewer than `small_below` groups - with each stage issuing its own loads (`lazy`,
// `lazy_small`) instead of the row issuing all of them first.  Overridable at compile time
// (-DGACT_QGEOM_F32=..., _F16, _BF16) for experiments.
struct QGeom { int sgr, threads, run, stage, stage_small, small_below; bool lazy, lazy_small; };
#ifndef GACT_QGEOM_F16
#define GACT_QGEOM_F16 {{1, 64, 0, 4, 4, 1 << 15, true, false}, {1, 64, 128, 2, 2, 1 << 17, true, true}, {1, 64, 128, 1, 1, 0, true, true}, {1, 64, 128, 0, 0, 0, false, false}}
#endif
#ifndef GACT_QGEOM_BF16
#define GACT_QGEOM_BF16 {{1, 64, 0, 4, 4, 1 << 15, true, false}, {1, 64, 128, 2, 2, 0, true, true}, {1, 64, 128, 1, 1, 0, true, true}, {1, 64, 128, 0, 0, 0, false, false}}
#endif
// Staging pays where few waves share a SIMD and costs its extra divisions elsewhere.  float, quantize alone:
//   1 bit, 4 groups at a time: 8 M elements 9.8 -> 8.4 us, 17 M 14.5 -> 13.6, 34 M unchanged, 43 M 32.0 -> 32.4;
//   2 bit, group by group: 4 M 5.70 -> 5.51 us, 103 M 69.0 -> 67.8; two at a time is 2 % better still at 4 M and
//     1-2 % worse from 17 M on;  4 bit, group by group: 4 M 5.88 -> 5.73 us, unchanged at 103 M.
// half: 1 bit, 4 groups at a time: 4 M elements 6.7 -> 6.3 us, 17 M 11.8 -> 10.5, 67 M 29.0 -> 28.3;  2 bit, two at a
//   time: 2 % faster up to 17 M, 2 % slower at 67 M and 134 M (group by group: 3-8 % slower);  4 bit: within 1 %.
//   8 bit in one-wave workgroups: 4 M elements 4.78 -> 4.41 us, 17 M 10.7 -> 10.5, 67 M 32.3 -> 31.8 (4 bit and float 8 bit lose 1-5 % that way).
//   stages that issue their own loads: 1 bit 4 M elements 6.27 -> 6.67 us, 17 M 10.4 -> 10.1, 34 M 16.3 -> 15.9, 134 M 49.8 -> 49.0
//   (hence from 2^15 groups on);  2 bit, two at a time: 4 M unchanged, 17 M 10.0 -> 9.2, 26 M 13.8 -> 12.9, 134 M 51.0 -> 49.5,
//   256 M 93.0 -> 91.5 (bfloat16 67 M: 27.8 -> 26.4);  4 bit, group by group: 8 M 6.66 -> 6.3, 67 M and 256 M within 1 %.
//   float: 1 bit, four at a time: 4 M 6.5 -> 7.5 us, 17 M 13.6 -> 12.8, 103 M 69.3 -> 67.5, 256 M 170 -> 167 (from 2^15 groups on);
//   4 bit group by group: 4 M 5.64 -> 5.41, 8 M 8.29 -> 8.15, larger within 1 %;  2 bit within 2 % either way: not used.
#ifndef GACT_QGEOM_F32
#define GACT_QGEOM_F32 {{1, 64, 0, 4, 4, 1 << 15, true, false}, {1, 64, 128, 1, 2, 1 << 15, false, false}, {1, 64, 128, 1, 1, 0, true, true}, {1, 256, 128, 0, 0, 0, false, false}}
#endif
template <typename T>
__host__ __device__ constexpr QGeom q_geom(int bits) {
  constexpr QGeom f32[4] = GACT_QGEOM_F32, f16[4] = GACT_QGEOM_F16, b16[4] = GACT_QGEOM_BF16;
  const int k = bits == 1 ? 0 : bits == 2 ? 1 : bits == 4 ? 2 : 3;
  return Elem<T>::kDtype == GACT_F32 ? f32[k] : Elem<T>::kDtype == GACT_F16 ? f16[k] : b16[k];
}

// Geometry of the single-tensor dequantize launch for 1, 2, 4 and 8 bit: super-groups per unit, parts a
// super-group is split into (sgs = 1 then), threads per workgroup, XCD-aware run of tiles - and the same pair
// (sgs, parts) for large tensors (`large_from` groups and more), with the bytes of dynamic LDS a workgroup
// of 256 threads asks for from `cap_from` groups on without touching them (0: none; see the occupancy caps below).
// Units are 4 or 8 groups; units of 1 or 2 groups cost 10-150 %: every unit pays its code loads, its table and its
// divisions.  Dequantize alone, us, units of 4 against units of 8 (no cap), by groups in the tensor:
//   float 1 bit  65 536: 13.95 / 12.29   100 000: 20.0 / 18.4    (2 and 4 bit alike: 8)
//   float 8 bit  65 536: 15.76 / 15.98   100 000: 23.2 / 23.7    (4, and 8 with the cap from 2^17 groups)
//   half  1 bit  16 384: 3.86 / 4.36   65 536: 6.8 / 7.4   81 920: 10.3 / 8.8   98 304: 10.4 / 10.4   130 000: 14.2 / 13.3
//                (8 from 73 728 groups; capped at 6 workgroups per CU from 2^18 groups: 67 M elements 25.7 -> 24.8 us, 134 M
//                48.8 -> 46.7, 268 M 98.3 -> 90.4, while the same cap costs 6-12 % at 29-34 M; 2 and 4 bit lose 2-30 % by any cap)
//   half  2 bit  16 384: 3.87 / 4.73   65 536: 7.41 / 8.15   130 000: 14.5 / 13.8   1 M: 94.6 / 99.4   (4 throughout)
//   half  4 bit  16 384: 4.39 / 5.05   65 536: 8.08 / 8.95   200 000: 24.0 / 24.0   401 408: 45.0 / 46.7   1 M: 105.1 / 106.7
//   half  8 bit  65 536: 9.21 / 9.40   130 000: 18.0 / 18.2
struct DqGeom { int sgs, parts, threads, run, sgs_large, parts_large; unsigned lds_large; int large_from, cap_from; };
#ifndef GACT_DQGEOM_F32
#define GACT_DQGEOM_F32 {{1, 1, 256, GACT_XCD_RUN_DQ, 1, 1, 53000u, 1 << 17, 1 << 17}, {2, 1, 256, GACT_XCD_RUN_DQ, 2, 1, 53000u, 1 << 17, 1 << 17}, \
                         {4, 1, 256, GACT_XCD_RUN_DQ, 4, 1, 53000u, 1 << 17, 1 << 17}, {4, 1, 256, GACT_XCD_RUN_DQ, 8, 1, 53000u, 1 << 17, 1 << 17}}
#endif
#ifndef GACT_DQGEOM_F16
#define GACT_DQGEOM_F16 {{1, 2, 256, GACT_XCD_RUN_DQ, 1, 1, 26000u, 9 << 13, 1 << 18}, {1, 1, 256, GACT_XCD_RUN_DQ, 1, 1, 0u, 1 << 17, 1 << 17}, \
                         {2, 1, 256, GACT_XCD_RUN_DQ, 2, 1, 0u, 3 << 15, 3 << 15}, {4, 1, 256, GACT_XCD_RUN_DQ, 8, 1, 40000u, 1 << 17, 1 << 17}}
#endif
template <typename T>
__host__ __device__ constexpr DqGeom dq_geom(int bits) {
  constexpr DqGeom f32[4] = GACT_DQGEOM_F32, f16[4] = GACT_DQGEOM_F16;
  const int k = bits == 1 ? 0 : bits == 2 ? 1 : bits == 4 ? 2 : 3;
  return sizeof(T) == 4 ? f32[k] : f16[k];
}
__host__ __device__ constexpr int dq_unit_groups(DqGeom d, int bits, bool large) {
  return (large ? d.sgs_large : d.sgs) * (8 / bits) / (large ? d.parts_large : d.parts);
}

// The seed, a structure, comes first: the library is built with the kernels' leading scalar arguments preloaded into
// registers, which pays for dequantize and costs the quantize kernels up to 0.5 % - a structure is not preloaded,
// nor is anything behind it.
template <typename T, int BITS, int NOISE, bool GIVEN, bool SMALL = false>
__global__ void __launch_bounds__(256)
quantize_kernel(SeedArg seed_arg, const T* __restrict__ x, int64_t numel, int64_t N, uint8_t* __restrict__ packed,
                typename Elem<T>::Stat* __restrict__ scale_out, T* mn_io, T* mx_io, const float* __restrict__ noise) {
  constexpr QGeom G = q_geom<T>(BITS);
  constexpr int STAGE = SMALL ? G.stage_small : G.stage;
  constexpr bool LAZY = SMALL ? G.lazy_small : G.lazy;
  constexpr int SGR = NOISE == GACT_NOISE_REF ? 1 : G.sgr;   // the reference stream's code is too long to lay out several times
  // Tiles are handed out last first: the tensor's last tile - the only one that can be ragged, and then slower than
  // the others (169 343 float groups at 1 bit: 33.4 us when it is dispatched last, 31.6 when first) - goes to the
  // first workgroup instead of being the one the end of the kernel waits for.
  const uint32_t tile = gridDim.x - 1u - xcd_tile<(uint32_t)G.run>(blockIdx.x, gridDim.x);
  const int64_t sg0 = ((int64_t)tile * (blockDim.x >> 4) + (threadIdx.x >> 4)) * SGR;
  if (sg0 * (8 / BITS) >= N) return;
  const uint64_t seed = seed_arg.value();
  // half at 2 bit: packed bytes leave registers for seven waves on a SIMD instead of five, which helps while a tensor does not fill the
  // chip for long and costs bandwidth on large ones (4 M elements 4.53 -> 4.35 us, 17 M 8.7 -> 8.4, 51 M and 72 M equal, 134 M 49.7 -> 51.3, 268 M 96 -> 100; a cap
  // by dynamic LDS at five or four waves gets half of that back)
  constexpr bool PACKS = SMALL || !(std::is_same<T, f16>::value && BITS == 2 && NOISE != GACT_NOISE_REF);
  // bfloat16 widens here: ordered minima leave registers for more waves than HBM bears (67 M elements 1 bit 26.7 -> 27.5 us, 2 bit 25.7 -> 26.9,
  // 8 M 5.58 -> 5.67), where batches (three waves on a SIMD instead of two: 686 M 562 -> 548 us a round trip, 83 M 97.5 -> 95.5), runs of
  // pieces (heads [64,12,512,64] 4 bit 14.1 -> 13.9) and tiles gain; strips are apart (see there)
  constexpr bool ORDERED = !std::is_same<T, bf16>::value;
  quantize_supergroup<T, BITS, NOISE, GIVEN, SGR, STAGE, LAZY, PACKS, ORDERED>(ContiguousSource<T>{x, numel}, N, sg0, threadIdx.x & 15, packed, scale_out, mn_io, mx_io,
                                                  (uint32_t)seed, (uint32_t)(seed >> 32), noise);
}

// ------------------------------------------------------------------------------------------------
// Quantize at 1 bit with a wave per super-group: row r takes groups 2r and 2r + 1 of the 8 whose codes share bytes, the
// four rows OR their partial bytes together (two ds_bpermute steps on 4 dwords) and each then stores its quarter of the
// super-group's 256 bytes.  A wave holds 8 KB (float) or 4 KB (half) where a row per super-group makes it hold 32 or
// 16 KB and, with its 175 registers, leaves room for two waves per SIMD: 65 536 float groups are exactly one round of
// such waves, and the row form's time steps up with every further round (65 536 groups 12.9 us, 69 632: 16.2) where
// this form grows evenly (13.5, 14.4).  Float, us, row form / this form, by groups: 8 192: 5.3 / 4.8   32 768: 9.5 / 8.3
// 49 152: 11.3 / 10.8   57 344 .. 65 536: 11.8 .. 12.9 / 12.1 .. 13.5   73 728: 16.8 / 14.9   98 304: 19.7 / 19.4
// 131 072: 25.2 / 24.2   169 343: 31.4 / 30.7   229 376: 40.9 / 40.4   262 144 and more: equal.  Half: 8 192: 5.1 / 4.7
// 16 384: 5.4 / 4.6   32 768: 6.7 / 6.6   49 152: 8.2 / 8.3   65 536 and more: 9.2 / 9.9 .. 48.8 / 51.2.  At 2 bit (one
// group per row) there is nothing in it at any size.  Same results as quantize_kernel; not for the reference stream.
// ------------------------------------------------------------------------------------------------
#ifndef GACT_W8_RUN
#define GACT_W8_RUN 32
#endif
__device__ __forceinline__ uint32_t pack4(const uint32_t* b) {
  // the reference accumulates in a uint8_t: keep the low 8 bits of every byte
  return (b[0] & 0xffu) | ((b[1] & 0xffu) << 8) | ((b[2] & 0xffu) << 16) | (b[3] << 24);
}
template <typename T, int BITS, int NOISE, typename SRC>
__device__ __forceinline__ void quantize_wave8(const SeedArg& seed_arg, const SRC& src, int64_t sg, int64_t N, uint8_t* __restrict__ packed,
                                               typename Elem<T>::Stat* __restrict__ scale_out, T* __restrict__ mn_out,
                                               T* __restrict__ mx_out, const float* __restrict__ noise) {
  static_assert(NOISE != GACT_NOISE_REF, "the reference stream draws per output byte");
  static_assert(BITS == 1 || BITS == 2, "four rows share a super-group: two groups a row at 1 bit, one at 2 bit");
  typedef typename Elem<T>::Stat Stat;
  constexpr int WPT = 8 / BITS, GR = WPT / 4, QMAX = (1 << BITS) - 1;   // GR: groups of a row
  constexpr int CH = Elem<T>::kQChunks, W = Elem<T>::kQWidth;
  const int64_t n0 = sg * WPT;
  if (n0 >= N) return;   // the whole wave
  const int lane = threadIdx.x & 63, r = lane >> 4, i = lane & 15;
  const int64_t na = n0 + GR * r;   // the row's first group
  const uint64_t seed = seed_arg.value();
  const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);

  typename Elem<T>::Store v[GR];
#pragma unroll
  for (int g = 0; g < GR; g++)
    if (na + g < N) src.load(na + g, i, v[g]);
  Stat lo[GR], hi[GR], sc[GR];
  constexpr bool ORDERED = !(std::is_same<T, bf16>::value && SRC::kContiguous);   // see quantize_kernel
  Elem<T>::template groups_minmax<GR, ORDERED>(v, lo, hi, N - na);
  {
    const int mine = i & (GR - 1);   // with two groups a row, odd lanes divide for the second
    const Stat lo_m = mine ? lo[GR - 1] : lo[0], hi_m = mine ? hi[GR - 1] : hi[0];
    const Stat s_m = Elem<T>::make_scale(lo_m, hi_m, QMAX);
    if (i < GR && na + i < N) {
      scale_out[na + i] = s_m;
      mn_out[na + i] = Elem<T>::elem_of(lo_m);
      if (mx_out) mx_out[na + i] = Elem<T>::elem_of(hi_m);
    }
    sc[0] = GR == 1 ? s_m : row_bcast<0>(s_m);
    if (GR > 1) sc[GR - 1] = row_bcast<1>(s_m);
  }

  constexpr bool PK = packs_bytes<T, BITS, NOISE, false>();
  uint32_t bytes[CH][W];
  uint32_t words[CH][W / 4];   // PK
#pragma unroll
  for (int k = 0; k < CH; k++) {
#pragma unroll
    for (int e = 0; e < W; e++) bytes[k][e] = 0;
#pragma unroll
    for (int d = 0; d < W / 4; d++) words[k][d] = 0;
  }
  FastRow<T, GR> fast;
#pragma unroll
  for (int g = 0; g < GR; g++) {
    const int64_t n = na + g;
    const uint32_t shift = (uint32_t)((GR * r + g) * BITS);   // the group's field within its bytes
    if (n < N) {
      if constexpr (PK) {
        float cd[CH / 2][W];
        if (NOISE == GACT_NOISE_FAST) fast.draws(g, na, i, k0, k1, cd);
#pragma unroll
        for (int k = 0; k < CH; k++) {
          uint32_t w[W / 4];
          chunk_words<T, NOISE>(v[g], k, lo[g], sc[g], cd, w);
#pragma unroll
          for (int d = 0; d < W / 4; d++) words[k][d] |= field_of<Elem<T>::kExactField>(w[d], shift);
        }
      } else {
#pragma unroll
        for (int k = 0; k < CH; k++) {
          float u[W];
          if (NOISE == GACT_NOISE_INJECT) {
            Elem<T>::load_noise(noise + n * GROUP + chunk_col<T>(k, i), u);
          } else {
#pragma unroll
            for (int e = 0; e < W; e++) u[e] = 0.5f;
          }
          uint32_t c[W];
          Elem<T>::template codes<NOISE == GACT_NOISE_CONST, false>(v[g], k, lo[g], sc[g], u, c);
#pragma unroll
          for (int e = 0; e < W; e++) bytes[k][e] |= c[e] << shift;
        }
      }
      if (!PK && Elem<T>::kRepairsInfiniteScale && Elem<T>::scale_is_inf(sc[g])) {   // rare, see Elem<T>::kRepairsInfiniteScale
#pragma unroll
        for (int k = 0; k < CH; k++)
#pragma unroll
          for (int e = 0; e < W; e++)
            if (Elem<T>::above(v[g], k, e, lo[g])) bytes[k][e] |= 0xffffffffu << shift;
      }
    }
  }

  // the lane's 16 bytes as 4 dwords in the order of their addresses, OR-ed over the four rows (every lane of the wave
  // is here: only whole waves left above)
  uint32_t pk[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    pk[j] = PK ? words[j * 4 / W][(j * 4) % W / 4] : pack4(&bytes[j * 4 / W][(j * 4) % W]);
    pk[j] |= (uint32_t)__shfl_xor((int)pk[j], 16, 64);
    pk[j] |= (uint32_t)__shfl_xor((int)pk[j], 32, 64);
  }
  // row r stores dword r of every lane: float chunk r; half chunk r / 2, its columns 4 (r % 2) .. - 256 contiguous
  // bytes per store instruction either way
  const uint32_t mine = r == 0 ? pk[0] : r == 1 ? pk[1] : r == 2 ? pk[2] : pk[3];
  const int col = W == 4 ? chunk_col<T>(r, i) : chunk_col<T>(r >> 1, i) + 4 * (r & 1);
  stream_store(mine, reinterpret_cast<uint32_t*>(packed + sg * GROUP + col));
}
template <typename T, int BITS, int NOISE>
__global__ void __launch_bounds__(256)
quantize_wave8_kernel(SeedArg seed_arg, const T* __restrict__ x, int64_t numel, int64_t N, uint8_t* __restrict__ packed,
                      typename Elem<T>::Stat* __restrict__ scale_out, T* __restrict__ mn_out, T* __restrict__ mx_out,
                      const float* __restrict__ noise) {
  const uint32_t tile = gridDim.x - 1u - xcd_tile<GACT_W8_RUN>(blockIdx.x, gridDim.x);   // last tile first, see quantize_kernel
  const int64_t sg = (int64_t)tile * (blockDim.x >> 6) + (threadIdx.x >> 6);               // the wave's super-group
  quantize_wave8<T, BITS, NOISE>(seed_arg, ContiguousSource<T>{x, numel}, sg, N, packed, scale_out, mn_out, mx_out, noise);
}

// ------------------------------------------------------------------------------------------------
// Quantize a tensor that is not contiguous, without a contiguous copy of it: groups are consecutive elements in the order of
// the tensor's indices, wherever they lie.  The copy these kernels replace is torch's element-wise one, 0.5-2 TB/s: half
// channels-last [64,256,56,56], 4 bit, 223 us of copy and 20 of quantize -> 37; [64,512,28,28] 107 + 12 -> 23; half heads
// [64,12,197,64] 14 + 7 -> 8; small tensors lose a launch ([2,12,197,64] 3.6 + 3.5 -> 4.6).
// ------------------------------------------------------------------------------------------------
// Innermost runs contiguous (GatherSource): quantize_kernel - at 1 and 2 bit quantize_wave8_kernel, whatever the size: a row
// of 8 or 4 groups would hold 8 to 32 addresses in flight (heads [2,12,197,64] float 2 bit 11.2 -> 4.9 us) - with an
// address per 16-byte piece.
template <typename T, int BITS, int NOISE>
__global__ void __launch_bounds__(256)
quantize_gather_kernel(SeedArg seed_arg, const T* __restrict__ x, int64_t numel, int64_t N, uint8_t* __restrict__ packed,
                       typename Elem<T>::Stat* __restrict__ scale_out, T* mn_out, T* mx_out, GatherShape shape) {
  const uint32_t tile = gridDim.x - 1u - xcd_tile<GACT_XCD_RUN_Q>(blockIdx.x, gridDim.x);
  if constexpr (BITS <= 2) {
    quantize_wave8<T, BITS, NOISE>(seed_arg, GatherSource<T>{x, numel, shape}, (int64_t)tile * (blockDim.x >> 6) + (threadIdx.x >> 6), N,
                                   packed, scale_out, mn_out, mx_out, nullptr);
    return;
  }
  const int64_t sg = (int64_t)tile * (blockDim.x >> 4) + (threadIdx.x >> 4);
  if (sg * (8 / BITS) >= N) return;
  const uint64_t seed = seed_arg.value();
  quantize_supergroup<T, BITS, NOISE, false>(GatherSource<T>{x, numel, shape}, N, sg, threadIdx.x & 15, packed, scale_out, mn_out, mx_out,
                                             (uint32_t)seed, (uint32_t)(seed >> 32), nullptr);
}

// Innermost dimension strided, the one before it contiguous (channels-last activations seen as [batch, channels, pixels], a
// transposed matrix): a workgroup owns `tile` consecutive elements of the tensor in index order - whole channels and parts
// of channels - and brings them into LDS in that order: it walks the memory rows (one pixel, all channels side by side) that hold
// them in 16-byte pieces and scatters each piece's elements, one channel each, to where they belong.  Rows of 16 lanes then
// quantize super-groups out of LDS.  Neighbouring tiles read other channels of the same memory rows; they run on one XCD at about
// the same time (xcd_tile), so a line that several of them share comes from HBM once and from that XCD's L2 afterwards.
// Bound by its two phases standing one behind the other: half [64,256,56,56] at 4 bit (which takes strips) 54 us, of which reading
// and scattering alone take 33 and quantizing out of LDS alone 27 (with more, smaller workgroups 41 and 21, together 51).  Half
// [64,512,28,28] at 4 bit, 21 us on one buffer, 32 from HBM: 2.1 waves per SIMD on average, which wait for memory and barriers 0.39
// and for their turn to issue 0.35 of their lives; the vector units issue 0.37 of the cycles, LDS conflicts take 0.09; it reads 1.24
// times its bytes from HBM.
struct TransposedShape {
  int64_t sb, sk;          // strides of batch and pixel, in elements
  uint32_t M, K;           // channels of a batch entry, pixels
  int64_t channels;        // of all batch entries
  int tile;                // elements of a workgroup, a multiple of 2048
};
// The tile in LDS: 16 bytes of padding after every group keep the elements of channels a power of two of pixels apart out of
// each other's banks.  `at` in elements; groups start on 16-byte boundaries.
template <typename T>
__host__ __device__ __forceinline__ constexpr uint32_t tile_byte(uint32_t at) { return at * (uint32_t)sizeof(T) + (at / GROUP) * 16u; }
template <typename T>
constexpr unsigned tile_bytes(int tile) { return tile_byte<T>((uint32_t)tile) + 16u; }   // and a spare place
template <typename T>
struct TileSource {
  static constexpr bool kContiguous = false;
  const uint8_t* tile;
  int64_t n_first;
  __device__ __forceinline__ void load(int64_t n, int i, typename Elem<T>::Store& st) const {
    const uint8_t* p = tile + (uint32_t)(n - n_first) * (GROUP * (uint32_t)sizeof(T) + 16u);
#pragma unroll
    for (int k = 0; k < Elem<T>::kQChunks; k++) Elem<T>::load_chunk(reinterpret_cast<const T*>(p) + chunk_col<T>(k, i), st, k);
  }
};
#define TRANSPOSED_THREADS 512
// ROWS neighbouring pixels of a piece per lane and step (the host picks as many as divide the number of pixels, up to 16
// bytes of them): turned around in registers, they are one LDS write per channel.
template <int ROWS> struct TransposedUnroll { static constexpr int value = ROWS >= 8 ? 1 : ROWS >= 4 ? 2 : 4; };   // steps in flight
template <typename T, int BITS, int NOISE, int ROWS>
__global__ void __launch_bounds__(TRANSPOSED_THREADS)
quantize_transposed_kernel(SeedArg seed_arg, const T* __restrict__ x, int64_t numel, int64_t N, uint8_t* __restrict__ packed,
                           typename Elem<T>::Stat* __restrict__ scale_out, T* mn_out, T* mx_out, TransposedShape g) {
  extern __shared__ u32x4 tile_lds[];
  uint8_t* const tile = reinterpret_cast<uint8_t*>(tile_lds);
  constexpr int W = Elem<T>::kQWidth, WPT = 8 / BITS, U = TransposedUnroll<ROWS>::value, WAVES = TRANSPOSED_THREADS / 64;
  constexpr uint32_t ES = sizeof(T);
  static_assert(ROWS * ES <= 16, "one LDS write per channel");
  const int64_t E0 = (int64_t)xcd_tile<GACT_XCD_RUN_TR>(blockIdx.x, gridDim.x) * g.tile;
  const int L = numel - E0 < g.tile ? (int)(numel - E0) : g.tile;   // the grid has no tile past the end: at least 1
  const int64_t ch0 = E0 / g.K, ch1 = (E0 + L - 1) / g.K;           // channels, counted over all batch entries
  // the pixels of the tile: all of them, or (a tile smaller than a channel) L of them from its first one on, around the end
  const uint32_t k_first = (uint32_t)L < g.K ? (uint32_t)(E0 - ch0 * g.K) : 0u;
  const uint32_t steps = ((uint32_t)L < g.K ? (uint32_t)L : g.K) / ROWS;
  const int64_t piece0 = ch0 / W;
  const uint32_t pieces = (uint32_t)(ch1 / W - piece0) + 1;         // 16-byte pieces of a memory row
  // a wave takes up to 8 pieces (128 bytes) side by side and as many rows as its lanes reach; the waves share the blocks
  const uint32_t side = pieces < 8 ? pieces : 8, lane = threadIdx.x & 63;
  const uint32_t rl = (uint32_t)(((float)lane + 0.5f) / (float)side), cl = lane - rl * side;
  const uint32_t steps_at_once = 64u / side;
  const uint32_t down = (steps + steps_at_once * U - 1) / (steps_at_once * U), across = (pieces + side - 1) / side;
  // memory offsets are 32-bit, from the batch entry of the tile's first channel on (the host makes sure that they suffice)
  const uint32_t b0 = (uint32_t)(ch0 / g.M);
  const uint8_t* const base = reinterpret_cast<const uint8_t*>(x) + (int64_t)b0 * g.sb * ES;
  const uint32_t row_bytes = (uint32_t)g.sk * ES, outside = (uint32_t)g.tile;
  for (uint32_t block = threadIdx.x >> 6; block < down * across; block += WAVES) {
    const uint32_t c0 = block / down, r0 = (block - c0 * down) * (steps_at_once * U) + rl;
    const int64_t ch = (piece0 + c0 * side + cl) * W;   // the piece's first channel; M is a multiple of W: one batch entry holds it
    const bool live = rl < steps_at_once && c0 * side + cl < pieces && ch < g.channels;
    const uint32_t b = live ? (uint32_t)ch / g.M : b0;
    const uint32_t column = ((b - b0) * (uint32_t)g.sb + (live ? (uint32_t)ch - b * g.M : 0u)) * ES;
    const int at0 = (int)(ch * (int64_t)g.K - E0);      // where the first channel's pixel 0 belongs (may lie outside)
    u32x4 v[U][ROWS];
    uint32_t k[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint32_t r = r0 + u * steps_at_once;
      k[u] = k_first + ROWS * r;
      k[u] = k[u] >= g.K ? k[u] - g.K : k[u];
      if (live && r < steps) {
        const uint32_t from = column + k[u] * row_bytes;
#pragma unroll
        for (int j = 0; j < ROWS; j++) v[u][j] = *reinterpret_cast<const u32x4*>(base + (from + j * row_bytes));
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (live && r0 + u * steps_at_once < steps) {
#pragma unroll
        for (int e = 0; e < W; e++) {
          // channels of other tiles (before this one: a huge unsigned number) go to a spare place behind the tile
          const uint32_t at = (uint32_t)(at0 + (int)(e * g.K)) + k[u];
          uint8_t* const to = tile + tile_byte<T>(at < outside ? at : outside);
          if constexpr (ES == 4 && ROWS == 4) {
            *reinterpret_cast<u32x4*>(to) = u32x4{v[u][0][e], v[u][1][e], v[u][2][e], v[u][3][e]};
          } else if constexpr (ES == 4) {
            *reinterpret_cast<uint32_t*>(to) = v[u][0][e];
          } else if constexpr (ROWS == 1) {
            *reinterpret_cast<uint16_t*>(to) = (uint16_t)(v[u][0][e / 2] >> (16 * (e & 1)));
          } else {
            uint32_t pair[ROWS / 2];
#pragma unroll
            for (int j = 0; j < ROWS / 2; j++)
              pair[j] = __builtin_amdgcn_perm(v[u][2 * j + 1][e / 2], v[u][2 * j][e / 2], e & 1 ? 0x07060302u : 0x05040100u);
            if constexpr (ROWS == 8) *reinterpret_cast<u32x4*>(to) = u32x4{pair[0], pair[1], pair[2], pair[3]};
            else *reinterpret_cast<u32x2*>(to) = u32x2{pair[0], pair[1]};
          }
        }
      }
    }
  }
  for (uint32_t at = (uint32_t)L + threadIdx.x; at < (uint32_t)g.tile; at += TRANSPOSED_THREADS)   // the padding of the last group
    *reinterpret_cast<T*>(tile + tile_byte<T>(at)) = (T)0.0f;
  __syncthreads();
  const TileSource<T> src{tile, E0 / GROUP};
  if constexpr (BITS == 1) {
    // A wave per super-group: a tile of 64 KB holds 8 (float) or 16 of them, fewer than the workgroup has rows.  A row per super-group / this,
    // us: float [64,512,28,28] 50.2 / 33.7, [110,512,32,32] 98.5 / 58.5, [128,512,14,14] 28.2 / 18.8, [16,64,14,14] 6.7 / 4.7; half equal, and
    // with tiles of 48 KB [256,512,14,14] 22.9 / 19.0.  2 bit: float equal to 5 % slower, half 10 % slower: rows.
    for (int sg = (int)(threadIdx.x >> 6); sg * WPT * GROUP < L; sg += WAVES)
      quantize_wave8<T, BITS, NOISE>(seed_arg, src, E0 / (WPT * GROUP) + sg, N, packed, scale_out, mn_out, mx_out, (const float*)nullptr);
  } else {
    const uint64_t seed = seed_arg.value();
    for (int sg = (int)(threadIdx.x >> 4); sg * WPT * GROUP < L; sg += TRANSPOSED_THREADS / 16)
      // bfloat16 with ordered minima, whose registers let three workgroups onto a CU: [256,512,14,14] 2 bit 24.3 -> 20.3 us, 4 bit 20.2 -> 19.4
      quantize_supergroup<T, BITS, NOISE, false>(
          src, N, E0 / (WPT * GROUP) + sg, threadIdx.x & 15, packed, scale_out, mn_out, mx_out, (uint32_t)seed, (uint32_t)(seed >> 32), nullptr);
  }
}

// The same layout where channels are long (K pixels hold a super-group and more): a workgroup owns a strip of channels, 64 bytes
// of every memory row, and walks along the pixels in steps of GS chunks of 256, the next step's loads in flight while it works on
// the one before.  It quantizes the units - a super-group, or GS groups where that is more - that begin in its channels.  These
// begin at another pixel in every channel (first_pixel), so a step completes GS groups of each channel whose head came with
// the step before: LDS holds two steps' groups per channel, in turn.  A unit that runs past its channel's last pixel ends in
// the next channel: past the end the walk goes on at the first pixels with every column belonging to the channel before it.  A
// strip can be cut into segments of whole units, for more workgroups than there are strips; a segment reads up to a unit of
// pixels beyond its own.
// Bound by the chain of a step - loads, scatter, barrier, quantize, barrier - with few waves to overlap it: half [64,256,56,56] at
// 4 bit 37 us with inputs in rotation, 32 on one buffer, 56 from HBM.  256 CUs hold its 512 workgroups at once (of the two on a CU
// the one dispatched second takes a fifth longer): 1.4 waves per SIMD on average, waiting 0.46 of their lives (from HBM 0.63), with
// 0.44 of the cycles issuing vector instructions and LDS conflicts 0.06; it reads 1.18 times its bytes from HBM.  With GS = 1 it
// took 42; more waves through more segments cost more reading than they hide (44), and dropping one of the two barriers by a
// ring of four slots changed nothing (41.8).  (36.8 since codes are packed by conversions, [64,64,112,112] 1 bit 53.0 -> 48.8.)
// What its 37 us are made of, each part taken out of a copy: the walk's reads alone 24.7 (a linear read of the tensor 16.5), with the
// scatter 26.6, with everything but the stores 31 to 33.  Of the two workgroups on a CU the first takes 2.8 us a step and the
// second 6, until the first has ended at 22 us and leaves the second 3.1 us a step and the CU half empty.  None of these changed it by more than 1 %:
// twice the waves (512 threads), strips of 128 bytes (one workgroup of 1024), no reading beyond the channel's end (the first step's
// pixels kept in registers), the stores held back until the next loads have arrived, priorities by progress.
// What did: the loads of a step behind all of its scatter, and the four elements of the column behind the strip asked for together
// (each had a test and a wait of its own: three round trips to memory a chunk, at the end of every strip).  Before -> now, us, inputs in
// rotation: half [64,256,56,56] 1 bit 47.1 -> 42.8, 2 bit 39.4 -> 37.7, 4 bit 36.8 -> 36.0, 8 bit 42.8 -> 41.8, [64,64,112,112] 1 bit 48.6 -> 45.9,
// [8,256,56,56] 4 bit 11.5 -> 10.9, [2,64,128,128] 5.8 -> 5.3; float equal, small tensors -2 to +2.5 %.
#define STRIP_PIECES 4    /* 16-byte pieces of a memory row in a strip (8: half [2,64,128,128] 4 bit 7.6 -> 9.5 us, large tensors equal) */
#define STRIP_CHUNK 256   /* pixels: a thread takes four of one piece */
#define STRIP_THREADS (STRIP_PIECES * STRIP_CHUNK / 4)
struct StripShape {
  int64_t sb, sk;
  uint32_t M, K, strips;   // strips of a batch entry
  uint32_t batch, segments, segment;   // segment: units of a channel in a segment
};
// whole super-groups, and whole steps of GS groups
template <int BITS, int GS> struct StripUnit { static constexpr int value = 8 / BITS > GS ? 8 / BITS * GROUP : GS * GROUP; };
template <typename T, int BITS, int NOISE, int GS>
__global__ void __launch_bounds__(STRIP_THREADS, 4 / GS)
quantize_strips_kernel(SeedArg seed_arg, const T* __restrict__ x, int64_t numel, int64_t N, uint8_t* __restrict__ packed,
                       typename Elem<T>::Stat* __restrict__ scale_out, T* __restrict__ mn_out, T* __restrict__ mx_out, StripShape g) {
  static_assert(GS <= 8 / BITS, "a super-group holds a step's groups: past the tensor's last group there may be none to store");
  typedef typename Elem<T>::Stat Stat;
  constexpr int CH = Elem<T>::kQChunks, W = Elem<T>::kQWidth, WPT = 8 / BITS, QMAX = (1 << BITS) - 1;
  constexpr uint32_t ES = sizeof(T), UNIT = StripUnit<BITS, GS>::value, STEP = GS * GROUP;
  constexpr int STRIP = STRIP_PIECES * W;             // channels of a strip
  constexpr int OWN = STRIP / (STRIP_THREADS / 16);   // channels of a row of 16 lanes: 2 (16-bit types), 1 (float)
  // LDS: two steps' groups per channel; 16 bytes behind every channel and 64 behind every 8 half channels keep the channels, and the
  // pieces, that a wave writes at once out of each other's banks
  constexpr uint32_t SLOT = STEP * ES, CHANNEL = 2 * SLOT + 16, PIECE = W * CHANNEL + (ES == 2 ? 64 : 0);
  __shared__ u32x4 ring_lds[STRIP_PIECES * PIECE / 16];
  uint8_t* const ring = reinterpret_cast<uint8_t*>(ring_lds);
  const uint32_t id = xcd_tile<GACT_XCD_RUN_TR>(blockIdx.x, gridDim.x);
  const uint32_t seg = id / (g.strips * g.batch), strip = id - seg * (g.strips * g.batch);
  const uint32_t b = strip / g.strips, m0 = (strip - b * g.strips) * STRIP;
  const uint32_t width = g.M - m0 < (uint32_t)STRIP ? g.M - m0 : (uint32_t)STRIP;   // a multiple of W
  const T* const entry = x + (int64_t)b * g.sb;
  const uint32_t K = g.K;
  // the column behind the strip's last one, where that channel's units may end: the next channel, perhaps of the next entry
  const T* const behind = m0 + width < g.M ? entry + m0 + width : b + 1 < g.batch ? x + (int64_t)(b + 1) * g.sb : nullptr;

  // this thread's part of a step: four pixels of one piece in each of its chunks
  const uint32_t piece = threadIdx.x % STRIP_PIECES, quad = threadIdx.x / STRIP_PIECES;
  const bool has_piece = piece * W < width;
  const bool last_piece = (piece + 1) * W == width;
  const T* const from = entry + m0 + piece * W;
  const uint32_t P0 = (uint32_t)(((uint64_t)b * g.M + m0) * K);   // element index of the strip's first channel, low bits
  const auto first_pixel = [&](uint32_t channel) { return (0u - (P0 + channel * K)) & (UNIT - 1); };   // of its first unit
  uint32_t first_of[W];
#pragma unroll
  for (int e = 0; e < W; e++) first_of[e] = first_pixel(piece * W + e);
  struct Chunk { u32x4 v[4]; uint32_t beyond[4]; };   // beyond: the elements' bits
  const uint32_t j_first = seg * g.segment * (UNIT / STEP);        // first step's groups of the segment within a channel
  const uint32_t j_end = j_first + g.segment * (UNIT / STEP);
  auto load = [&](uint32_t chunk, Chunk& q) {
    const uint32_t at = chunk * STRIP_CHUNK + 4 * quad;            // four pixels on one side of K: both are multiples of four
    const uint32_t k = at < K ? at : at - K;
    if (has_piece && at < K + UNIT) {
      const T* const p = from + (int64_t)k * g.sk;
#pragma unroll
      for (int j = 0; j < 4; j++) q.v[j] = *reinterpret_cast<const u32x4*>(p + j * g.sk);
      if (at >= K && last_piece) {
        // into registers of their own and under one test, so that all four are asked for before any is waited for
        if (behind) {
          typedef typename std::conditional<ES == 4, uint32_t, uint16_t>::type Bits;
          const Bits* const p1 = reinterpret_cast<const Bits*>(behind) + (int64_t)k * g.sk;
#pragma unroll
          for (int j = 0; j < 4; j++) q.beyond[j] = p1[j * g.sk];
        } else {
#pragma unroll
          for (int j = 0; j < 4; j++) q.beyond[j] = 0u;
        }
      }
    }
  };
  // four elements of a channel (16-bit types: in lo) to their place in the channel's two slots.  A step holds a slot's number of
  // consecutive elements of a channel, so what comes before the first unit cannot reach a slot that is being filled.
  auto put = [&](uint32_t base, uint32_t pos, u32x2 lo, u32x2 hi) {
    uint8_t* const to = ring + base + (pos & (2 * STEP - 1)) * ES;
    if constexpr (ES == 4) *reinterpret_cast<u32x4*>(to) = u32x4{lo.x, lo.y, hi.x, hi.y};
    else *reinterpret_cast<u32x2*>(to) = lo;
  };
  auto column = [&](const Chunk& q, int e, u32x2& lo, u32x2& hi) {   // channel e of the piece: its four pixels side by side
    if constexpr (ES == 4) {
      lo = u32x2{q.v[0][e], q.v[1][e]};
      hi = u32x2{q.v[2][e], q.v[3][e]};
    } else {
      const uint32_t sel = e & 1 ? 0x07060302u : 0x05040100u;
      lo = u32x2{__builtin_amdgcn_perm(q.v[1][e / 2], q.v[0][e / 2], sel), __builtin_amdgcn_perm(q.v[3][e / 2], q.v[2][e / 2], sel)};
      hi = u32x2{0u, 0u};
    }
  };
  auto scatter = [&](uint32_t chunk, const Chunk& q) {
    const uint32_t at = chunk * STRIP_CHUNK + 4 * quad;
    if (!has_piece) return;
    u32x2 lo, hi;
    if (at < K) {
#pragma unroll
      for (int e = 0; e < W; e++) {
        column(q, e, lo, hi);
        put(piece * PIECE + e * CHANNEL, at - first_of[e], lo, hi);
      }
    } else if (at < K + UNIT) {   // past the end: a column belongs to the channel before it
#pragma unroll
      for (int e = 0; e < W; e++) {
        column(q, e, lo, hi);
        if (e > 0) put(piece * PIECE + (e - 1) * CHANNEL, at - first_of[e > 0 ? e - 1 : 0], lo, hi);
        else if (piece > 0) put((piece - 1) * PIECE + (W - 1) * CHANNEL, at - first_pixel(piece * W - 1), lo, hi);
      }
      if (last_piece) {
        hi = u32x2{0u, 0u};
        if constexpr (ES == 4) {
          lo = u32x2{q.beyond[0], q.beyond[1]};
          hi = u32x2{q.beyond[2], q.beyond[3]};
        } else {
          lo = u32x2{q.beyond[0] | q.beyond[1] << 16, q.beyond[2] | q.beyond[3] << 16};
        }
        put(piece * PIECE + (W - 1) * CHANNEL, at - first_of[W - 1], lo, hi);
      }
    }
  };

  // this lane's 16 bytes of the super-group that group n belongs to
  auto store_bytes = [&](int64_t n, const uint32_t (&b4)[4]) {
#pragma unroll
    for (int k = 0; k < CH; k++) {
      uint8_t* const to = packed + n / WPT * GROUP + chunk_col<T>(k, threadIdx.x & 15);
      if constexpr (W == 4) stream_store(b4[k], reinterpret_cast<uint32_t*>(to));
      else stream_store(u32x2{b4[2 * k], b4[2 * k + 1]}, reinterpret_cast<u32x2*>(to));
    }
  };
  // this row's channels
  const uint64_t seed = seed_arg.value();
  const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
  const int row = threadIdx.x >> 4, i = threadIdx.x & 15;
  uint32_t delay[OWN], last[OWN];   // step t completes groups (t - delay) * GS .. of the channel; end of the segment's (t - delay)
  int64_t n_first[OWN];
#pragma unroll
  for (int c = 0; c < OWN; c++) {
    const uint32_t m = row * OWN + c, first = first_pixel(m);
    last[c] = m < width ? (K - first + UNIT - 1) / UNIT * (UNIT / STEP) : 0u;
    last[c] = last[c] < j_end ? last[c] : j_end;
    delay[c] = (first + STEP - 1) / STEP;
    n_first[c] = (((int64_t)b * g.M + m0 + m) * K + first) / GROUP;
  }
  uint32_t bytes[OWN][4];   // the lane's 16 bytes of each channel's super-group, in the order of their addresses
  // Scale and minimum stay in the row until its 16 lanes hold those of STATS steps (or the channel ends): a step's own are pieces of a
  // few bytes, one for every channel, and each costs the memory system what a whole line does.  Lane G * k + r keeps group r of
  // the step k of its turn.  Stored step by step / by turns, us: half [64,256,56,56] 1 bit 42.6 / 41.0, 2 bit 37.5 / 36.7, 4 and 8 bit
  // equal, float 2 bit 67.5 / 66.1, 4 bit 64.0 / 62.9, [32,64,112,112] 1 bit 38.9 / 37.9; tensors of 2 M elements and fewer equal, but
  // float 1-2 % slower (0.05-0.1 us of 4 to 7).
  constexpr uint32_t STATS = 16 / (OWN * GS);
  Stat kept_scale = (Stat)0.0f, kept_lo = (Stat)0.0f;

  const uint32_t most = (K + UNIT - 1) / STEP + 1;   // no channel has anything left after so many steps
  const uint32_t end = j_end + UNIT / STEP < most ? j_end + UNIT / STEP : most;
  // `ahead` steps further on the same registers are loaded again
  auto step = [&](uint32_t t, Chunk (&q)[GS], uint32_t ahead) {
#pragma unroll
    for (int h = 0; h < GS; h++) scatter(t * GS + h, q[h]);
    // after the last of the step's registers is read: a wait between two chunks would be one for the loads issued in between
    if (t + ahead < end) {
#pragma unroll
      for (int h = 0; h < GS; h++) load((t + ahead) * GS + h, q[h]);
    }
    __syncthreads();
    uint32_t j[OWN];
    bool due[OWN], any = false;
#pragma unroll
    for (int c = 0; c < OWN; c++) {
      j[c] = t - delay[c];
      due[c] = t >= delay[c] && j[c] < last[c] && j[c] >= j_first;
      any |= due[c];
    }
    if (__builtin_amdgcn_ballot_w64(any) == 0) {
      __syncthreads();
      return;
    }
    constexpr int G = OWN * GS;   // groups of the row: group s of channel c is number c * GS + s
    typename Elem<T>::Store st[G];
    Stat lo[G], hi[G], sc[G];
#pragma unroll
    for (int r = 0; r < G; r++) {
      const uint32_t m = row * OWN + r / GS;
      const uint8_t* p = ring + (m / W) * PIECE + (m % W) * CHANNEL + (j[r / GS] & 1) * SLOT + (r % GS) * (GROUP * ES);
#pragma unroll
      for (int k = 0; k < CH; k++) Elem<T>::load_chunk(reinterpret_cast<const T*>(p) + chunk_col<T>(k, i), st[r], k);
    }
    // bfloat16 widens its elements for two groups at 4 bit only.  With one group a step the statistics that wait for their turn leave no
    // registers for that: 128 and up to 37 spilled, against 126 and none with ordered minima.  Widened / ordered, us: one group [40,256,56,56]
    // 4 bit 36.8 / 30.4, 2 bit 43.4 / 32.4, 1 bit 59.0 / 39.6, [22,256,56,56] 4 bit 27.9 / 21.7, [64,256,56,56] 8 bit 41.2 / 40.5; two groups
    // [64,256,56,56] 1 bit 41.7 / 41.4, 2 bit 36.9 / 36.8, 4 bit 36.0 / 36.0, [16,256,56,56] 4 bit 14.5 / 14.7.
    Elem<T>::template groups_minmax<G, !std::is_same<T, bf16>::value || GS == 1 || BITS != 4>(st, lo, hi);
    {
      // one division per lane: lane r of the row takes group r % G
      const int mine = i & (G - 1);
      Stat lo_m = lo[0], hi_m = hi[0];
#pragma unroll
      for (int r = 1; r < G; r++) {
        lo_m = mine == r ? lo[r] : lo_m;
        hi_m = mine == r ? hi[r] : hi_m;
      }
      const bool second = OWN > 1 && mine >= GS;   // the group is one of the row's second channel
      const uint32_t j_m = second ? j[OWN - 1] : j[0], last_m = second ? last[OWN - 1] : last[0];
      const bool due_m = second ? due[OWN - 1] : due[0];
      const int64_t n_m = (second ? n_first[OWN - 1] : n_first[0]) + mine % GS;
      const Stat s_m = Elem<T>::make_scale(lo_m, hi_m, QMAX);
      const uint32_t turn = (uint32_t)i / G;
      if ((j_m & (STATS - 1)) == turn) {
        kept_scale = s_m;
        kept_lo = lo_m;
      }
      if (due_m && ((j_m & (STATS - 1)) == STATS - 1 || j_m + 1 == last_m)) {
        const uint32_t at = (j_m & ~(STATS - 1)) + turn;
        const int64_t n = n_m + (int64_t)at * GS;
        if (at <= j_m && at >= j_first && n < N) {
          scale_out[n] = kept_scale;
          mn_out[n] = Elem<T>::elem_of(kept_lo);
        }
      }
      if (mx_out && i < G && due_m && n_m + (int64_t)j_m * GS < N) mx_out[n_m + (int64_t)j_m * GS] = Elem<T>::elem_of(hi_m);
      sc[0] = G == 1 ? s_m : row_bcast<0>(s_m);
      if (G > 1) sc[1 % G] = row_bcast<1>(s_m);
      if (G > 2) {
        sc[2 % G] = row_bcast<2>(s_m);
        sc[3 % G] = row_bcast<3>(s_m);
      }
    }
#pragma unroll
    for (int c = 0; c < OWN; c++) {
      if (due[c]) {
        const int64_t n0 = n_first[c] + j[c] * GS;
        constexpr bool WHOLE = WPT <= GS;                                   // a step completes its super-groups
        const uint32_t before = WHOLE ? 0u : (j[c] * GS) % WPT;             // groups of the super-group before this step's
        FastRow<T, GS> fast;
        uint32_t sum[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int s = 0; s < GS; s++) {
          const int r = c * GS + s;
          const uint32_t field_shift = (s % WPT) * BITS;
          float cd[CH / 2][W];
          if (NOISE == GACT_NOISE_FAST) fast.draws(s, n0, i, k0, k1, cd);
#pragma unroll
          for (int k = 0; k < CH; k++) {
            uint32_t w[W / 4];
            if constexpr (packs_bytes<T, BITS, NOISE, false>()) {
              chunk_words<T, NOISE>(st[r], k, lo[r], sc[r], cd, w);
            } else {
              uint32_t code[W];
              if (NOISE == GACT_NOISE_FAST) {
                if (k < CH / 2) Elem<T>::template codes<false, false, true, false>(st[r], k, lo[r], sc[r], cd[k % (CH / 2)], code);
                else Elem<T>::template codes<false, false, true, true>(st[r], k, lo[r], sc[r], cd[k % (CH / 2)], code);
              } else {
                float u[W];
#pragma unroll
                for (int e = 0; e < W; e++) u[e] = 0.5f;
                Elem<T>::template codes<true, false>(st[r], k, lo[r], sc[r], u, code);
              }
              if (Elem<T>::kRepairsInfiniteScale && Elem<T>::scale_is_inf(sc[r])) {   // rare, see Elem<T>::kRepairsInfiniteScale
#pragma unroll
                for (int e = 0; e < W; e++)
                  if (Elem<T>::above(st[r], k, e, lo[r])) code[e] = 0xffu;
              }
#pragma unroll
              for (int d = 0; d < W / 4; d++) w[d] = pack4(code + 4 * d);
            }
#pragma unroll
            for (int d = 0; d < W / 4; d++) {
              const uint32_t field = field_of<Elem<T>::kExactField>(w[d], field_shift);
              uint32_t& byte4 = sum[k * (W / 4) + d];
              byte4 = s % WPT == 0 ? field : byte4 | field;
            }
          }
          if (WHOLE && s % WPT == WPT - 1) store_bytes(n0 + s, sum);
        }
        if (!WHOLE) {
          const uint32_t shift = before * BITS;
#pragma unroll
          for (int d = 0; d < 4; d++) {
            const uint32_t w = field_of<Elem<T>::kExactField>(sum[d], shift);
            bytes[c][d] = before == 0 ? w : bytes[c][d] | w;
          }
          if (before == WPT - GS) store_bytes(n0, bytes[c]);
        }
      }
    }
    __syncthreads();
  };
  if constexpr (GS == 1) {   // two steps' loads in flight
    Chunk even[1], odd[1];
    load(j_first, even[0]);
    if (j_first + 1 < end) load(j_first + 1, odd[0]);
    for (uint32_t t = j_first; t < end; t += 2) {
      step(t, even, 2);
      if (t + 1 < end) step(t + 1, odd, 2);
    }
  } else {                   // one step's, as many bytes (two steps': half [64,256,56,56] 4 bit 37.8 -> 39.9 us, 2 bit 40.4 -> 44.5,
                             // float 4 bit 63.9 -> 66.5, half [16,256,56,56] 15.9 -> 17.4; nothing gained)
    Chunk q[GS];
#pragma unroll
    for (int h = 0; h < GS; h++) load(j_first * GS + h, q[h]);
    for (uint32_t t = j_first; t < end; t++) step(t, q, 1);
  }
}

template <typename T, int BITS, bool LARGE = false>
__global__ void __launch_bounds__(256)
dequantize_kernel(const uint8_t* __restrict__ packed, const typename Elem<T>::Stat* __restrict__ scale,
                  const T* __restrict__ mn,
                  int64_t numel, int64_t N, T* __restrict__ out) {
  constexpr DqGeom D = dq_geom<T>(BITS);
  constexpr int LPU = GROUP / Elem<T>::kDqWidth;  // lanes per unit: 64 (float) or 32 (half)
  const int64_t unit = ((int64_t)xcd_tile<(uint32_t)D.run>(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x) / LPU;
  if (unit * dq_unit_groups(D, BITS, LARGE) >= N) return;
  dequantize_unit<T, BITS, LARGE ? D.sgs_large : D.sgs, LARGE ? D.parts_large : D.parts, LARGE>(packed, scale, mn, numel, N,
                                                                                              unit, threadIdx.x % LPU, out);
}

// ------------------------------------------------------------------------------------------------
// Groups of 64, 128 and 512 elements (config.group_size), float and half, in one pass each way.
//
// Quantize.  Whatever the group size, a row of 16 lanes takes spans of 512 consecutive elements in the layout of
// quantize_kernel's pairs of groups (two halves of 256, the lane's chunks 16 chunk widths apart), because that is what a
// block of the fast stream serves: one Philox block per lane and span.  A group is then one, two, four or eight of the
// lane's chunks - at 64 half elements half a row's chunk, and neighbouring groups sit in the two halves of the row.  Where
// the 8/BITS groups that share their bytes fill more than a span, two or four rows of the wave share them (ROWS) and OR
// their bytes together at the end; a row then takes SPR spans.
//
// HBM-bound, as the kernels for groups of 256.  Against minimax + scale + pack (three launches, the data read twice and
// ragged tensors copied to whole groups first): half [16384,1024], 4 bit, groups of 128: 26.7 -> 9.8 us quantize
// (4.3 TB/s), 11.6 -> 8.7 dequantize; 67 M float elements, 8 bit: quantize 57 us (0.74 of 8 TB/s; groups of 256: 52).
// ------------------------------------------------------------------------------------------------
#define GROUPS_SPAN 512
template <int LANE>
__device__ __forceinline__ uint32_t quad_bcast_u32(uint32_t v) {   // value of lane LANE of the quad
  return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, LANE * 0x55, 0xf, 0xf, false);
}
// scale of the lane's group G from the lane that divided for it (QUAD: lane G of every quad, else lane G of the row)
template <int G, bool QUAD>
__device__ __forceinline__ float groups_bcast(float v) {
  return QUAD ? __builtin_bit_cast(float, quad_bcast_u32<G & 3>(__builtin_bit_cast(uint32_t, v))) : row_bcast<G>(v);
}
template <int G, bool QUAD>
__device__ __forceinline__ f16 groups_bcast(f16 v) {
  return QUAD ? __builtin_bit_cast(f16, (uint16_t)quad_bcast_u32<G & 3>((uint32_t)__builtin_bit_cast(uint16_t, v))) : row_bcast<G>(v);
}

template <typename T, int D, int BITS>
struct GroupsShape {
  static constexpr int WPT = 8 / BITS;
  static constexpr int CH = Elem<T>::kQChunks, W = Elem<T>::kQWidth;
  static constexpr int CPS = 2 * CH;                                        // chunks of a span per lane
  static constexpr int GPS = GROUPS_SPAN / D;                               // groups of a span
  static constexpr bool HALF = D < 16 * W;                                  // a chunk of the row holds two groups
  static constexpr int GL = HALF ? GPS / 2 : GPS;                           // groups of a span a lane has elements of
  static constexpr int CPG = CPS / GL;                                      // chunks of a group per lane
  static constexpr int SPANS = D * WPT > GROUPS_SPAN ? D * WPT / GROUPS_SPAN : 1;   // spans of a unit: whole super-groups
  static constexpr int ROWS = SPANS < 4 ? SPANS : 4, SPR = SPANS / ROWS;
  static constexpr int UNIT_GROUPS = SPANS * GPS;
  static_assert(D == 64 || D == 128 || D == 512, "group sizes of the one-pass kernels");
};

// of the lane's chunks of every group: ORDERED by lane_ordered, which may ask (nan) for the other way
template <typename T, int D, int BITS, bool ORDERED, int G = 0>
__device__ __forceinline__ void groups_lane_minmax(const typename Elem<T>::Store (&v)[2], T (&lo)[GroupsShape<T, D, BITS>::GL],
                                                   T (&hi)[GroupsShape<T, D, BITS>::GL], bool& nan) {
  typedef GroupsShape<T, D, BITS> S;
  constexpr int C0 = G * S::CPG, CH = S::CH, CPG = S::CPG <= CH ? S::CPG : CH;
  if constexpr (G < S::GL) {
    if constexpr (ORDERED) Elem<T>::template lane_ordered<C0 % CH, C0 % CH + CPG>(v[C0 / CH], lo[G], hi[G], nan);
    else Elem<T>::template lane_minmax<C0 % CH, C0 % CH + CPG>(v[C0 / CH], lo[G], hi[G]);
    if constexpr (S::CPG > CH) {   // a group of 512: both halves
      T lo2, hi2;
      if constexpr (ORDERED) Elem<T>::template lane_ordered<0, CH>(v[1], lo2, hi2, nan);
      else Elem<T>::template lane_minmax<0, CH>(v[1], lo2, hi2);
      lo[G] = lo2 < lo[G] ? lo2 : lo[G];   // no NaN that lane_ordered has not told of; the other way's start values are none
      hi[G] = hi2 > hi[G] ? hi2 : hi[G];
    }
    groups_lane_minmax<T, D, BITS, ORDERED, G + 1>(v, lo, hi, nan);
  }
}
template <typename T, int D, int BITS>
__device__ __forceinline__ void groups_stats(const typename Elem<T>::Store (&v)[2], T (&lo)[GroupsShape<T, D, BITS>::GL],
                                             T (&hi)[GroupsShape<T, D, BITS>::GL]) {
  typedef GroupsShape<T, D, BITS> S;
  bool nan = false;
  groups_lane_minmax<T, D, BITS, true>(v, lo, hi, nan);
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(nan) != 0, 0)) groups_lane_minmax<T, D, BITS, false>(v, lo, hi, nan);
#pragma unroll
  for (int g = 0; g < S::GL; g++) {
    if constexpr (S::HALF) half_row_all_minmax(lo[g], hi[g]);
    else row_all_minmax(lo[g], hi[g]);
  }
}
template <typename T, int D, int BITS, int G = 0>
__device__ __forceinline__ void groups_share_scale(T mine, T (&sc)[GroupsShape<T, D, BITS>::GL]) {
  typedef GroupsShape<T, D, BITS> S;
  if constexpr (G < S::GL) {
    sc[G] = S::GL == 1 ? mine : groups_bcast<G, S::HALF>(mine);
    groups_share_scale<T, D, BITS, G + 1>(mine, sc);
  }
}

template <typename T, int D, int BITS, int NOISE, bool PACKS = true>
__global__ void __launch_bounds__(64)
quantize_groups_kernel(SeedArg seed_arg, const T* __restrict__ x, int64_t numel, int64_t N, uint8_t* __restrict__ packed,
                       T* __restrict__ scale_out, T* __restrict__ mn_out, T* __restrict__ mx_out,
                       const float* __restrict__ noise) {
  static_assert(NOISE != GACT_NOISE_REF, "the reference stream draws per output byte");
  typedef GroupsShape<T, D, BITS> S;
  constexpr int WPT = S::WPT, CH = S::CH, W = S::W, QMAX = (1 << BITS) - 1;
  const uint32_t tile = gridDim.x - 1u - xcd_tile<GACT_XCD_RUN_Q>(blockIdx.x, gridDim.x);   // last tile first, see quantize_kernel
  const int row = (int)(threadIdx.x >> 4), i = threadIdx.x & 15;
  const int64_t unit = (int64_t)tile * (4 / S::ROWS) + row / S::ROWS;
  const int part = row % S::ROWS;   // the row's share of its unit
  if (unit * S::UNIT_GROUPS >= N) return;   // all rows of the unit
  const uint64_t seed = seed_arg.value();
  const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
  const int half = S::HALF ? i >> 3 : 0;

  constexpr bool PK = PACKS && packs_bytes<T, BITS, NOISE, false>();
  typename Elem<T>::Store v[2];
  uint32_t acc[S::CPG][W];
  uint32_t words_of[S::CPG][W / 4];   // PK: the same bytes, packed
#pragma unroll
  for (int s = 0; s < S::SPR; s++) {
    const int64_t span = unit * S::SPANS + part * S::SPR + s;
    load_group<T>(x, numel, span * 2, i, v[0]);
    load_group<T>(x, numel, span * 2 + 1, i, v[1]);
    T lo[S::GL], hi[S::GL], sc[S::GL];
    groups_stats<T, D, BITS>(v, lo, hi);
    {
      // one division per lane: lane j of the row (half rows: of every quad) takes the lane group j
      const int mine = i & (S::GL - 1);
      T lo_m = lo[0], hi_m = hi[0];
#pragma unroll
      for (int g = 1; g < S::GL; g++) {
        lo_m = mine == g ? lo[g] : lo_m;
        hi_m = mine == g ? hi[g] : hi_m;
      }
      const T s_m = Elem<T>::make_scale(lo_m, hi_m, QMAX);
      const int64_t n = span * S::GPS + (S::HALF ? 2 * mine + half : mine);
      if ((S::HALF ? i & 7 : i) < S::GL && n < N) {
        scale_out[n] = s_m;
        mn_out[n] = lo_m;
        if (mx_out) mx_out[n] = hi_m;
      }
      groups_share_scale<T, D, BITS>(s_m, sc);
    }
    uint32_t words[2][2];
    if (NOISE == GACT_NOISE_FAST) fast_pair_words<T>(span, i, k0, k1, words);

    u32x2 held = {0u, 0u};   // half rows: the finished bytes of an even super-group, until the odd one joins them
#pragma unroll
    for (int g = 0; g < S::GL; g++) {
      const int first = S::HALF ? 2 * g : s * S::GPS + g;   // the (first) group within the row's unit
      const int64_t n = span * S::GPS + (S::HALF ? 2 * g + half : g);
      const uint32_t shift = (uint32_t)((first % WPT + (S::HALF && WPT > 1 ? half : 0) + part * S::SPR * S::GPS) * BITS);
      if (S::ROWS > 1 ? s == 0 && g == 0 : first % WPT == 0) {
#pragma unroll
        for (int c = 0; c < S::CPG; c++) {
#pragma unroll
          for (int e = 0; e < W; e++) acc[c][e] = 0;
#pragma unroll
          for (int d = 0; d < W / 4; d++) words_of[c][d] = 0;
        }
      }
      const bool overflowed = !PK && Elem<T>::kRepairsInfiniteScale && Elem<T>::scale_is_inf(sc[g]);
#pragma unroll
      for (int c = 0; c < S::CPG; c++) {
        const int h = (g * S::CPG + c) / CH, k = (g * S::CPG + c) % CH;
        if constexpr (PK) {   // a group past the last one holds zeros, whose codes are zero
          float cd[CH / 2][W];
          if (NOISE == GACT_NOISE_FAST) fast_centred_draws<T>(words[h], cd);
          uint32_t w[W / 4];
          chunk_words<T, NOISE>(v[h], k, lo[g], sc[g], cd, w);
#pragma unroll
          for (int d = 0; d < W / 4; d++) words_of[c][d] |= field_of<Elem<T>::kExactField>(w[d], shift);
          continue;
        }
        uint32_t code[W];
        if (NOISE == GACT_NOISE_FAST) {
          float cd[CH / 2][W];
          fast_centred_draws<T>(words[h], cd);
          if (k < CH / 2) Elem<T>::template codes<false, false, true, false>(v[h], k, lo[g], sc[g], cd[k % (CH / 2)], code);
          else Elem<T>::template codes<false, false, true, true>(v[h], k, lo[g], sc[g], cd[k % (CH / 2)], code);
        } else {
          float u[W];
#pragma unroll
          for (int e = 0; e < W; e++) u[e] = 0.5f;
          if (NOISE == GACT_NOISE_INJECT && n < N)
            Elem<T>::load_noise(noise + span * GROUPS_SPAN + h * GROUP + chunk_col<T>(k, i), u);
          Elem<T>::template codes<NOISE == GACT_NOISE_CONST, false>(v[h], k, lo[g], sc[g], u, code);
        }
        // a group past the last one holds zeros, whose codes are zero
#pragma unroll
        for (int e = 0; e < W; e++) acc[c][e] |= code[e] << shift;
        if (__builtin_amdgcn_ballot_w64(overflowed) != 0 && overflowed) {   // rare, see Elem<T>::kRepairsInfiniteScale
#pragma unroll
          for (int e = 0; e < W; e++)
            if (Elem<T>::above(v[h], k, e, lo[g])) acc[c][e] |= 0xffffffffu << shift;
        }
      }
      if constexpr (S::ROWS > 1) {
        // the bytes go out below, when the row has gone through its share
      } else if constexpr (!S::HALF) {
        if (first % WPT == WPT - 1) {
          const int64_t sg = (unit * S::UNIT_GROUPS + first) / WPT;
          if (sg * WPT < N) {
#pragma unroll
            for (int c = 0; c < S::CPG; c++) {
              if constexpr (PK) Elem<T>::store_words(packed + sg * D + chunk_col<T>(c, i), words_of[c]);
              else Elem<T>::store_codes(packed + sg * D + chunk_col<T>(c, i), acc[c]);
            }
          }
        }
      } else if (WPT == 1) {
        if (n < N) {
          if constexpr (PK) Elem<T>::store_words(packed + n * D + W * (i & 7), words_of[0]);
          else Elem<T>::store_codes(packed + n * D + W * (i & 7), acc[0]);
        }
      } else if ((first + 1) % WPT == WPT - 1) {
        // the two halves of the row hold different fields of the same bytes; super-groups go out in pairs, one per half
        // row, so that a row writes 128 contiguous bytes
        u32x2 w;
        w.x = PK ? words_of[0][0] : pack4(acc[0]);
        w.y = PK ? words_of[0][W / 4 - 1] : pack4(acc[0] + 4);
        w.x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w.x, 0x128, 0xf, 0xf, false);   // row_ror:8
        w.y |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w.y, 0x128, 0xf, 0xf, false);
        const int q = first / WPT;   // super-group of the span
        if (WPT == 8 || (q & 1)) {
          const int64_t sg = (span * S::GPS) / WPT + (WPT == 8 ? 0 : q - 1 + half);
          const u32x2 out = {WPT == 8 || half ? w.x : held.x, WPT == 8 || half ? w.y : held.y};
          if ((WPT < 8 || half == 0) && sg * WPT < N) stream_store(out, reinterpret_cast<u32x2*>(packed + sg * D + W * (i & 7)));
        } else {
          held = w;
        }
      }
    }
  }
  if constexpr (S::ROWS > 1) {
    // the unit is one super-group.  The lane's dwords in the order of their columns, OR-ed over the rows (every row of the
    // unit is here); each row stores its share of them.
    constexpr int DW = S::CPG * W / 4, OWN = DW / S::ROWS;
    static_assert(DW % S::ROWS == 0, "rows store equal shares");
    uint32_t pk[DW];
#pragma unroll
    for (int j = 0; j < DW; j++) {
      pk[j] = PK ? words_of[j * 4 / W][(j * 4) % W / 4] : pack4(&acc[j * 4 / W][(j * 4) % W]);
#pragma unroll
      for (int off = 16; off < 16 * S::ROWS; off <<= 1) pk[j] |= (uint32_t)__shfl_xor((int)pk[j], off, 64);
    }
#pragma unroll
    for (int j = 0; j < OWN; j++) {
      uint32_t mine = pk[j];
#pragma unroll
      for (int r = 1; r < S::ROWS; r++) mine = part == r ? pk[r * OWN + j] : mine;
      const int at = part * OWN + j;   // W = 4: chunk; W = 8: half a chunk
      const int col = W == 4 ? chunk_col<T>(at, i) : chunk_col<T>(at >> 1, i) + 4 * (at & 1);
      stream_store(mine, reinterpret_cast<uint32_t*>(packed + unit * D + col));
    }
  }
}

// Dequantize.  A lane takes P 16-byte pieces of the columns of super-groups - it loads the code bytes of these columns once and
// writes that piece of each of the super-group's 8/BITS groups - and the wave's 64 lanes cover neighbouring pieces, so a store
// instruction writes whole groups.  Codes, scales and minima of all the pieces are asked for first.
// WPT consecutive values from a + n0 on, in loads of up to 16 bytes where the array is aligned
template <typename T, int WPT>
__device__ __forceinline__ void load_stats(const T* __restrict__ a, int64_t n0, int64_t N, bool aligned, T (&v)[WPT]) {
  if (WPT > 1 && aligned && n0 + WPT <= N) {
    constexpr int VL = WPT * (int)sizeof(T) > 16 ? 16 / (int)sizeof(T) : (WPT > 1 ? WPT : 2);
    typedef T vec __attribute__((ext_vector_type(VL)));
#pragma unroll
    for (int c = 0; c < WPT / VL; c++) {
      const vec q = reinterpret_cast<const vec*>(a + n0)[c];
#pragma unroll
      for (int e = 0; e < VL; e++) v[c * VL + e] = q[e];
    }
  } else {
#pragma unroll
    for (int ni = 0; ni < WPT; ni++) v[ni] = n0 + ni < N ? a[n0 + ni] : (T)1.0f;
  }
}
template <typename T, int D, int BITS, int P>
__global__ void __launch_bounds__(256)
dequantize_groups_kernel(const uint8_t* __restrict__ packed, const T* __restrict__ scale, const T* __restrict__ mn,
                         int64_t numel, int64_t N, T* __restrict__ out) {
  constexpr int WPT = 8 / BITS, W = Elem<T>::kDqWidth;
  const uint32_t tile = xcd_tile<GACT_XCD_RUN_DQ>(blockIdx.x, gridDim.x);
  const int64_t wave = (int64_t)tile * (blockDim.x >> 6) + wave_first(threadIdx.x >> 6);
  const int64_t byte0 = wave * (P * 64 * W);   // the wave's first code byte
  const int64_t n_first = byte0 / D * WPT;
  if (n_first >= N) return;   // the whole wave
  const OutWindow window(out + n_first * D, (numel - n_first * D) * (int64_t)sizeof(T));
  const int lane = threadIdx.x & 63;
  const bool aligned = ((reinterpret_cast<uintptr_t>(scale) | reinterpret_cast<uintptr_t>(mn)) & 15u) == 0;
  uint32_t w[P][W / 4];
  T s[P][WPT], m[P][WPT];
#pragma unroll
  for (int p = 0; p < P; p++) {
    const int64_t at = byte0 + (p * 64 + lane) * W;   // the piece's code bytes
    const int64_t n0 = at / D * WPT;
#pragma unroll
    for (int k = 0; k < W / 4; k++) w[p][k] = 0u;
    if (n0 < N) {
      if constexpr (W == 4) {
        w[p][0] = stream_load(reinterpret_cast<const uint32_t*>(packed + at));
      } else {
        const u32x2 q = stream_load(reinterpret_cast<const u32x2*>(packed + at));
        w[p][0] = q.x;
        w[p][W / 4 - 1] = q.y;
      }
    }
    load_stats<T, WPT>(scale, n0, N, aligned, s[p]);
    load_stats<T, WPT>(mn, n0, N, aligned, m[p]);
  }
#pragma unroll
  for (int p = 0; p < P; p++) {
    const int64_t at = byte0 + (p * 64 + lane) * W;
    const int64_t n0 = at / D * WPT;
    const int col = (int)(at % D);
#pragma unroll
    for (int ni = 0; ni < WPT; ni++) {
      const typename Elem<T>::Dq dq = Elem<T>::dq_prepare(s[p][ni], m[p][ni]);
      T v[W];
      if (__builtin_amdgcn_ballot_w64(!dq.fast) == 0) {
#pragma unroll
        for (int e = 0; e < W; e++)
          v[e] = Elem<T>::finish(div_by_reciprocal((float)__builtin_amdgcn_ubfe(w[p][e >> 2], 8 * (e & 3) + ni * BITS, BITS), dq.s, dq.r), dq.mn);
      } else {
#pragma unroll
        for (int e = 0; e < W; e++)
          v[e] = Elem<T>::finish((float)__builtin_amdgcn_ubfe(w[p][e >> 2], 8 * (e & 3) + ni * BITS, BITS) / dq.s, dq.mn);
      }
      const int64_t first = (n0 + ni) * D + col;   // the piece's first element of this group
      if (first + W <= numel) {
        Elem<T>::template store_dq<GACT_STORE_NT_SYSTEM>(window, (uint32_t)((first - n_first * D) * (int64_t)sizeof(T)), v);
      } else {
#pragma unroll
        for (int e = 0; e < W; e++)
          if (first + e < numel) out[first + e] = v[e];
      }
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(256)
minimax256_kernel(const T* __restrict__ x, int64_t N, T* __restrict__ mn, T* __restrict__ mx) {
  const int64_t row = (int64_t)xcd_tile<GACT_XCD_RUN_Q>(blockIdx.x, gridDim.x) * (blockDim.x >> 4) + (threadIdx.x >> 4);
  if (row * MINIMAX_ROW_GROUPS >= N) return;
  minimax_row<T>(x, N, row, threadIdx.x & 15, mn, mx);
}

// ------------------------------------------------------------------------------------------------
// General shapes (any D for minimax; any G, D for pack / unpack).  These keep the operator surface
// complete; the path the library is built for is G = 1, D = 256 above.
// ------------------------------------------------------------------------------------------------
// Row min/max for any D.  2^lpr_log2 lanes share a row (8..64: as many as the row has 16-byte pieces, so
// short rows put several rows in a wave) and a lane group takes R consecutive rows, all of whose loads are
// issued before the first reduction.  VEC = false (a base address that is not 16-byte aligned) reads
// element by element.
template <typename T, bool VEC, int R>
__global__ void __launch_bounds__(256)
minimax_any_kernel(const T* __restrict__ x, int64_t N, int64_t D, int lpr_log2, T* __restrict__ mn,
                   T* __restrict__ mx) {
  constexpr int W = VEC ? 16 / (int)sizeof(T) : 1;
  typedef T vecw __attribute__((ext_vector_type(VEC ? W : 2)));
  typedef typename std::conditional<VEC, vecw, T>::type vec;
  const int lpr = 1 << lpr_log2;
  const int64_t group = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> lpr_log2;
  const int sub = threadIdx.x & (lpr - 1);
  const int64_t V = D / W;
  float lo[R], hi[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    lo[r] = Elem<T>::init_lo();
    hi[r] = Elem<T>::init_hi();
    const int64_t n = group * R + r;
    if (n < N) {
      const vec* row = reinterpret_cast<const vec*>(x + n * D);
#pragma unroll 4
      for (int64_t v = sub; v < V; v += lpr) {
        const vec q = stream_load(row + v);
#pragma unroll
        for (int e = 0; e < W; e++) {
          float f;
          if constexpr (VEC) f = (float)q[e]; else f = (float)q;
          lo[r] = __builtin_fminf(lo[r], f);
          hi[r] = __builtin_fmaxf(hi[r], f);
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; r++) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
      if (off < lpr) {  // uniform over the launch
        lo[r] = __builtin_fminf(lo[r], __shfl_xor(lo[r], off, 64));
        hi[r] = __builtin_fmaxf(hi[r], __shfl_xor(hi[r], off, 64));
      }
    const int64_t n = group * R + r;
    if (sub == 0 && n < N) {
      mn[n] = Elem<T>::from_float(lo[r]);
      mx[n] = Elem<T>::from_float(hi[r]);
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(256)
scale_kernel(const T* __restrict__ mn, const T* __restrict__ mx, int bits, int64_t count, T* __restrict__ scale) {
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id < count) scale[id] = Elem<T>::make_scale(mn[id], mx[id], (1 << bits) - 1);
}

// one thread per output byte j = (no*G + g)*D + d
template <typename T, int NOISE>
__global__ void __launch_bounds__(256)
pack_any_kernel(const T* __restrict__ data, const T* __restrict__ mn, const T* __restrict__ scale, int bits,
                int64_t N, int64_t G, int64_t D, uint64_t seed, const float* __restrict__ noise,
                uint8_t* __restrict__ packed, int64_t total_bytes) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= total_bytes) return;
  const int wpt = 8 / bits;
  const int64_t d = j % D;
  const int64_t g = (j / D) % G;
  const int64_t no = j / (D * G);
  const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
  uint32_t r[4];
  uint32_t byte = 0;
  for (int ni = 0; ni < wpt; ni++) {
    const int64_t n = no * wpt + ni;
    if (n >= N) break;
    const int64_t id = (n * G + g) * D + d;
    const int64_t sid = n * G + g;
    float u = 0.5f;
    if (NOISE == GACT_NOISE_INJECT) {
      u = noise[id];
    } else if (NOISE == GACT_NOISE_REF) {
      if ((ni & 3) == 0) philox4x32<PHILOX_REF_ROUNDS>(ni >> 2, 0u, (uint32_t)j, (uint32_t)((uint64_t)j >> 32), k0, k1, r);
      u = curand_uniform_map(r[ni & 3]);
    } else if (NOISE == GACT_NOISE_FAST) {
      const uint64_t blk = fast_block_of((uint64_t)id);
      philox4x32<PHILOX_FAST_ROUNDS>(0u, 0u, (uint32_t)blk, (uint32_t)(blk >> 32), k0, k1, r);
      u = fast_centred_of(r, (uint64_t)id);
    }
    typename Elem<T>::Store one;
    Elem<T>::set(one, 0, 0, data[id]);
    byte |= Elem<T>::template code1<true, NOISE == GACT_NOISE_FAST>(one, 0, 0, mn[sid], scale[sid], u) << (ni * bits);
  }
  packed[j] = (uint8_t)byte;
}

template <typename T>
__global__ void __launch_bounds__(256)
unpack_any_kernel(const uint8_t* __restrict__ packed, int bits, const T* __restrict__ scale,
                  const T* __restrict__ mn, int64_t N, int64_t G, int64_t D, T* __restrict__ out,
                  int64_t total_bytes) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= total_bytes) return;
  const int wpt = 8 / bits;
  const int64_t d = j % D;
  const int64_t g = (j / D) % G;
  const int64_t no = j / (D * G);
  const uint32_t byte = packed[j];
  for (int ni = 0; ni < wpt; ni++) {
    const int64_t n = no * wpt + ni;
    if (n >= N) break;
    const int64_t sid = n * G + g;
    int c = (int)((byte >> (ni * bits)) & ((1u << bits) - 1u));
    out[(n * G + g) * D + d] = Elem<T>::decode(c, Elem<T>::dq_prepare(scale[sid], mn[sid]));
  }
}

// G = 1 and D a multiple of 8 (every group size config.group_size can take): a thread owns 8 consecutive
// columns of one super-group - 8 output bytes, 8 elements of each of its 8/bits groups with 16-byte loads -
// and no thread divides 64-bit indices.  Same arithmetic and the same noise streams as pack_any_kernel.
template <typename T, int NOISE>
__global__ void __launch_bounds__(256)
pack_rows8_kernel(const T* __restrict__ data, const T* __restrict__ mn, const T* __restrict__ scale, int bits,
                  int64_t N, uint32_t tpr /* threads per super-group = D / 8 */, uint32_t total_threads, uint64_t seed,
                  const float* __restrict__ noise, uint8_t* __restrict__ packed) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total_threads) return;
  const int wpt = 8 / bits;
  const uint32_t no = t / tpr, c8 = t - no * tpr;
  const int64_t D = (int64_t)tpr * 8;
  const int64_t j0 = (int64_t)no * D + (int64_t)c8 * 8;  // first output byte
  const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
  typedef T vec8 __attribute__((ext_vector_type(8)));
  uint32_t bytes[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
  uint32_t r[8][4];
  for (int ni = 0; ni < wpt; ni++) {
    const int64_t n = (int64_t)no * wpt + ni;
    if (n >= N) break;
    const int64_t id0 = n * D + (int64_t)c8 * 8;
    const vec8 x = stream_load(reinterpret_cast<const vec8*>(data + id0));
    const T lo = mn[n], sc = scale[n];
    float u[8];
    if (NOISE == GACT_NOISE_INJECT) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(noise + id0), b = *reinterpret_cast<const f32x4*>(noise + id0 + 4);
      u[0] = a.x; u[1] = a.y; u[2] = a.z; u[3] = a.w; u[4] = b.x; u[5] = b.y; u[6] = b.z; u[7] = b.w;
    } else if (NOISE == GACT_NOISE_REF) {
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const uint64_t j = (uint64_t)(j0 + e);
        if ((ni & 3) == 0) philox4x32<PHILOX_REF_ROUNDS>(ni >> 2, 0u, (uint32_t)j, (uint32_t)(j >> 32), k0, k1, r[e]);
        u[e] = curand_uniform_map(r[e][ni & 3]);
      }
    } else if (NOISE == GACT_NOISE_FAST) {
      // the thread's 8 consecutive elements share a block (id0 is a multiple of 8)
      const uint64_t blk = fast_block_of((uint64_t)id0);
      philox4x32<PHILOX_FAST_ROUNDS>(0u, 0u, (uint32_t)blk, (uint32_t)(blk >> 32), k0, k1, r[0]);
#pragma unroll
      for (int e = 0; e < 8; e++) u[e] = fast_centred_of(r[0], (uint64_t)id0 + e);
    } else {
#pragma unroll
      for (int e = 0; e < 8; e++) u[e] = 0.5f;
    }
#pragma unroll
    for (int e = 0; e < 8; e++) {
      typename Elem<T>::Store one;
      Elem<T>::set(one, 0, 0, x[e]);
      bytes[e] |= Elem<T>::template code1<true, NOISE == GACT_NOISE_FAST>(one, 0, 0, lo, sc, u[e]) << (ni * bits);
    }
  }
  u32x2 w;
  w.x = (bytes[0] & 0xffu) | ((bytes[1] & 0xffu) << 8) | ((bytes[2] & 0xffu) << 16) | (bytes[3] << 24);
  w.y = (bytes[4] & 0xffu) | ((bytes[5] & 0xffu) << 8) | ((bytes[6] & 0xffu) << 16) | (bytes[7] << 24);
  stream_store(w, reinterpret_cast<u32x2*>(packed + j0));
}

template <typename T>
__global__ void __launch_bounds__(256)
unpack_rows8_kernel(const uint8_t* __restrict__ packed, int bits, const T* __restrict__ scale,
                    const T* __restrict__ mn, int64_t N, uint32_t tpr, uint32_t total_threads, T* __restrict__ out) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total_threads) return;
  const int wpt = 8 / bits;
  const uint32_t no = t / tpr, c8 = t - no * tpr;
  const int64_t D = (int64_t)tpr * 8;
  const u32x2 w = stream_load(reinterpret_cast<const u32x2*>(packed + (int64_t)no * D + (int64_t)c8 * 8));
  typedef T vec8 __attribute__((ext_vector_type(8)));
  for (int ni = 0; ni < wpt; ni++) {
    const int64_t n = (int64_t)no * wpt + ni;
    if (n >= N) break;
    const typename Elem<T>::Dq dq = Elem<T>::dq_prepare(scale[n], mn[n]);
    vec8 v;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const uint32_t byte = ((e < 4 ? w.x : w.y) >> (8 * (e & 3))) & 0xffu;
      v[e] = Elem<T>::decode((int)((byte >> (ni * bits)) & ((1u << bits) - 1u)), dq);
    }
    stream_store(v, reinterpret_cast<vec8*>(out + n * D + (int64_t)c8 * 8));
  }
}

// ------------------------------------------------------------------------------------------------
// Dropout-mask bit packing.  Within each 512-element block, element e = k*16 + w is bit k of word w
// (quantization_cuda_kernel.cu:228-252): with one 16-byte load per lane, lane k holds elements
// 16k .. 16k+15, so word w is the ballot over lanes of "byte w is nonzero"; one wave packs two blocks
// (low and high half of each ballot).  A partial last block is packed sequentially (element e -> word
// e/32, bit e%32), which is the plain ballot of one byte per lane and fits the ceil(n/32)-word output.  It belongs to the
// kernel's last wave, whose time everybody waits for: its loads are asked for together and its bytes leave four at a time (a load per
// element made unpack of 3 M elements 5.3 us, of 103 M 21.4; now 2.7 and 18.0).
// ------------------------------------------------------------------------------------------------
// A wave takes MASK_PAIRS consecutive pairs of blocks (4 KB of mask bytes) and issues all its loads first.
#ifndef MASK_PAIRS
#define MASK_PAIRS 4
#endif
__global__ void __launch_bounds__(256)
mask_pack_kernel(const uint8_t* __restrict__ data, int64_t n, int32_t* __restrict__ mask) {
  const int64_t wave = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int64_t full_blocks = n / 512;
  const int64_t pairs = (full_blocks + 1) / 2;
  const int64_t pair0 = wave * MASK_PAIRS;
  if (pair0 < pairs) {
    u32x4 q[MASK_PAIRS];
#pragma unroll
    for (int j = 0; j < MASK_PAIRS; j++) {
      const int64_t blk = (pair0 + j) * 2 + (lane >> 5);  // lanes 0..31 hold the pair's first block
      q[j] = u32x4{0u, 0u, 0u, 0u};
      if (blk < full_blocks) q[j] = stream_load(reinterpret_cast<const u32x4*>(data + (blk * 32 + (lane & 31)) * 16));
    }
    // word w of a block is the ballot of "byte w is nonzero" over the block's 32 lanes.  The 32 words of
    // pair j are collected in lanes 32 * (j & 1) ..: one store then writes two pairs.
    uint32_t mine[MASK_PAIRS / 2];
#pragma unroll
    for (int j = 0; j < MASK_PAIRS; j++) {
      uint32_t sel = 0;
#pragma unroll
      for (int w = 0; w < 16; w++) {
        const uint32_t word = w < 4 ? q[j].x : w < 8 ? q[j].y : w < 12 ? q[j].z : q[j].w;
        const uint64_t b = __ballot(((word >> (8 * (w & 3))) & 0xffu) != 0u);
        if ((lane & 15) == w) sel = (lane & 16) ? (uint32_t)(b >> 32) : (uint32_t)b;
      }
      if ((j & 1) == 0) mine[j >> 1] = sel;
      else if (lane >= 32) mine[j >> 1] = sel;
    }
#pragma unroll
    for (int jj = 0; jj < MASK_PAIRS / 2; jj++) {
      const int64_t word = (pair0 + 2 * jj) * 32 + lane;  // 16 words per block
      if ((word >> 4) < full_blocks) stream_store(mine[jj], reinterpret_cast<uint32_t*>(mask) + word);
    }
  }
  // the partial block goes to the wave after the last one that packs full blocks
  if (wave == (pairs + MASK_PAIRS - 1) / MASK_PAIRS) {
    const int64_t base = full_blocks * 512;
    const int64_t words = (n + 31) / 32;
    uint8_t v[8];   // all of it asked for before the first word is written
#pragma unroll
    for (int c = 0; c < 8; c++) {
      const int64_t e = base + 64 * c + lane;
      v[c] = e < n ? data[e] : 0;
    }
    uint32_t word = 0;   // lane w: word w of the block
#pragma unroll
    for (int c = 0; c < 8; c++) {
      const uint64_t b = __ballot(v[c] != 0);
      if (lane >> 1 == c) word = lane & 1 ? (uint32_t)(b >> 32) : (uint32_t)b;
    }
    if (full_blocks * 16 + lane < words) mask[full_blocks * 16 + lane] = (int32_t)word;   // 16 words at most
  }
}

// Unpack: a 16-lane row takes one block of 512 elements per step.  Lane r loads word r of the block (one
// 4-byte load, 64 contiguous bytes per row and 256 per wave), the row shares the 16 words by DPP broadcast,
// and lane r writes elements 16 r .. 16 r + 15 (bit r of every word) and 16 (r + 16) .. (bit r + 16): two 16-byte
// stores, each covering 256 contiguous bytes per row.  A wave takes MASK_STEPS steps (4 blocks each), all loads
// first.  (An earlier form let every lane load all 64 bytes of its block - 4 KB of requests per KB written: 75 us
// for 268 M elements against 47 us now, buffers cold in every cache.)
#ifndef MASK_STEPS
#define MASK_STEPS 2 /* 268 M elements: 49.1 us with 1, 47.4 with 2, 50.9 with 4, 55.2 with 8 */
#endif
template <int I>
__device__ __forceinline__ void mask_words_of_row(uint32_t mine, uint32_t (&w)[16]) {
  if constexpr (I < 16) {
    w[I] = row_bcast_u32<I>(mine);
    mask_words_of_row<I + 1>(mine, w);
  }
}
__global__ void __launch_bounds__(256)
mask_unpack_kernel(const int32_t* __restrict__ mask, int64_t n, uint8_t* __restrict__ out) {
  const int64_t wave = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int row = lane >> 4, r = lane & 15;
  const int64_t full_blocks = n / 512;
  const int64_t blk0 = wave * (MASK_STEPS * 4);
  if (blk0 > full_blocks) return;
  // the wave's stores go through a window that starts at its first block (see OutWindow)
  const int64_t window_first = blk0 * 512;
  const OutWindow window(out + window_first, n - window_first);
  uint32_t mine[MASK_STEPS];
#pragma unroll
  for (int j = 0; j < MASK_STEPS; j++) {
    const int64_t blk = blk0 + j * 4 + row;
    mine[j] = blk < full_blocks ? (uint32_t)mask[blk * 16 + r] : 0u;
  }
#pragma unroll
  for (int j = 0; j < MASK_STEPS; j++) {
    const int64_t blk = blk0 + j * 4 + row;
    uint32_t w[16];
    mask_words_of_row<0>(mine[j], w);   // every lane of the wave takes part in the broadcasts
    if (blk < full_blocks) {
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int k = r + 16 * h;
        uint32_t q[4];
#pragma unroll
        for (int c = 0; c < 4; c++)
          q[c] = ((w[4 * c] >> k) & 1u) | (((w[4 * c + 1] >> k) & 1u) << 8) | (((w[4 * c + 2] >> k) & 1u) << 16) |
                 (((w[4 * c + 3] >> k) & 1u) << 24);
        window.store16<GACT_STORE_NT_SYSTEM>(u32x4{q[0], q[1], q[2], q[3]}, (uint32_t)((blk - blk0) * 512 + k * 16));
      }
    } else if (blk == full_blocks) {
      // the partial block, in order: lane r of this row takes word r, elements 32 r .. 32 r + 31
      const int64_t first = full_blocks * 512 + r * 32;
      if (first < n) {
        const uint32_t word = (uint32_t)mask[full_blocks * 16 + r];
#pragma unroll
        for (int c = 0; c < 8; c++) {
          const uint32_t four = (word >> (4 * c)) & 15u;
          const uint32_t bytes = (four * 0x00204081u) & 0x01010101u;   // bit i of the four to byte i
          if (first + 4 * c + 4 <= n) {
            *reinterpret_cast<uint32_t*>(out + first + 4 * c) = bytes;
          } else {
#pragma unroll
            for (int e = 0; e < 3; e++)
              if (first + 4 * c + e < n) out[first + 4 * c + e] = (uint8_t)(bytes >> (8 * e));
          }
        }
      }
    }
  }
}

// ------------------------------------------------------------------------------------------------
// Greedy bit allocation.  calc_precision.cc:66-118: a max-heap of (float key, index) compared
// lexicographically; indices are distinct, so the pop order is the descending total order and an
// argmax restates it.  Keys are doubles narrowed to float exactly as the heap's pair<float, int64> does.
// ------------------------------------------------------------------------------------------------
__host__ __device__ inline int prec_next_bits(int b) { return b == 32 ? 8 : b == 8 ? 4 : b == 4 ? 2 : b == 2 ? 1 : 0; }
// Widths by level: 1, 2, 4, 8, 32.  The key of the step down from a level, which saves so many bits.
__host__ __device__ inline int prec_level(int bits) { return bits == 32 ? 4 : bits == 8 ? 3 : bits == 4 ? 2 : bits == 2 ? 1 : 0; }
__host__ __device__ inline int prec_width(int level) { return level == 4 ? 32 : 1 << level; }
__host__ __device__ inline float prec_level_key(float C, int level, int64_t saving) {
  double obj;
  if (level == 4) obj = -(double)C / 65025;
  else obj = C * (level == 3 ? 1.0 / 65025 - 1.0 / 225 : level == 2 ? 1.0 / 225 - 1.0 / 9 : 1.0 / 9 - 1.0 / 1);
  return (float)(obj / (double)saving);
}
__host__ __device__ inline float prec_key(float C, int b, int64_t w) { return prec_level_key(C, prec_level(b), w * (int64_t)(b - prec_next_bits(b))); }
__host__ __device__ inline bool prec_valid_bits(int b) { return b == 1 || b == 2 || b == 4 || b == 8 || b == 32; }

#define PREC_MAX_L 4096      /* tensors the device kernel handles (LDS tables, 12 bits of a candidate's key) */
#define PREC_THREADS 1024    /* largest workgroup the kernel is launched with */
#define PREC_BINS 256        /* bins of a histogram, four per lane of a wave */

// The sequential restatement of the heap loop by one wave: each step is a 64-lane argmax.  Used when a
// tensor's step keys do not decrease (never the case for the finite positive sensitivities the callers
// produce).
__device__ void calc_precision_sequential(int32_t* __restrict__ b_s, float* __restrict__ key_s,
                                          const float* __restrict__ C, const int64_t* __restrict__ w, int L,
                                          double b_sum, double target, int* rc_out) {
  const int lane = threadIdx.x;  // threadIdx.x < 64
  for (int idx = lane; idx < L; idx += 64)
    if (b_s[idx] > 1) key_s[idx] = prec_key(C[idx], b_s[idx], w[idx]);
  __builtin_amdgcn_wave_barrier();
  int rc = 0;
  while (b_sum > target) {
    float best_key = 0.0f;
    int best = -1;
    for (int idx = lane; idx < L; idx += 64) {
      if (b_s[idx] > 1) {
        const float k = key_s[idx];
        if (best < 0 || best_key < k || (!(k < best_key) && idx > best)) { best_key = k; best = idx; }
      }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      const float ok = __shfl_xor(best_key, off, 64);
      const int oi = __shfl_xor(best, off, 64);
      if (oi >= 0 && (best < 0 || best_key < ok || (!(ok < best_key) && oi > best))) { best_key = ok; best = oi; }
    }
    if (best < 0) { rc = GACT_EBUDGET; break; }
    const int cur = b_s[best];
    const int nb = prec_next_bits(cur);
    const int64_t wb = w[best];
    __builtin_amdgcn_wave_barrier();
    if (lane == 0) {
      b_s[best] = nb;
      if (nb > 1) key_s[best] = prec_key(C[best], nb, wb);
    }
    b_sum -= (double)(wb * (int64_t)(cur - nb));
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  *rc_out = rc;
}

// order-preserving map of a float key to an unsigned integer (+0 and -0 compare equal in the heap)
__device__ __forceinline__ uint32_t sortable_key(float k) {
  if (k == 0.0f) k = 0.0f;
  const uint32_t u = __builtin_bit_cast(uint32_t, k);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Over the lanes of a wave by DPP moves (rows, then the last lane of a row into the next ones): a running sum, and the least or
// greatest value, which ends up in the last lane.
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t lane_before(uint32_t v, uint32_t none) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ uint64_t add_lane_before(uint64_t v) {
  return v + (((uint64_t)lane_before<CTRL, ROWS>((uint32_t)(v >> 32), 0u) << 32) | lane_before<CTRL, ROWS>((uint32_t)v, 0u));
}
__device__ __forceinline__ uint64_t wave_running_sum(uint64_t v) {
  v = add_lane_before<0x111, 0xf>(v);   // row_shr:1, 2, 4, 8
  v = add_lane_before<0x112, 0xf>(v);
  v = add_lane_before<0x114, 0xf>(v);
  v = add_lane_before<0x118, 0xf>(v);
  v = add_lane_before<0x142, 0xa>(v);   // row_bcast:15 into rows 1 and 3
  return add_lane_before<0x143, 0xc>(v);   // row_bcast:31 into rows 2 and 3
}
template <bool MOST>
__device__ __forceinline__ uint32_t wave_extreme(uint32_t v) {
  const auto pick = [](uint32_t a, uint32_t b) { return MOST ? (a > b ? a : b) : (a < b ? a : b); };
  v = pick(v, lane_before<0x111, 0xf>(v, v));
  v = pick(v, lane_before<0x112, 0xf>(v, v));
  v = pick(v, lane_before<0x114, 0xf>(v, v));
  v = pick(v, lane_before<0x118, 0xf>(v, v));
  v = pick(v, lane_before<0x142, 0xa>(v, v));
  v = pick(v, lane_before<0x143, 0xc>(v, v));
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ __forceinline__ uint64_t read_lane(uint64_t v, int lane) {
  return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), lane) << 32) | (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
}

// The greedy pops candidates (tensor i, step s) in descending (key, i) order.  A tensor's steps have
// strictly decreasing keys, so that order is the descending order of ALL candidate steps by
// (key, index, earlier step first); the loop `while (b_sum > target) pop` then takes the candidates down to the one whose saving
// brings the sum to the target.  One workgroup, a thread per candidate (four a tensor, R a thread beyond 1024), looks for that one: the
// candidates' savings go into a histogram over the range of the keys left, a running sum over its bins from the top says in which bin the
// target is met, and that bin is the next range, until it holds one candidate (two or three histograms; six at most, the
// keys have 48 bits).  Then every candidate with a key not below that one's is taken.  Savings are integers: their
// sums are exact in any order.  Falls back to the sequential loop where the order argument does not hold.
// Bound by its chain of latencies - the loads, a double division, and per histogram the additions in LDS, a barrier and a scan that every
// wave does for itself.  Sorting all candidates (bitonic, slots in registers) and summing along the sorted order took, in graph replay, us, that /
// this: 3 tensors 5.6 / 2.7, 24 7.0 / 3.3, 69 9.3 / 3.8, 120 9.4 / 3.7, 160 13.4 / 4.5, 300 21.3 / 7.5, 1000 39.7 / 8.8, 4000 176 / 31.
template <int R>
__global__ void __launch_bounds__(PREC_THREADS)
calc_precision_kernel(int32_t* __restrict__ b, const float* __restrict__ C, const int64_t* __restrict__ w,
                      int L, double target, int32_t* __restrict__ status) {
  constexpr int WAVES = PREC_THREADS / 64;
  __shared__ __align__(16) uint64_t sum_s[3][PREC_BINS];
  __shared__ __align__(16) uint32_t count_s[3][PREC_BINS];
  __shared__ int64_t total_s[WAVES];
  __shared__ uint32_t least_s[WAVES], most_s[WAVES], flag_s[WAVES];   // flags: 1 not in order, 2 a width that is none
  __shared__ int32_t b_s[PREC_MAX_L];   // the sequential path's
  __shared__ float key_s[PREC_MAX_L];
  const int tid = threadIdx.x, NT = blockDim.x, lane = tid & 63, wave = tid >> 6, waves = NT >> 6;
  const auto clear = [&](int h) {
    for (int bin = tid; bin < PREC_BINS; bin += NT) {
      sum_s[h][bin] = 0;
      count_s[h][bin] = 0;
    }
  };

  uint64_t key[R];      // float key (ordered), index, earlier steps above later ones; 0: no candidate
  int64_t saving[R];
  int level[R];         // of the tensor's width
  int64_t total = 0;    // bits of all tensors that can take a step
  uint32_t least = 0xffffffffu, most = 0u;
  bool bad_order = false, bad_width = false;
  int32_t given[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int slot = r * NT + tid, idx = slot >> 2;
    given[r] = idx < L ? b[idx] : 1;
    saving[r] = idx < L ? w[idx] : 1;
  }
  float Ci[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int idx = (r * NT + tid) >> 2;
    Ci[r] = idx < L ? C[idx] : 0.0f;
  }
  clear(0);
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int slot = r * NT + tid, idx = slot >> 2, st = slot & 3;
    const int64_t wi = saving[r];
    bad_width |= !prec_valid_bits(given[r]);
    level[r] = prec_level(given[r]);
    const int from = level[r] - st;
    const bool step = from > 0;
    if (level[r] > 0 && st == 0) total += (int64_t)given[r] * wi;
    saving[r] = wi * (int64_t)(prec_width(step ? from : 1) - prec_width(step ? from - 1 : 0));
    const float k = prec_level_key(Ci[r], step ? from : 1, saving[r]);
    const float before = __builtin_bit_cast(float, lane_before<0x90, 0xf>(__builtin_bit_cast(uint32_t, k), 0u));   // quad_perm [0,0,1,2]
    const float prev = st == 0 ? __builtin_inff() : before;
    const uint32_t order = sortable_key(k);
    if (step) {
      // keys that do not decrease (NaN among them), or a size that is no size
      if ((!(k < prev) && !(k == prev && k == 0.0f)) || wi <= 0) bad_order = true;
      least = order < least ? order : least;
      most = order > most ? order : most;
    }
    key[r] = step ? ((uint64_t)order << 16) | ((uint32_t)idx << 4) | (uint32_t)(3 - st) : 0;
  }
  total = (int64_t)read_lane(wave_running_sum((uint64_t)total), 63);
  least = wave_extreme<false>(least);
  most = wave_extreme<true>(most);
  const uint32_t flags = (__builtin_amdgcn_ballot_w64(bad_order) != 0 ? 1u : 0u) | (__builtin_amdgcn_ballot_w64(bad_width) != 0 ? 2u : 0u);
  if (lane == 0) {
    total_s[wave] = total;
    least_s[wave] = least;
    most_s[wave] = most;
    flag_s[wave] = flags;
  }
  __syncthreads();
  int64_t b_sum = 0;
  uint32_t flag = 0;
  for (int v = 0; v < waves; v++) {
    b_sum += total_s[v];
    least = least_s[v] < least ? least_s[v] : least;
    most = most_s[v] > most ? most_s[v] : most;
    flag |= flag_s[v];
  }
  if (flag & 2) {  // a width outside {1,2,4,8,32}: leave b as it is
    if (status && tid == 0) *status = GACT_EINVAL;
    return;
  }
  int rc = 0;
  if (flag) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int slot = r * NT + tid;
      if ((slot & 3) == 0 && (slot >> 2) < L) b_s[slot >> 2] = given[r];
    }
    __syncthreads();
    if (tid < 64) calc_precision_sequential(b_s, key_s, C, w, L, (double)b_sum, target, &rc);
    __syncthreads();
    for (int idx = tid; idx < L; idx += NT) b[idx] = b_s[idx];
    if (status && tid == 0) *status = rc;
    return;
  }

  uint64_t last = ~0ull;   // candidates from this key on are taken
  if ((double)b_sum > target) {
    uint64_t from = (uint64_t)least << 16, span = ((((uint64_t)most << 16) | 0xffffu) - from);   // the keys left: from .. from + span
    if (most < least) span = 0;                                                                  // no candidate at all
    int64_t left = b_sum;                                                                        // without what lies above the range
    // three histograms in turn: the next one is cleared while this one fills, and two levels back everybody has passed a barrier since
    for (int h = 0;; h = h == 2 ? 0 : h + 1) {
      const int bits = 64 - __builtin_clzll(span | 1), shift = bits > 8 ? bits - 8 : 0;
#pragma unroll
      for (int r = 0; r < R; r++) {
        const uint64_t at = key[r] - from;
        if (key[r] != 0 && at <= span) {
          const uint32_t bin = (uint32_t)(at >> shift);
          atomicAdd((unsigned long long*)&sum_s[h][bin], (unsigned long long)saving[r]);
          atomicAdd(&count_s[h][bin], 1u);
        }
      }
      clear(h == 2 ? 0 : h + 1);
      __syncthreads();
      // lane l: bins 255 - 4 l and the three below, the higher ones first
      int64_t s4[4];
      uint32_t c4[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        s4[j] = (int64_t)sum_s[h][PREC_BINS - 1 - 4 * lane - j];
        c4[j] = count_s[h][PREC_BINS - 1 - 4 * lane - j];
      }
      const int64_t mine = s4[0] + s4[1] + s4[2] + s4[3];
      const int64_t incl = (int64_t)wave_running_sum((uint64_t)mine);
      const uint64_t meets = __builtin_amdgcn_ballot_w64(!((double)(left - incl) > target));
      if (meets == 0) {   // every step taken and still over budget
        last = 0;
        rc = GACT_EBUDGET;
        break;
      }
      const int where = __builtin_ctzll(meets);   // the first lane after whose bins the target is met
      int64_t running = left - (incl - mine), above = running;
      int bin = 0;
      uint32_t count = 0;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if ((double)running > target) {
          bin = j;
          above = running;
          count = c4[j];
        }
        running -= s4[j];
      }
      left = (int64_t)read_lane((uint64_t)above, where);
      from += (uint64_t)(PREC_BINS - 1 - 4 * where - __builtin_amdgcn_readlane(bin, where)) << shift;
      span = (1ull << shift) - 1;
      if (__builtin_amdgcn_readlane((int)count, where) <= 1) {
        last = from;
        break;
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int slot = r * NT + tid;
    const uint64_t taken = __builtin_amdgcn_ballot_w64(key[r] != 0 && key[r] >= last);   // a tensor's: its first so many
    if ((slot & 3) == 0 && (slot >> 2) < L) b[slot >> 2] = prec_width(level[r] - __builtin_popcount((uint32_t)(taken >> lane) & 15u));
  }
  if (status && tid == 0) *status = rc;
}

// ------------------------------------------------------------------------------------------------
// Batched launch over a table of tensors with device-resident bits.
// ------------------------------------------------------------------------------------------------
// The workspace of a batched launch (device memory the caller brings, or the library's static array):
//   BatchHeader                      what the plan found
//   int32 block_tensor[total_blocks] tensor of every block of the grid
struct BatchHeader {
  int64_t need;            // arena bytes the table needs
  int64_t ok;              // 1: every width and element type valid and need <= capacity
  int64_t tensors_at[4];   // tensors at width 1, 2, 4, 8
  int64_t reserved[26];
};
static_assert(sizeof(BatchHeader) == 256, "the header is 32 int64");
struct BatchWorkspace {
  BatchHeader* hdr;
  int32_t* block_tensor;
};
__host__ __device__ inline int64_t batch_workspace_need(int64_t L, int64_t total_blocks) {
  (void)L;
  return (int64_t)sizeof(BatchHeader) + (total_blocks + 3) / 4 * 16;
}
__host__ __device__ inline BatchWorkspace batch_workspace(void* base) {
  BatchWorkspace w;
  w.hdr = (BatchHeader*)base;
  w.block_tensor = (int32_t*)((uint8_t*)base + sizeof(BatchHeader));
  return w;
}
__device__ __forceinline__ int width_index(int bits) { return bits == 1 ? 0 : bits == 2 ? 1 : bits == 4 ? 2 : 3; }

template <typename FIRST>
__device__ __forceinline__ int batch_find(const FIRST& first_block, int L, int64_t block) {
  int lo = 0, hi = L - 1;  // last entry with first_block <= block
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (first_block(mid) <= block) lo = mid; else hi = mid - 1;
  }
  return lo;
}
// The plan's workgroups behind the first note the tensor of 256 blocks each.  The tensors' first blocks come into LDS at once (up to
// PLAN_LDS_L of them): a search in memory is a chain of loads, one for every bit of L, and was what the plan's launch took longest for
// (graph replay, a launch: 3 tensors 4.0 -> 2.6 us, 45 4.0 -> 2.55, 120 4.1 -> 2.7, 190 4.3 -> 2.9, 400 4.1 -> 3.2, 800 5.3 -> 4.6, 2048 9.2 -> 7.9,
// from one block a tensor to 512).
#define PLAN_THREADS 256
#define PLAN_LDS_L 2048
__device__ __forceinline__ void batch_plan_blocks(const gact_batch_entry* __restrict__ table, int L, int64_t total_blocks, const BatchWorkspace& ws) {
  __shared__ int32_t first_s[PLAN_LDS_L];   // a grid has fewer than 2^31 blocks
  const int64_t g = (int64_t)(blockIdx.x - 1) * PLAN_THREADS + threadIdx.x;
  if (L <= PLAN_LDS_L) {
    for (int t = threadIdx.x; t < L; t += PLAN_THREADS) first_s[t] = (int32_t)table[t].first_block;
    __syncthreads();
    if (g < total_blocks) ws.block_tensor[g] = batch_find([&](int t) { return (int64_t)first_s[t]; }, L, g);
  } else if (g < total_blocks) {
    ws.block_tensor[g] = batch_find([&](int t) { return table[t].first_block; }, L, g);
  }
}

// Bytes of the arena a tensor of N groups takes at a width, as the plan counts them
__device__ __forceinline__ int64_t batch_span(int width, int64_t N) {
  const int wpt = 8 / width;
  const int64_t n_round = (N + wpt - 1) / wpt * wpt;
  return ((int64_t)width * n_round * (GROUP / 8) + 255) / 256 * 256;
}

// What the plan's workgroup 0 does: thread t sizes tensors t, t + 256, ...; the running packed-arena offset is carried across rounds of
// 256 with an inclusive scan of each wave and the waves' totals.  One round, with the loads of all tensors under way at once, where a
// wave alone took two (65 to 128 tensors).  entry(t) loads all that is needed of a tensor, place(t, entry, offset) takes that and what
// the plan finds for it.
template <typename ENTRY, typename PLACE>
__device__ __forceinline__ void batch_plan_sizes(const int32_t* __restrict__ bits, int L, int64_t capacity, const BatchWorkspace& ws,
                                                 int64_t* __restrict__ verdict, const ENTRY& entry, const PLACE& place) {
  constexpr int WAVES = PLAN_THREADS / 64;
  __shared__ int64_t total_s[WAVES];
  __shared__ int bad_s, count_s[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (threadIdx.x == 0) bad_s = 0;
  if (threadIdx.x < 4) count_s[threadIdx.x] = 0;
  __syncthreads();
  int64_t base = 0;
  for (int t0 = 0; t0 < L; t0 += PLAN_THREADS) {
    const int t = t0 + threadIdx.x;
    int64_t bytes = 0;
    int width = 0;
    gact_batch_entry e = {};
    if (t < L) {
      const int given = bits[t];
      e = entry(t);
      const bool valid = given == 1 || given == 2 || given == 4 || given == 8;
      width = valid ? given : 8;
      if (!valid || e.dtype < 0 || e.dtype > 2) bad_s = 1;
      atomicAdd(&count_s[width_index(width)], 1);
      bytes = batch_span(width, (e.numel + GROUP - 1) / GROUP);
    }
    const int64_t incl = (int64_t)wave_running_sum((uint64_t)bytes);
    if (lane == 63) total_s[wave] = incl;
    __syncthreads();
    int64_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
      before += w < wave ? total_s[w] : 0;
      all += total_s[w];
    }
    if (t < L) place(t, e, base + before + incl - bytes);
    base += all;
    __syncthreads();
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const int64_t ok = (!bad_s && base <= capacity) ? 1 : 0;
    ws.hdr->need = base;
    ws.hdr->ok = ok;
    if (verdict) {   // the same two words where the caller can see them: written through, for a host that looks at them before the kernel's end
      __hip_atomic_store(verdict, base, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __hip_atomic_store(verdict + 1, ok, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
#pragma unroll
    for (int k = 0; k < 4; k++) ws.hdr->tensors_at[k] = count_s[k];
  }
}

// The plan, one launch.  Workgroup 0: batch_plan_sizes.  The other workgroups, one thread per
// block of the grid: find the block's tensor and note it, so that a work kernel's block needs one load for it
// (this part depends on the geometry only, not on the widths).
__global__ void __launch_bounds__(PLAN_THREADS)
batch_plan_kernel(gact_batch_entry* table, const int32_t* __restrict__ bits, int L, int64_t total_blocks,
                  int64_t capacity, BatchWorkspace ws, int64_t* __restrict__ verdict) {
  if (blockIdx.x > 0) {
    batch_plan_blocks(table, L, total_blocks, ws);
    return;
  }
  batch_plan_sizes(bits, L, capacity, ws, verdict, [&](int t) { return table[t]; },
                   [&](int t, const gact_batch_entry&, int64_t offset) { table[t].packed_offset = offset; });
}

// The plan of a table that the launch itself brings: what changes from call to call - a tensor's address and its seed - arrives in the
// kernel's arguments, everything else of the entries is read from `geometry` on the GPU.  The table, a copy of the widths and the
// verdict (which may lie in pinned host memory) are written by the same launch, where three copies stood around it, four launches and the
// Python between them.  69 half tensors, 16 M elements together: host time of a quantize call 68 -> 26 us; with the dequantize call's plan
// brought the same way calc_precision, quantize and dequantize together 116 -> 62; 142 float tensors, 67 M elements, 165 -> 144.
struct BatchArgs {
  const void* x[GACT_BATCH_ARGS];
  uint64_t seed[GACT_BATCH_ARGS];
};
__global__ void __launch_bounds__(PLAN_THREADS)
batch_plan_args_kernel(BatchArgs args, const gact_batch_entry* __restrict__ geometry, gact_batch_entry* __restrict__ table,
                       const int32_t* __restrict__ bits, int32_t* __restrict__ kept, int L, int64_t total_blocks, int64_t capacity,
                       BatchWorkspace ws, int64_t* __restrict__ verdict) {
  if (blockIdx.x > 0) {
    batch_plan_blocks(geometry, L, total_blocks, ws);
    return;
  }
  if (kept)
    for (int t = threadIdx.x; t < L; t += PLAN_THREADS) kept[t] = bits[t];
  batch_plan_sizes(bits, L, capacity, ws, verdict,
                   [&](int t) {
                     gact_batch_entry e = geometry[t];
                     e.x = args.x[t];
                     e.seed = args.seed[t];
                     return e;
                   },
                   [&](int t, gact_batch_entry e, int64_t offset) {
                     e.packed_offset = offset;
                     table[t] = e;
                   });
}

// Quantize, one launch per element type over all blocks of the grid: the width of a block's tensor is read from
// device memory and selects the code path (a row takes 8 groups whatever the width, so every path holds the same
// amount of data in registers); blocks of tensors of another element type leave at once.  PACKED: the sum of the widths below 8 whose
// codes are packed as bytes where packs_bytes allows it (see batch_packs).
template <typename T, int NOISE, int PACKED>
__global__ void __launch_bounds__(256)
quantize_batched_kernel(const gact_batch_entry* __restrict__ table, const int32_t* __restrict__ bits,
                        BatchWorkspace ws, uint8_t* __restrict__ packed_arena, uint8_t* __restrict__ scale_arena,
                        uint8_t* __restrict__ min_arena) {
  if (ws.hdr->ok == 0) return;  // the plan did not fit the arena or held an invalid width
  const int64_t block = xcd_tile<GACT_XCD_RUN_QB>(blockIdx.x, gridDim.x);
  const int t = ws.block_tensor[block];
  const gact_batch_entry ent = table[t];
  if (ent.dtype != Elem<T>::kDtype) return;
  const int64_t N = (ent.numel + GROUP - 1) / GROUP;
  const int64_t lb = block - ent.first_block;
  const T* x = (const T*)ent.x;
  uint8_t* packed = packed_arena + ent.packed_offset;
  typename Elem<T>::Stat* sc = (typename Elem<T>::Stat*)(scale_arena + ent.stats_offset * 4);
  T* mn = (T*)(min_arena + ent.stats_offset * 4);
  switch (bits[t]) {
    case 1: quantize_block128<T, 1, NOISE, (PACKED & 1) != 0>(x, ent.numel, N, lb, packed, sc, mn, ent.seed); break;
    case 2: quantize_block128<T, 2, NOISE, (PACKED & 2) != 0>(x, ent.numel, N, lb, packed, sc, mn, ent.seed); break;
    case 4: quantize_block128<T, 4, NOISE, (PACKED & 4) != 0>(x, ent.numel, N, lb, packed, sc, mn, ent.seed); break;
    default: quantize_block128<T, 8, NOISE>(x, ent.numel, N, lb, packed, sc, mn, ent.seed); break;
  }
}

// Dequantize, one launch for all widths (every width fits 60 registers): the width of a block's tensor is read
// from device memory and selects the code path, so no workgroup is launched only to leave.
template <int BITS>
__device__ __forceinline__ void dequantize_batched_block(const gact_batch_entry& ent, int64_t lb, int quarter,
                                                         const uint8_t* packed, const uint8_t* sc, const uint8_t* mn) {
  const int64_t N = (ent.numel + GROUP - 1) / GROUP;
  if (ent.dtype == GACT_F32)
    dequantize_block128<float, BITS>(packed, (const float*)sc, (const float*)mn, ent.numel, N, lb, quarter, (float*)ent.x);
  else if (ent.dtype == GACT_F16)
    dequantize_block128<f16, BITS>(packed, (const f16*)sc, (const f16*)mn, ent.numel, N, lb, quarter, (f16*)ent.x);
  else
    dequantize_block128<bf16, BITS>(packed, (const float*)sc, (const bf16*)mn, ent.numel, N, lb, quarter, (bf16*)ent.x);
}
// grid: four workgroups per block of 128 groups; workgroups on a CU: batch_dequantize_lds
__device__ __forceinline__ void dequantize_batched(const gact_batch_entry* __restrict__ table, const void* const* outs,
                                                   const int32_t* __restrict__ bits, const BatchWorkspace& ws,
                                                   const uint8_t* __restrict__ packed_arena, const uint8_t* __restrict__ scale_arena,
                                                   const uint8_t* __restrict__ min_arena) {
  if (ws.hdr->ok == 0) return;
  // the XCD-aware order of the single-tensor kernel (715 -> 709 us on 120 half tensors)
  const uint32_t tile = xcd_tile<GACT_XCD_RUN_DQB>(blockIdx.x, gridDim.x);
  const int64_t block = tile >> 2;
  const int quarter = tile & 3;   // which quarter of the block
  const int t = ws.block_tensor[block];
  gact_batch_entry ent = table[t];
  if (outs) ent.x = outs[t];
  const int width = bits[t];
  // the plan may be older than this launch: a width written over since must not lead past the codes
  if (outs) {
    const int64_t N = (ent.numel + GROUP - 1) / GROUP;
    const int64_t span = width == 1 ? batch_span(1, N) : width == 2 ? batch_span(2, N) : width == 4 ? batch_span(4, N) : batch_span(8, N);
    if (ent.packed_offset + span > ws.hdr->need) return;
  }
  const int64_t lb = block - ent.first_block;
  const uint8_t* packed = packed_arena + ent.packed_offset;
  const uint8_t* sc = scale_arena + ent.stats_offset * 4;
  const uint8_t* mn = min_arena + ent.stats_offset * 4;
  switch (width) {
    case 1: dequantize_batched_block<1>(ent, lb, quarter, packed, sc, mn); break;
    case 2: dequantize_batched_block<2>(ent, lb, quarter, packed, sc, mn); break;
    case 4: dequantize_batched_block<4>(ent, lb, quarter, packed, sc, mn); break;
    default: dequantize_batched_block<8>(ent, lb, quarter, packed, sc, mn); break;
  }
}
__global__ void __launch_bounds__(256)
dequantize_batched_kernel(const gact_batch_entry* __restrict__ table, const int32_t* __restrict__ bits,
                          BatchWorkspace ws, const uint8_t* __restrict__ packed_arena,
                          const uint8_t* __restrict__ scale_arena, const uint8_t* __restrict__ min_arena) {
  dequantize_batched(table, nullptr, bits, ws, packed_arena, scale_arena, min_arena);
}
// With the outputs' addresses in the launch's arguments: the table and the plan of the quantize call serve as they are, where a plan of
// the outputs' own table stood before this launch (3.8 us on the GPU and a launch).  A block's address is one more scalar load beside its
// entry.  69 half tensors, 16 M elements: calc_precision, quantize and dequantize 61.5 -> 53.7 us, 142 float tensors 140 -> 131; 120 half
// tensors, 1.83 G elements, 1360 -> 1351.
struct BatchOutputs {
  const void* x[GACT_BATCH_ARGS];
};
__global__ void __launch_bounds__(256)
dequantize_batched_to_kernel(const gact_batch_entry* __restrict__ table, const int32_t* __restrict__ bits,
                             BatchWorkspace ws, const uint8_t* __restrict__ packed_arena,
                             const uint8_t* __restrict__ scale_arena, const uint8_t* __restrict__ min_arena, BatchOutputs outs) {
  dequantize_batched(table, outs.x, bits, ws, packed_arena, scale_arena, min_arena);
}

// ------------------------------------------------------------------------------------------------
// Host side of the C ABI.
// ------------------------------------------------------------------------------------------------
namespace {

inline bool valid_bits(int bits) { return bits == 1 || bits == 2 || bits == 4 || bits == 8; }
inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
// hipGetLastError returns and clears the thread's last error, which may be one an earlier call of the caller's left
// behind: an entry point clears it before its first launch (fresh_launch) and reports what its own launches left.
inline void fresh_launch() { (void)hipGetLastError(); }
inline int launch_status() { return hipGetLastError() == hipSuccess ? GACT_OK : GACT_ELAUNCH; }

// one 16-lane row per unit of work (a super-group for quantize / dequantize, 8 groups for minimax);
// 16 rows per 256-thread block
inline void row_grid(int64_t rows, dim3* grid, dim3* block, int threads = 256) {
  const int rows_per_block = threads / 16;
  *grid = dim3((unsigned)((rows + rows_per_block - 1) / rows_per_block));
  *block = dim3(threads);
}
inline int64_t supergroups(int64_t N, int bits) { return (N + 8 / bits - 1) / (8 / bits); }

// Fewer resident waves per CU for some kernels on large tensors.  These streams mix a minority of traffic in
// the other direction into their main direction, and past a point more requests in flight make that mix more
// expensive for the memory system, not cheaper (a stand-alone kernel that writes 8 KB and reads 1 KB per
// wave: 88 us for 411 MB at full occupancy, 70 us at 2 waves per SIMD).  The cap is a request for dynamic
// LDS that the kernels never touch - a CU has 160 KB of it, so 53 000 bytes admit 3 workgroups.  What counts is
// the bytes in flight per CU: the cap goes with units of 8 groups (8 KB of stores per float wave); with units of 4
// it starves the CU (float 1 bit, 103 M elements: 66 us with units of 8 and the cap, 71 with units of 4 and no cap,
// 98 with units of 4 and the cap; float 8 bit: 80, 82, 96; half 8 bit, 256 M elements, 4 workgroups per CU: 119, 129,
// 147).  Hence the geometry table's own entries for large tensors.
// Interleaved A/B in both orders on a 411 MB float tensor (us, full occupancy -> capped), units of 8 groups:
// dequantize with 3 workgroups of 4 waves per CU 1 bit 76.3 -> 66.1, 2 bit 76.4 -> 69.6, 4 bit 77.6 -> 74.5,
// 8 bit 81.7 -> 79.9; quantize float 4 bit with 16 one-wave workgroups 76.1 -> 71.1.
// The other kernels (all half quantize, float quantize at 1, 2 and 8 bit) and small tensors gain nothing or
// lose, and keep full occupancy.
// From 2^17 groups (34 M elements) on (`large_from` in the geometry table): with buffers that are cold in every cache
// the cap costs 3-12 % at 8-26 M elements, is neutral at 31-34 M and gains 1-7 % from 43 M, 3-13 % at 84 M.
// Quantize, float: 4 bit capped at 16 one-wave workgroups per CU from 98 304 groups on (100 000 groups: 21.1 -> 20.9 us,
// 200 000: 40.1 -> 37.9, 401 408: 77.4 -> 72.6, 1 M: 191.5 -> 177.8; 65 536: 14.6 -> 14.65), 2 bit at 8 from 196 608 groups on
// (262 144 groups: 47.6 -> 46.2 us, 401 408: 72.2 -> 69.1, 1 M: 177.3 -> 165.3; 131 072: 25.3 -> 26.1).  Buffers cold in
// every cache.  1 and 8 bit gain 1-2 % at most, half loses at 4 and 8 bit and gains 1-2 % at 1 and 2 bit: left alone.
#ifndef GACT_QCAP_FROM_GROUPS
#define GACT_QCAP_FROM_GROUPS (3 << 15)
#endif
#ifndef GACT_QCAP2_FROM_GROUPS
#define GACT_QCAP2_FROM_GROUPS (3 << 16)
#endif
inline unsigned quantize_lds_cap(size_t elem_size, int bits, int64_t N) {
  if (elem_size != 4) return 0u;
  if (bits == 4) return N >= GACT_QCAP_FROM_GROUPS ? 10000u : 0u;
  if (bits == 2) return N >= GACT_QCAP2_FROM_GROUPS ? 20000u : 0u;
  return 0u;
}

// Below how many groups a 1-bit quantize takes the wave-per-super-group kernel (0: never), by element size.  (The kernel
// also exists at 2 bit - four rows of one group each, 4 KB per float wave - and is not launched there: float [4096,1024]
// at 2 bit, deterministic, 5.22 us with a row per super-group against 5.37-5.52 us that way, in workgroups of one or
// four waves, with or without the XCD-aware tile order; 13 M elements 11.3 against 11.4-11.8 us; 103 M 68.1 / 67.6-68.8.)
#ifndef GACT_W8_BELOW_F32
#define GACT_W8_BELOW_F32 (1 << 18)
#endif
#ifndef GACT_W8_BELOW_F16
#define GACT_W8_BELOW_F16 40960
#endif
#ifndef GACT_W8_THREADS
#define GACT_W8_THREADS 256
#endif

// What a single-tensor launch is made of: the kernel, its grid, and the dynamic LDS it asks for.  Planning and
// launching are separate so that gact_launch_geometry reports exactly what a launch would use.
struct LaunchPlan {
  const void* kernel = nullptr;   // null: the arguments name no kernel (an unknown noise mode or width)
  dim3 grid, block;
  unsigned lds = 0;
};

// the quantize kernel of a noise mode: its small-tensor form where the geometry has one (staging is for fused
// min/max and not for the reference stream)
template <typename T, int BITS, int NOISE, bool GIVEN>
const void* quantize_kernel_of(bool small) {
  constexpr QGeom G = q_geom<T>(BITS);
  // small tensors have a kernel of their own where it differs: in its stages, or (half at 2 bit) in how it packs
  constexpr bool PACKS_WHEN_SMALL = std::is_same<T, f16>::value && BITS == 2 && NOISE != GACT_NOISE_INJECT;
  if constexpr (!GIVEN && NOISE != GACT_NOISE_REF && (G.stage_small != G.stage || G.lazy_small != G.lazy || PACKS_WHEN_SMALL)) {
    if (small) return (const void*)quantize_kernel<T, BITS, NOISE, GIVEN, true>;
  }
  return (const void*)quantize_kernel<T, BITS, NOISE, GIVEN, false>;
}

template <typename T, int BITS, bool GIVEN>
LaunchPlan plan_quantize(int64_t N, int noise_mode) {
  LaunchPlan p;
  constexpr QGeom G = q_geom<T>(BITS);
  if constexpr (!GIVEN && BITS == 1) {
    if (noise_mode != GACT_NOISE_REF && N < (sizeof(T) == 4 ? GACT_W8_BELOW_F32 : GACT_W8_BELOW_F16)) {
      const unsigned per_block = GACT_W8_THREADS / 64;
      p.grid = dim3((unsigned)((supergroups(N, BITS) + per_block - 1) / per_block));
      p.block = dim3(GACT_W8_THREADS);
      switch (noise_mode) {
        case GACT_NOISE_CONST: p.kernel = (const void*)quantize_wave8_kernel<T, BITS, GACT_NOISE_CONST>; break;
        case GACT_NOISE_INJECT: p.kernel = (const void*)quantize_wave8_kernel<T, BITS, GACT_NOISE_INJECT>; break;
        case GACT_NOISE_FAST: p.kernel = (const void*)quantize_wave8_kernel<T, BITS, GACT_NOISE_FAST>; break;
      }
      return p;
    }
  }
  const int sgr = noise_mode == GACT_NOISE_REF ? 1 : G.sgr;
  row_grid((supergroups(N, BITS) + sgr - 1) / sgr, &p.grid, &p.block, G.threads);
  // the reference stream's one Philox block per byte makes the kernel instruction-bound: it wants every wave
  p.lds = noise_mode == GACT_NOISE_REF ? 0u : quantize_lds_cap(sizeof(T), BITS, N);
  const bool small = N < G.small_below;
  switch (noise_mode) {
    case GACT_NOISE_CONST: p.kernel = quantize_kernel_of<T, BITS, GACT_NOISE_CONST, GIVEN>(small); break;
    case GACT_NOISE_INJECT: p.kernel = quantize_kernel_of<T, BITS, GACT_NOISE_INJECT, GIVEN>(small); break;
    case GACT_NOISE_REF: p.kernel = quantize_kernel_of<T, BITS, GACT_NOISE_REF, GIVEN>(small); break;
    case GACT_NOISE_FAST: p.kernel = quantize_kernel_of<T, BITS, GACT_NOISE_FAST, GIVEN>(small); break;
  }
  return p;
}

template <typename T, bool GIVEN>
LaunchPlan plan_quantize_bits(int bits, int64_t N, int noise_mode) {
  switch (bits) {
    case 1: return plan_quantize<T, 1, GIVEN>(N, noise_mode);
    case 2: return plan_quantize<T, 2, GIVEN>(N, noise_mode);
    case 4: return plan_quantize<T, 4, GIVEN>(N, noise_mode);
    case 8: return plan_quantize<T, 8, GIVEN>(N, noise_mode);
  }
  return LaunchPlan();
}

// every quantize kernel takes the same arguments
template <typename T, bool GIVEN>
int dispatch_quantize(int bits, const T* x, int64_t numel, int64_t N, uint8_t* packed, typename Elem<T>::Stat* scale,
                      T* mn, T* mx,
                      int noise_mode, SeedArg seed, const float* noise, hipStream_t stream) {
  const LaunchPlan p = plan_quantize_bits<T, GIVEN>(bits, N, noise_mode);
  if (!p.kernel) return GACT_EINVAL;
  void* args[] = {(void*)&seed, (void*)&x, (void*)&numel, (void*)&N, (void*)&packed, (void*)&scale, (void*)&mn, (void*)&mx, (void*)&noise};
  return hipLaunchKernel(p.kernel, p.grid, p.block, args, p.lds, stream) == hipSuccess ? GACT_OK : GACT_ELAUNCH;
}

template <typename T>
LaunchPlan plan_dequantize(int bits, int64_t N) {
  LaunchPlan p;
  // a unit takes 256 / (16 / sizeof(T)) lanes
  const DqGeom d = dq_geom<T>(bits);
  const bool large = N >= d.large_from;
  const int64_t units_per_block = d.threads / (GROUP / (16 / (int64_t)sizeof(T)));
  const int64_t unit_groups = dq_unit_groups(d, bits, large);
  // the caps are stated for workgroups of 256 threads
  p.lds = N >= d.cap_from ? d.lds_large * (unsigned)d.threads / 256u : 0u;
  p.grid = dim3((unsigned)(((N + unit_groups - 1) / unit_groups + units_per_block - 1) / units_per_block));
  p.block = dim3((unsigned)d.threads);
#define GACT_DQ_KERNEL(B) (large ? (const void*)dequantize_kernel<T, B, true> : (const void*)dequantize_kernel<T, B, false>)
  switch (bits) {
    case 1: p.kernel = GACT_DQ_KERNEL(1); break;
    case 2: p.kernel = GACT_DQ_KERNEL(2); break;
    case 4: p.kernel = GACT_DQ_KERNEL(4); break;
    case 8: p.kernel = GACT_DQ_KERNEL(8); break;
  }
#undef GACT_DQ_KERNEL
  return p;
}

template <typename T>
int dispatch_dequantize(int bits, const uint8_t* packed, const typename Elem<T>::Stat* scale, const T* mn,
                        int64_t numel, int64_t N, T* out,
                        hipStream_t stream) {
  const LaunchPlan p = plan_dequantize<T>(bits, N);
  if (!p.kernel) return GACT_EINVAL;
  void* args[] = {(void*)&packed, (void*)&scale, (void*)&mn, (void*)&numel, (void*)&N, (void*)&out};
  return hipLaunchKernel(p.kernel, p.grid, p.block, args, p.lds, stream) == hipSuccess ? GACT_OK : GACT_ELAUNCH;
}

// ---- group sizes of the one-pass kernels other than 256 ----
inline bool one_pass_group(int64_t group) { return group == 64 || group == 128 || group == 512; }

template <typename T, int D, int BITS>
LaunchPlan plan_quantize_groups(int64_t N, int noise_mode) {
  typedef GroupsShape<T, D, BITS> S;
  LaunchPlan p;
  row_grid((N + S::UNIT_GROUPS - 1) / S::UNIT_GROUPS * S::ROWS, &p.grid, &p.block, 64);
  switch (noise_mode) {
    case GACT_NOISE_CONST:
      p.kernel = (const void*)quantize_groups_kernel<T, D, BITS, GACT_NOISE_CONST>;
      // half at 1 bit in groups of 512: packed bytes take 80 registers instead of 94, six waves on a SIMD instead of five, which costs
      // bandwidth from 16 M elements on (a cap at five or four waves does not help).  Joined per byte / packed, us: 2 M 4.31 / 4.02,
      // 4 M 4.57 / 4.30, 8 M 5.50 / 5.53, 12 M 6.96 / 7.22, 17 M 8.3 / 8.9, 34 M 14.6 / 15.0, 67 M 25.1 / 26.0, 134 M 46.7 / 48.1
      if constexpr (std::is_same<T, f16>::value && D == 512 && BITS == 1) {
        if (N >= 1 << 14) p.kernel = (const void*)quantize_groups_kernel<T, D, BITS, GACT_NOISE_CONST, false>;
      }
      break;
    case GACT_NOISE_INJECT: p.kernel = (const void*)quantize_groups_kernel<T, D, BITS, GACT_NOISE_INJECT>; break;
    case GACT_NOISE_FAST: p.kernel = (const void*)quantize_groups_kernel<T, D, BITS, GACT_NOISE_FAST>; break;
  }
  return p;
}
template <typename T, int D>
LaunchPlan plan_quantize_groups_bits(int bits, int64_t N, int noise_mode) {
  switch (bits) {
    case 1: return plan_quantize_groups<T, D, 1>(N, noise_mode);
    case 2: return plan_quantize_groups<T, D, 2>(N, noise_mode);
    case 4: return plan_quantize_groups<T, D, 4>(N, noise_mode);
    case 8: return plan_quantize_groups<T, D, 8>(N, noise_mode);
  }
  return LaunchPlan();
}
template <typename T>
int dispatch_quantize_groups(int64_t group, int bits, const T* x, int64_t numel, int64_t N, uint8_t* packed, T* scale, T* mn,
                             T* mx, int noise_mode, SeedArg seed, const float* noise, hipStream_t stream) {
  const LaunchPlan p = group == 64    ? plan_quantize_groups_bits<T, 64>(bits, N, noise_mode)
                       : group == 128 ? plan_quantize_groups_bits<T, 128>(bits, N, noise_mode)
                                      : plan_quantize_groups_bits<T, 512>(bits, N, noise_mode);
  if (!p.kernel) return GACT_EINVAL;
  void* args[] = {(void*)&seed, (void*)&x, (void*)&numel, (void*)&N, (void*)&packed, (void*)&scale, (void*)&mn, (void*)&mx, (void*)&noise};
  return hipLaunchKernel(p.kernel, p.grid, p.block, args, p.lds, stream) == hipSuccess ? GACT_OK : GACT_ELAUNCH;
}

// One piece per lane keeps the most waves and the shortest chain in each, two keep more in flight per wave and are better once
// the tensor fills the chip several times over.  Dequantize of groups of 128, us, buffers cold in every cache, one piece / two
// (four and eight lose 5-100 % everywhere but float 8 bit, where they gain nothing):
//   float 1 M elements  2 bit 2.6 / 3.3  4 bit 2.6 / 2.9  8 bit 2.6 / 2.6    4 M  2 bit 4.46 / 4.42  4 bit 4.5 / 4.9  8 bit 5.7 / 4.4
//         17 M  2 bit 14.3 / 12.8  4 bit 15.6 / 15.4  8 bit 19.3 / 15.7    100 M  2 bit 76 / 73  4 bit 87 / 79  8 bit 101 / 78
//   half  4 M  2 bit 3.8 / 4.9  4 bit 3.5 / 4.4  8 bit 3.7 / 4.0    17 M  2 bit 7.6 / 8.1  4 bit 9.9 / 8.5  8 bit 12.4 / 10.6
//         50 M  1 bit 21.1 / 21.0  2 bit 23.1 / 22.1  4 bit 26.3 / 24.1  8 bit 33.1 / 28.9    100 M  1 bit 43.1 / 40.3
// Float at 1 bit has eight stores per piece already (two pieces: 50 M 37.2 / 38.4) and gains from the occupancy cap instead
// (40 000 bytes: 50 M 37.2 -> 35.8, 100 M 71.3 -> 66.6, 17 M 13.8 -> 13.2); the others lose by it (float 4 bit 17 %, half 20-30 %).
template <typename T>
constexpr int64_t groups_two_pieces_from(int bits) {   // elements
  return sizeof(T) == 4 ? (bits == 1 ? INT64_MAX : bits == 2 ? 1LL << 22 : bits == 4 ? 1LL << 23 : 1LL << 21)
                        : (bits == 1 ? 1LL << 26 : bits == 2 ? 1LL << 25 : bits == 4 ? 1LL << 23 : 1LL << 23);
}
#define GROUPS_DQ_CAP_FROM (1LL << 24)
template <typename T, int D, int BITS>
LaunchPlan plan_dequantize_groups_bits(int64_t N) {
  LaunchPlan p;
  const bool two = N * D >= groups_two_pieces_from<T>(BITS);
  const int64_t per_wave = (two ? 2 : 1) * 64 * Elem<T>::kDqWidth;   // code bytes
  const int64_t waves = (supergroups(N, BITS) * D + per_wave - 1) / per_wave;
  p.kernel = two ? (const void*)dequantize_groups_kernel<T, D, BITS, 2> : (const void*)dequantize_groups_kernel<T, D, BITS, 1>;
  p.grid = dim3((unsigned)((waves + 3) / 4));
  p.block = dim3(256);
  p.lds = sizeof(T) == 4 && BITS == 1 && N * D >= GROUPS_DQ_CAP_FROM ? 40000u : 0u;
  return p;
}
template <typename T, int D>
LaunchPlan plan_dequantize_groups(int bits, int64_t N) {
  switch (bits) {
    case 1: return plan_dequantize_groups_bits<T, D, 1>(N);
    case 2: return plan_dequantize_groups_bits<T, D, 2>(N);
    case 4: return plan_dequantize_groups_bits<T, D, 4>(N);
    case 8: return plan_dequantize_groups_bits<T, D, 8>(N);
  }
  return LaunchPlan();
}
template <typename T>
int dispatch_dequantize_groups(int64_t group, int bits, const uint8_t* packed, const T* scale, const T* mn, int64_t numel,
                               int64_t N, T* out, hipStream_t stream) {
  const LaunchPlan p = group == 64    ? plan_dequantize_groups<T, 64>(bits, N)
                       : group == 128 ? plan_dequantize_groups<T, 128>(bits, N)
                                      : plan_dequantize_groups<T, 512>(bits, N);
  if (!p.kernel) return GACT_EINVAL;
  void* args[] = {(void*)&packed, (void*)&scale, (void*)&mn, (void*)&numel, (void*)&N, (void*)&out};
  return hipLaunchKernel(p.kernel, p.grid, p.block, args, p.lds, stream) == hipSuccess ? GACT_OK : GACT_ELAUNCH;
}

// ---- tensors that are not contiguous ----
inline Divisor divisor(uint32_t d) {   // for numerators below 2^31
  Divisor r{d, 0u, 0u};
  if (d > 1) {
    uint32_t l = 0;
    while ((1ull << l) < d) l++;
    r.m = (uint32_t)((1ull << (31 + l)) / d + 1);
    r.s = l - 1;
  }
  return r;
}
// sizes and strides with dimensions of one element dropped and dimensions that lie one inside the other joined
inline int joined_dims(int ndim, const int64_t* sizes, const int64_t* strides, int64_t (&size)[8], int64_t (&stride)[8]) {
  int n = 0;
  for (int d = 0; d < ndim; d++) {
    if (sizes[d] == 1) continue;
    if (n > 0 && stride[n - 1] == sizes[d] * strides[d]) {
      size[n - 1] *= sizes[d];
      stride[n - 1] = strides[d];
    } else {
      if (n == 8) return -1;
      size[n] = sizes[d];
      stride[n] = strides[d];
      n++;
    }
  }
  return n;
}
// Strips or tiles.  A tile's workgroup reads a piece of its own of every memory row: the longer the channels (K pixels), the
// narrower that piece; a strip's always reads 64 bytes, but it walks its pixels one step after the other - of a channel at least
// four super-groups, at 1 and 2 bit one and a half - and reads up to a super-group of pixels beyond its own.  us, tiles / strips:
//   half [64,256,56,56] 8 bit 57 / 41  4 bit 55 / 37  2 bit 52 / 40  1 bit 54 / 48    float 4 bit 80 / 63  1 bit 155 / 78
//   half [64,64,112,112] 8 bit 101 / 37  4 bit 99 / 35  1 bit 94 / 52    half [64,512,28,28] 8 bit 26 / 26  4 bit 23 / 31
//   half [33,128,52,52] 8 bit 18 / 13  4 bit 18 / 14  2 bit 17 / 19    [40,96,64,64] 2 bit 16 / 19    [2,256,56,56] 2 bit 10 / 14
//   half [8,64,112,112] 2 bit 31 / 14  1 bit 32 / 26    [1,64,112,112] 2 bit 9 / 13
//   float [16,256,56,56] 2 bit 28 / 21  1 bit 30 / 28    [2,256,56,56] 2 bit 14 / 10  1 bit 15 / 16    [8,64,112,112] 1 bit 39 / 20
inline bool takes_strips(size_t elem_size, int bits, int64_t numel, int64_t K) {
  if (K % 4 != 0) return false;
  const int64_t sge = 8 / bits * GROUP;
  if (bits >= 4) return K >= 4 * sge;
  if (K < 3 * sge / 2) return false;
  if (elem_size == 4) return bits == 2 || numel >= (1 << 22);
  return numel >= (K >= 8192 ? 1 << 22 : 1 << 24);
}
// How strips are worked through: GS groups of a channel per step, and the segments they are cut into.  Two groups share a Philox
// block and a division sequence and have half the barriers, in 66 KB of LDS, two workgroups to a CU: half [64,256,56,56] 4 bit
// 42 -> 37 us, 2 bit 45 -> 40, float 4 bit 69 -> 63, half [16,256,56,56] 4 bit 16.4 -> 14.2.  At 8 bit, whose super-group is one
// group, there is nothing in it and smaller tensors lose half their segments (half [2,256,56,56] 5.8 -> 7.5), so it keeps one
// group.  So do strips that two to a CU would leave a quarter of the CUs' places empty (float [33,128,52,52] 4 bit,
// 264 strips: 19.1 against 19.8).
#define STRIP_WORKGROUPS 512
struct StripCut { int gs; int64_t segment, segments; };   // segment: units
inline StripCut strip_cut(int bits, int64_t strips, int64_t K) {
  StripCut c;
  c.gs = bits == 8 ? 1 : 2;
  for (;;) {
    const int64_t unit = 8 / bits > c.gs ? 8 / bits * GROUP : c.gs * GROUP, per_channel = (K + unit - 1) / unit;
    // one group: at least so many workgroups (more would read more beyond their own); two: what the CUs hold at once
    int64_t segments = c.gs == 1 ? (STRIP_WORKGROUPS + strips - 1) / strips : STRIP_WORKGROUPS / strips;
    segments = segments < 1 ? 1 : segments;
    if (c.gs == 2 && segments <= per_channel && strips * segments < STRIP_WORKGROUPS * 3 / 4) {
      c.gs = 1;
      continue;
    }
    segments = segments < per_channel ? segments : per_channel;
    c.segment = (per_channel + segments - 1) / segments;
    c.segments = (per_channel + c.segment - 1) / c.segment;
    return c;
  }
}
// Elements of a workgroup's tile: as many tiles as the workgroups that the GPU holds, or a multiple of that, in whole super-groups.  Up to
// 48 KB, three workgroups to a CU that load and quantize by turns, where that leaves a tile 21 channels in the end, and either 28 KB or
// the CU that gets most no more than the other way; up to 64 KB, two workgroups, where those would leave 16 channels before the rounds are
// cut (half [64,512,28,28] 4 bit 23 us against 28 with one of 144 KB), else one of up to 144 KB (half [64,256,56,56] 1 bit 54 against 64;
// [2,256,56,56] 9 against 13).  64 / 48 KB, us, with what the latter leaves: half 4 bit [512,512,7,7] 15.0 / 13.6 (36 KB, 376 channels),
// [256,512,14,14] 22.4 / 19.0 (36 KB, 94), [64,512,20,20] 13.2 / 12.2 (36 KB, 46), [64,512,28,28] 21.5 / 20.4 (36 KB, 23); float 4 bit
// [2000,256,7,7] 37.1 / 32.0 (48 KB, 251), [128,512,14,14] 18.8 / 17.1 (40 KB, 52), [64,512,20,20] 20.1 / 17.0 (40 KB, 26).  Fewer
// channels: half [64,256,32,32] 4 bit 14.5 / 16.6 (44 KB, 22), [87,256,876] 2 bit 17.6 / 19.6, 4 bit 18.0 / 19.1 (28 KB, 16).  Smaller
// tiles: half 4 bit [311,256,49] 6.9 / 7.7 (12 KB, 635 tiles: 36 KB for some CUs, where 477 of 16 KB are 32), [2164,256,9] 8.1 / 9.1 (16 KB,
// 609: 48, 487 of 20 KB: 40), but [273,128,179] 9.5 / 8.1 (16 KB, 764: 48, 509 of 24 KB: 48).  Over 3900 layouts of 9 to 1225 pixels
// and 1.3 to 64 M elements at the four widths this rule is 1.0 % behind the better way on average, one of 28 channels before the rounds are
// cut 2.2, the 64 KB everywhere 4.7; the worst is float [974,256,49] 4 bit 19.5 / 23.2 (32 KB).
// Float at 2 bit has registers for two workgroups only (106): [2000,256,7,7] 38.0 / 39.2.
inline int transposed_tile(size_t elem_size, int bits, int64_t numel, int64_t K) {
  const auto cut = [&](int64_t slots, int64_t most) {
    const int64_t rounds = (numel + slots * most - 1) / (slots * most);
    return ((numel + slots * rounds - 1) / (slots * rounds) + 2047) / 2048 * 2048;
  };
  const auto busiest = [&](int64_t tile) { return ((numel + tile - 1) / tile + 255) / 256 * tile; };   // CU, elements
  const int64_t size = (int64_t)elem_size, most = 65536 / size, three = cut(768, 49152 / size);
  const int64_t two = (most < numel / 512 ? most : numel / 512) < 16 * K ? cut(256, 147456 / size) : cut(512, most);
  const bool by_threes = !(elem_size == 4 && bits == 2) && three >= 21 * K && (three * size >= 28672 || busiest(three) <= busiest(two));
  return (int)(by_threes ? three : two);
}
// Where the tile kernel gains over the contiguous copy before quantize_kernel; elsewhere the caller makes that copy.  us, in place
// / copy and quantize:
//   Few pixels: a step of the walk is wider than a channel, most lanes idle, and at 1 bit float few super-groups are in flight:
//     33 M elements of 2 pixels, half 4 bit 72 / 60  1 bit 109 / 60  float 4 bit 115 / 75  1 bit 206 / 75
//     of 3, half 1 bit 77 / 62  float 4 bit 84 / 76  1 bit 152 / 77;  of 8, float 1 bit 1.16-1.19 times;  of 12, 0.95
//   Long channels: a tile of c channels reads (c + W - 1) / c times its bytes (W elements of a piece), the copy always once.  4 bit:
//     half [1,64,50257] 35 / 39  [5,64,12321] 34 / 25  [42,64,12321] 75 / 148  [3,64,20001] 50 / 27  [26,64,20001] 101 / 168
//     [3,64,169343] 553 / 453  [42,8,12321] 29 / 15  [24,8,169343] 245 / 65    float [1,256,50257] 220 / 165  [26,64,20001] 167 / 233
//     [340,8,12321] 94 / 110  [10,64,50257] 504 / 403
//   Below about a million elements both are bound by their launches, of which this is one less.
// Of 4851 layouts of 2 to 1000004 pixels, 8 to 1024 channels and 2^15 to 2^26 elements, at the four widths each, 2220 were slower in
// place by 3 % and more without these lines and the one on channels of one piece in dispatch_quantize_strided; with them fewer than
// 200 are, 45 of these by more than a tenth.
inline bool tiles_pay(size_t elem_size, int bits, int64_t numel, int64_t M, int64_t K, int64_t tile) {
  const bool word = elem_size == 4;
  int fewest = 0;   // pixels
  if (numel >= 1 << 24) fewest = bits == 1 ? (word ? 10 : 5) : (word ? 4 : 3);
  else if (numel >= (bits == 1 ? 1 << 21 : 1 << 23)) fewest = bits == 1 ? (word ? 6 : 3) : (word ? 3 : 0);
  if (K < fewest) return false;
  if (numel < (K % 4 != 0 ? (bits == 1 ? 3 << 17 : 1 << 20) : (bits == 1 ? 1 << 20 : 1 << 21))) return true;
  // the longest channel, in sixteenths of a tile; the copy of narrow memory rows is the faster one (one piece: M is W)
  int longest = word ? (numel < 1 << 24 ? 11 : 14) : M < 64 ? 6 : numel < 3 << 22 ? 11 : 16;
  if (!word && M == 8) longest = K % 4 == 0 ? 6 : 3;
  if (numel < 3 << 20) {
    if (K % 4 == 0) longest = 17;
    else if (M == 8) longest = 11;
  }
  return 16 * K <= longest * tile;
}
template <typename T, int BITS>
const void* quantize_gather_of(int noise_mode) {
  return noise_mode == GACT_NOISE_CONST ? (const void*)quantize_gather_kernel<T, BITS, GACT_NOISE_CONST>
                                        : (const void*)quantize_gather_kernel<T, BITS, GACT_NOISE_FAST>;
}
template <typename T, int BITS, int ROWS>
const void* quantize_transposed_rows_of(int noise_mode) {
  return noise_mode == GACT_NOISE_CONST ? (const void*)quantize_transposed_kernel<T, BITS, GACT_NOISE_CONST, ROWS>
                                        : (const void*)quantize_transposed_kernel<T, BITS, GACT_NOISE_FAST, ROWS>;
}
template <typename T, int BITS>
const void* quantize_transposed_of(int noise_mode, uint32_t K) {
  if constexpr (sizeof(T) == 2)
    if (K % 8 == 0) return quantize_transposed_rows_of<T, BITS, 8>(noise_mode);
  if (K % 4 == 0) return quantize_transposed_rows_of<T, BITS, 4>(noise_mode);
  return quantize_transposed_rows_of<T, BITS, 1>(noise_mode);
}
template <typename T, int BITS, int GS>
const void* quantize_strips_of(int noise_mode) {
  return noise_mode == GACT_NOISE_CONST ? (const void*)quantize_strips_kernel<T, BITS, GACT_NOISE_CONST, GS>
                                        : (const void*)quantize_strips_kernel<T, BITS, GACT_NOISE_FAST, GS>;
}
template <typename T>
int dispatch_quantize_strided(int n, const int64_t (&size)[8], const int64_t (&stride)[8], const T* x, int64_t numel, int bits,
                              int noise_mode, SeedArg seed, uint8_t* packed, typename Elem<T>::Stat* scale, T* mn, T* mx,
                              hipStream_t stream) {
  constexpr int W = Elem<T>::kQWidth;
  const int64_t N = (numel + GROUP - 1) / GROUP;
  LaunchPlan p;
  GatherShape gs;
  TransposedShape ts;
  StripShape ss;
  void* shape = nullptr;
  bool pieces = true;   // every stride but the 1 in whole pieces
  for (int d = 0; d < n; d++) pieces = pieces && (stride[d] == 1 || stride[d] % W == 0);
  if (!pieces || !aligned16(x) || n < 2) return GACT_ESHAPE;
  if (stride[n - 1] == 1 && n <= 4 && size[n - 1] % W == 0 && numel / W < 0x7fffffffLL) {
    int64_t sz[3] = {1, 1, 1}, st[3] = {0, 0, 0};   // the outer dimensions, right-aligned
    for (int d = 0; d < n - 1; d++) {
      if (stride[d] == 1) return GACT_ESHAPE;
      sz[3 - (n - 1) + d] = size[d];
      st[3 - (n - 1) + d] = stride[d] / W;
    }
    gs.run = divisor((uint32_t)(size[n - 1] / W));
    gs.n2 = divisor((uint32_t)sz[2]);
    gs.n1 = divisor((uint32_t)sz[1]);
    gs.s0 = st[0];
    gs.s1 = st[1];
    gs.s2 = st[2];
    shape = &gs;
    row_grid(supergroups(N, bits) * (bits <= 2 ? 4 : 1), &p.grid, &p.block, bits <= 2 ? GACT_W8_THREADS : 64);
    switch (bits) {
      case 1: p.kernel = quantize_gather_of<T, 1>(noise_mode); break;
      case 2: p.kernel = quantize_gather_of<T, 2>(noise_mode); break;
      case 4: p.kernel = quantize_gather_of<T, 4>(noise_mode); break;
      case 8: p.kernel = quantize_gather_of<T, 8>(noise_mode); break;
    }
  } else if (stride[n - 2] == 1 && stride[n - 1] != 1 && n <= 3 && (n == 2 || stride[0] != 1) && size[n - 2] % W == 0 &&
             size[n - 1] < (1 << 24) && numel / size[n - 1] < 0x7fffffffLL) {
    const int tile = transposed_tile(sizeof(T), bits, numel, size[n - 1]);
    const bool tiles = tiles_pay(sizeof(T), bits, numel, size[n - 2], size[n - 1], tile);
    // channels of one piece leave three quarters of a strip's lanes without work: half [1091,8,3844] 4 bit strips 77, copy 68 us,
    // [1551,8,2704] 2 bit 90, 63, where tiles (as odd numbers of pixels take) need half of the copy's time
    const bool one_piece = size[n - 2] == W && bits < 8;
    if (takes_strips(sizeof(T), bits, numel, size[n - 1]) && !(one_piece && tiles)) {
      if (one_piece && bits == 1 && size[n - 1] < 32768) return GACT_ESHAPE;   // half [83,8,12544] 36, copy 24; [83,8,50176] 68, 102
      ss.M = (uint32_t)size[n - 2];
      ss.K = (uint32_t)size[n - 1];
      ss.sk = stride[n - 1];
      ss.sb = n == 3 ? stride[0] : 0;
      ss.batch = n == 3 ? (uint32_t)size[0] : 1;
      ss.strips = (ss.M + STRIP_PIECES * W - 1) / (STRIP_PIECES * W);
      const int64_t strips = (int64_t)ss.strips * ss.batch;
      const StripCut cut = strip_cut(bits, strips, ss.K);
      ss.segment = (uint32_t)cut.segment;
      ss.segments = (uint32_t)cut.segments;
      shape = &ss;
      p.grid = dim3((unsigned)(strips * ss.segments));
      p.block = dim3(STRIP_THREADS);
      switch (bits) {
        case 1: p.kernel = cut.gs == 1 ? quantize_strips_of<T, 1, 1>(noise_mode) : quantize_strips_of<T, 1, 2>(noise_mode); break;
        case 2: p.kernel = cut.gs == 1 ? quantize_strips_of<T, 2, 1>(noise_mode) : quantize_strips_of<T, 2, 2>(noise_mode); break;
        case 4: p.kernel = cut.gs == 1 ? quantize_strips_of<T, 4, 1>(noise_mode) : quantize_strips_of<T, 4, 2>(noise_mode); break;
        case 8: p.kernel = quantize_strips_of<T, 8, 1>(noise_mode); break;
      }
      void* args[] = {(void*)&seed, (void*)&x, (void*)&numel, (void*)&N, (void*)&packed, (void*)&scale, (void*)&mn, (void*)&mx, shape};
      return hipLaunchKernel(p.kernel, p.grid, p.block, args, p.lds, stream) == hipSuccess ? GACT_OK : GACT_ELAUNCH;
    }
    if (!tiles) return GACT_ESHAPE;
    ts.M = (uint32_t)size[n - 2];
    ts.K = (uint32_t)size[n - 1];
    ts.sk = stride[n - 1];
    ts.sb = n == 3 ? stride[0] : 0;
    ts.channels = numel / size[n - 1];
    ts.tile = tile;
    // a tile's rows and batch entries have to lie within 4 GB of its first entry
    const int64_t entries = ts.tile / ((int64_t)ts.M * ts.K) + 2;
    if ((entries * ts.sb + (int64_t)ts.K * ts.sk + ts.M) * (int64_t)sizeof(T) > 0xffffffffLL) return GACT_ESHAPE;
    shape = &ts;
    p.lds = tile_bytes<T>(ts.tile);
    p.grid = dim3((unsigned)((numel + ts.tile - 1) / ts.tile));
    p.block = dim3(TRANSPOSED_THREADS);
    switch (bits) {
      case 1: p.kernel = quantize_transposed_of<T, 1>(noise_mode, ts.K); break;
      case 2: p.kernel = quantize_transposed_of<T, 2>(noise_mode, ts.K); break;
      case 4: p.kernel = quantize_transposed_of<T, 4>(noise_mode, ts.K); break;
      case 8: p.kernel = quantize_transposed_of<T, 8>(noise_mode, ts.K); break;
    }
    if (p.lds > 65536 &&
        hipFuncSetAttribute(p.kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds) != hipSuccess)
      return GACT_ELAUNCH;
  } else {
    return GACT_ESHAPE;
  }
  void* args[] = {(void*)&seed, (void*)&x, (void*)&numel, (void*)&N, (void*)&packed, (void*)&scale, (void*)&mn, (void*)&mx, shape};
  return hipLaunchKernel(p.kernel, p.grid, p.block, args, p.lds, stream) == hipSuccess ? GACT_OK : GACT_ELAUNCH;
}

template <typename T>
void launch_minimax_any(const T* x, int64_t N, int64_t D, T* mn, T* mx, hipStream_t stream) {
  const bool vec = aligned16(x);  // D % 32 == 0 keeps every row 16-byte aligned once the base is
  const int64_t pieces = vec ? D / (16 / (int64_t)sizeof(T)) : D;
  int lpr_log2 = 3;
  while (lpr_log2 < 6 && (2LL << lpr_log2) <= pieces) lpr_log2++;
  const bool several = pieces <= (64LL << 1);  // short rows: 4 rows per lane group
  const int64_t groups = several ? (N + 3) / 4 : N;
  const dim3 grid((unsigned)(((groups << lpr_log2) + 255) / 256)), block(256);
  if (vec && several)
    hipLaunchKernelGGL((minimax_any_kernel<T, true, 4>), grid, block, 0, stream, x, N, D, lpr_log2, mn, mx);
  else if (vec)
    hipLaunchKernelGGL((minimax_any_kernel<T, true, 1>), grid, block, 0, stream, x, N, D, lpr_log2, mn, mx);
  else if (several)
    hipLaunchKernelGGL((minimax_any_kernel<T, false, 4>), grid, block, 0, stream, x, N, D, lpr_log2, mn, mx);
  else
    hipLaunchKernelGGL((minimax_any_kernel<T, false, 1>), grid, block, 0, stream, x, N, D, lpr_log2, mn, mx);
}

// the 8-columns-per-thread kernels take G = 1, D % 8 == 0, 16-byte aligned rows, and a thread count that fits 32 bits
inline bool rows8_ok(int bits, int64_t N, int64_t G, int64_t D, uint32_t* tpr, uint32_t* total) {
  if (G != 1 || D % 8 != 0 || D / 8 > 0x7fffffffLL) return false;
  const int64_t rows = supergroups(N, bits), threads = rows * (D / 8);
  if (threads <= 0 || threads > 0xffffff00LL) return false;
  *tpr = (uint32_t)(D / 8);
  *total = (uint32_t)threads;
  return true;
}

template <typename T>
int pack_any(const T* data, const T* mn, const T* scale, int bits, int64_t N, int64_t G, int64_t D, int noise_mode,
             uint64_t seed, const float* noise, uint8_t* packed, hipStream_t stream) {
  uint32_t tpr = 0, threads = 0;
  const bool rows8 = rows8_ok(bits, N, G, D, &tpr, &threads) && aligned16(data) && aligned16(packed) &&
                     (D * (int64_t)sizeof(T)) % 16 == 0 && (noise_mode != GACT_NOISE_INJECT || aligned16(noise));
  const int64_t total = gact_packed_bytes(bits, N, G, D);
  const dim3 grid((unsigned)(rows8 ? (threads + 255u) / 256u : (total + 255) / 256)), block(256);
#define GACT_LAUNCH_PACK(M)                                                                                          \
  do {                                                                                                               \
    if (rows8)                                                                                                       \
      hipLaunchKernelGGL((pack_rows8_kernel<T, M>), grid, block, 0, stream, data, mn, scale, bits, N, tpr, threads,   \
                         seed, noise, packed);                                                                       \
    else                                                                                                             \
      hipLaunchKernelGGL((pack_any_kernel<T, M>), grid, block, 0, stream, data, mn, scale, bits, N, G, D, seed,       \
                         noise, packed, total);                                                                      \
  } while (0)
  switch (noise_mode) {
    case GACT_NOISE_CONST: GACT_LAUNCH_PACK(GACT_NOISE_CONST); break;
    case GACT_NOISE_INJECT: GACT_LAUNCH_PACK(GACT_NOISE_INJECT); break;
    case GACT_NOISE_REF: GACT_LAUNCH_PACK(GACT_NOISE_REF); break;
    case GACT_NOISE_FAST: GACT_LAUNCH_PACK(GACT_NOISE_FAST); break;
    default: return GACT_EINVAL;
  }
#undef GACT_LAUNCH_PACK
  return launch_status();
}

template <typename T>
int unpack_any(const uint8_t* packed, int bits, const T* scale, const T* mn, int64_t N, int64_t G, int64_t D, T* out,
               hipStream_t stream) {
  uint32_t tpr = 0, threads = 0;
  if (rows8_ok(bits, N, G, D, &tpr, &threads) && aligned16(out) && (reinterpret_cast<uintptr_t>(packed) & 7u) == 0 &&
      (D * (int64_t)sizeof(T)) % 16 == 0) {
    hipLaunchKernelGGL((unpack_rows8_kernel<T>), dim3((threads + 255u) / 256u), dim3(256), 0, stream, packed, bits, scale,
                       mn, N, tpr, threads, out);
  } else {
    const int64_t total = gact_packed_bytes(bits, N, G, D);
    hipLaunchKernelGGL((unpack_any_kernel<T>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, packed, bits,
                       scale, mn, N, G, D, out, total);
  }
  return launch_status();
}

}  // namespace

extern "C" {

const char* gact_strerror(int code) {
  switch (code) {
    case GACT_OK: return "ok";
    case GACT_EINVAL: return "invalid argument";
    case GACT_EALIGN: return "pointer is not 16-byte aligned";
    case GACT_ESHAPE: return "unsupported shape";
    case GACT_ELAUNCH: return "HIP launch failed";
    case GACT_EBUDGET: return "bit budget unreachable: every tensor is already at 1 bit";
    case GACT_ELIMIT: return "beyond the limit of the library's own workspace (262144 blocks of 128 groups)";
  }
  return "unknown error";
}

int gact_abi_version(void) { return GACT_ABI_VERSION; }

int64_t gact_packed_bytes(int bits, int64_t N, int64_t G, int64_t D) {
  if (!valid_bits(bits) || N < 0 || G < 0 || D < 0) return GACT_EINVAL;
  const int wpt = 8 / bits;
  const int64_t n_round = (N + wpt - 1) / wpt * wpt;
  return (int64_t)bits * n_round * G * D / 8;
}

int gact_minimax(const void* data, int dtype, int64_t N, int64_t D, void* mn, void* mx, void* stream) {
  if (dtype != GACT_F32 && dtype != GACT_F16) return GACT_EINVAL;
  if (N < 0 || !(D % 32 == 0 && D > 32)) return GACT_ESHAPE;  // minimax_cuda_kernel.cu:80
  if (N == 0) return GACT_OK;
  if (!data || !mn || !mx) return GACT_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  fresh_launch();
  if (D == GROUP && aligned16(data)) {
    dim3 grid, block;
    row_grid((N + MINIMAX_ROW_GROUPS - 1) / MINIMAX_ROW_GROUPS, &grid, &block, MINIMAX_THREADS);
    if (dtype == GACT_F32)
      hipLaunchKernelGGL((minimax256_kernel<float>), grid, block, 0, s, (const float*)data, N, (float*)mn, (float*)mx);
    else
      hipLaunchKernelGGL((minimax256_kernel<f16>), grid, block, 0, s, (const f16*)data, N, (f16*)mn, (f16*)mx);
  } else {
    if (dtype == GACT_F32)
      launch_minimax_any<float>((const float*)data, N, D, (float*)mn, (float*)mx, s);
    else
      launch_minimax_any<f16>((const f16*)data, N, D, (f16*)mn, (f16*)mx, s);
  }
  return launch_status();
}

int gact_pack(const void* data, const void* mn, const void* mx, int dtype, int bits, int64_t N, int64_t G, int64_t D,
              int noise_mode, uint64_t seed, const float* noise, void* packed, void* scale, void* stream) {
  if (dtype != GACT_F32 && dtype != GACT_F16) return GACT_EINVAL;
  if (!valid_bits(bits)) return GACT_EINVAL;  // quantization_cuda_kernel.cu:86
  if (N < 0 || G < 0 || D < 0) return GACT_EINVAL;
  if (noise_mode < GACT_NOISE_CONST || noise_mode > GACT_NOISE_FAST) return GACT_EINVAL;
  if (N * G * D == 0) return GACT_OK;
  if (!data || !mn || !mx || !packed || !scale) return GACT_EINVAL;
  if (noise_mode == GACT_NOISE_INJECT && !noise) return GACT_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  fresh_launch();
  if (G == 1 && D == GROUP && aligned16(data) && aligned16(packed) && (noise_mode != GACT_NOISE_INJECT || aligned16(noise))) {
    // the fused row kernel with min/max taken from the caller
    if (dtype == GACT_F32)
      return dispatch_quantize<float, true>(bits, (const float*)data, N * GROUP, N, (uint8_t*)packed, (float*)scale,
                                            (float*)const_cast<void*>(mn), (float*)const_cast<void*>(mx), noise_mode, SeedArg{seed, nullptr}, noise, s);
    return dispatch_quantize<f16, true>(bits, (const f16*)data, N * GROUP, N, (uint8_t*)packed, (f16*)scale,
                                        (f16*)const_cast<void*>(mn), (f16*)const_cast<void*>(mx), noise_mode, SeedArg{seed, nullptr}, noise, s);
  }
  const int64_t count = N * G;
  const dim3 sgrid((unsigned)((count + 255) / 256)), sblock(256);
  if (dtype == GACT_F32) {
    hipLaunchKernelGGL((scale_kernel<float>), sgrid, sblock, 0, s, (const float*)mn, (const float*)mx, bits, count, (float*)scale);
    return pack_any<float>((const float*)data, (const float*)mn, (const float*)scale, bits, N, G, D, noise_mode, seed, noise, (uint8_t*)packed, s);
  }
  hipLaunchKernelGGL((scale_kernel<f16>), sgrid, sblock, 0, s, (const f16*)mn, (const f16*)mx, bits, count, (f16*)scale);
  return pack_any<f16>((const f16*)data, (const f16*)mn, (const f16*)scale, bits, N, G, D, noise_mode, seed, noise, (uint8_t*)packed, s);
}

int gact_unpack(const void* packed, int bits, const void* scale, const void* mn, int dtype, int64_t N, int64_t G,
                int64_t D, void* out, void* stream) {
  if (dtype != GACT_F32 && dtype != GACT_F16) return GACT_EINVAL;
  if (!valid_bits(bits)) return GACT_EINVAL;  // quantization_cuda_kernel.cu:191
  if (N < 0 || G < 0 || D < 0) return GACT_EINVAL;
  if (N * G * D == 0) return GACT_OK;
  if (!packed || !scale || !mn || !out) return GACT_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  fresh_launch();
  if (G == 1 && D == GROUP && aligned16(out) && aligned16(packed)) {
    if (dtype == GACT_F32)
      return dispatch_dequantize<float>(bits, (const uint8_t*)packed, (const float*)scale, (const float*)mn, N * GROUP, N, (float*)out, s);
    return dispatch_dequantize<f16>(bits, (const uint8_t*)packed, (const f16*)scale, (const f16*)mn, N * GROUP, N, (f16*)out, s);
  }
  if (G == 1 && one_pass_group(D) && aligned16(out) && aligned16(packed)) {
    if (dtype == GACT_F32)
      return dispatch_dequantize_groups<float>(D, bits, (const uint8_t*)packed, (const float*)scale, (const float*)mn, N * D, N, (float*)out, s);
    return dispatch_dequantize_groups<f16>(D, bits, (const uint8_t*)packed, (const f16*)scale, (const f16*)mn, N * D, N, (f16*)out, s);
  }
  if (dtype == GACT_F32)
    return unpack_any<float>((const uint8_t*)packed, bits, (const float*)scale, (const float*)mn, N, G, D, (float*)out, s);
  return unpack_any<f16>((const uint8_t*)packed, bits, (const f16*)scale, (const f16*)mn, N, G, D, (f16*)out, s);
}

int gact_quantize_seeded(const void* x, int dtype, int64_t numel, int bits, int noise_mode, uint64_t seed,
                         const uint64_t* seed_add, const float* noise, void* packed, void* scale, void* mn, void* mx,
                         void* stream) {
  if (dtype != GACT_F32 && dtype != GACT_F16 && dtype != GACT_BF16) return GACT_EINVAL;
  if (!valid_bits(bits) || numel < 0) return GACT_EINVAL;
  if (noise_mode < GACT_NOISE_CONST || noise_mode > GACT_NOISE_FAST) return GACT_EINVAL;
  if (numel == 0) return GACT_OK;
  if (!x || !packed || !scale || !mn) return GACT_EINVAL;
  if (noise_mode == GACT_NOISE_INJECT && !noise) return GACT_EINVAL;
  if (!aligned16(x) || !aligned16(packed) || (noise_mode == GACT_NOISE_INJECT && !aligned16(noise))) return GACT_EALIGN;
  if (reinterpret_cast<uintptr_t>(seed_add) & 7u) return GACT_EALIGN;
  const int64_t N = (numel + GROUP - 1) / GROUP;
  hipStream_t s = (hipStream_t)stream;
  fresh_launch();
  const SeedArg sa{seed, seed_add};
  if (dtype == GACT_F32)
    return dispatch_quantize<float, false>(bits, (const float*)x, numel, N, (uint8_t*)packed, (float*)scale, (float*)mn, (float*)mx, noise_mode, sa, noise, s);
  if (dtype == GACT_BF16)
    return dispatch_quantize<bf16, false>(bits, (const bf16*)x, numel, N, (uint8_t*)packed, (float*)scale, (bf16*)mn, (bf16*)mx, noise_mode, sa, noise, s);
  return dispatch_quantize<f16, false>(bits, (const f16*)x, numel, N, (uint8_t*)packed, (f16*)scale, (f16*)mn, (f16*)mx, noise_mode, sa, noise, s);
}

int gact_quantize(const void* x, int dtype, int64_t numel, int bits, int noise_mode, uint64_t seed, const float* noise,
                  void* packed, void* scale, void* mn, void* mx, void* stream) {
  return gact_quantize_seeded(x, dtype, numel, bits, noise_mode, seed, nullptr, noise, packed, scale, mn, mx, stream);
}

int gact_dequantize(const void* packed, int bits, const void* scale, const void* mn, int dtype, int64_t numel, void* out,
                    void* stream) {
  if (dtype != GACT_F32 && dtype != GACT_F16 && dtype != GACT_BF16) return GACT_EINVAL;
  if (!valid_bits(bits) || numel < 0) return GACT_EINVAL;
  if (numel == 0) return GACT_OK;
  if (!packed || !scale || !mn || !out) return GACT_EINVAL;
  if (!aligned16(out) || !aligned16(packed)) return GACT_EALIGN;
  const int64_t N = (numel + GROUP - 1) / GROUP;
  hipStream_t s = (hipStream_t)stream;
  fresh_launch();
  if (dtype == GACT_F32)
    return dispatch_dequantize<float>(bits, (const uint8_t*)packed, (const float*)scale, (const float*)mn, numel, N, (float*)out, s);
  if (dtype == GACT_BF16)
    return dispatch_dequantize<bf16>(bits, (const uint8_t*)packed, (const float*)scale, (const bf16*)mn, numel, N, (bf16*)out, s);
  return dispatch_dequantize<f16>(bits, (const uint8_t*)packed, (const f16*)scale, (const f16*)mn, numel, N, (f16*)out, s);
}

int gact_quantize_groups(const void* x, int dtype, int64_t numel, int group, int bits, int noise_mode, uint64_t seed,
                         const uint64_t* seed_add, const float* noise, void* packed, void* scale, void* mn, void* mx,
                         void* stream) {
  if (group == GROUP)
    return gact_quantize_seeded(x, dtype, numel, bits, noise_mode, seed, seed_add, noise, packed, scale, mn, mx, stream);
  if (dtype != GACT_F32 && dtype != GACT_F16) return GACT_EINVAL;
  if (!valid_bits(bits) || numel < 0) return GACT_EINVAL;
  if (noise_mode < GACT_NOISE_CONST || noise_mode > GACT_NOISE_FAST) return GACT_EINVAL;
  if (!one_pass_group(group) || noise_mode == GACT_NOISE_REF) return GACT_ESHAPE;
  if (numel == 0) return GACT_OK;
  if (!x || !packed || !scale || !mn) return GACT_EINVAL;
  if (noise_mode == GACT_NOISE_INJECT && !noise) return GACT_EINVAL;
  if (!aligned16(x) || !aligned16(packed) || (noise_mode == GACT_NOISE_INJECT && !aligned16(noise))) return GACT_EALIGN;
  if (reinterpret_cast<uintptr_t>(seed_add) & 7u) return GACT_EALIGN;
  const int64_t N = (numel + group - 1) / group;
  hipStream_t s = (hipStream_t)stream;
  fresh_launch();
  const SeedArg sa{seed, seed_add};
  if (dtype == GACT_F32)
    return dispatch_quantize_groups<float>(group, bits, (const float*)x, numel, N, (uint8_t*)packed, (float*)scale, (float*)mn, (float*)mx, noise_mode, sa, noise, s);
  return dispatch_quantize_groups<f16>(group, bits, (const f16*)x, numel, N, (uint8_t*)packed, (f16*)scale, (f16*)mn, (f16*)mx, noise_mode, sa, noise, s);
}

int gact_dequantize_groups(const void* packed, int bits, const void* scale, const void* mn, int dtype, int64_t numel, int group,
                           void* out, void* stream) {
  if (group == GROUP) return gact_dequantize(packed, bits, scale, mn, dtype, numel, out, stream);
  if (dtype != GACT_F32 && dtype != GACT_F16) return GACT_EINVAL;
  if (!valid_bits(bits) || numel < 0) return GACT_EINVAL;
  if (!one_pass_group(group)) return GACT_ESHAPE;
  if (numel == 0) return GACT_OK;
  if (!packed || !scale || !mn || !out) return GACT_EINVAL;
  if (!aligned16(out) || !aligned16(packed)) return GACT_EALIGN;
  const int64_t N = (numel + group - 1) / group;
  hipStream_t s = (hipStream_t)stream;
  fresh_launch();
  if (dtype == GACT_F32)
    return dispatch_dequantize_groups<float>(group, bits, (const uint8_t*)packed, (const float*)scale, (const float*)mn, numel, N, (float*)out, s);
  return dispatch_dequantize_groups<f16>(group, bits, (const uint8_t*)packed, (const f16*)scale, (const f16*)mn, numel, N, (f16*)out, s);
}

int gact_quantize_strided(const void* x, int dtype, int ndim, const int64_t* sizes, const int64_t* strides, int bits, int noise_mode,
                          uint64_t seed, const uint64_t* seed_add, void* packed, void* scale, void* mn, void* mx, void* stream) {
  if (dtype != GACT_F32 && dtype != GACT_F16 && dtype != GACT_BF16) return GACT_EINVAL;
  if (!valid_bits(bits) || ndim < 0 || (ndim > 0 && (!sizes || !strides))) return GACT_EINVAL;
  if (noise_mode < GACT_NOISE_CONST || noise_mode > GACT_NOISE_FAST) return GACT_EINVAL;
  if (noise_mode != GACT_NOISE_CONST && noise_mode != GACT_NOISE_FAST) return GACT_ESHAPE;
  int64_t numel = 1;
  for (int d = 0; d < ndim; d++) {
    if (sizes[d] < 0 || strides[d] < 0) return GACT_EINVAL;
    numel *= sizes[d];
  }
  if (numel == 0) return GACT_OK;
  int64_t size[8], stride[8];
  const int n = joined_dims(ndim, sizes, strides, size, stride);
  if (n < 0) return GACT_ESHAPE;
  if (n == 0 || (n == 1 && stride[0] == 1))
    return gact_quantize_seeded(x, dtype, numel, bits, noise_mode, seed, seed_add, nullptr, packed, scale, mn, mx, stream);
  if (!x || !packed || !scale || !mn) return GACT_EINVAL;
  if (!aligned16(packed) || (reinterpret_cast<uintptr_t>(seed_add) & 7u)) return GACT_EALIGN;
  hipStream_t s = (hipStream_t)stream;
  fresh_launch();
  const SeedArg sa{seed, seed_add};
  if (dtype == GACT_F32)
    return dispatch_quantize_strided<float>(n, size, stride, (const float*)x, numel, bits, noise_mode, sa, (uint8_t*)packed, (float*)scale, (float*)mn, (float*)mx, s);
  if (dtype == GACT_BF16)
    return dispatch_quantize_strided<bf16>(n, size, stride, (const bf16*)x, numel, bits, noise_mode, sa, (uint8_t*)packed, (float*)scale, (bf16*)mn, (bf16*)mx, s);
  return dispatch_quantize_strided<f16>(n, size, stride, (const f16*)x, numel, bits, noise_mode, sa, (uint8_t*)packed, (f16*)scale, (f16*)mn, (f16*)mx, s);
}

int gact_launch_geometry(int kind, int dtype, int bits, int64_t N, int* threads, int* lds_bytes, int* workgroups_per_cu) {
  if (dtype != GACT_F32 && dtype != GACT_F16 && dtype != GACT_BF16) return GACT_EINVAL;
  if (!valid_bits(bits) || N <= 0 || (kind != 0 && kind != 1)) return GACT_EINVAL;
  LaunchPlan p;
  if (kind == 0)
    p = dtype == GACT_F32 ? plan_quantize_bits<float, false>(bits, N, GACT_NOISE_FAST)
        : dtype == GACT_F16 ? plan_quantize_bits<f16, false>(bits, N, GACT_NOISE_FAST)
                            : plan_quantize_bits<bf16, false>(bits, N, GACT_NOISE_FAST);
  else
    p = dtype == GACT_F32 ? plan_dequantize<float>(bits, N)
        : dtype == GACT_F16 ? plan_dequantize<f16>(bits, N) : plan_dequantize<bf16>(bits, N);
  if (!p.kernel) return GACT_EINVAL;
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, p.kernel, (int)p.block.x, (size_t)p.lds) != hipSuccess) {
    (void)hipGetLastError();
    return GACT_ELAUNCH;
  }
  if (threads) *threads = (int)p.block.x;
  if (lds_bytes) *lds_bytes = (int)p.lds;
  if (workgroups_per_cu) *workgroups_per_cu = per_cu;
  return GACT_OK;
}

int gact_mask_pack(const uint8_t* data, int64_t n, int32_t* mask, void* stream) {
  if (n < 0) return GACT_EINVAL;
  if (n == 0) return GACT_OK;
  if (!data || !mask) return GACT_EINVAL;
  if (!aligned16(data)) return GACT_EALIGN;
  fresh_launch();
  const int64_t pairs = (n / 512 + 1) / 2;  // pairs of full blocks
  const int64_t waves = (pairs + MASK_PAIRS - 1) / MASK_PAIRS + 1;  // plus the wave that takes the partial block
  hipLaunchKernelGGL(mask_pack_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, (hipStream_t)stream, data, n, mask);
  return launch_status();
}

int gact_mask_unpack(const int32_t* mask, int64_t n, uint8_t* out, void* stream) {
  if (n < 0) return GACT_EINVAL;
  if (n == 0) return GACT_OK;
  if (!mask || !out) return GACT_EINVAL;
  if (!aligned16(out)) return GACT_EALIGN;
  fresh_launch();
  const int64_t blocks = n / 512 + 1;  // the partial block included
  const int64_t waves = (blocks + MASK_STEPS * 4 - 1) / (MASK_STEPS * 4);
  hipLaunchKernelGGL(mask_unpack_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, (hipStream_t)stream, mask, n, out);
  return launch_status();
}

int gact_calc_precision(int32_t* b, const float* C, const int64_t* w, int64_t L, double target) {
  if (L < 0) return GACT_EINVAL;
  if (L == 0) return GACT_OK;
  if (!b || !C || !w) return GACT_EINVAL;
  for (int64_t i = 0; i < L; i++)
    if (!prec_valid_bits(b[i])) return GACT_EINVAL;
  std::priority_queue<std::pair<float, int64_t>> q;
  double b_sum = 0;
  for (int64_t i = 0; i < L; i++)
    if (b[i] > 1) {
      q.push(std::make_pair(prec_key(C[i], b[i], w[i]), i));
      b_sum += (double)((int64_t)b[i] * w[i]);
    }
  while (b_sum > target) {
    if (q.empty()) return GACT_EBUDGET;
    const int64_t i = q.top().second;
    q.pop();
    const int nb = prec_next_bits(b[i]);
    b_sum -= (double)(w[i] * (int64_t)(b[i] - nb));
    b[i] = nb;
    if (nb > 1) q.push(std::make_pair(prec_key(C[i], nb, w[i]), i));
  }
  return GACT_OK;
}

int gact_calc_precision_device(int32_t* b, const float* C, const int64_t* w, int64_t L, double target, int32_t* status,
                               void* stream) {
  if (L < 0) return GACT_EINVAL;
  if (L > PREC_MAX_L) return GACT_ESHAPE;
  if (L == 0) return GACT_OK;
  if (!b || !C || !w) return GACT_EINVAL;
  fresh_launch();
  // one thread per candidate up to the largest workgroup
  const int64_t candidates = 4 * L;
  const dim3 threads((unsigned)(candidates >= PREC_THREADS ? PREC_THREADS : (candidates + 63) / 64 * 64));
  hipStream_t s = (hipStream_t)stream;
  const int each = (int)((candidates + PREC_THREADS - 1) / PREC_THREADS);
  if (each <= 1) hipLaunchKernelGGL((calc_precision_kernel<1>), dim3(1), threads, 0, s, b, C, w, (int)L, target, status);
  else if (each <= 4) hipLaunchKernelGGL((calc_precision_kernel<4>), dim3(1), threads, 0, s, b, C, w, (int)L, target, status);
  else hipLaunchKernelGGL((calc_precision_kernel<16>), dim3(1), threads, 0, s, b, C, w, (int)L, target, status);
  return launch_status();
}

int64_t gact_batch_workspace_bytes(int64_t L, int64_t total_blocks) {
  if (L < 0 || L > (1 << 30) || total_blocks < 0 || total_blocks > 0x1fffffffLL) return GACT_EINVAL;
  return batch_workspace_need(L, total_blocks);
}

namespace {
// Fewer workgroups on a CU, by a request for dynamic LDS that nobody touches (see quantize_lds_cap), for two of the batched kernels.
// Quantize, half: three.  Where codes are packed as bytes (batch_packs) its registers admit four, which is one too many from 10^8 elements
// on.  120 half tensors, four / three workgroups, us: 29 M elements, 1, 2 and 4 bit mixed 15.1 / 14.9, 114 M 46.3 / 44.9, 229 M 89.0 / 84.7,
// 343 M 132 / 126;  at 4 bit 15.7 / 15.4, 50.3 / 48.9, 97.8 / 94.3, 145 / 141;  57 M at 1 bit 23.8 / 24.6, the one loss seen.  Two
// lose 5 % up to 0.23 G.  Without packed bytes three or four make no difference (1.83 G mixed 669 / 666).  Float and bfloat16 hold
// two by their registers.
#define BATCHED_CAP_LDS 53000u
// Dequantize: batches that are known to hold float tensors only, by their size; half and bfloat16 lose by any cap (mixed 673 us, four on a
// CU 856, three 1010).  Whatever the widths, which the host does not know: the cap taken is one that loses at none of them.
// us with eight (no cap) / four / three workgroups, at 1 bit, 2 bit, 4 bit, 8 bit, and 1, 2 and 4 mixed:
//   8 M elements  7.6 / 8.4 / 7.7   7.6 / 8.3 / 8.7   7.9 / 8.8 / 9.4   9.2 / 10.6 / 11.0   8.1 / 9.3 / 9.9
//   14 M  13.1 / 12.7 / 12.0   13.0 / 13.2 / 13.8   13.7 / 13.7 / 14.1   16.3 / 16.6 / 16.4   13.7 / 14.4 / 14.6
//   29 M  23.4 / 22.0 / 22.2   23.3 / 22.2 / 23.3   24.3 / 23.3 / 24.3   28.1 / 27.5 / 29.0 (in 12 tensors 26.6 / 27.1 / 27.8)   24.5 / 23.1 / 24.1
//   43 M  33.9 / 32.3 / 32.6   33.9 / 32.4 / 33.7   35.5 / 33.6 / 34.5   39.4 / 39.4 / 41.5   36.2 / 33.8 / 34.8    -> four from 2^10 blocks (34 M) on
//   114 M  89.4 / 81.9 / 79.5   88.0 / 79.6 / 81.7   92.6 / 84.6 / 84.3   96.8 / 94.7 / 102.1   92.8 / 84.1 / 84.7
//   286 M, 8 bit 238 / 229 / 246, all four widths mixed 233 / 212 / 222
//   343 M  262 / 240 / 229   265 / 239 / 241   276 / 251 / 243   296 / 276 / 296   277 / 251 / 245    -> three from 10 * 2^10 (336 M)
//   915 M  689 / 639 / 603   697 / 639 / 633   737 / 671 / 641   813 / 744 / 793   730 / 663 / 634
unsigned batch_dequantize_lds(int dtypes, int64_t total_blocks) {
  return dtypes != GACT_DTYPES_F32 || total_blocks < 1 << 10 ? 0u : total_blocks < 10 << 10 ? 40000u : BATCHED_CAP_LDS;
}
// Whose codes the batched quantize of half tensors packs as bytes (fast stream), a sum of widths.  Bytes are fewer instructions and
// registers, which pays while a batch does not fill the chip for long and costs bandwidth where HBM bounds it, at 4 bit first; whatever
// the widths turn out to be, the line lies where the form taken loses to neither of the others.  120 tensors, us, all packed / all but
// 4 bit / none:
//   14 M elements  1 bit 11.2 / 11.2 / 11.8, 2 bit 11.4 / 11.4 / 12.1, 4 bit 11.4 / 12.5 / 12.5, the three mixed 11.3 / 11.7 / 12.1
//   57 M           24.6 / 24.6 / 25.2, 25.7 / 25.7 / 26.5, 27.3 / 28.6 / 28.5, 25.9 / 26.6 / 27.0
//   114 M          42.2 / 42.1 / 42.7, 44.2 / 44.1 / 45.1, 49.1 / 48.8 / 48.8, 45.1 / 45.7 / 45.8     -> all up to 2^12 blocks (134 M)
//   229 M          77.1 / 77.7 / 78.4, 82.1 / 82.3 / 83.3, 93.8 / 92.1 / 92.1, 84.9 / 85.0 / 85.6
//   343 M          113 / 113 / 115, 122.2 / 121.6 / 122.5, 141.7 / 134.8 / 134.8, 124.8 / 124.3 / 124.1  -> all but 4 bit below 12 * 2^10 (403 M)
//   458 M          149 / 150 / 153, 162.0 / 161.3 / 160.6, 187.6 / 179.6 / 179.1, 168.4 / 166.8 / 165.1  -> none from there on
//   1.83 G         600 / 610 / 602, 657 / 657 / 640, 757 / 739 / 743, 677 / 671 / 661
int batch_packs(int64_t total_blocks) { return total_blocks < (1 << 12) ? 7 : total_blocks < 12 << 10 ? 3 : 0; }
int batch_plan_on(gact_batch_entry* table, const int32_t* bits, int64_t L, int64_t total_blocks, int64_t capacity,
                  void* workspace, int64_t* verdict, hipStream_t s) {
  const BatchWorkspace ws = batch_workspace(workspace);
  hipLaunchKernelGGL(batch_plan_kernel, dim3((unsigned)(1 + (total_blocks + PLAN_THREADS - 1) / PLAN_THREADS)), dim3(PLAN_THREADS), 0, s, table, bits, (int)L,
                     total_blocks, capacity, ws, verdict);
  return launch_status();
}

int quantize_batched_on(const gact_batch_entry* table, const int32_t* bits, int64_t total_blocks, int noise_mode,
                        int dtypes, void* workspace, void* packed_arena, void* scale_arena, void* min_arena,
                        hipStream_t s) {
  const BatchWorkspace ws = batch_workspace(workspace);
  const dim3 grid((unsigned)total_blocks), block(256);
#define GACT_LAUNCH_QB(T, M, PACKED)                                                                          \
  hipLaunchKernelGGL((quantize_batched_kernel<T, M, PACKED>), grid, block, (Elem<T>::kDtype == GACT_F16 ? BATCHED_CAP_LDS : 0u), s, table, bits, ws, \
                     (uint8_t*)packed_arena, (uint8_t*)scale_arena, (uint8_t*)min_arena)
#define GACT_LAUNCH_QB_ALL(M, LAUNCH_F16)                                                                     \
  do {                                                                                                        \
    if (dtypes & GACT_DTYPES_F32) GACT_LAUNCH_QB(float, M, 7);                                                \
    if (dtypes & GACT_DTYPES_F16) LAUNCH_F16;                                                                 \
    if (dtypes & GACT_DTYPES_BF16) GACT_LAUNCH_QB(bf16, M, 7);                                                \
  } while (0)
  switch (noise_mode) {
    case GACT_NOISE_CONST: GACT_LAUNCH_QB_ALL(GACT_NOISE_CONST, GACT_LAUNCH_QB(f16, GACT_NOISE_CONST, 7)); break;
    case GACT_NOISE_REF: GACT_LAUNCH_QB_ALL(GACT_NOISE_REF, GACT_LAUNCH_QB(f16, GACT_NOISE_REF, 7)); break;
    default:
      GACT_LAUNCH_QB_ALL(GACT_NOISE_FAST, switch (batch_packs(total_blocks)) {
        case 7: GACT_LAUNCH_QB(f16, GACT_NOISE_FAST, 7); break;
        case 3: GACT_LAUNCH_QB(f16, GACT_NOISE_FAST, 3); break;
        default: GACT_LAUNCH_QB(f16, GACT_NOISE_FAST, 0); break;
      });
      break;
  }
#undef GACT_LAUNCH_QB_ALL
#undef GACT_LAUNCH_QB
  return launch_status();
}

inline int batched_args_ok(int64_t L, int64_t total_blocks) {
  return !(L < 0 || L > (1 << 30) || total_blocks < 0 || total_blocks > 0x1fffffffLL);   // the dequantize grid is 4 * total_blocks
}
}  // namespace

int gact_batch_plan(gact_batch_entry* table, const int32_t* bits, int64_t L, int64_t total_blocks, int64_t capacity,
                    void* workspace, void* stream) {
  if (!batched_args_ok(L, total_blocks) || capacity < 0) return GACT_EINVAL;
  if (!workspace) return GACT_EINVAL;
  if (!aligned16(workspace)) return GACT_EALIGN;
  if (L > 0 && (!table || !bits)) return GACT_EINVAL;
  fresh_launch();
  return batch_plan_on(table, bits, L, total_blocks, capacity, workspace, nullptr, (hipStream_t)stream);
}

int gact_batch_plan_args(const gact_batch_entry* geometry, const void* const* x, const uint64_t* seeds, gact_batch_entry* table,
                         const int32_t* bits, int32_t* kept, int64_t L, int64_t total_blocks, int64_t capacity, void* workspace,
                         int64_t* verdict, void* stream) {
  if (!batched_args_ok(L, total_blocks) || capacity < 0) return GACT_EINVAL;
  if (L > GACT_BATCH_ARGS) return GACT_ELIMIT;
  if (!workspace || (L > 0 && (!geometry || !x || !seeds || !table || !bits))) return GACT_EINVAL;
  if (!aligned16(workspace) || (reinterpret_cast<uintptr_t>(verdict) & 7u) != 0) return GACT_EALIGN;
  BatchArgs args = {};
  for (int64_t t = 0; t < L; t++) {
    args.x[t] = x[t];
    args.seed[t] = seeds[t];
  }
  fresh_launch();
  hipLaunchKernelGGL(batch_plan_args_kernel, dim3((unsigned)(1 + (total_blocks + PLAN_THREADS - 1) / PLAN_THREADS)), dim3(PLAN_THREADS), 0,
                     (hipStream_t)stream, args, geometry, table, bits, kept, (int)L, total_blocks, capacity, batch_workspace(workspace), verdict);
  return launch_status();
}

int gact_quantize_batched(const gact_batch_entry* table, const int32_t* bits, int64_t L, int64_t total_blocks,
                          int noise_mode, int dtypes, const void* workspace, void* packed_arena, void* scale_arena,
                          void* min_arena, void* stream) {
  if (!batched_args_ok(L, total_blocks)) return GACT_EINVAL;
  if (noise_mode != GACT_NOISE_CONST && noise_mode != GACT_NOISE_REF && noise_mode != GACT_NOISE_FAST)
    return GACT_EINVAL;  // injected noise is a single-tensor test mode
  if (dtypes < 0 || dtypes > GACT_DTYPES_ALL) return GACT_EINVAL;
  if (dtypes == 0) dtypes = GACT_DTYPES_ALL;
  if (L == 0 || total_blocks == 0) return GACT_OK;
  if (!table || !bits || !workspace || !packed_arena || !scale_arena || !min_arena) return GACT_EINVAL;
  if (!aligned16(packed_arena) || !aligned16(workspace)) return GACT_EALIGN;
  fresh_launch();
  return quantize_batched_on(table, bits, total_blocks, noise_mode, dtypes, const_cast<void*>(workspace), packed_arena,
                             scale_arena, min_arena, (hipStream_t)stream);
}

int gact_dequantize_batched(const gact_batch_entry* table, const int32_t* bits, int64_t L, int64_t total_blocks,
                            const void* workspace, const void* packed_arena, const void* scale_arena,
                            const void* min_arena, void* stream) {
  return gact_dequantize_batched_types(table, bits, L, total_blocks, GACT_DTYPES_ALL, workspace, packed_arena, scale_arena, min_arena, stream);
}
int gact_dequantize_batched_types(const gact_batch_entry* table, const int32_t* bits, int64_t L, int64_t total_blocks, int dtypes,
                                  const void* workspace, const void* packed_arena, const void* scale_arena, const void* min_arena,
                                  void* stream) {
  if (!batched_args_ok(L, total_blocks) || dtypes < 0 || dtypes > GACT_DTYPES_ALL) return GACT_EINVAL;
  if (L == 0 || total_blocks == 0) return GACT_OK;
  if (!table || !bits || !workspace || !packed_arena || !scale_arena || !min_arena) return GACT_EINVAL;
  if (!aligned16(packed_arena) || !aligned16(workspace)) return GACT_EALIGN;
  fresh_launch();
  const dim3 grid((unsigned)(4 * total_blocks)), block(256);
  hipLaunchKernelGGL(dequantize_batched_kernel, grid, block, batch_dequantize_lds(dtypes, total_blocks), (hipStream_t)stream, table, bits,
                     batch_workspace(const_cast<void*>(workspace)), (const uint8_t*)packed_arena,
                     (const uint8_t*)scale_arena, (const uint8_t*)min_arena);
  return launch_status();
}

int gact_dequantize_batched_to(const gact_batch_entry* table, void* const* x, const int32_t* bits, int64_t L, int64_t total_blocks, int dtypes,
                               const void* workspace, const void* packed_arena, const void* scale_arena, const void* min_arena,
                               void* stream) {
  if (!batched_args_ok(L, total_blocks) || dtypes < 0 || dtypes > GACT_DTYPES_ALL) return GACT_EINVAL;
  if (L > GACT_BATCH_ARGS) return GACT_ELIMIT;
  if (L == 0 || total_blocks == 0) return GACT_OK;
  if (!table || !x || !bits || !workspace || !packed_arena || !scale_arena || !min_arena) return GACT_EINVAL;
  if (!aligned16(packed_arena) || !aligned16(workspace)) return GACT_EALIGN;
  BatchOutputs outs = {};
  for (int64_t t = 0; t < L; t++) outs.x[t] = x[t];
  fresh_launch();
  const dim3 grid((unsigned)(4 * total_blocks)), block(256);
  hipLaunchKernelGGL(dequantize_batched_to_kernel, grid, block, batch_dequantize_lds(dtypes, total_blocks), (hipStream_t)stream, table,
                     bits, batch_workspace(const_cast<void*>(workspace)), (const uint8_t*)packed_arena, (const uint8_t*)scale_arena,
                     (const uint8_t*)min_arena, outs);
  return launch_status();
}

// ------------------------------------------------------------------------------------------------
// The batched quantize for callers that cannot allocate: plan + quantize with the workspace in a device array
// of the library's own.  Every GPU the library runs on holds its own copy of the array, at its own address,
// until the process ends; the address is looked up once per device (the array's name is only a host-side
// handle) and that pointer is what the kernels get.  Calls on one GPU share the array: they must not overlap.
// Nothing in it has to start at zero - the plan kernel writes every field the work kernels read, the verdict
// (`ok`) included, on every call: a void plan left behind by an earlier call cannot leak into the next one.
// The verdict of a call is also written to the caller's `verdict` words, since the array itself is out of reach.
// ------------------------------------------------------------------------------------------------
#define GACT_STATIC_MAX_BLOCKS 262144
#define GACT_STATIC_WORKSPACE_BYTES (256 + GACT_STATIC_MAX_BLOCKS * 4)
#define GACT_MAX_DEVICES 64
static __device__ __align__(256) __attribute__((used)) unsigned char scratch[GACT_STATIC_WORKSPACE_BYTES];

namespace {
std::mutex g_scratch_mutex;
void* g_scratch_ptr[GACT_MAX_DEVICES];  // device address of `scratch` on each device, once looked up

int static_workspace(void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= GACT_MAX_DEVICES) return GACT_ELAUNCH;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return GACT_ELAUNCH;
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return GACT_OK;
}
}  // namespace

int gact_quantize_batched_static(gact_batch_entry* table, const int32_t* bits, int64_t L, int64_t total_blocks,
                                 int64_t capacity, int noise_mode, int dtypes, void* packed_arena, void* scale_arena,
                                 void* min_arena, int64_t* verdict, void* stream) {
  if (!batched_args_ok(L, total_blocks) || capacity < 0) return GACT_EINVAL;
  if (noise_mode != GACT_NOISE_CONST && noise_mode != GACT_NOISE_REF && noise_mode != GACT_NOISE_FAST) return GACT_EINVAL;
  if (dtypes < 0 || dtypes > GACT_DTYPES_ALL) return GACT_EINVAL;
  if (dtypes == 0) dtypes = GACT_DTYPES_ALL;
  if (total_blocks > GACT_STATIC_MAX_BLOCKS) return GACT_ELIMIT;
  if (L == 0 || total_blocks == 0) return GACT_OK;
  if (!table || !bits || !packed_arena || !scale_arena || !min_arena) return GACT_EINVAL;
  if (!aligned16(packed_arena)) return GACT_EALIGN;
  if (reinterpret_cast<uintptr_t>(verdict) & 7u) return GACT_EALIGN;
  void* ws = nullptr;
  const int rc = static_workspace(&ws);
  if (rc != GACT_OK) return rc;
  hipStream_t s = (hipStream_t)stream;
  fresh_launch();
  const int planned = batch_plan_on(table, bits, L, total_blocks, capacity, ws, verdict, s);
  if (planned != GACT_OK) return planned;
  return quantize_batched_on(table, bits, total_blocks, noise_mode, dtypes, ws, packed_arena, scale_arena, min_arena, s);
}

}  // extern "C"
