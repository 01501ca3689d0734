// gfx950 (CDNA4) kernels of the int8 KV-cache decode path, written for
// 64-wide wavefronts. Built ahead of time into a code object
// (hipcc --genco --offload-arch=gfx950) and launched by ppk_abi.cpp.
//
//   ppk_quantize_d{64,128,256}         quantize rows densely or append into arenas
//   ppk_dequantize                     codes * scales -> f32/bf16/f16
//   ppk_decode[_bf16h]_d{..}           decode attention (+ fused append, + in-block merge), up to 8 waves per
//                                      block
//   ppk_attn_merge_d{..}               cross-group merge + current token
//   ppk_decode_flat[_bf16h]_d{..}      decode attention over a balanced work list (ragged batches, + fused append)
//   ppk_attn_merge_flat_d{..}          merge of the balanced work list's records + current token
//   ppk_fdecode_{bf16,f32}_d{..}       decode attention over float (bf16/f32) K/V
//   ppk_fmerge_d{..}                   cross-group merge of the float path
//   ppk_fdecode_flat_{bf16,f32}_d{..}  float-path decode over a balanced work list (ragged batches)
//   ppk_fstep[_flat]_{bf16,f32}_d{..}  the float path's fused step: write the current token, then attend
//   ppk_fmerge_flat_d{..}              merge of the float balanced work list's records
//   ppk_renyi_sample                   CFG + Renyi effective-support sampler
//   ppk_kv_scatter_u{16,4,2}           float-store append of token records into arena slots
//   ppk_copy2d_batch                   batched rectangle copies + zero fill (arena joins, growth, copy-on-write)
//
// Semantics follow app/src/model/int8_kv_ops.rs:11-40 and
// app/src/model/int8_kv.cu:8-59; the design (wave-per-row quantize, one-wave
// split blocks streaming 1 KiB per load, scale folding) is this file's own.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "ppk_kernel_args.h"

namespace {

#ifdef PPK_WAVE_CLOCK
// Wave-clock diagnostics build (ppk_kernels_clock.hsaco, -DPPK_WAVE_CLOCK):
// the real-time clock at fixed points of a wave, kept in scalar registers and
// appended as one record at the wave's end (layout in ppk_kernel_args.h). A
// point "after x" first makes the wave wait for x (an empty asm that reads
// it), then reads the clock.
#define PPK_CLK_DECL uint64_t clk_[ppk::kWaveClockPoints] = {0, 0, 0, 0, 0, 0, 0, 0}
#define PPK_CLK(i) (clk_[i] = __builtin_amdgcn_s_memrealtime())
#define PPK_CLK_AFTER(i, dep)           \
  do {                                  \
    __asm__ volatile("" ::"v"(dep));    \
    PPK_CLK(i);                         \
  } while (0)
#define PPK_CLK_AT(var, dep)            \
  do {                                  \
    __asm__ volatile("" ::"v"(dep));    \
    (var) = __builtin_amdgcn_s_memrealtime(); \
  } while (0)
#define PPK_CLK_RECORD(args, kind, block, wave) \
  clock_record(args.clock, args.clock_seq, args.clock_cap, kind, block, wave, clk_)
// The buffer's own capacity word is honoured only up to the capacity the host
// derived from the buffer's size, so a wrong word cannot send a record past it.
__device__ __forceinline__ void clock_record(uint64_t* clock, uint32_t seq, uint32_t cap, uint32_t kind,
                                             uint32_t block, uint32_t wave,
                                             const uint64_t (&t)[ppk::kWaveClockPoints]) {
  if (!clock || (threadIdx.x & 63) != 0) return;
  const uint64_t per = clock[0], local = uint64_t(block) * (blockDim.x >> 6) + wave;
  const uint64_t slot = (uint64_t(seq) * 2 + kind - 1) * per + local;
  if (local >= per || slot >= clock[1] || slot >= cap) return;
  uint64_t* r = clock + ppk::kWaveClockWords * (slot + 1);
  const uint32_t hw = __builtin_amdgcn_s_getreg((31 << 11) | 4);    // HW_ID
  const uint32_t xcc = __builtin_amdgcn_s_getreg((15 << 11) | 20);  // XCC_ID
  r[0] = (uint64_t(kind) << 56) | (uint64_t(seq) << 32) | (uint64_t(block) << 8) | wave;
  r[1] = (uint64_t(xcc) << 32) | hw;
#pragma unroll
  for (int i = 0; i < ppk::kWaveClockPoints; ++i) r[2 + i] = t[i];
}
#else
#define PPK_CLK_DECL
#define PPK_CLK(i)
#define PPK_CLK_AFTER(i, dep)
#define PPK_CLK_AT(var, dep)
#define PPK_CLK_RECORD(args, kind, block, wave)
#endif

using u2 = uint32_t __attribute__((ext_vector_type(2)));
using u4 = uint32_t __attribute__((ext_vector_type(4)));
using f4 = float __attribute__((ext_vector_type(4)));
// Views of LDS that the compiler may not reorder against accesses of another type.
typedef uint16_t __attribute__((may_alias)) u16_alias;
typedef uint32_t __attribute__((may_alias)) u32_alias;
typedef uint32_t __attribute__((ext_vector_type(4), may_alias)) u4_alias;

enum { kF32 = 0, kBF16 = 1, kF16 = 2 };

__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float(uint32_t(h) << 16); }
__device__ __forceinline__ float f16_to_f32(uint16_t h) { return float(__builtin_bit_cast(_Float16, h)); }

// N consecutive elements starting at element i, widened to f32: one dtype
// branch, then N independent loads in flight together.
template <int N>
__device__ __forceinline__ void load_vec(const void* p, size_t i, uint32_t dtype, float (&out)[N]) {
  if (dtype == kF32) {
    const float* f = static_cast<const float*>(p) + i;
#pragma unroll
    for (int e = 0; e < N; ++e) out[e] = f[e];
  } else {
    const uint16_t* h = static_cast<const uint16_t*>(p) + i;
    uint16_t b[N];
#pragma unroll
    for (int e = 0; e < N; ++e) b[e] = h[e];
    if (dtype == kBF16) {
#pragma unroll
      for (int e = 0; e < N; ++e) out[e] = bf16_to_f32(b[e]);
    } else {
#pragma unroll
      for (int e = 0; e < N; ++e) out[e] = f16_to_f32(b[e]);
    }
  }
}

// The same elements as they are stored, to be widened later: one load (per
// dtype branch) whose result no instruction of the branch reads. A widening
// inside the branch makes the wave wait for the load there, and for every
// load before it, so a kernel that reads several small operands in both
// 16-bit dtypes that way pays one memory round trip after another before its
// stream starts; raw words let them all travel together.
template <int N>
struct RawVec {
  uint32_t w[N];  // f32: one element each; 16-bit: element e in half e % 2 of word e / 2
};
template <int N>
__device__ __forceinline__ void load_raw(const void* p, size_t i, uint32_t dtype, RawVec<N>& r) {
  if (dtype == kF32) {
    __builtin_memcpy(r.w, __builtin_assume_aligned(static_cast<const float*>(p) + i, 4), 4 * N);
  } else if constexpr (N == 1) {
    r.w[0] = static_cast<const uint16_t*>(p)[i];
  } else {
    __builtin_memcpy(r.w, __builtin_assume_aligned(static_cast<const uint16_t*>(p) + i, 2), 2 * N);
  }
}
// Waits for r's loads here. A kernel that loads an operand on some of its
// paths only settles it before its streaming loop: the compiler would
// otherwise keep those loads pending into the loop and, when it reuses their
// registers there, wait for everything in flight.
template <int N>
__device__ __forceinline__ void settle(const RawVec<N>& r) {
#pragma unroll
  for (int e = 0; e < N; ++e) __asm__ volatile("" ::"v"(r.w[e]));
}
template <int N>
__device__ __forceinline__ void widen(const RawVec<N>& r, uint32_t dtype, float (&x)[N]) {
#pragma unroll
  for (int e = 0; e < N; ++e) {
    // All three readings are formed and one is selected: no branch per element.
    const uint16_t h = uint16_t(r.w[e / 2] >> (16 * (e % 2)));
    const float as_f32 = __uint_as_float(r.w[e]), as_bf16 = bf16_to_f32(h), as_f16 = f16_to_f32(h);
    const float as_half = dtype == kBF16 ? as_bf16 : as_f16;
    x[e] = dtype == kF32 ? as_f32 : as_half;
  }
}

// Round-to-nearest-even to bfloat16, returned as the 16 stored bits. NaN stays
// a quiet NaN (the carry trick alone could turn some NaN payloads into Inf).
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float x) {
  const uint32_t u = __float_as_uint(x);
  const uint32_t rounded = (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
  return uint16_t(x != x ? 0x7fc0u : rounded);
}
// The same rounding kept in fp32 (the value a bf16 tensor would hold).
__device__ __forceinline__ float round_bf16(float x) {
  uint32_t u = __float_as_uint(x);
  u += 0x7fffu + ((u >> 16) & 1u);
  return __uint_as_float(u & 0xffff0000u);
}
// Two values rounded to bfloat16 (nearest even) by one v_cvt_pk_bf16_f32 and
// widened back to fp32: for finite inputs the bits of round_bf16 on each.
__device__ __forceinline__ void round_bf16_pair(float a, float b, float& ra, float& rb) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 h2 __attribute__((ext_vector_type(2)));
  const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{a, b}, h2));
  ra = __uint_as_float(u << 16);
  rb = __uint_as_float(u & 0xffff0000u);
}
// f32 -> f16, round to nearest even, from a materialised f32 value: the empty
// asm keeps the backend from folding a producing multiply into one fused
// multiply-to-f16 (v_fma_mixlo_f16), which rounds once where the reference
// semantics (an f32 product, then a conversion) round twice.
__device__ __forceinline__ uint16_t f32_to_f16_bits(float x) {
  __asm__("" : "+v"(x));
  return __builtin_bit_cast(uint16_t, static_cast<_Float16>(x));
}

__device__ __forceinline__ void store_elem(void* p, size_t i, uint32_t dtype, float x) {
  if (dtype == kF32) static_cast<float*>(p)[i] = x;
  else static_cast<uint16_t*>(p)[i] = dtype == kBF16 ? f32_to_bf16_bits(x) : f32_to_f16_bits(x);
}

// Loads above this line are issued before anything below it (both the
// optimiser and the scheduler would otherwise move them down to their use).
__device__ __forceinline__ void issue_here() {
  __asm__ volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
using ppk::fast_div;
using ppk::row_scale;
// A zero the compiler takes for a per-lane value: added to a uniform index it
// makes the load a vector load, which waits in order with the wave's other
// vector loads. A scalar load of the same word shares its counter with the
// kernel-argument loads, which can only be waited for all together.
__device__ __forceinline__ uint32_t lane_zero() {
  uint32_t z;
  __asm__("v_mov_b32 %0, 0" : "=v"(z));
  return z;
}

// Signed byte k of a dword as float; hipcc folds the sign-extension into an
// SDWA operand of v_cvt_f32_i32 (one VALU op per byte).
__device__ __forceinline__ float sbyte(uint32_t w, int k) { return float(int(int8_t(w >> (8 * k)))); }

template <int CTRL>
__device__ __forceinline__ float dpp_f32(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float dpp_xor1(float x) { return dpp_f32<0xB1>(x); }  // quad_perm [1,0,3,2]
__device__ __forceinline__ float dpp_xor2(float x) { return dpp_f32<0x4E>(x); }  // quad_perm [2,3,0,1]
__device__ __forceinline__ float dpp_half_mirror(float x) { return dpp_f32<0x141>(x); }
__device__ __forceinline__ float dpp_mirror(float x) { return dpp_f32<0x140>(x); }

// Sum over the LPT consecutive lanes that hold one token (LPT in {4, 8, 16});
// every lane of the group receives the total. DPP adds, no LDS traffic.
template <int LPT>
__device__ __forceinline__ float group_sum(float x) {
  x += dpp_xor1(x);
  x += dpp_xor2(x);
  if constexpr (LPT >= 8) x += dpp_half_mirror(x);
  if constexpr (LPT >= 16) x += dpp_mirror(x);
  return x;
}

// The same over ints (exact: no rounding at any step).
template <int CTRL>
__device__ __forceinline__ int dpp_i32(int x) {
  return __builtin_amdgcn_mov_dpp(x, CTRL, 0xF, 0xF, true);
}
template <int LPT>
__device__ __forceinline__ int group_sum_i32(int x) {
  x += dpp_i32<0xB1>(x);
  x += dpp_i32<0x4E>(x);
  if constexpr (LPT >= 8) x += dpp_i32<0x141>(x);
  if constexpr (LPT >= 16) x += dpp_i32<0x140>(x);
  return x;
}

// Reductions over the whole wave, every lane receiving the result, without
// LDS: DPP within rows of 16 lanes (quad swaps, half-row and row mirrors),
// then gfx950's lane swaps across rows (v_permlane16_swap) and halves
// (v_permlane32_swap); each swap of a value with itself hands every lane its
// partner's value beside its own.
template <class Op>
__device__ __forceinline__ float wave_reduce(float x, Op op) {
  x = op(x, dpp_f32<0xB1>(x));   // quad_perm [1,0,3,2]
  x = op(x, dpp_f32<0x4E>(x));   // quad_perm [2,3,0,1]
  x = op(x, dpp_f32<0x141>(x));  // row_half_mirror
  x = op(x, dpp_f32<0x140>(x));  // row_mirror
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = op(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float wave_max(float x) {
  return wave_reduce(x, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float wave_sum(float x) {
  return wave_reduce(x, [](float a, float b) { return a + b; });
}
// The same over a wave's token groups only (lanes that differ in the bits at
// and above log2(LPT)): each lane receives the reduction over the lanes of
// its position within a token.
template <int LPT, class Op>
__device__ __forceinline__ float groups_reduce(float x, Op op) {
  if constexpr (LPT <= 4) x = op(x, __shfl_xor(x, 4));
  if constexpr (LPT <= 8) x = op(x, dpp_f32<0x128>(x));  // row_ror:8, lane i ^ 8 of a row
  if constexpr (LPT <= 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = op(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  if constexpr (LPT <= 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = op(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  return x;
}
template <int LPT>
__device__ __forceinline__ float groups_max(float x) {
  return groups_reduce<LPT>(x, [](float a, float b) { return fmaxf(a, b); });
}

// Sum over a wave's token groups (lanes that differ in the bits at and above
// log2(LPT)) of each lane's N per-channel partial sums, scattered: one step
// per token-group bit, from bit 5 down, in which the two lanes that differ in
// that bit swap half of their values and add, so the values held halve each
// step and lane l ends with N >> steps totals, of its chunk's channels
// scatter_base<LPT, N>(l) + e, in acc[e]. Bits 5 and 4 use gfx950's lane
// swaps (v_permlane32_swap, v_permlane16_swap), bit 3 a DPP rotate by 8
// within a row, bit 2 one swizzle: VALU moves, where the butterfly over
// every value (__shfl_xor per value and bit) took one LDS permute each, 64
// per lane at D = 64 in every wave's epilogue.
template <int LPT, int N>
__device__ __forceinline__ int scatter_base(int lane) {
  int base = 0, n = N;
  if constexpr (LPT <= 32) { n >>= 1; base += ((lane >> 5) & 1) * n; }
  if constexpr (LPT <= 16) { n >>= 1; base += ((lane >> 4) & 1) * n; }
  if constexpr (LPT <= 8) { n >>= 1; base += ((lane >> 3) & 1) * n; }
  if constexpr (LPT <= 4) { n >>= 1; base += ((lane >> 2) & 1) * n; }
  return base;
}
template <int LPT, int N>
__device__ __forceinline__ void reduce_scatter_groups(float (&acc)[N], int lane) {
  if constexpr (LPT <= 32) {
    static_assert(N % 2 == 0, "a value per lane half");
    // Lanes 0-31 keep values [0, N/2), lanes 32-63 values [N/2, N).
#pragma unroll
    for (int k = 0; k < N / 2; ++k) {
      const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[k]), __float_as_uint(acc[N / 2 + k]),
                                                     false, false);
      acc[k] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
  }
  if constexpr (LPT <= 16) {
    static_assert(N % 4 == 0, "a value per lane quarter");
    // Even rows of 16 lanes keep [0, N/4), odd rows [N/4, N/2).
#pragma unroll
    for (int k = 0; k < N / 4; ++k) {
      const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[k]), __float_as_uint(acc[N / 4 + k]),
                                                     false, false);
      acc[k] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
  }
  if constexpr (LPT <= 8) {
    static_assert(N % 8 == 0, "a value per lane eighth");
    // Lanes i and i ^ 8 of a row: a rotate by 8 within the row pairs them.
    const bool hi = ((lane >> 3) & 1) != 0;
#pragma unroll
    for (int k = 0; k < N / 8; ++k) {
      const float keep = hi ? acc[N / 8 + k] : acc[k];
      const float give = hi ? acc[k] : acc[N / 8 + k];
      acc[k] = keep + dpp_f32<0x128>(give);  // row_ror:8
    }
  }
  if constexpr (LPT <= 4) {
    static_assert(N % 16 == 0, "a value per lane sixteenth");
    const bool hi = ((lane >> 2) & 1) != 0;
#pragma unroll
    for (int k = 0; k < N / 16; ++k) {
      const float keep = hi ? acc[N / 16 + k] : acc[k];
      const float give = hi ? acc[k] : acc[N / 16 + k];
      acc[k] = keep + __shfl_xor(give, 4);
    }
  }
}

// Largest |x| of a lane's values with f32::max / fmaxf semantics (NaNs of
// either kind skipped); the result is >= +0 and never NaN. Written on the bit
// patterns: the hardware float max quiets a signalling NaN and returns it,
// which would drop the max of the values before it.
template <int N>
__device__ __forceinline__ float lane_absmax(const float (&x)[N]) {
  uint32_t m = 0;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const uint32_t a = __float_as_uint(x[k]) & 0x7fffffffu;
    m = max(m, a > 0x7f800000u ? 0u : a);
  }
  return __uint_as_float(m);
}

// ---------------------------------------------------------------------------
// Kernel 1: quantize (dense) / quantize-and-append (arena).
// One wave per (tensor, row); D/64 channels per lane.
// Bit-exact contract (int8_kv_ops.rs:17-18, int8_kv.cu:13,17):
//   s = max(absmax / 127, 1e-12); code = clamp(rne(x / s), -127, 127).
// NaN quotients become code 0 (as a float->int conversion of NaN does on
// the reference GPU path); the absmax ignores NaN like fmaxf / f32::max.
// ---------------------------------------------------------------------------
// ORs `bits` (PPK_FLAG_*, uniform) into *flags, if there is one and any bit is
// set. Every lane issues the atomic (the same bits; a rare path): see
// quantize_values on branches on the lane, which the compiler's own atomic
// would bring back.
__device__ __forceinline__ void raise_flags(uint32_t* flags, uint32_t bits) {
  if (flags && bits) __asm__ volatile("global_atomic_or %0, %1, off" ::"v"(flags), "v"(bits) : "memory");
}

// Quantise one row of D values into codes[0..D) and *scale; the whole wave
// participates, lane l holding elements l*D/64 ... (l+1)*D/64 - 1 of the
// row. Returns whether a value of the lane was non-finite. Every lane stores the scale
// (one value at one address): a lane-0 branch here would make the compiler
// restructure the control flow around it, and the decode kernels' streaming
// loops then wait for loads of paths that never reach them.
template <int D, bool ONE = false>
__device__ __forceinline__ bool quantize_values(const float (&x)[D / ppk::kWave], uint8_t* codes, float* scale,
                                                int lane) {
#pragma clang fp contract(off)
  constexpr int EPL = D / ppk::kWave;
  bool finite = true;
#pragma unroll
  for (int e = 0; e < EPL; ++e) finite = finite && __builtin_isfinite(x[e]);
  const float amax = wave_max(lane_absmax(x));
  const float s = fmaxf(amax / 127.0f, 1e-12f);
  uint32_t packed = 0;
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    const float qf = rintf(x[e] / s);
    const int qi = (qf != qf) ? 0 : int(fminf(fmaxf(qf, -127.f), 127.f));
    packed |= (uint32_t(qi) & 0xffu) << (8 * e);
  }
  uint8_t* out = codes + size_t(lane) * EPL;
  if constexpr (EPL == 1) *out = uint8_t(packed);
  else if constexpr (EPL == 2) *reinterpret_cast<uint16_t*>(out) = uint16_t(packed);
  else *reinterpret_cast<uint32_t*>(out) = packed;
  if (!ONE || lane == 0) *scale = s;
  return !finite;
}

// The same for row src_row of src[rows, D] in dtype.
template <int D>
__device__ __forceinline__ void quantize_row(const void* src, size_t src_row, uint32_t dtype, uint8_t* codes,
                                             float* scale, uint32_t* flags, int lane) {
  constexpr int EPL = D / ppk::kWave;
  float x[EPL];
  load_vec<EPL>(src, src_row * D + size_t(lane) * EPL, dtype, x);
  const bool bad = quantize_values<D, true>(x, codes, scale, lane);
  if (flags && __any(bad) && lane == 0) atomicOr(flags, 1u);
}

template <int D>
__device__ __forceinline__ void quantize_body(const ppk::QuantizeArgs& a) {
  const int lane = threadIdx.x & 63;
  const uint64_t wave = uint64_t(blockIdx.x) * (blockDim.x / 64) + threadIdx.x / 64;
  if (wave >= a.rows * a.ntensors) return;  // uniform per wave
  const uint32_t tensor = wave >= a.rows ? 1u : 0u;
  const uint64_t r = wave - (tensor ? a.rows : 0);
  const void* src = tensor ? a.src[1] : a.src[0];
  size_t dst = r;
  if (a.capacity) {
    const uint64_t bh = r / a.tokens;
    const uint32_t tok = uint32_t(r - bh * a.tokens);
    const uint64_t slot = uint64_t(a.past ? a.past[bh / a.heads] : a.uniform_past) + tok;
    if (slot >= a.capacity) {
      if (lane == 0 && a.flags) atomicOr(a.flags, 2u);
      return;
    }
    dst = bh * a.capacity + slot;
  }
  quantize_row<D>(src, r, a.src_dtype, (tensor ? a.codes[1] : a.codes[0]) + dst * D,
                  (tensor ? a.scales[1] : a.scales[0]) + dst, a.flags, lane);
}

// ---------------------------------------------------------------------------
// Dequantize
// ---------------------------------------------------------------------------
// Dequantization in units of one 16-byte output chunk: E = 8 codes for a
// 16-bit output, 4 for f32. A wave takes chunks of R * 64 consecutive units,
// all loads of a chunk before its first store: each load instruction reads
// 64*E consecutive code bytes, each store instruction writes 1 KiB, and the
// chunk's output is one piece of R KiB. Addresses are a scalar base, the lane
// and constants. Bound by memory, mostly by its writes (two thirds of the
// bytes for a 16-bit output): where a wave's units lay a grid apart (and the
// next batch was loaded before the stores), 1 M rows of D = 128 to bf16 took
// 77 us, now 64. Eight units per lane measured the same. The host sizes the
// grid for one chunk per wave up to 128 blocks per CU.
template <int E, uint32_t OUT, bool ROUND>
__device__ __forceinline__ void dequantize_units(const ppk::DequantizeArgs& a) {
#pragma clang fp contract(off)
  constexpr uint32_t R = ppk::kDequantizeUnits;
  using Raw = typename std::conditional<E == 8, u2, uint32_t>::type;
  const uint64_t units = a.rows * (a.head_dim / E);
  const uint32_t row_shift = __builtin_ctz(a.head_dim / E);  // units per token row: a power of two up to 64
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
  const uint64_t step = uint64_t(gridDim.x) * 4 * R * 64;
  for (uint64_t u0 = (uint64_t(blockIdx.x) * 4 + wave) * R * 64; u0 < units; u0 += step) {
    const uint32_t left = uint32_t(min(units - u0, uint64_t(R * 64)));
    const bool full = left == R * 64;
    const Raw* codes = reinterpret_cast<const Raw*>(a.codes) + u0;
    const float* scales = a.scales + (u0 >> row_shift);
    Raw raw[R];
    float sc[R];
    if (full) {
#pragma unroll
      for (uint32_t r = 0; r < R; ++r) raw[r] = __builtin_nontemporal_load(codes + (lane + r * 64));
#pragma unroll
      for (uint32_t r = 0; r < R; ++r) sc[r] = (scales + ((r * 64) >> row_shift))[lane >> row_shift];
    } else {
#pragma unroll
      for (uint32_t r = 0; r < R; ++r) {
        const uint32_t u = min(lane + r * 64, left - 1);  // clamped: in bounds, masked for storing
        raw[r] = __builtin_nontemporal_load(codes + u);
        sc[r] = scales[u >> row_shift];
      }
    }
#pragma unroll
    for (uint32_t r = 0; r < R; ++r) {
      float f[E];
#pragma unroll
      for (int k = 0; k < E; ++k) {
        uint32_t w;
        if constexpr (E == 8) w = raw[r][k / 4];
        else w = raw[r];
        const float v = sbyte(w, k % 4) * sc[r];
        f[k] = ROUND ? round_bf16(v) : v;
      }
      u4 out;
      if constexpr (E == 4) {
#pragma unroll
        for (int k = 0; k < 4; ++k) out[k] = __float_as_uint(f[k]);
      } else {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const uint16_t lo = OUT == kBF16 ? f32_to_bf16_bits(f[2 * w]) : f32_to_f16_bits(f[2 * w]);
          const uint16_t hi = OUT == kBF16 ? f32_to_bf16_bits(f[2 * w + 1]) : f32_to_f16_bits(f[2 * w + 1]);
          out[w] = uint32_t(lo) | (uint32_t(hi) << 16);
        }
      }
      if (full || lane + r * 64 < left)
        __builtin_nontemporal_store(out, static_cast<u4*>(a.out) + u0 + (lane + r * 64));
    }
  }
}

// Output type and the bf16 pre-rounding are fixed per instantiation (a bf16
// output already rounds to bf16, so it needs no pre-rounding).
__device__ __forceinline__ void dequantize_body(const ppk::DequantizeArgs& a) {
  if (a.out_dtype == kF32) {
    if (a.round_bf16) dequantize_units<4, kF32, true>(a);
    else dequantize_units<4, kF32, false>(a);
  } else if (a.out_dtype == kBF16) {
    dequantize_units<8, kBF16, false>(a);
  } else {
    if (a.round_bf16) dequantize_units<8, kF16, true>(a);
    else dequantize_units<8, kF16, false>(a);
  }
}

// ---------------------------------------------------------------------------
// Kernel 2a: decode attention. A row is covered by G blocks (groups) of W waves
// of S tokens each; its waves take its batches in turn (Batches below), the
// block combines its waves through LDS. With one group per row
// the block also scores the current token and writes the final output, so a
// decode step is a single launch; otherwise it writes a partial (m, z, y)
// record for the merge kernel. Optionally the block first quantises the new
// K/V token of its row into slot past[b] (a slot attention never reads).
//
// Lane layout inside a wave: LPT = D/16 lanes share one token, each holding
// 16 channels, so one dwordx4 load per lane moves 1 KiB = TPL = 64/LPT whole
// tokens. The dot product is 16 FMAs per lane plus a DPP group sum; the
// per-token scale is applied once to the sum (default) instead of to every
// element. Phase K streams K codes and scales and leaves log2-domain scores
// in LDS; phase V streams V codes and scales and accumulates
// p_t * vscale_t * code_t per channel. The exact wave max is known before
// phase V, so no running rescale is needed. Each wave keeps two batches of
// loads in flight (the next batch is issued before the current is consumed).
// ---------------------------------------------------------------------------
struct WavePartial {
  float m;         // max log2-domain score (-inf if the wave had no tokens)
  float z;         // sum of 2^(s - m)
  float acc[16];   // sum of 2^(s - m) * v: while streaming over this lane's 16 channels; at the end the wave's
                   // totals of channels c * 16 + scatter_base<LPT, 16>(lane) + e in acc[e], e < D / 64
#ifdef PPK_WAVE_CLOCK
  uint64_t t_first = 0;  // the clock when the stream's first K data had arrived
#endif
};

// One batch = U load tiles = U*TPL consecutive tokens of this wave's range.
// Codes come as one dwordx4 per lane per tile; the batch's per-token scales
// come as one coalesced dword per lane (lane l holds token l of the batch)
// and reach each token's lane group through a cross-lane read.
template <int D, int U>
__device__ __forceinline__ void load_batch(const uint8_t* base, const float* scales, uint32_t t0, uint32_t n, int j,
                                           int lane, u4 (&raw)[U], float& scale) {
  constexpr int TPL = ppk::kWave / (D / 16);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t tc = min((t0 + u) * TPL + j, n - 1);  // clamp: always in bounds
    raw[u] = __builtin_nontemporal_load(reinterpret_cast<const u4*>(base + size_t(tc) * D));
  }
  // Scales stay cacheable: a batch's 4*TPL scales need not start on a cache
  // line (capacity is arbitrary), and the next batch reuses the shared line.
  scale = scales[min(t0 * TPL + uint32_t(lane % (U * TPL)), n - 1)];
}

// q in exact integer form for the K-phase dot products: every lane's 16
// channels become q_int = rne(q / qmax * Q), Q = 127 * 2^21, split into four
// signed bytes hi*2^21 + m1*2^14 + m2*2^7 + lo (each in [-127, 127]) packed
// four channels per dword. <codes, part> is then an exact v_dot4_i32_i8 sum;
// the four partial sums pair up exactly in int32 (hi*2^7 + m1, m2*2^7 + lo),
// are summed over the token's lanes in int32 (exact), and meet in one fp32
// multiply-add, so q_int . codes carries fp32 rounding only. q_int keeps 29
// bits of q relative to the row's max |q|: with 22 bits (three slices) the
// rounding of q was the largest error on heavy-tailed history (max relative
// error 7.9e-3 at D = 64 against the f64 oracle, 1.2e-3 with 29 bits; the
// time per step the same).
struct QInt {
  int hi[4], m1[4], m2[4], lo[4];
  float unscale;  // qmax / Q (NaN if q held a non-finite value)
};

// Max over G consecutive lanes (G a power of two <= 64) of values that are
// >= +0 and never NaN: such floats order like their bit patterns, so the
// reduction runs as unsigned integer max (the DPP move folds into the max,
// and no NaN canonicalisation is needed).
template <int G>
__device__ __forceinline__ float group_max_nonneg(float x) {
  uint32_t b = __float_as_uint(x);
  auto step = [&](uint32_t o) { b = max(b, o); };
  step(uint32_t(__builtin_amdgcn_mov_dpp(int(b), 0xB1, 0xF, 0xF, true)));
  step(uint32_t(__builtin_amdgcn_mov_dpp(int(b), 0x4E, 0xF, 0xF, true)));
  if constexpr (G >= 8) step(uint32_t(__builtin_amdgcn_mov_dpp(int(b), 0x141, 0xF, 0xF, true)));
  if constexpr (G >= 16) step(uint32_t(__builtin_amdgcn_mov_dpp(int(b), 0x140, 0xF, 0xF, true)));
#pragma unroll
  for (int o = 16; o < G; o <<= 1) step(uint32_t(__shfl_xor(int(b), o)));
  return __uint_as_float(b);
}

// Quantization at streaming rates: dense (int8_kv_ops::quantize over [rows,
// D]) and quantize-and-append into arenas (rows of K and V written at slot
// past[b] + t). A row's D values are split over G = D / E lanes, 16 bytes (E
// values) per lane, so one wave-wide load covers 64 / G whole rows and the
// row's absmax is a G-lane reduction; each lane then forms the E codes of
// quantize_row's arithmetic (IEEE division, ties-to-even, clamp, NaN quotient
// -> 0), see below. A wave takes chunks of R * 64 consecutive units of one
// tensor: all its addresses are one scalar base plus the lane plus constants,
// its loads cover 4 KiB and its code stores 2 KiB (1 KiB for f32 sources) in
// one piece, and its R * 64 / G scales leave in one store. An append's chunk
// that lies in one row of the arena and within its capacity (a scalar test)
// stores like a dense one; others index per lane.
//
// Bound by vector instructions before this split (each unit paid 64-bit
// addresses and three divisions by runtime sizes, an IEEE division, and five
// to six instructions per value: ~230 per unit, now ~65). Appends of K and V, bf16 -> int8, 32 x 16 x 1000 tokens
// of D = 128: 92.3 -> 65.0 us (6.1 TB/s), 8 x 16 x 3000 of D = 256: 133.6 ->
// 90.9; dense 1 M rows of D = 128: 77 -> 70 us.
template <int D, int E, uint32_t DT, bool ARENA>
__device__ __forceinline__ void quantize_stream_units(const ppk::StreamQuantizeArgs& a) {
#pragma clang fp contract(off)
  constexpr int G = D / E;
  constexpr int R = 4;
  constexpr uint32_t RU = 64 / G;    // rows per wave-wide load
  constexpr uint32_t ROWS = R * RU;  // rows per chunk
  static_assert(64 % G == 0 && G >= R, "a row's lanes stay inside one wave");
  using Code = typename std::conditional<E == 8, u2, uint32_t>::type;
  const int lane = threadIdx.x & 63;
  const uint32_t gl = uint32_t(lane) % G, gr = uint32_t(lane) / G;
  const uint32_t rows = uint32_t(a.rows);  // per tensor
  const uint32_t per_tensor = (rows + ROWS - 1) / ROWS;  // chunks; one never crosses from K to V
  const uint32_t chunks = per_tensor * a.ntensors;
  const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
  bool any_bad = false, any_over = false;
  for (uint32_t chunk = blockIdx.x * 4 + wave; chunk < chunks; chunk += gridDim.x * 4) {
    const bool second = chunk >= per_tensor;
    const uint32_t row0 = (second ? chunk - per_tensor : chunk) * ROWS;
    const uint32_t left = rows - row0;  // rows of the tensor from here on, at least one
    const u4* src = static_cast<const u4*>(second ? a.src[1] : a.src[0]) + uint64_t(row0) * G;
    u4 raw[R];
    if (left >= ROWS) {
#pragma unroll
      for (int r = 0; r < R; ++r) raw[r] = __builtin_nontemporal_load(src + (lane + r * 64));
    } else {  // the tensor's last rows: clamped for loading, masked for storing
#pragma unroll
      for (int r = 0; r < R; ++r)
        raw[r] = __builtin_nontemporal_load(src + min(uint32_t(lane + r * 64), left * G - 1));
    }
    // Appends: the arena row of the chunk's first row, and whether all the
    // chunk's rows follow it there.
    uint64_t dst0 = row0;
    bool plain = left >= ROWS;
    uint32_t past_of[R];
    bool one_row = true;
    if constexpr (ARENA) {
      const uint32_t bh = fast_div(row0, a.token_div);
      const uint32_t t0 = row0 - bh * a.tokens;
      one_row = left >= ROWS && uint64_t(t0) + ROWS <= a.tokens;
      if (one_row) {
        const uint64_t slot = uint64_t(a.past ? a.past[fast_div(bh, a.head_div)] : a.uniform_past) + t0;
        plain = slot + ROWS <= a.capacity;
        dst0 = uint64_t(bh) * a.capacity + slot;
      } else {
        plain = false;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const uint32_t row = row0 + min(r * RU + gr, left - 1);
          past_of[r] = a.past ? a.past[fast_div(fast_div(row, a.token_div), a.head_div)] : a.uniform_past;
        }
      }
    }
    Code code[R];
    float scale[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float x[E];
      if constexpr (DT == kF32) {
#pragma unroll
        for (int k = 0; k < E; ++k) x[k] = __uint_as_float(raw[r][k]);
      } else {
#pragma unroll
        for (int k = 0; k < E; ++k) {
          const uint16_t h = uint16_t(raw[r][k / 2] >> (16 * (k % 2)));
          x[k] = DT == kBF16 ? bf16_to_f32(h) : f16_to_f32(h);
        }
      }
      // Fast row max: the float max chain is exact unless the lane holds a
      // NaN (a signalling one can drop the values before it); such a lane is
      // seen below, and the wave recomputes.
      float m = 0.f;
#pragma unroll
      for (int k = 0; k < E; ++k) m = fmaxf(m, fabsf(x[k]));
      float sc = row_scale(group_max_nonneg<G>(m));
      // Rounded quotients in fixed point: u = 384 + x / sc from one fused
      // multiply-add with the hardware reciprocal (at most 1 ulp off 1/sc).
      // |x/sc| <= 127 (1 + 2^-24), so u lies in [256, 512), where a float's
      // grid is 2^-15 and its mantissa is the quotient + 128 in 8.15 bits; u
      // is within 2^-16 (its rounding) + 1.52e-5 (the reciprocal) + 3.9e-6
      // (the quotient's own rounding) < 1.2 grid steps of RN(x/sc). Half a
      // unit and 2 steps are added and the word shifted one up: byte 2 then
      // holds the rounded quotient + 128, and the low 16 bits, in half
      // steps, the distance above the half-integer less 2 steps. At 9 or more
      // the rounding is that of RN(x/sc) (and needs no clamp: the value is
      // clear of 127.5); at 8 or less (5 steps of 2^15: one value in 6500) the
      // value is divided. A NaN or infinite u is the largest word (u is
      // positive otherwise).
      const float rcp = __builtin_amdgcn_rcpf(sc);
      constexpr uint32_t kStep = 2, kNear = 8;
      uint32_t w[E];
      uint32_t top = 0;
      uint16_t low = 0xffff;
#pragma unroll
      for (int k = 0; k < E; ++k) {
        const uint32_t u = __float_as_uint(__builtin_fmaf(x[k], rcp, 384.0f));
        w[k] = (u + (0x4000u + kStep)) << 1;
        top = max(top, u);
        low = min(low, uint16_t(w[k]));
      }
      uint32_t packed[E / 4];
#pragma unroll
      for (int i = 0; i < E / 4; ++i) {
        // v_perm: bytes 2 of (a, b) and of (c, d), then the two byte pairs.
        const uint32_t ab = __builtin_amdgcn_perm(w[4 * i + 1], w[4 * i], 0x0c0c0602u);
        const uint32_t cd = __builtin_amdgcn_perm(w[4 * i + 3], w[4 * i + 2], 0x0c0c0602u);
        packed[i] = __builtin_amdgcn_perm(cd, ab, 0x05040100u) ^ 0x80808080u;
      }
      if (__any(low <= kNear || top >= 0x7f800000u)) {  // wave-uniform
        bool finite = true;
#pragma unroll
        for (int k = 0; k < E; ++k) finite = finite && __builtin_isfinite(x[k]);
        // A non-finite input may have spoilt the fast max of its row: the
        // wave then recomputes every row it holds with the NaN-skipping max
        // and the division (the reduction needs all lanes). With finite rows
        // the scale stands and only the flagged values divide.
        const bool all = __any(!finite);
        if (all) sc = fmaxf(group_max_nonneg<G>(lane_absmax(x)) / 127.0f, 1e-12f);
#pragma unroll
        for (int k = 0; k < E; ++k) {
          if (all || uint16_t(w[k]) <= kNear) {
            const float t = rintf(x[k] / sc);
            const uint32_t q = t != t ? 0u : uint32_t(int(__builtin_amdgcn_fmed3f(t, -127.f, 127.f)));
            const int at = 8 * (k % 4);
            packed[k / 4] = (packed[k / 4] & ~(0xffu << at)) | ((q & 0xffu) << at);
          }
        }
        any_bad = any_bad || (!finite && r * RU + gr < left);
      }
      scale[r] = sc;
      if constexpr (E == 8) code[r] = u2{packed[0], packed[1]};
      else code[r] = packed[0];
    }
    uint8_t* codes = second ? a.codes[1] : a.codes[0];
    float* scales = second ? a.scales[1] : a.scales[0];
    if (plain) {
      Code* out = reinterpret_cast<Code*>(codes + dst0 * D);
#pragma unroll
      for (int r = 0; r < R; ++r) __builtin_nontemporal_store(code[r], out + (lane + r * 64));
      float s = scale[0];
#pragma unroll
      for (int r = 1; r < R; ++r) s = gl == r ? scale[r] : s;
      if (gl < R) (scales + dst0)[gl * RU + gr] = s;
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const uint32_t in = r * RU + gr;
        bool store = in < left;
        uint64_t dst = dst0 + in;
        if constexpr (ARENA) {
          const uint32_t row = row0 + min(in, left - 1);
          const uint32_t bh = fast_div(row, a.token_div);
          uint64_t slot = dst - uint64_t(bh) * a.capacity;  // one arena row: from its first slot
          if (!one_row) {
            slot = uint64_t(past_of[r]) + (row - bh * a.tokens);
            dst = uint64_t(bh) * a.capacity + slot;
          }
          any_over = any_over || (store && slot >= a.capacity);
          store = store && slot < a.capacity;
        }
        if (store) {
          __builtin_nontemporal_store(code[r], reinterpret_cast<Code*>(codes + dst * D) + gl);
          if (gl == 0) scales[dst] = scale[r];
        }
      }
    }
  }
  if (a.flags) {
    const bool bad = __any(any_bad), over = __any(any_over);
    if (lane == 0 && (bad || over)) atomicOr(a.flags, (bad ? 1u : 0u) | (over ? 2u : 0u));
  }
}

template <int D, bool ARENA>
__device__ __forceinline__ void quantize_stream_dtype(const ppk::StreamQuantizeArgs& a) {
  if (a.src_dtype == kF32) quantize_stream_units<D, 4, kF32, ARENA>(a);
  else if (a.src_dtype == kBF16) quantize_stream_units<D, 8, kBF16, ARENA>(a);
  else quantize_stream_units<D, 8, kF16, ARENA>(a);
}


// The query of one wave, from x = channels lane * D/64 ... of q: each lane
// forms the slices of its own D/64 channels and the wave exchanges them
// through `region` (LDS of this wave alone, 4 * D bytes, 16-byte aligned), so
// that every lane ends with the slices of its 16-channel chunk. Quantising
// the whole chunk in every lane instead, 64/LPT times the same work, was ~380
// instructions on the critical path of every wave: at two waves per SIMD over
// 1 us of a launch that takes 4-6 us for short rows.
template <int D>
__device__ __forceinline__ QInt quantize_query(const float (&x)[D / ppk::kWave], void* region, int lane) {
  constexpr float Q = 266338304.0f;  // 127 * 2^21
  constexpr int EPL = D / ppk::kWave;
  float amax = 0.f;
  bool finite = true;
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    amax = fmaxf(amax, fabsf(x[e]));
    finite = finite && __builtin_isfinite(x[e]);
  }
  amax = wave_max(amax);
  const bool bad = __any(!finite);
  const float inv = amax > 0.f ? Q / amax : 0.f;
  QInt r;
  r.unscale = bad ? __builtin_nanf("") : amax / Q;
  uint32_t part[4] = {0, 0, 0, 0};
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    const float v = fminf(fmaxf(rintf(x[e] * inv), -Q), Q);
    const int qi = finite ? int(v) : 0;
    const int hi = (qi + (1 << 20)) >> 21;  // [-127, 127]
    const int r1 = qi - hi * (1 << 21);     // [-2^20, 2^20)
    const int m1 = (r1 + 8192) >> 14;       // [-64, 64]
    const int r2 = r1 - m1 * 16384;         // [-8192, 8191]
    const int m2 = (r2 + 64) >> 7;          // [-64, 64]
    const int lo = r2 - m2 * 128;           // [-64, 63]
    part[0] |= (uint32_t(hi) & 0xffu) << (8 * e);
    part[1] |= (uint32_t(m1) & 0xffu) << (8 * e);
    part[2] |= (uint32_t(m2) & 0xffu) << (8 * e);
    part[3] |= (uint32_t(lo) & 0xffu) << (8 * e);
  }
  uint8_t* b = static_cast<uint8_t*>(region);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint8_t* to = b + i * D + lane * EPL;
    if constexpr (EPL == 1) *to = uint8_t(part[i]);
    else if constexpr (EPL == 2) *reinterpret_cast<u16_alias*>(to) = uint16_t(part[i]);
    else *reinterpret_cast<u32_alias*>(to) = part[i];
  }
  __builtin_amdgcn_wave_barrier();  // LDS serves a wave's accesses in order
  const u4_alias* from = reinterpret_cast<const u4_alias*>(b + (lane % (D / 16)) * 16);
  const u4 h = from[0], m1 = from[D / 16], m2 = from[2 * (D / 16)], l = from[3 * (D / 16)];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    r.hi[w] = int(h[w]);
    r.m1[w] = int(m1[w]);
    r.m2[w] = int(m2[w]);
    r.lo[w] = int(l[w]);
  }
  __builtin_amdgcn_wave_barrier();
  return r;
}

// What phase K needs of the query: the integer slices (fp32 history) or the
// lane's 16 channels (bf16 history), and the factor of its scores.
template <bool BF16H>
struct Query {
  QInt qi;
  float qr[16];
  float sl2;
};
template <int D, bool BF16H>
__device__ __forceinline__ void make_query(const float (&x)[D / ppk::kWave], float scale_log2, void* region, int lane,
                                           Query<BF16H>& q) {
  if constexpr (BF16H) {
    constexpr int EPL = D / ppk::kWave;
    float* f = static_cast<float*>(region);
#pragma unroll
    for (int e = 0; e < EPL; ++e) f[lane * EPL + e] = x[e];
    __builtin_amdgcn_wave_barrier();
    const float* from = f + (lane % (D / 16)) * 16;
#pragma unroll
    for (int i = 0; i < 16; ++i) q.qr[i] = from[i];
    __builtin_amdgcn_wave_barrier();
    q.sl2 = scale_log2;
  } else {
    q.qi = quantize_query<D>(x, region, lane);
    q.sl2 = scale_log2 * q.qi.unscale;
  }
}

// One tile's K codes against the query: the log2-domain score of the lane
// group's token (the same in each of its LPT lanes).
template <int D, bool BF16H>
__device__ __forceinline__ float tile_score(const u4& raw, float kscale, const Query<BF16H>& q) {
  constexpr int LPT = D / 16;
  if constexpr (BF16H) {
    // pp_i8_load semantics: every element is bf16(code * scale) before the fp32 dot.
    float d = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
      for (int k = 0; k < 4; k += 2) {
        float e0, e1;
        round_bf16_pair(sbyte(raw[w], k) * kscale, sbyte(raw[w], k + 1) * kscale, e0, e1);
        d = fmaf(q.qr[4 * w + k], e0, d);
        d = fmaf(q.qr[4 * w + k + 1], e1, d);
      }
    return group_sum<LPT>(d) * q.sl2;
  } else {
    int sh = 0, s1 = 0, s2 = 0, sl = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      sh = __builtin_amdgcn_sdot4(int(raw[w]), q.qi.hi[w], sh, false);
      s1 = __builtin_amdgcn_sdot4(int(raw[w]), q.qi.m1[w], s1, false);
      s2 = __builtin_amdgcn_sdot4(int(raw[w]), q.qi.m2[w], s2, false);
      sl = __builtin_amdgcn_sdot4(int(raw[w]), q.qi.lo[w], sl, false);
    }
    const int hm = group_sum_i32<LPT>(sh * 128 + s1);
    const int lm = group_sum_i32<LPT>(s2 * 128 + sl);
    return fmaf(float(hm), 16384.f, float(lm)) * (kscale * q.sl2);
  }
}

// One tile's V codes added with weight p (the lane group's token).
template <bool BF16H>
__device__ __forceinline__ void tile_accumulate(const u4& raw, float p, float vscale, float (&acc)[16]) {
  if constexpr (BF16H) {
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
      for (int k = 0; k < 4; k += 2) {
        float e0, e1;
        round_bf16_pair(sbyte(raw[w], k) * vscale, sbyte(raw[w], k + 1) * vscale, e0, e1);
        acc[4 * w + k] = fmaf(p, e0, acc[4 * w + k]);
        acc[4 * w + k + 1] = fmaf(p, e1, acc[4 * w + k + 1]);
      }
  } else {
    const float wgt = p * vscale;
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
      for (int k = 0; k < 4; ++k) acc[4 * w + k] = fmaf(wgt, sbyte(raw[w], k), acc[4 * w + k]);
  }
}

// Phase K for one batch of U tiles: scores (log2 domain) into LDS, running
// max. The tiles' scales are fetched together and the lanes of chunk c store
// tile c % 4's scores, one unmasked write for the batch: with a fetch and a
// masked write per tile, each tile waited for its own LDS round trip, and the
// branch on the lane made the compiler restructure the kernel (see
// quantize_values).
template <int D, bool BF16H, int U>
__device__ __forceinline__ float score_batch(const u4 (&raw)[U], float scale_lane, uint32_t t0, uint32_t n, int j,
                                             int c, const Query<BF16H>& q, float* s_batch, float mloc) {
  constexpr int LPT = D / 16;
  constexpr int TPL = ppk::kWave / LPT;
  static_assert(U == 4 && LPT >= U, "a lane of each token per tile");
  float kscale[U], s[U];
#pragma unroll
  for (int u = 0; u < U; ++u) kscale[u] = __shfl(scale_lane, u * TPL + j);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const float x = tile_score<D, BF16H>(raw[u], kscale[u], q);
    s[u] = (t0 + u) * TPL + j < n ? x : -INFINITY;
    mloc = fmaxf(mloc, s[u]);
  }
  const float lo = (c & 1) ? s[1] : s[0], hi = (c & 1) ? s[3] : s[2];
  s_batch[(c & 3) * TPL + j] = (c & 2) ? hi : lo;
  return mloc;
}

// Phase V for one batch: lane l owns token l of the batch (the layout of the
// scale load), turns its score into p = 2^(s - m) once, adds it to z and
// forms the weight p * vscale; each tile's token groups then fetch their
// token's weight with one cross-lane read and accumulate weight * code.
template <int D, bool BF16H, int U>
__device__ __forceinline__ void accumulate_batch(const u4 (&raw)[U], float scale_lane, uint32_t t0, uint32_t n, int j,
                                                 int lane, float m, const float* s_batch, float& z,
                                                 float (&acc)[16]) {
  constexpr int LPT = D / 16;
  constexpr int TPL = ppk::kWave / LPT;
  constexpr int TPB = U * TPL;  // tokens per batch (<= 64)
  static_assert(TPB <= ppk::kWave, "one scale per lane per batch");
  const float e = __builtin_amdgcn_exp2f(s_batch[lane % TPB] - m);
  const float pr = (t0 * TPL + uint32_t(lane % TPB) < n && lane < TPB) ? e : 0.f;
  z += pr;
  const float w_lane = BF16H ? pr : pr * scale_lane;
  float wgt[U], vscale[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {  // all four fetched before the first is used
    wgt[u] = __shfl(w_lane, u * TPL + j);
    vscale[u] = BF16H ? __shfl(scale_lane, u * TPL + j) : 1.f;
  }
#pragma unroll
  for (int u = 0; u < U; ++u) tile_accumulate<BF16H>(raw[u], wgt[u], vscale[u], acc);
}

// The wave's batches of a row of n tokens (DecodeArgs::turn): chunks of 2^shift
// batches, the row's waves taking the row's chunks in turn. Every wave of every
// block of the row then has the same share whatever the row's length (a short
// row of a ragged batch no longer fills its first waves and leaves the others
// idle until the block's join), and at any time a block's waves read one
// contiguous stretch, where ranges of a power of two bytes per wave moved
// through the same memory channels in step. One chunk per wave (shift 31)
// gives each wave a contiguous range of `chunk` batches. The host picks by
// the waves' share, see plan_attention.
struct Batches {
  uint32_t first, step, shift;  // chunk k starts at batch first + k * step
  uint32_t count;               // batches of this wave
  uint32_t end;                 // batches of the row: the place past the last one
  // The first tile of batch i; past this wave's last one, the first tile past the row's end.
  __device__ __forceinline__ uint32_t tile(uint32_t i) const {
    const uint32_t k = i >> shift;
    return 4 * (i < count ? first + k * step + (i - (k << shift)) : end);
  }
};
template <int TPB>
__device__ __forceinline__ Batches row_batches(const ppk::Turns& t, uint32_t n, uint32_t place, uint32_t turns) {
  const uint32_t end = n / TPB + (n % TPB != 0 ? 1u : 0u);
  if (t.shift == 31) {
    const uint32_t first = place * t.chunk;
    return Batches{first, 0, 31, end > first ? min(end - first, t.chunk) : 0u, end};
  }
  const uint32_t chunks = (end + t.chunk - 1) >> t.shift;
  uint32_t count = 0;
  if (chunks > place) {
    const uint32_t last = fast_div(chunks - place - 1, t.div);  // this wave's last chunk
    count = (last + 1) << t.shift;
    if (place + last * turns == chunks - 1) count -= (chunks << t.shift) - end;  // the row's last, cut short
  }
  return Batches{place << t.shift, turns << t.shift, t.shift, count, end};
}

// A stream of at most NBATCH batches per phase, K and V already requested:
// scores, weights and sums stay in the registers of the token groups (no LDS
// round trip between the phases). Tokens at or past the row's length n may
// hold anything: their scores are masked and their V scales zeroed.
template <int D, bool BF16H, int NBATCH, int NB>
__device__ __forceinline__ void short_attention(const u4 (&k)[NB][4], const float (&ks)[NB], const u4 (&v)[2][4],
                                                const float (&vs)[2], const Batches& bt, uint32_t n, int lane,
                                                const Query<BF16H>& q, WavePartial& out) {
  constexpr int LPT = D / 16;
  constexpr int TPL = ppk::kWave / LPT;
  constexpr int TPB = 4 * TPL;
  const int j = lane / LPT;
  PPK_CLK_AT(out.t_first, k[0][0][0]);
  uint32_t tok[NBATCH];  // the batches' first tokens
#pragma unroll
  for (int b = 0; b < NBATCH; ++b) tok[b] = bt.tile(uint32_t(b)) * TPL;
  float sc[NBATCH][4], vsc[NBATCH][4];
  float m = -INFINITY;
#pragma unroll
  for (int b = 0; b < NBATCH; ++b) {
    const float vl = tok[b] + uint32_t(lane % TPB) < n ? vs[b] : 0.f;
#pragma unroll
    for (int u = 0; u < 4; ++u) vsc[b][u] = __shfl(vl, u * TPL + j);
  }
#pragma unroll
  for (int b = 0; b < NBATCH; ++b) {
    float kscale[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) kscale[u] = __shfl(ks[b], u * TPL + j);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float x = tile_score<D, BF16H>(k[b][u], kscale[u], q);
      sc[b][u] = tok[b] + uint32_t(u * TPL + j) < n ? x : -INFINITY;
      m = fmaxf(m, sc[b][u]);
    }
  }
  m = groups_max<LPT>(m);
  float z = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) out.acc[i] = 0.f;
#pragma unroll
  for (int b = 0; b < NBATCH; ++b)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float e = __builtin_amdgcn_exp2f(sc[b][u] - m);
      const float p = tok[b] + uint32_t(u * TPL + j) < n ? e : 0.f;
      z += p;
      tile_accumulate<BF16H>(v[b][u], p, vsc[b][u], out.acc);
    }
  out.m = m;
  out.z = groups_reduce<LPT>(z, [](float x, float y) { return x + y; });
  reduce_scatter_groups<LPT, 16>(out.acc, lane);
}

// Streams this wave's batches (more than two) of a row of n tokens: phase K
// scores, phase V accumulation. A ring of NB batches (rr[b], rs[b]) keeps NB -
// 1 batches' loads in flight while one is consumed: batch i of the sequence
// K_0 .. K_{nb-1}, (padding to a whole ring), V_0 .. V_{nb-1} lives in slot
// i % NB, and each slot is refilled with batch i + NB as soon as batch i is
// used, so phase V's first batches are requested during phase K's last ones.
// The caller has issued the first NB K batches, clamped to tokens of the
// same arena row. Addresses past the end clamp to the last token and those
// tokens are masked out. Every ring load is issued unconditionally (batches
// past the end clamp to the row's last token, a cached line) so that each
// wait is for exactly the oldest batch: a conditional load leaves the
// compiler's count of loads in flight unknown on one path, and it then waits
// for all of them (vmcnt(0)), which drains the ring every batch. Only the
// arithmetic of batches past the end is skipped (uniform branches).
template <int D, bool BF16H, int NB>
__device__ __forceinline__ void ring_attention(const uint8_t* kb, const uint8_t* vb, const float* ksb,
                                               const float* vsb, const Batches& bt, uint32_t n,
                                               const Query<BF16H>& q, float* s_lds, int lane, WavePartial& out,
                                               u4 (&rr)[NB][4], float (&rs)[NB]) {
  constexpr int LPT = D / 16;
  constexpr int TPL = ppk::kWave / LPT;
  constexpr int U = 4;  // tiles per batch
  constexpr int TPB = U * TPL;
  const int j = lane / LPT;  // token within a load tile
  const int c = lane % LPT;  // 16-channel chunk
#pragma unroll
  for (int i = 0; i < 16; ++i) out.acc[i] = 0.f;
  float mloc = -INFINITY, z = 0.f;
  const uint32_t nb = bt.count;                  // K batches (and V batches)
  const uint32_t nbp = (nb + NB - 1) / NB * NB;  // rounded up to whole rings
  PPK_CLK_AT(out.t_first, rr[0][0][0]);
  for (uint32_t k0 = 0; k0 < nbp; k0 += NB) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const uint32_t i = k0 + uint32_t(b);
      if (i < nb) mloc = score_batch<D, BF16H, U>(rr[b], rs[b], bt.tile(i), n, j, c, q, s_lds + i * TPB, mloc);
      // Refill slot b with item i + NB: K batch i + NB, or V batch i + NB - nbp.
      const bool isv = i + NB >= nbp;
      load_batch<D, U>(isv ? vb : kb, isv ? vsb : ksb, bt.tile(isv ? i + NB - nbp : i + NB), n, j, lane, rr[b],
                       rs[b]);
      issue_here();  // the refill goes out before the next batch is used
    }
  }
  const float m = groups_max<LPT>(mloc);
  __builtin_amdgcn_wave_barrier();
  for (uint32_t v0 = 0; v0 < nbp; v0 += NB) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const uint32_t i = v0 + uint32_t(b);
      if (i < nb) accumulate_batch<D, BF16H, U>(rr[b], rs[b], bt.tile(i), n, j, lane, m, s_lds + i * TPB, z, out.acc);
      load_batch<D, U>(vb, vsb, bt.tile(i + NB), n, j, lane, rr[b], rs[b]);  // past the end on the last ring
      issue_here();
    }
  }
  // Each token's p was added once, by its owning lane: sum over the wave.
  out.m = m;
  out.z = wave_sum(z);
  reduce_scatter_groups<LPT, 16>(out.acc, lane);
}

// A wave's record for its block: m, z, two pad floats, y[D] (16-byte aligned)
// at `rec`; this lane holds the totals of channels ch .. ch + D/64 - 1.
template <int D, int N>
__device__ __forceinline__ void write_block_record(float* rec, int ch, int lane, float m, float z,
                                                   const float (&acc)[N]) {
#pragma unroll
  for (int e = 0; e < D / ppk::kWave; ++e) rec[4 + ch + e] = acc[e];
  rec[0] = m;  // the same in every lane, as below wherever a wave's (m, z) is stored
  rec[1] = z;
}

// Log-sum-exp combine of a block's W <= MAXW records (stride floats apart) and
// a score s0 that joins the maximum (-inf for none), by one wave: lane w takes
// record w's (m, z), the y rows of this lane's channels are requested eight
// records at a time (past W: the last record again, with weight 0). One LDS
// round trip for the weights and one for the rows; a loop over the records
// took two per record, ~0.7 us at the end of every 8-wave block. MAYBE_INF: a
// y may be infinite (a float store that holds infinities; codes times finite
// scales are not), and the places past W count as 0, since a weight of 0 alone
// would make it NaN.
template <int D, int MAXW, bool MAYBE_INF>
__device__ __forceinline__ void combine_block(const float* recs, uint32_t stride, uint32_t W, int lane, float s0,
                                              float& m, float& z, float (&y)[D / ppk::kWave]) {
  constexpr int EPL = D / ppk::kWave;
  const float* mine = recs + min(uint32_t(lane), W - 1) * stride;
  float mw = mine[0], zw = mine[1];
  float v[8][EPL];
  auto rows = [&](uint32_t w0) {
#pragma unroll
    for (int k = 0; k < 8; ++k)
#pragma unroll
      for (int e = 0; e < EPL; ++e) v[k][e] = recs[min(w0 + uint32_t(k), W - 1) * stride + 4 + lane * EPL + e];
  };
  rows(0);
  if (uint32_t(lane) >= W) {
    mw = -INFINITY;
    zw = 0.f;
  }
  m = fmaxf(wave_max(mw), s0);
  const float wt = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - m);
  z = wave_sum(wt * zw);
#pragma unroll
  for (int e = 0; e < EPL; ++e) y[e] = 0.f;
  auto add1 = [&](uint32_t w0, int k, bool there) {
    const float wk = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wt), int(w0) + k));
#pragma unroll
    for (int e = 0; e < EPL; ++e) y[e] = fmaf(wk, there ? v[k][e] : 0.f, y[e]);
  };
  auto add = [&](uint32_t w0) {
    if constexpr (MAYBE_INF) {
      // One and two records by themselves, the rest of eight without a branch
      // each (a branch per record cost blocks of eight waves 0.1-0.2 us).
      add1(w0, 0, true);
      if (W - w0 < 2) return;  // uniform
      add1(w0, 1, true);
      if (W - w0 < 3) return;
#pragma unroll
      for (int k = 2; k < 8; ++k) add1(w0, k, w0 + uint32_t(k) < W);
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) add1(w0, k, true);
    }
  };
  add(0);
  if constexpr (MAXW > 8) {
    if (W > 8) {  // uniform
      rows(8);
      add(8);
    }
  }
}

template <int D, bool BF16H, int NB, bool EARLY>
__device__ __forceinline__ void decode_body(const ppk::DecodeArgs& a) {
  constexpr int LPT = D / 16;
  constexpr int TPL = ppk::kWave / LPT;
  constexpr int U = 4;  // tiles per batch
  constexpr int EPL = D / ppk::kWave;
  static_assert(NB >= 2, "a short stream keeps its K batches in ring slots 0 and 1");
  PPK_CLK_DECL;
  PPK_CLK(0);
  extern __shared__ __attribute__((aligned(16))) float lds[];
  // The arguments on the way to the first loads, requested together (the
  // compiler would load each where it is first used, one round trip after
  // another).
  __asm__ volatile("" ::"s"(a.q), "s"(a.k), "s"(a.v), "s"(a.ks), "s"(a.vs), "s"(a.sk), "s"(a.sv), "s"(a.past),
                   "s"(a.k_new), "s"(a.v_new), "s"(a.rows), "s"(a.capacity), "s"(a.split_tokens), "s"(a.ngroups),
                   "s"(a.q_dtype), "s"(a.scratch_dtype), "s"(a.new_dtype), "s"(a.append),
                   "s"(a.row_div.mul), "s"(a.row_div.shift), "s"(a.head_div.mul), "s"(a.head_div.shift),
                   "s"(a.turn.div.mul), "s"(a.turn.div.shift), "s"(a.turn.shift), "s"(a.turn.chunk), "s"(blockDim.x));
  const int lane = threadIdx.x & 63;
  // The wave index is uniform: in a scalar register, every quantity derived
  // from it (the wave's range, its length, its batch counts) is too, and the
  // stream's loop and batch conditions become scalar branches.
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int W = blockDim.x >> 6;
  const int j = lane / LPT;
  const int c = lane % LPT;
  // Blocks are numbered group-major: consecutive blocks belong to different
  // rows, so the short blocks of short rows (with contiguous ranges, their
  // empty tail groups) spread over the CUs.
  const uint32_t group = fast_div(blockIdx.x, a.row_div);
  const uint32_t row = blockIdx.x - group * a.rows;
  const uint32_t S = a.split_tokens;

  // Everything the wave reads is requested first, in one round trip: the
  // row's length, q, the current token (wave 0 of a block that covers its
  // row), the new K/V row of the fused commit (waves 0 and 1 of group 0), all
  // as raw words, and the stream's first batches, clamped to the arena (not
  // to the row's length, which arrives with them; the tokens past it are
  // masked). The commit, the current token's score and the query's slices
  // are then formed while the batches are in flight. What bounds short rows
  // is this chain of round trips, not bytes; with the small operands widened
  // where they were loaded (each load waited for before the next), the row's
  // length and late kernel arguments read in between and the query quantised
  // by every lane group: H = 16, 512 tokens f32 at D = 64 5.88 us, now 4.43;
  // 24 layers of 2048 tokens at D = 128 204.8, now 187.8; B = 16 x 1500 at D =
  // 64 11.16, now 10.62; B = 32 x 8192 unchanged (162.2). The slot the commit
  // writes is past every wave's length, so the speculative reads of it are
  // masked. The host turns the early batches off (the kernel without EARLY) when it
  // knows many waves have no history (ragged host lengths, or waves past the
  // span): their speculative reads would be wasted bandwidth (config 4: 9 %
  // more HBM traffic than the history, 18.7 -> 18.3 us without).
  const uint32_t p_raw = a.past[fast_div(row, a.head_div) + lane_zero()];
  const bool final_out = a.ngroups == 1;
  const bool cur = final_out && wave == 0;
  const bool kw = a.append && group == 0 && wave == 0;
  const bool vw = a.append && group == 0 && wave == (W > 1 ? 1 : 0);
  const size_t first = size_t(row) * D + size_t(lane) * EPL;
  RawVec<EPL> q_raw, sk_raw, sv_raw, kn_raw, vn_raw;
  load_raw<EPL>(a.q, first, a.q_dtype, q_raw);
  if (cur) {
    load_raw<EPL>(a.sk, first, a.scratch_dtype, sk_raw);
    load_raw<EPL>(a.sv, first, a.scratch_dtype, sv_raw);
  }
  if (kw) load_raw<EPL>(a.k_new, first, a.new_dtype, kn_raw);
  if (vw) load_raw<EPL>(a.v_new, first, a.new_dtype, vn_raw);

  // This wave's batches of the row: those of the longest row the plan covers,
  // until the length is known.
  constexpr int TPB = U * TPL;
  const uint32_t place = group * W + wave, turns = a.ngroups * W;
  const uint64_t cover = uint64_t(turns) * S;
  uint32_t nspec = uint32_t(min(uint64_t(a.capacity), cover));
  const size_t tok0 = size_t(row) * a.capacity;
  const uint8_t* kb = a.k + tok0 * D + size_t(c) * 16;
  const uint8_t* vb = a.v + tok0 * D + size_t(c) * 16;
  const float* ksb = a.ks + tok0;
  const float* vsb = a.vs + tok0;
  // LDS of this wave alone: the query's exchange, then a score per token of
  // its range, at last its (m, z, pad, pad, y[D]) record.
  const uint32_t lds_stride = max(a.turn.tokens, uint32_t(D + 4));
  float* s_lds = lds + size_t(wave) * lds_stride;

  float s_cur = -INFINITY, sv[EPL];
  bool valid = false;
  uint32_t n = 0;  // the row's live history
  Batches bt{};
  uint32_t raise = 0;  // PPK_FLAG_* bits, uniform; reported at the end (a branch on the lane here, see quantize_values)
  Query<BF16H> query;
  auto settle_all = [&]() {
    settle(q_raw);
    settle(sk_raw);
    settle(sv_raw);
    settle(kn_raw);
    settle(vn_raw);
  };
  // Everything that waits for the small loads; runs with the stream's first
  // batches in flight.
  uint32_t p = 0;
  auto length_here = [&]() {
    issue_here();
    PPK_CLK(1);
    p = __builtin_amdgcn_readfirstlane(p_raw);
    PPK_CLK_AFTER(2, p_raw);
    valid = p <= a.capacity && uint64_t(p) <= cover;
    n = valid ? p : 0u;
    bt = row_batches<TPB>(a.turn, n, place, turns);
  };
  auto operands_here = [&]() {
    issue_here();
    settle_all();
    float x[EPL];
    widen<EPL>(q_raw, a.q_dtype, x);
    if (bt.count > 0) make_query<D, BF16H>(x, a.scale_log2, s_lds, lane, query);
    if (cur) {
      // Log2-domain score of the current token, which comes from the scratch copy, not the arena.
      float kv[EPL], d = 0.f;
      widen<EPL>(sk_raw, a.scratch_dtype, kv);
      widen<EPL>(sv_raw, a.scratch_dtype, sv);
#pragma unroll
      for (int e = 0; e < EPL; ++e) d = fmaf(x[e], kv[e], d);
      s_cur = wave_sum(d) * a.scale_log2;
    }
    // A length within the caller's span that the plan does not cover: the plan
    // was sized from a stale host copy of the lengths (the row gives NaN).
    if (kw && p <= a.capacity && p <= a.span && uint64_t(p) > cover) raise |= 4u;
    if (kw || vw) {
      if (p >= a.capacity) {
        raise |= 2u;
      } else {
        const size_t slot = size_t(row) * a.capacity + p;
        float t[EPL];
        if (kw) {
          widen<EPL>(kn_raw, a.new_dtype, t);
          if (__any(quantize_values<D>(t, a.k + slot * D, a.ks + slot, lane))) raise |= 1u;
        }
        if (vw) {
          widen<EPL>(vn_raw, a.new_dtype, t);
          if (__any(quantize_values<D>(t, a.v + slot * D, a.vs + slot, lane))) raise |= 1u;
        }
      }
    }
  };

  WavePartial part;
  part.m = -INFINITY;
  part.z = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) part.acc[i] = 0.f;
  u4 rr[NB][U], va[2][U];
  float rs[NB], vsa[2];
  auto load_k = [&](int b, const Batches& of, uint32_t limit) {
    load_batch<D, U>(kb, ksb, of.tile(uint32_t(b)), limit, j, lane, rr[b], rs[b]);
  };
  auto load_v = [&](int b, const Batches& of, uint32_t limit) {
    load_batch<D, U>(vb, vsb, of.tile(uint32_t(b)), limit, j, lane, va[b], vsa[b]);
  };
  // The batches to request: the covered row's, or, without speculation, the
  // row's own (then its length is waited for here; the operands that came with
  // it wait until the batches are on their way). Either way a wave of one or
  // two batches requests K and V together, and does no arithmetic on a batch
  // that is not there: with ragged host lengths and the bf16 history, which
  // that arithmetic bounds, one-batch waves took 8.4 us where they did both
  // (64 rows of 181..362 tokens at D = 64), now 6.0.
  if constexpr (!EARLY) {
    length_here();
    nspec = n;
  }
  const Batches early = row_batches<TPB>(a.turn, nspec, place, turns);
  auto prologue = [&]() {
    if constexpr (EARLY) length_here();
    operands_here();
  };
  // The paths differ in what is in flight when the prologue runs; each runs
  // its own copy of it, so that its waits count that path's loads only.
  if (early.count == 1) {
    // At most one batch: K and V at once, one memory round trip in all.
    load_k(0, early, nspec);
    load_v(0, early, nspec);
    prologue();
    if (bt.count > 0) short_attention<D, BF16H, 1>(rr, rs, va, vsa, early, n, lane, query, part);
  } else if (early.count == 2) {
    load_k(0, early, nspec);
    load_k(1, early, nspec);
    load_v(0, early, nspec);
    load_v(1, early, nspec);
    prologue();
    if (bt.count == 2) short_attention<D, BF16H, 2>(rr, rs, va, vsa, early, n, lane, query, part);
    else if (bt.count == 1) short_attention<D, BF16H, 1>(rr, rs, va, vsa, early, n, lane, query, part);
  } else if (early.count == 0) {
    prologue();
  } else {
#pragma unroll
    for (int b = 0; b < NB; ++b) load_k(b, early, nspec);
    prologue();
    if (bt.count > 2) {
      settle_all();  // long done, but not on every edge the compiler gives this block
      ring_attention<D, BF16H, NB>(kb, vb, ksb, vsb, bt, n, query, s_lds, lane, part, rr, rs);
    } else if (bt.count == 2) {
      load_v(0, bt, n);
      load_v(1, bt, n);
      short_attention<D, BF16H, 2>(rr, rs, va, vsa, bt, n, lane, query, part);
    } else if (bt.count == 1) {
      load_v(0, bt, n);
      short_attention<D, BF16H, 1>(rr, rs, va, vsa, bt, n, lane, query, part);
    }
  }
  PPK_CLK(4);
#ifdef PPK_WAVE_CLOCK
  clk_[3] = part.t_first;
#endif

  // Combine the block's waves through LDS: each wave's record replaces its
  // scores (its own LDS, so no barrier is needed before).
  write_block_record<D>(s_lds, c * 16 + scatter_base<LPT, 16>(lane), lane, part.m, part.z, part.acc);
  raise_flags(a.flags, raise);
  __syncthreads();
  PPK_CLK(5);
  if (wave != 0) {
    PPK_CLK_RECORD(a, ppk::kWaveClockDecode, blockIdx.x, uint32_t(wave));
    return;
  }

  float m, y[EPL], zsum;
  combine_block<D, 8, false>(lds, lds_stride, uint32_t(W), lane, s_cur, m, zsum, y);
  if (final_out) {
    const float wc = __builtin_amdgcn_exp2f(s_cur - m);
    zsum += wc;
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      const float o = valid ? fmaf(wc, sv[e], y[e]) / zsum : __builtin_nanf("");
      store_elem(a.out, size_t(row) * D + size_t(lane) * EPL + e, a.out_dtype, o);
    }
  } else {
    const size_t rec = size_t(row) * a.ngroups + group;
#pragma unroll
    for (int e = 0; e < EPL; ++e) a.part_y[rec * D + size_t(lane) * EPL + e] = y[e];
    a.part_mz[rec * 2] = m;
    a.part_mz[rec * 2 + 1] = zsum;
  }
  PPK_CLK(6);
  PPK_CLK_RECORD(a, ppk::kWaveClockDecode, blockIdx.x, 0u);
}

// ---------------------------------------------------------------------------
// Kernel 2b: merge. One wave per row: scores the current (unquantised) token,
// combines it with every split's (m, z, y) by log-sum-exp weights, divides.
// Rows with past > capacity (or beyond the launched coverage) give NaN.
// ---------------------------------------------------------------------------
// Log-sum-exp combine of one row's `nsplits` partial records, one wave: the
// combined max m, the sum z of 2^(m_s - m) z_s, and y for this lane's D/64
// channels, sum_s 2^(m_s - m) y_s, added in split order. Lane s loads record
// s's (m, z); the y rows load eight splits at a time with all eight loads
// issued before the first use, so the chain costs one memory round trip per
// eight splits instead of one per split. request() issues whatever else the
// caller loads (as raw words: nothing in it may wait), score() then returns
// the extra score that joins the max (-inf for none).
template <int D, class Request, class Score>
__device__ __forceinline__ void combine_records(const float* mz, const float* py, uint32_t nsplits, int lane,
                                                Request request, Score score, float& m, float& z,
                                                float (&y)[D / ppk::kWave]) {
  constexpr int EPL = D / ppk::kWave;
  // Everything that does not depend on the max is requested first, in one
  // round trip, in the order of use: the (m, z) pairs of the first 64 splits
  // (kept in registers for the weights), the caller's operands, the y rows of
  // the first sixteen splits.
  const uint32_t s_first = min(uint32_t(lane), nsplits - 1);
  float m_first = mz[2 * s_first], z_first = mz[2 * s_first + 1];
  request();
  float first[16][EPL];
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const uint32_t si = min(uint32_t(k), nsplits - 1);  // clamp: always a loaded record
#pragma unroll
    for (int e = 0; e < EPL; ++e) first[k][e] = py[size_t(si) * D + size_t(lane) * EPL + e];
  }
  if (uint32_t(lane) >= nsplits) {
    m_first = -INFINITY;
    z_first = 0.f;
  }
  float mm = m_first;
  for (uint32_t s = lane + ppk::kWave; s < nsplits; s += ppk::kWave) mm = fmaxf(mm, mz[2 * s]);
  m = fmaxf(wave_max(mm), score());
  z = 0.f;
#pragma unroll
  for (int e = 0; e < EPL; ++e) y[e] = 0.f;
  for (uint32_t s0 = 0; s0 < nsplits; s0 += ppk::kWave) {
    const uint32_t s = s0 + uint32_t(lane);
    float ms = m_first, zs = z_first;
    if (s0 != 0) {
      ms = s < nsplits ? mz[2 * s] : -INFINITY;
      zs = s < nsplits ? mz[2 * s + 1] : 0.f;
    }
    const float w = ms == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms - m);
    z = fmaf(w, zs, z);
    const uint32_t cnt = min(uint32_t(ppk::kWave), nsplits - s0);
    for (uint32_t i = 0; i < cnt; i += 8) {
      float v[8][EPL];
      if (s0 == 0 && i < 16) {
#pragma unroll
        for (int k = 0; k < 8; ++k)
#pragma unroll
          for (int e = 0; e < EPL; ++e) v[k][e] = i == 0 ? first[k][e] : first[8 + k][e];
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const uint32_t si = s0 + min(i + uint32_t(k), cnt - 1);  // clamp: always a loaded record
#pragma unroll
          for (int e = 0; e < EPL; ++e) v[k][e] = py[size_t(si) * D + size_t(lane) * EPL + e];
        }
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        // Record i + k's weight sits in that lane (a uniform index, 0 past the
        // last record): one readlane, no LDS. Past it the y row counts as 0
        // too (0 times an infinite y would be NaN); selected, not branched: a
        // branch per record would hold the next eight records' loads back
        // (36 records, 8 rows of D = 128: 10.4 us against 8.9).
        const bool live = i + uint32_t(k) < cnt;
        const float wk = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), int(i) + k));
#pragma unroll
        for (int e = 0; e < EPL; ++e) y[e] = fmaf(wk, live ? v[k][e] : 0.f, y[e]);
      }
    }
  }
  z = wave_sum(z);
}

// The current token of an int8 merge: q, sk and sv of one row as raw words,
// then the log2-domain score q . sk (sv widened beside it).
template <int D>
struct MergeCurrent {
  static constexpr int EPL = D / ppk::kWave;
  RawVec<EPL> q, sk, sv_raw;
  float sv[EPL], s_cur;
  __device__ __forceinline__ void request(const ppk::MergeArgs& a, size_t base) {
    load_raw<EPL>(a.q, base, a.q_dtype, q);
    load_raw<EPL>(a.sk, base, a.scratch_dtype, sk);
    load_raw<EPL>(a.sv, base, a.scratch_dtype, sv_raw);
  }
  __device__ __forceinline__ float score(const ppk::MergeArgs& a) {
    float qv[EPL], kv[EPL], d = 0.f;
    widen<EPL>(q, a.q_dtype, qv);
    widen<EPL>(sk, a.scratch_dtype, kv);
    widen<EPL>(sv_raw, a.scratch_dtype, sv);
#pragma unroll
    for (int e = 0; e < EPL; ++e) d = fmaf(qv[e], kv[e], d);
    s_cur = wave_sum(d) * a.scale_log2;
    return s_cur;
  }
};

template <int D>
__device__ __forceinline__ void attn_merge_body(const ppk::MergeArgs& a) {
  constexpr int EPL = D / ppk::kWave;
  PPK_CLK_DECL;
  PPK_CLK(0);
  // Every argument on the way to the loads, requested together.
  __asm__ volatile("" ::"s"(a.q), "s"(a.sk), "s"(a.sv), "s"(a.past), "s"(a.part_y), "s"(a.part_mz), "s"(a.out),
                   "s"(a.capacity), "s"(a.split_tokens), "s"(a.nsplits), "s"(a.q_dtype), "s"(a.scratch_dtype),
                   "s"(a.out_dtype), "s"(a.scale_log2), "s"(a.head_div.mul), "s"(a.head_div.shift));
  const int lane = threadIdx.x;
  const uint32_t row = blockIdx.x;
  const size_t base = size_t(row) * D + size_t(lane) * EPL;
  // The row's length travels with the records (as a vector load, see lane_zero).
  MergeCurrent<D> cur;
  uint32_t p_raw = 0;
  auto request = [&]() {
    cur.request(a, base);
    p_raw = a.past[fast_div(row, a.head_div) + lane_zero()];
  };
  float m, zsum, y[EPL];
  combine_records<D>(a.part_mz + size_t(row) * a.nsplits * 2, a.part_y + size_t(row) * a.nsplits * D, a.nsplits,
                     lane, request, [&]() { return cur.score(a); }, m, zsum, y);
  PPK_CLK_AFTER(1, y[0]);
  const uint32_t p = __builtin_amdgcn_readfirstlane(p_raw);
  const bool valid = p <= a.capacity && uint64_t(p) <= uint64_t(a.nsplits) * a.split_tokens;
  const float wc = __builtin_amdgcn_exp2f(cur.s_cur - m);
  zsum += wc;
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    const float o = valid ? fmaf(wc, cur.sv[e], y[e]) / zsum : __builtin_nanf("");
    store_elem(a.out, base + e, a.out_dtype, o);
  }
  PPK_CLK(2);
  PPK_CLK_RECORD(a, ppk::kWaveClockMerge, blockIdx.x, 0u);
}

// ---------------------------------------------------------------------------
// Kernel 2c: decode attention over a balanced work list (ragged batches). The
// per-row plan above gives every row the same number of blocks, sized for
// the longest row, so in a ragged batch the CUs holding long rows run on
// while the others idle. Here the host, from its copy of the lengths, cuts
// the live history into units of at most Q tokens, each inside one row (row
// r of len_r tokens is max(1, ceil(len_r / Q)) units, Q = max(ceil(T /
// (waves - rows)), 64) for T live tokens in all, so the units fit the
// waves: sum <= T / Q + rows <= waves), and wave i takes unit i: no unit
// exceeds the mean share by more than waves / (waves - rows). The table
// travels in the kernel arguments, so every wave issues all of its loads at
// once, the device lengths among them (they are compared with the table
// before anything is written). A row of one unit is finished by its wave
// (current token included); the units of a longer row leave log-sum-exp
// records that the balanced merge kernel joins.
//
// A unit is streamed as (K, V) pairs of batches through a window of NP pairs
// in registers with an online softmax (running max per token group, one
// rescale per batch that raises it). What bounds a unit is its waves' latency
// more than its bytes: the table is searched with two dependent scalar loads,
// every small operand travels as raw words beside the window's first pairs,
// and the window's refills are unconditional (past the end they read the
// unit's last token again), so that each wait is for the oldest pair only.
// Against a per-lane table search, loads widened one after another and
// conditional refills (H = 16, host lengths): B = 8 of 256..4096 at D = 128
// 24.5 -> 21.1 us, at D = 64 16.0 -> 14.1; B = 24 of 200..3000 at D = 64 25.0
// -> 20.5; B = 32 of 256..4096 at D = 128 60.9 -> 56.5. Three or four pairs
// were 1 and 5 % slower.
// ---------------------------------------------------------------------------
// One (K, V) batch pair of a unit under the online softmax. Token group j
// (the LPT lanes holding one token of each tile) keeps its own running max m,
// sum z and 16-channel accumulator: the batch's four scores are formed, the
// state is rescaled to the new max if any group of the wave has one, then
// each tile's V codes are added with weight 2^(s - m) * vscale.
template <int D, bool BF16H>
__device__ __forceinline__ void online_pair(const u4 (&kraw)[4], const u4 (&vraw)[4], float ks_lane, float vs_lane,
                                            uint32_t t0, uint32_t n, int j, const Query<BF16H>& q, float& m, float& z,
                                            float (&acc)[16]) {
  constexpr int LPT = D / 16;
  constexpr int TPL = ppk::kWave / LPT;
  float s[4], kscale[4], vscale[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) kscale[u] = __shfl(ks_lane, u * TPL + j);
#pragma unroll
  for (int u = 0; u < 4; ++u) vscale[u] = __shfl(vs_lane, u * TPL + j);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const float sc = tile_score<D, BF16H>(kraw[u], kscale[u], q);
    s[u] = (t0 + u) * TPL + j < n ? sc : -INFINITY;
  }
  const float mb = fmaxf(fmaxf(m, fmaxf(s[0], s[1])), fmaxf(s[2], s[3]));
  if (__any(mb > m)) {  // a new max somewhere (always on a group's first token)
    const float f = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mb);
    z *= f;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] *= f;
    m = mb;
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const float p = s[u] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(s[u] - m);
    z += p;
    tile_accumulate<BF16H>(vraw[u], p, vscale[u], acc);
  }
}

// Streams tokens [0, n) (n >= 1) of the given K / V / scale ranges through the
// window of NP (K, V) pairs; returns the wave's partial as short_attention
// does. early() runs once the window's first loads are in flight and leaves
// the query.
template <int D, bool BF16H, int NP, class Early>
__device__ __forceinline__ void wave_attention_window(const uint8_t* kb, const uint8_t* vb, const float* ksb,
                                                      const float* vsb, uint32_t n, const Query<BF16H>& q, int lane,
                                                      WavePartial& out, Early early) {
  constexpr int LPT = D / 16;
  constexpr int TPL = ppk::kWave / LPT;
  constexpr int U = 4;
  const int j = lane / LPT;
  const uint32_t nb = (n + U * TPL - 1) / (U * TPL);  // batches per phase
  u4 kr[NP][U], vr[NP][U];
  float ksl[NP], vsl[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    load_batch<D, U>(kb, ksb, uint32_t(p) * U, n, j, lane, kr[p], ksl[p]);
    load_batch<D, U>(vb, vsb, uint32_t(p) * U, n, j, lane, vr[p], vsl[p]);
  }
  early();
  float m = -INFINITY, z = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) out.acc[i] = 0.f;
  for (uint32_t b0 = 0; b0 < nb; b0 += NP) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const uint32_t bi = b0 + uint32_t(p);
      // Scales of tokens at or past n are never used (their scores are -inf).
      if (bi < nb) online_pair<D, BF16H>(kr[p], vr[p], ksl[p], vsl[p], bi * U, n, j, q, m, z, out.acc);
      load_batch<D, U>(kb, ksb, (bi + NP) * U, n, j, lane, kr[p], ksl[p]);
      load_batch<D, U>(vb, vsb, (bi + NP) * U, n, j, lane, vr[p], vsl[p]);
      issue_here();
    }
  }
  // Join the token groups: common max, then sums across groups.
  const float mm = groups_max<LPT>(m);
  const float w = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mm);
  z *= w;
#pragma unroll
  for (int i = 0; i < 16; ++i) out.acc[i] *= w;
  out.m = mm;
  out.z = groups_reduce<LPT>(z, [](float a, float b) { return a + b; });
  reduce_scatter_groups<LPT, 16>(out.acc, lane);
}

// The table's entry of unit `unit` (< units_total, uniform): the last
// sequence whose first unit is at most `unit`. Counting the group heads and
// then the group's eight first units costs two dependent scalar loads.
struct FlatUnit {
  uint32_t b, past, len, units;
  uint32_t head, slot;  // the unit's head, its place within the head's row
};
__device__ __forceinline__ FlatUnit flat_unit(const ppk::FlatTable& t, uint32_t unit) {
  uint32_t g = 0;
#pragma unroll
  for (int i = 1; i < ppk::kFlatMaxBatch / 8; ++i) g += t.pivot[i] <= unit ? 1u : 0u;
  uint32_t first = t.first[8 * g], b = 8 * g;
#pragma unroll
  for (int i = 1; i < 8; ++i) {
    const uint32_t f = t.first[8 * g + i];
    if (f <= unit) {
      first = f;
      ++b;
    }
  }
  const ppk::FlatSequence s = t.seq[b];
  FlatUnit u;
  u.b = b;
  u.past = s.past;
  u.len = s.len;
  u.units = s.units & 0xffffffu;
  u.head = fast_div(unit - first, ppk::FastDiv{s.div_mul, s.units >> 24});
  u.slot = unit - first - u.head * u.units;
  return u;
}

template <int D, bool BF16H>
__device__ __forceinline__ void decode_flat_body(const ppk::DecodeFlatArgs& fa) {
  const ppk::DecodeArgs& a = fa.d;
  const ppk::FlatTable& t = fa.t;
  constexpr int LPT = D / 16;
  constexpr int EPL = D / ppk::kWave;
  __shared__ u4 s_query[8][D / 4];  // per wave: the query's exchange
  // The arguments on the way to the first loads, requested together.
  __asm__ volatile("" ::"s"(a.q), "s"(a.k), "s"(a.v), "s"(a.ks), "s"(a.vs), "s"(a.sk), "s"(a.sv), "s"(a.past),
                   "s"(a.k_new), "s"(a.v_new), "s"(a.rows), "s"(a.heads), "s"(a.capacity), "s"(a.q_dtype),
                   "s"(a.scratch_dtype), "s"(a.new_dtype), "s"(a.append), "s"(a.head_div.mul), "s"(a.head_div.shift),
                   "s"(t.share), "s"(t.units_total), "s"(t.pivot[1]), "s"(t.pivot[2]), "s"(t.pivot[3]),
                   "s"(t.pivot[4]), "s"(blockDim.x));
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform, as everything derived from it
  const uint32_t W = blockDim.x >> 6;
  const uint32_t wid = blockIdx.x * W + wave;
  const int c = lane % LPT;

  // Append job (a decode step): wave q < 2 rows quantises tensor q & 1 of
  // row q >> 1 into slot past[b] (the device value) of the arenas. Its loads
  // are issued first, beside everything else this wave reads.
  const bool append = a.append && wid < 2 * a.rows;  // the host keeps waves >= 2 rows
  const uint32_t arow = wid >> 1;
  RawVec<EPL> new_raw;
  uint32_t ap_raw = 0;
  if (append) {
    ap_raw = a.past[fast_div(arow, a.head_div) + lane_zero()];
    load_raw<EPL>((wid & 1u) ? a.v_new : a.k_new, size_t(arow) * D + size_t(lane) * EPL, a.new_dtype, new_raw);
  }
  uint32_t raise = 0;  // PPK_FLAG_* bits, uniform; reported at the end
  auto commit = [&]() {
    if (!append) return;
    const uint32_t ap = __builtin_amdgcn_readfirstlane(ap_raw);
    if (ap >= a.capacity) {
      raise |= 2u;
    } else {
      const size_t dst = size_t(arow) * a.capacity + ap;
      const bool value = (wid & 1u) != 0;
      float x[EPL];
      widen<EPL>(new_raw, a.new_dtype, x);
      if (__any(quantize_values<D>(x, (value ? a.v : a.k) + dst * D, (value ? a.vs : a.ks) + dst, lane))) raise |= 1u;
    }
  };
  auto report = [&]() { raise_flags(a.flags, raise); };
  if (wid >= t.units_total) {
    commit();
    report();
    return;
  }
  const FlatUnit u = flat_unit(t, wid);
  const uint32_t row = u.b * a.heads + u.head;
  const uint32_t t0 = u.slot * t.share;
  const uint32_t n = u.len > t0 ? min(t.share, u.len - t0) : 0u;
  const int ch = c * 16 + scatter_base<LPT, 16>(lane);  // this lane's output channels: ch .. ch + EPL - 1
  const bool whole = u.units == 1;                      // the whole row: its current token too
  const uint32_t p_raw = a.past[u.b + lane_zero()];
  RawVec<EPL> q_raw, sk_raw, sv_raw;
  load_raw<EPL>(a.q, size_t(row) * D + size_t(lane) * EPL, a.q_dtype, q_raw);
  if (whole) {
    load_raw<EPL>(a.sk, size_t(row) * D + size_t(lane) * EPL, a.scratch_dtype, sk_raw);
    load_raw<EPL>(a.sv, size_t(row) * D + size_t(ch), a.scratch_dtype, sv_raw);
  }
  WavePartial part;
  part.m = -INFINITY;
  part.z = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) part.acc[i] = 0.f;
  float s_cur = -INFINITY;
  if (n > 0) {
    Query<BF16H> query;
    const size_t tok0 = size_t(row) * a.capacity + t0;
    auto early = [&]() {  // with the unit's first loads in flight
      issue_here();
      settle(new_raw);
      settle(sk_raw);
      settle(sv_raw);
      float x[EPL];
      widen<EPL>(q_raw, a.q_dtype, x);
      make_query<D, BF16H>(x, a.scale_log2, s_query[wave], lane, query);
      if (whole) {
        float kv[EPL], d = 0.f;
        widen<EPL>(sk_raw, a.scratch_dtype, kv);
#pragma unroll
        for (int e = 0; e < EPL; ++e) d = fmaf(x[e], kv[e], d);
        s_cur = wave_sum(d) * a.scale_log2;
      }
      commit();
    };
    wave_attention_window<D, BF16H, 2>(a.k + tok0 * D + size_t(c) * 16, a.v + tok0 * D + size_t(c) * 16,
                                       a.ks + tok0, a.vs + tok0, n, query, lane, part, early);
  } else {
    commit();
  }
  // The row is valid when the host's length is in range and the device agrees.
  const bool host_ok = u.past <= a.capacity && u.past <= a.span;
  const bool fresh = __builtin_amdgcn_readfirstlane(p_raw) == u.past;
  if (!fresh) raise |= 4u;
  report();
  if (whole) {
    const bool valid = fresh && host_ok;
    const float m = fmaxf(part.m, s_cur);
    const float wp = n > 0 ? __builtin_amdgcn_exp2f(part.m - m) : 0.f;
    const float wc = n > 0 ? __builtin_amdgcn_exp2f(s_cur - m) : 1.f;
    const float zsum = n > 0 ? fmaf(wp, part.z, wc) : 1.f;
    float sv[EPL];
    widen<EPL>(sv_raw, a.scratch_dtype, sv);
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      const float o = valid ? fmaf(wc, sv[e], n > 0 ? wp * part.acc[e] : 0.f) / zsum : __builtin_nanf("");
      store_elem(a.out, size_t(row) * D + size_t(ch + e), a.out_dtype, o);
    }
  } else if (u.slot < a.ngroups) {  // always, by the host's count of slots
    const size_t rec = size_t(row) * a.ngroups + u.slot;
#pragma unroll
    for (int e = 0; e < EPL; ++e) a.part_y[rec * D + size_t(ch + e)] = part.acc[e];
    a.part_mz[rec * 2] = part.m;
    a.part_mz[rec * 2 + 1] = part.z;
  }
}

// Balanced merge: one wave per row of two or more units (the others were
// written by the decode launch): joins the row's records and the current
// token, or gives NaN when the row is invalid or the device length differs
// from the table's.
template <int D>
__device__ __forceinline__ void attn_merge_flat_body(const ppk::MergeFlatArgs& fa) {
  const ppk::MergeArgs& a = fa.m;
  const ppk::FlatTable& t = fa.t;
  constexpr int EPL = D / ppk::kWave;
  __asm__ volatile("" ::"s"(a.q), "s"(a.sk), "s"(a.sv), "s"(a.past), "s"(a.part_y), "s"(a.part_mz), "s"(a.out),
                   "s"(a.capacity), "s"(a.nsplits), "s"(a.q_dtype), "s"(a.scratch_dtype), "s"(a.out_dtype),
                   "s"(a.scale_log2), "s"(a.head_div.mul), "s"(a.head_div.shift));
  const int lane = threadIdx.x;
  const uint32_t row = blockIdx.x;
  const uint32_t b = fast_div(row, a.head_div);
  const ppk::FlatSequence seq = t.seq[b];
  const uint32_t units = seq.units & 0xffffffu;
  if (units < 2) return;  // uniform per wave
  const uint32_t phost = seq.past;
  const size_t base = size_t(row) * D + size_t(lane) * EPL;
  MergeCurrent<D> cur;
  uint32_t p_raw = 0;
  auto request = [&]() {
    cur.request(a, base);
    p_raw = a.past[b + lane_zero()];
  };
  float m, zsum, y[EPL];
  combine_records<D>(a.part_mz + size_t(row) * a.nsplits * 2, a.part_y + size_t(row) * a.nsplits * D,
                     min(units, a.nsplits), lane, request, [&]() { return cur.score(a); }, m, zsum, y);
  const uint32_t pdev = __builtin_amdgcn_readfirstlane(p_raw);
  const bool valid = pdev == phost && phost <= a.capacity && phost <= a.span;
  const float wc = __builtin_amdgcn_exp2f(cur.s_cur - m);
  zsum += wc;
#pragma unroll
  for (int e = 0; e < EPL; ++e)
    store_elem(a.out, base + e, a.out_dtype, valid ? fmaf(wc, cur.sv[e], y[e]) / zsum : __builtin_nanf(""));
}

// ---------------------------------------------------------------------------
// Float-KV decode attention: the reference's non-int8 decode path
// (app/src/model/decode_attention.hip:9-66, fused_attention.rs:8-30) on the
// block geometry of the int8 kernel. K/V are stored bf16 or f32; row r attends
// its first n = lengths ? lengths[r / heads] : size tokens (the current token
// is already in the store) and gives NaN if n == 0 or n > span (max_length,
// or size).
//
// Lane layout: a lane holds one 16-byte chunk of a token, EPC = 8 (bf16) or 4
// (f32) channels; LPT = D / EPC lanes share a token and a wave-wide dwordx4
// load moves TPL = 64 / LPT whole tokens (1 KiB). Scores go to LDS in the
// log2 domain, exactly as in the int8 kernel, and phase V weights each token's
// chunk by p = 2^(s - m) broadcast from the lane that owns the token.
// ---------------------------------------------------------------------------
template <int LPT>
__device__ __forceinline__ float token_sum(float x) {
  if constexpr (LPT <= 16) {
    return group_sum<LPT>(x);
  } else {
    x = group_sum<16>(x);
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    if constexpr (LPT >= 64) {
      r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
      x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    return x;
  }
}

template <bool BF16KV>
__device__ __forceinline__ void unpack_chunk(const u4& r, float (&x)[BF16KV ? 8 : 4]) {
  if constexpr (BF16KV) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      x[2 * w] = __uint_as_float(r[w] << 16);
      x[2 * w + 1] = __uint_as_float(r[w] & 0xffff0000u);
    }
  } else {
#pragma unroll
    for (int w = 0; w < 4; ++w) x[w] = __uint_as_float(r[w]);
  }
}

template <int D, bool BF16KV>
struct FloatGeom {
  static constexpr int kElemBytes = BF16KV ? 2 : 4;
  static constexpr int kEpc = ppk::kLaneBytes / kElemBytes;  // channels per lane
  static constexpr int kLpt = D / kEpc;                       // lanes per token
  static constexpr int kTpl = ppk::kWave / kLpt;              // tokens per wave load
  static constexpr int kTokenBytes = D * kElemBytes;
  static_assert(kLpt >= 4 && kLpt <= ppk::kWave, "token must span 4..64 lanes");
};

template <int D, bool BF16KV, int U>
__device__ __forceinline__ void load_fbatch(const char* base, uint32_t t0, uint32_t n, int j, u4 (&raw)[U]) {
  using G = FloatGeom<D, BF16KV>;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t tc = min((t0 + u) * G::kTpl + j, n - 1);  // clamp: always in bounds
    raw[u] = __builtin_nontemporal_load(reinterpret_cast<const u4*>(base + size_t(tc) * G::kTokenBytes));
  }
}

template <int D, bool BF16KV, int U>
__device__ __forceinline__ float fscore_batch(const u4 (&raw)[U], uint32_t t0, uint32_t n, int j, int c,
                                              const float (&qr)[FloatGeom<D, BF16KV>::kEpc], float sl2,
                                              float* s_batch, float mloc) {
  using G = FloatGeom<D, BF16KV>;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t tok = (t0 + u) * G::kTpl + j;
    float x[G::kEpc];
    unpack_chunk<BF16KV>(raw[u], x);
    float d = 0.f;
#pragma unroll
    for (int e = 0; e < G::kEpc; ++e) d = fmaf(qr[e], x[e], d);
    float sc = token_sum<G::kLpt>(d) * sl2;
    sc = tok < n ? sc : -INFINITY;
    mloc = fmaxf(mloc, sc);
    if (c == 0) s_batch[u * G::kTpl + j] = sc;
  }
  return mloc;
}

template <int D, bool BF16KV, int U>
__device__ __forceinline__ void faccumulate_batch(const u4 (&raw)[U], uint32_t t0, uint32_t n, int j, int lane,
                                                  float m, const float* s_batch, float& z,
                                                  float (&acc)[FloatGeom<D, BF16KV>::kEpc]) {
  using G = FloatGeom<D, BF16KV>;
  constexpr int TPB = U * G::kTpl;  // tokens per batch (<= 64)
  static_assert(TPB <= ppk::kWave, "one token per lane per batch");
  const uint32_t tl = t0 * G::kTpl + uint32_t(lane % TPB);
  const float e = __builtin_amdgcn_exp2f(s_batch[lane % TPB] - m);
  const float pr = (tl < n && lane < TPB) ? e : 0.f;
  z += pr;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const float wgt = __shfl(pr, u * G::kTpl + j);
    float x[G::kEpc];
    unpack_chunk<BF16KV>(raw[u], x);
#pragma unroll
    for (int e = 0; e < G::kEpc; ++e) acc[e] = fmaf(wgt, x[e], acc[e]);
  }
}

template <int D, bool BF16KV>
struct FloatWavePartial {
  float m, z;
  // While streaming: this lane's chunk; at the end the wave's totals of channels
  // c * kEpc + scatter_base<kLpt, kEpc>(lane) + e in acc[e], e < D / 64.
  float acc[FloatGeom<D, BF16KV>::kEpc];
};

// One wave streams n tokens of a row from `begin`: phase K scores into LDS,
// phase V accumulation; A/B batches ping-pong, and the last phase-K iteration
// already fetches the first V batches. early() leaves the query chunk in qr,
// with the first two batches in flight.
template <int D, bool BF16KV, class Early>
__device__ __forceinline__ void fwave_attention(const ppk::FloatDecodeArgs& a, uint32_t row, uint32_t begin,
                                                uint32_t n, const float (&qr)[FloatGeom<D, BF16KV>::kEpc],
                                                float* s_lds, int lane, FloatWavePartial<D, BF16KV>& out,
                                                Early early) {
  using G = FloatGeom<D, BF16KV>;
  constexpr int U = 4;
  constexpr int TPB = U * G::kTpl;
  const int j = lane / G::kLpt;
  const int c = lane % G::kLpt;
  out.m = -INFINITY;
  out.z = 0.f;
#pragma unroll
  for (int i = 0; i < G::kEpc; ++i) out.acc[i] = 0.f;
  const uint32_t nb = (n + TPB - 1) / TPB;
  if (nb == 0) {  // uniform per wave
    early();
    return;
  }

  const char* kb = static_cast<const char*>(a.k) +
                   (size_t(row) * a.k_stride + size_t(begin) * D) * G::kElemBytes + size_t(c) * ppk::kLaneBytes;
  const char* vb = static_cast<const char*>(a.v) +
                   (size_t(row) * a.v_stride + size_t(begin) * D) * G::kElemBytes + size_t(c) * ppk::kLaneBytes;
  const float sl2 = a.scale_log2;
  // Each wave takes its batches in a rotated order: it starts at batch rot of
  // its nb batches and wraps, and phase V follows the same order. Waves that
  // start at the same offset of rows a power of two apart (a store of 4096 or
  // 8192 tokens) otherwise move through the same HBM channels in step. rot is
  // a multiplicative hash of the wave's global index scaled into [0, nb) (no
  // division), uniform per wave, so the remapping is scalar work. Scores land
  // in LDS by token and phase V reads them by token, so only the order of
  // phase V's fp32 sums changes. Logical batches past nb (the padding to
  // whole ping-pong pairs) keep their place past the end, where loads clamp
  // and tokens are masked. Measured with bf16 stores of exactly the sequence
  // length (power-of-two strides): B=8 x 4096 D=64 30.0 -> 21.7 us, B=4 x
  // 4096 D=128 26.3 -> 21.7 us, B=16 x 1024 D=128 23.3 -> 20.1 us; B=32 x
  // 8192 D=128 310.5 -> 309.0 us. It costs where a few long rows stream one
  // wave per CU: 4 x 8192 + 28 x 512 tokens on the per-row plan 112.2 ->
  // 115.7 us (the balanced plan, which host lengths select, does not rotate).
  // Contiguous at any share: taking a row's batches in turn, as the int8 kernel
  // does, gained up to 3 % on uniform rows of a power of two tokens (B=32 x
  // 8192 D=128 309.9 -> 301.1 us) and lost up to 12 % on ragged ones (B=32 of
  // 256..8192 175.2 -> 181.8); over 544 shapes it was 2-3 % slower.
  const uint32_t wave_id = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
  const uint32_t rot = ((wave_id * 0x9E37u & 0xFFFFu) * nb) >> 16;
  // Logical batch b -> its place in the range; past the end: past the range.
  auto place = [&](uint32_t b) { return b < nb ? (b + rot >= nb ? b + rot - nb : b + rot) : b; };

  u4 ra[U], rb[U];
  float mloc = -INFINITY;
  auto score = [&](const u4 (&r)[U], uint32_t b) {
    if (b < nb)
      mloc = fscore_batch<D, BF16KV, U>(r, place(b) * U, n, j, c, qr, sl2, s_lds + place(b) * TPB, mloc);
  };
  // Both first batches go out before anything waits for the query: with the
  // second behind that wait, rows of a few batches paid up to one more memory
  // round trip (captured sequences, us: 8 rows x 1145 tokens at D = 128 7.58 /
  // 7.43, step 7.93 / 7.70; 256 rows of up to 28 at D = 128 4.34 / 4.25).
  load_fbatch<D, BF16KV, U>(kb, place(0) * U, n, j, ra);
  load_fbatch<D, BF16KV, U>(kb, place(1) * U, n, j, rb);
  issue_here();
  early();
  for (uint32_t b = 0; b < nb; b += 2) {
    const bool last = b + 2 >= nb;
    score(ra, b);
    load_fbatch<D, BF16KV, U>(last ? vb : kb, place(last ? 0 : b + 2) * U, n, j, ra);
    score(rb, b + 1);
    load_fbatch<D, BF16KV, U>(last ? vb : kb, place(last ? 1 : b + 3) * U, n, j, rb);
  }
  float m = mloc;
  m = groups_max<G::kLpt>(m);
  __builtin_amdgcn_wave_barrier();

  float z = 0.f;
  auto accumulate = [&](const u4 (&r)[U], uint32_t b) {
    if (b < nb)
      faccumulate_batch<D, BF16KV, U>(r, place(b) * U, n, j, lane, m, s_lds + place(b) * TPB, z, out.acc);
  };
  for (uint32_t b = 0; b < nb; b += 2) {
    accumulate(ra, b);
    load_fbatch<D, BF16KV, U>(vb, place(b + 2) * U, n, j, ra);
    accumulate(rb, b + 1);
    load_fbatch<D, BF16KV, U>(vb, place(b + 3) * U, n, j, rb);
  }
  z = wave_sum(z);
  reduce_scatter_groups<G::kLpt, G::kEpc>(out.acc, lane);
  out.m = m;
  out.z = z;
}

// The fused step's current token, widened from its raw words and rounded to
// the store's dtype (the value a stored token would hold).
template <int N, bool BF16KV>
__device__ __forceinline__ void widen_current(const RawVec<N>& raw, uint32_t dtype, float (&x)[N]) {
  widen<N>(raw, dtype, x);
  if constexpr (BF16KV) {
#pragma unroll
    for (int e = 0; e < N; ++e) x[e] = bf16_to_f32(f32_to_bf16_bits(x[e]));
  }
}

// The fused step's write of one current-token tensor of `row` at slot p of
// the store; returns PPK_FLAG_OVERFLOW when the slot is past the store.
template <int EPL, bool BF16KV>
__device__ __forceinline__ uint32_t write_current(void* store, uint64_t stride, uint32_t row, uint32_t p,
                                                  uint32_t size, const float (&x)[EPL], int lane) {
  if (p >= size) return 2u;
  const size_t base = size_t(row) * stride + size_t(p) * (EPL * ppk::kWave) + size_t(lane) * EPL;
#pragma unroll
  for (int e = 0; e < EPL; ++e) store_elem(store, base + e, BF16KV ? kBF16 : kF32, x[e]);
  return 0;
}

template <int D, bool BF16KV, bool STEP>
__device__ __forceinline__ void fdecode_body(const ppk::FloatDecodeArgs& a) {
  using G = FloatGeom<D, BF16KV>;
  constexpr int EPL = D / ppk::kWave;
  extern __shared__ float lds[];
  const int lane = threadIdx.x & 63;
  // Uniform: the wave's range, length and loop bounds stay in scalar registers.
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane % G::kLpt;
  // Blocks are numbered group-major: consecutive blocks belong to different
  // rows, so the empty tail groups of short rows (ragged batches) spread over
  // the CUs instead of leaving some CUs with only live blocks.
  const uint32_t group = fast_div(blockIdx.x, a.row_div);
  const uint32_t row = blockIdx.x - group * a.rows;
  // The stored tokens a row streams: lengths[b] (the step's current token
  // comes from k_new / v_new instead). The wave's first loads wait for it: the
  // other arguments they need are requested beside it (the compiler would
  // load each where it is first used, one scalar round trip after another).
  const uint32_t seq = fast_div(row, a.head_div);
  const uint32_t len = a.lengths ? a.lengths[seq] : a.size;
  __asm__ volatile("" ::"s"(seq), "s"(a.q), "s"(a.k), "s"(a.v), "s"(a.k_new), "s"(a.v_new), "s"(a.q_stride), "s"(a.k_stride),
                   "s"(a.v_stride), "s"(a.size), "s"(a.split_tokens), "s"(a.ngroups), "s"(a.q_dtype),
                   "s"(a.new_dtype), "s"(a.scale_log2), "s"(a.span), "s"(blockDim.x));
  const int W = blockDim.x >> 6;
  const uint32_t S = a.split_tokens;
  bool valid;
  if constexpr (STEP)
    valid = len < a.size && len + 1 <= a.span && uint64_t(len) <= uint64_t(a.ngroups) * W * S;
  else
    valid = len > 0 && len <= a.span && len <= a.size && uint64_t(len) <= uint64_t(a.ngroups) * W * S;

  // The step: group 0's waves 0 and 1 write the current key and value at slot
  // len (never read here: every stream stops before it); wave 0 of a block
  // that finishes its row also folds the current token into the result. The
  // operands travel as raw words beside the stream's first batch.
  const bool final_out = a.ngroups == 1;
  const bool kw = STEP && group == 0 && wave == 0;
  const bool vw = STEP && group == 0 && wave == (W > 1 ? 1 : 0);
  const bool cur = STEP && final_out && wave == 0;
  RawVec<G::kEpc> q_raw;
  RawVec<EPL> qc_raw, kn_raw, vn_raw;
  load_raw<G::kEpc>(a.q, size_t(row) * a.q_stride + size_t(c) * G::kEpc, a.q_dtype, q_raw);
  const size_t own = size_t(row) * D + size_t(lane) * EPL;
  if (kw || cur) load_raw<EPL>(a.k_new, own, a.new_dtype, kn_raw);
  if (vw || cur) load_raw<EPL>(a.v_new, own, a.new_dtype, vn_raw);
  if (cur) load_raw<EPL>(a.q, size_t(row) * a.q_stride + size_t(lane) * EPL, a.q_dtype, qc_raw);
  const uint32_t begin = (group * W + wave) * S;
  const uint32_t n = (valid && begin < len) ? min(S, len - begin) : 0u;

  float qr[G::kEpc], kcur[EPL], vcur[EPL];
  float s_cur = -INFINITY;
  uint32_t raise = 0;
  auto early = [&]() {
    settle(q_raw);
    settle(kn_raw);
    settle(vn_raw);
    settle(qc_raw);
    widen<G::kEpc>(q_raw, a.q_dtype, qr);
    if (kw || cur) widen_current<EPL, BF16KV>(kn_raw, a.new_dtype, kcur);
    if (vw || cur) widen_current<EPL, BF16KV>(vn_raw, a.new_dtype, vcur);
    if (cur) {
      float qcur[EPL], d = 0.f;
      widen<EPL>(qc_raw, a.q_dtype, qcur);
#pragma unroll
      for (int e = 0; e < EPL; ++e) d = fmaf(qcur[e], kcur[e], d);
      s_cur = wave_sum(d) * a.scale_log2;
    }
    // A stored length within the span that the plan does not cover: the plan
    // was sized from a stale host copy of the lengths (the row gives NaN).
    if (kw && len < a.size && len + 1 <= a.span && uint64_t(len) > uint64_t(a.ngroups) * W * S) raise |= 4u;
    if (kw) raise |= write_current<EPL, BF16KV>(const_cast<void*>(a.k), a.k_stride, row, len, a.size, kcur, lane);
    if (vw) raise |= write_current<EPL, BF16KV>(const_cast<void*>(a.v), a.v_stride, row, len, a.size, vcur, lane);
  };
  FloatWavePartial<D, BF16KV> part;
  // LDS of this wave alone: a score per token of its batches, then its record.
  constexpr uint32_t TPB = 4 * G::kTpl;
  const uint32_t lds_stride = max((S + TPB - 1) / TPB * TPB, uint32_t(D + 4));
  float* s_lds = lds + size_t(wave) * lds_stride;
  fwave_attention<D, BF16KV>(a, row, begin, n, qr, s_lds, lane, part, early);

  // Combine the block's waves through LDS: each wave's record replaces its
  // scores (its own LDS, so no barrier is needed before).
  write_block_record<D>(s_lds, c * G::kEpc + scatter_base<G::kLpt, G::kEpc>(lane), lane, part.m, part.z, part.acc);
  raise_flags(a.flags, raise);
  __syncthreads();
  if (wave != 0) return;

  float m, y[EPL], zsum;
  combine_block<D, 16, true>(lds, lds_stride, uint32_t(W), lane, s_cur, m, zsum, y);
  if (cur) {
    const float wc = __builtin_amdgcn_exp2f(s_cur - m);
    zsum += wc;
#pragma unroll
    for (int e = 0; e < EPL; ++e) y[e] = fmaf(wc, vcur[e], y[e]);
  }
  if (a.ngroups == 1) {
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      const float o = (valid && zsum > 0.f) ? y[e] / zsum : __builtin_nanf("");
      store_elem(a.out, size_t(row) * D + size_t(lane) * EPL + e, a.out_dtype, o);
    }
  } else {
    const size_t rec = size_t(row) * a.ngroups + group;
#pragma unroll
    for (int e = 0; e < EPL; ++e) a.part_y[rec * D + size_t(lane) * EPL + e] = y[e];
    a.part_mz[rec * 2] = m;
    a.part_mz[rec * 2 + 1] = zsum;
  }
}

// Cross-group merge of the float path (pp_attention_merge,
// decode_attention.hip:55-66): one wave per row, log-sum-exp weights, NaN for
// invalid rows or a non-positive total weight.
// The fused step's current token in a merge: its row as raw words, then q .
// k_new (rounded to the store's dtype) as a log2-domain score, with v_new kept
// for the fold. Nothing without the step.
template <int D>
struct FloatMergeCurrent {
  static constexpr int EPL = D / ppk::kWave;
  RawVec<EPL> q, k, v;
  float vcur[EPL], s_cur = -INFINITY;
  __device__ __forceinline__ void request(const ppk::FloatMergeArgs& a, uint32_t row, int lane) {
    if (!a.step) return;  // uniform
    const size_t own = size_t(lane) * EPL;
    load_raw<EPL>(a.q, size_t(row) * a.q_stride + own, a.q_dtype, q);
    load_raw<EPL>(a.k_new, size_t(row) * D + own, a.new_dtype, k);
    load_raw<EPL>(a.v_new, size_t(row) * D + own, a.new_dtype, v);
  }
  __device__ __forceinline__ float score(const ppk::FloatMergeArgs& a) {
    if (!a.step) return s_cur;
    float qv[EPL], kv[EPL], d = 0.f;
    widen<EPL>(q, a.q_dtype, qv);
    widen<EPL>(k, a.new_dtype, kv);
    widen<EPL>(v, a.new_dtype, vcur);
    if (a.kv_bf16) {
#pragma unroll
      for (int e = 0; e < EPL; ++e) {
        kv[e] = bf16_to_f32(f32_to_bf16_bits(kv[e]));
        vcur[e] = bf16_to_f32(f32_to_bf16_bits(vcur[e]));
      }
    }
#pragma unroll
    for (int e = 0; e < EPL; ++e) d = fmaf(qv[e], kv[e], d);
    s_cur = wave_sum(d) * a.scale_log2;
    return s_cur;
  }
};

template <int D>
__device__ __forceinline__ void fmerge_body(const ppk::FloatMergeArgs& a) {
  constexpr int EPL = D / ppk::kWave;
  // Every argument on the way to the loads, requested together.
  __asm__ volatile("" ::"s"(a.lengths), "s"(a.part_y), "s"(a.part_mz), "s"(a.out), "s"(a.q), "s"(a.k_new),
                   "s"(a.v_new), "s"(a.size), "s"(a.split_tokens), "s"(a.nsplits), "s"(a.out_dtype), "s"(a.span),
                   "s"(a.step), "s"(a.q_dtype), "s"(a.new_dtype), "s"(a.kv_bf16), "s"(a.scale_log2),
                   "s"(a.head_div.mul), "s"(a.head_div.shift));
  const int lane = threadIdx.x;
  const uint32_t row = blockIdx.x;
  float m, zsum, y[EPL];
  FloatMergeCurrent<D> cur;
  // The row's length travels with the records (as a vector load, see lane_zero).
  uint32_t len_raw = a.size;
  auto request = [&]() {
    cur.request(a, row, lane);
    if (a.lengths) len_raw = a.lengths[fast_div(row, a.head_div) + lane_zero()];
  };
  combine_records<D>(a.part_mz + size_t(row) * a.nsplits * 2, a.part_y + size_t(row) * a.nsplits * D, a.nsplits,
                     lane, request, [&]() { return cur.score(a); }, m, zsum, y);
  const uint32_t len = __builtin_amdgcn_readfirstlane(len_raw);
  const bool cover = uint64_t(len) <= uint64_t(a.nsplits) * a.split_tokens;
  const bool valid = a.step ? (len < a.size && len + 1 <= a.span && cover)
                            : (len > 0 && len <= a.span && len <= a.size && cover);
  if (a.step) {
    const float wc = __builtin_amdgcn_exp2f(cur.s_cur - m);
    zsum += wc;
#pragma unroll
    for (int e = 0; e < EPL; ++e) y[e] = fmaf(wc, cur.vcur[e], y[e]);
  }
  const size_t base = size_t(row) * D + size_t(lane) * EPL;
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    const float o = (valid && zsum > 0.f) ? y[e] / zsum : __builtin_nanf("");
    store_elem(a.out, base + e, a.out_dtype, o);
  }
}

// ---------------------------------------------------------------------------
// Float-KV decode over the balanced work list (ragged batches with the host's
// copy of the lengths): the int8 path's table (units of at most Q tokens of
// one row, one unit per wave), each unit streamed as (K, V) batch
// pairs through a window of two pairs with an online softmax. A row of one
// unit is finished in the decode launch; longer rows leave one record per
// unit for ppk_fmerge_flat_d*. A row whose host length lies outside
// (0, min(size, max_length)], or whose device lengths[b] differs from the
// table's, gives NaN.
// ---------------------------------------------------------------------------
// One (K, V) batch pair under the online softmax: token group j (the lanes
// of one token of each tile) keeps its running max m, sum z and channel
// accumulators; the batch's four scores, a rescale if any group of the wave
// has a new max, then the V rows.
template <int D, bool BF16KV>
__device__ __forceinline__ void fonline_pair(const u4 (&kraw)[4], const u4 (&vraw)[4], uint32_t t0, uint32_t n, int j,
                                             const float (&qr)[FloatGeom<D, BF16KV>::kEpc], float sl2, float& m,
                                             float& z, float (&acc)[FloatGeom<D, BF16KV>::kEpc]) {
  using G = FloatGeom<D, BF16KV>;
  float s[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const uint32_t tok = (t0 + u) * G::kTpl + j;
    float x[G::kEpc];
    unpack_chunk<BF16KV>(kraw[u], x);
    float d = 0.f;
#pragma unroll
    for (int e = 0; e < G::kEpc; ++e) d = fmaf(qr[e], x[e], d);
    const float sc = token_sum<G::kLpt>(d) * sl2;
    s[u] = tok < n ? sc : -INFINITY;
  }
  const float mb = fmaxf(fmaxf(m, fmaxf(s[0], s[1])), fmaxf(s[2], s[3]));
  if (__any(mb > m)) {
    const float f = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mb);
    z *= f;
#pragma unroll
    for (int e = 0; e < G::kEpc; ++e) acc[e] *= f;
    m = mb;
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const float pr = s[u] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(s[u] - m);
    z += pr;
    float x[G::kEpc];
    unpack_chunk<BF16KV>(vraw[u], x);
#pragma unroll
    for (int e = 0; e < G::kEpc; ++e) acc[e] = fmaf(pr, x[e], acc[e]);
  }
}

// Streams tokens [begin, begin + n) of one row (n >= 1) through the window
// of NP (K, V) pairs; the partial as fwave_attention returns it. The refills
// are unconditional, as in the int8 window (wave_attention_window). early()
// leaves the query chunk in qr, with the window's first loads in flight.
template <int D, bool BF16KV, int NP, class Early>
__device__ __forceinline__ void fwave_attention_window(const ppk::FloatDecodeArgs& a, uint32_t row, uint32_t begin,
                                                       uint32_t n, const float (&qr)[FloatGeom<D, BF16KV>::kEpc],
                                                       int lane, FloatWavePartial<D, BF16KV>& out, Early early) {
  using G = FloatGeom<D, BF16KV>;
  constexpr int U = 4;
  const int j = lane / G::kLpt;
  const int c = lane % G::kLpt;
  const char* kb = static_cast<const char*>(a.k) +
                   (size_t(row) * a.k_stride + size_t(begin) * D) * G::kElemBytes + size_t(c) * ppk::kLaneBytes;
  const char* vb = static_cast<const char*>(a.v) +
                   (size_t(row) * a.v_stride + size_t(begin) * D) * G::kElemBytes + size_t(c) * ppk::kLaneBytes;
  const uint32_t nb = (n + U * G::kTpl - 1) / (U * G::kTpl);  // batches per phase
  u4 kr[NP][U], vr[NP][U];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    load_fbatch<D, BF16KV, U>(kb, uint32_t(p) * U, n, j, kr[p]);
    load_fbatch<D, BF16KV, U>(vb, uint32_t(p) * U, n, j, vr[p]);
  }
  early();
  float m = -INFINITY, z = 0.f, acc[G::kEpc];
#pragma unroll
  for (int e = 0; e < G::kEpc; ++e) acc[e] = 0.f;
  for (uint32_t b0 = 0; b0 < nb; b0 += NP) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const uint32_t bi = b0 + uint32_t(p);
      if (bi < nb) fonline_pair<D, BF16KV>(kr[p], vr[p], bi * U, n, j, qr, a.scale_log2, m, z, acc);
      load_fbatch<D, BF16KV, U>(kb, (bi + NP) * U, n, j, kr[p]);
      load_fbatch<D, BF16KV, U>(vb, (bi + NP) * U, n, j, vr[p]);
      issue_here();
    }
  }
  const float mm = groups_max<G::kLpt>(m);
  const float w = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mm);
  z *= w;
#pragma unroll
  for (int e = 0; e < G::kEpc; ++e) acc[e] *= w;
  z = groups_reduce<G::kLpt>(z, [](float a, float b) { return a + b; });
  reduce_scatter_groups<G::kLpt, G::kEpc>(acc, lane);
  out.m = mm;
  out.z = z;
#pragma unroll
  for (int e = 0; e < G::kEpc; ++e) out.acc[e] = acc[e];
}

template <int D, bool BF16KV, bool STEP>
__device__ __forceinline__ void fdecode_flat_body(const ppk::FloatDecodeFlatArgs& fa) {
  const ppk::FloatDecodeArgs& a = fa.d;
  const ppk::FlatTable& t = fa.t;
  using G = FloatGeom<D, BF16KV>;
  constexpr int EPL = D / ppk::kWave;
  // The arguments on the way to the first loads, requested together.
  __asm__ volatile("" ::"s"(a.q), "s"(a.k), "s"(a.v), "s"(a.lengths), "s"(a.q_stride), "s"(a.k_stride),
                   "s"(a.v_stride), "s"(a.rows), "s"(a.heads), "s"(a.q_dtype), "s"(a.new_dtype), "s"(a.scale_log2),
                   "s"(t.share), "s"(t.units_total), "s"(t.pivot[1]), "s"(t.pivot[2]), "s"(t.pivot[3]),
                   "s"(t.pivot[4]), "s"(gridDim.x));
  const int lane = threadIdx.x & 63;
  // Wave w of block x takes unit w * blocks + x: the waves that share a CU
  // take units far apart in the list (rows of different lengths, idle waves
  // spread over the CUs), which evens the bytes each CU streams. Measured on
  // MI355X (H = 16, bf16, D = 128, against unit 4x + w): 8 sequences of 4096
  // tokens beside 24 of 1024, 87.5 -> 78.1 us; 4 of 8192 beside 28 of 512,
  // 68.9 -> 67.0 us; f32 1 of 8192 beside 31 of 256, 52.5 -> 48.0 us;
  // within 2 % elsewhere. (The int8 kernel keeps consecutive units per
  // block: this mapping did not help it.)
  const uint32_t wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * gridDim.x + blockIdx.x;
  // The step's writes: wave q < 2 rows writes tensor q & 1 of row q >> 1 at
  // slot lengths[b] (the device value; every stream stops before it).
  const bool put = STEP && wid < 2 * a.rows;  // the host keeps waves >= 2 rows
  const uint32_t arow = wid >> 1;
  const bool value = (wid & 1u) != 0;
  RawVec<EPL> new_raw;
  uint32_t slot_raw = 0;
  if (put) {
    slot_raw = a.lengths[fast_div(arow, a.head_div) + lane_zero()];
    load_raw<EPL>(value ? a.v_new : a.k_new, size_t(arow) * D + size_t(lane) * EPL, a.new_dtype, new_raw);
  }
  auto write = [&]() {
    if (!put) return;
    float x[EPL];
    widen<EPL>(new_raw, a.new_dtype, x);
    raise_flags(a.flags, write_current<EPL, BF16KV>(const_cast<void*>(value ? a.v : a.k),
                                                    value ? a.v_stride : a.k_stride, arow,
                                                    __builtin_amdgcn_readfirstlane(slot_raw), a.size, x, lane));
  };
  if (wid >= t.units_total) {
    write();
    return;
  }
  const FlatUnit u = flat_unit(t, wid);
  const int c = lane % G::kLpt;
  const int ch = c * G::kEpc + scatter_base<G::kLpt, G::kEpc>(lane);  // this lane's output channels
  const uint32_t row = u.b * a.heads + u.head;
  const uint32_t t0 = u.slot * t.share;
  const uint32_t n = u.len > t0 ? min(t.share, u.len - t0) : 0u;
  const uint32_t l_raw = a.lengths[u.b + lane_zero()];
  // The step's current token, folded by the wave of a one-unit row (longer
  // rows: by the merge), in this kernel's lane layout and token arithmetic.
  const bool whole = u.units == 1;
  const bool cur = STEP && whole;
  RawVec<G::kEpc> q_raw, kx_raw;
  RawVec<EPL> vx_raw;
  load_raw<G::kEpc>(a.q, size_t(row) * a.q_stride + size_t(c) * G::kEpc, a.q_dtype, q_raw);
  if (cur) {
    load_raw<G::kEpc>(a.k_new, size_t(row) * D + size_t(c) * G::kEpc, a.new_dtype, kx_raw);
    load_raw<EPL>(a.v_new, size_t(row) * D + size_t(ch), a.new_dtype, vx_raw);
  }
  FloatWavePartial<D, BF16KV> part;
  part.m = -INFINITY;
  part.z = 0.f;
#pragma unroll
  for (int e = 0; e < G::kEpc; ++e) part.acc[e] = 0.f;
  float qr[G::kEpc];
  auto early = [&]() {
    issue_here();
    settle(new_raw);
    settle(kx_raw);
    settle(vx_raw);
    widen<G::kEpc>(q_raw, a.q_dtype, qr);
    write();
  };
  if (n > 0) fwave_attention_window<D, BF16KV, 2>(a, row, t0, n, qr, lane, part, early);
  else early();
  const uint32_t ldev = __builtin_amdgcn_readfirstlane(l_raw);
  bool valid;
  if constexpr (STEP) {
    valid = ldev == u.past && u.past < a.size && u.past + 1 <= a.span;
    // A device length that differs from the host copy the table was built
    // from: the row gives NaN, and a decode step says why in its flags.
    if (ldev != u.past) raise_flags(a.flags, 4u);
  } else {
    valid = u.len > 0 && ldev == u.past;
  }
  if (cur) {
    float kx[G::kEpc], vx[EPL], d = 0.f;
    widen<G::kEpc>(kx_raw, a.new_dtype, kx);
    widen<EPL>(vx_raw, a.new_dtype, vx);
    if constexpr (BF16KV) {
#pragma unroll
      for (int e = 0; e < G::kEpc; ++e) kx[e] = bf16_to_f32(f32_to_bf16_bits(kx[e]));
#pragma unroll
      for (int e = 0; e < EPL; ++e) vx[e] = bf16_to_f32(f32_to_bf16_bits(vx[e]));
    }
#pragma unroll
    for (int e = 0; e < G::kEpc; ++e) d = fmaf(qr[e], kx[e], d);
    const float s_cur = token_sum<G::kLpt>(d) * a.scale_log2;
    const float m2 = fmaxf(part.m, s_cur);
    const float w1 = part.m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(part.m - m2);
    const float wc = __builtin_amdgcn_exp2f(s_cur - m2);
    part.z = fmaf(part.z, w1, wc);
#pragma unroll
    for (int e = 0; e < EPL; ++e) part.acc[e] = fmaf(part.acc[e], w1, wc * vx[e]);
  }
  if (whole) {
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      const float o = (valid && part.z > 0.f) ? part.acc[e] / part.z : __builtin_nanf("");
      store_elem(a.out, size_t(row) * D + size_t(ch + e), a.out_dtype, o);
    }
  } else if (u.slot < a.ngroups) {  // always, by the host's count of slots
    const size_t rec = size_t(row) * a.ngroups + u.slot;
#pragma unroll
    for (int e = 0; e < EPL; ++e) a.part_y[rec * D + size_t(ch + e)] = part.acc[e];
    a.part_mz[rec * 2] = part.m;
    a.part_mz[rec * 2 + 1] = part.z;
  }
}

// Merge of the float balanced work list: one wave per row of two or more
// units (the others were written by the decode launch).
template <int D>
__device__ __forceinline__ void fmerge_flat_body(const ppk::FloatMergeFlatArgs& fa) {
  const ppk::FloatMergeArgs& a = fa.m;
  const ppk::FlatTable& t = fa.t;
  constexpr int EPL = D / ppk::kWave;
  __asm__ volatile("" ::"s"(a.lengths), "s"(a.part_y), "s"(a.part_mz), "s"(a.out), "s"(a.q), "s"(a.k_new),
                   "s"(a.v_new), "s"(a.size), "s"(a.nsplits), "s"(a.out_dtype), "s"(a.span), "s"(a.step),
                   "s"(a.q_dtype), "s"(a.new_dtype), "s"(a.kv_bf16), "s"(a.scale_log2), "s"(a.head_div.mul),
                   "s"(a.head_div.shift));
  const int lane = threadIdx.x;
  const uint32_t row = blockIdx.x;
  const uint32_t b = fast_div(row, a.head_div);
  const ppk::FlatSequence seq = t.seq[b];
  const uint32_t units = seq.units & 0xffffffu;
  if (units < 2) return;  // uniform per wave
  uint32_t l_raw = 0;
  float m, zsum, y[EPL];
  FloatMergeCurrent<D> cur;
  auto request = [&]() {
    cur.request(a, row, lane);
    l_raw = a.lengths[b + lane_zero()];
  };
  combine_records<D>(a.part_mz + size_t(row) * a.nsplits * 2, a.part_y + size_t(row) * a.nsplits * D,
                     min(units, a.nsplits), lane, request, [&]() { return cur.score(a); }, m, zsum, y);
  const uint32_t ldev = __builtin_amdgcn_readfirstlane(l_raw);
  if (a.step) {
    const float wc = __builtin_amdgcn_exp2f(cur.s_cur - m);
    zsum += wc;
#pragma unroll
    for (int e = 0; e < EPL; ++e) y[e] = fmaf(wc, cur.vcur[e], y[e]);
  }
  const bool valid = a.step ? (ldev == seq.past && seq.past < a.size && seq.past + 1 <= a.span)
                            : (seq.len > 0 && ldev == seq.past);
  const size_t base = size_t(row) * D + size_t(lane) * EPL;
#pragma unroll
  for (int e = 0; e < EPL; ++e)
    store_elem(a.out, base + e, a.out_dtype, (valid && zsum > 0.f) ? y[e] / zsum : __builtin_nanf(""));
}

// ---------------------------------------------------------------------------
// CFG + Renyi effective-support sampler (app/src/inference/renyi_sample.hip:23-204,
// hip_sampling.rs:89-105). Per logical row: v = u + cfg (c - u) over the whole
// head (every column must be finite), legal candidates [start, start + count),
// H = log Z + max(0, log Z - log Z_alpha) / (alpha - 1) clamped to [0, ln count],
// support = clamp((u32)(exp(H) + 0.5), 1, count), rank = min((u32)(uniform *
// support), support - 1), token = the rank-th candidate by (value descending,
// index ascending).
//
// The arithmetic that decides support keeps the reference's order: 256
// strided partial sums of exp(v - m) and exp(alpha (v - m)) in candidate
// order, then the halving tree (steps 128, 64 through LDS, 32..1 by lane
// swaps within each wave: the same pairs added in the same order), with
// the device expf/logf. The candidate selection is this file's own: the
// reference sorts the whole legal range (a bitonic network of ~66 barrier
// phases at 2048 candidates); here the values are counted into 512 equal bins
// beside the sums, and the few candidates of the bin that holds the rank are
// ordered by comparison. Where that bin is crowded, a 4-pass radix select over
// a 32-bit order-preserving key of the value finds the selected value and a
// ballot count orders equal values by index. All name the same candidate.
// The kernel is a chain of barriers and round trips (one block per row, one
// wave per SIMD): three barriers now, where four radix passes took twenty and
// the support two more: 32 rows x 2048 choices with guidance 10.3 -> 6.3 us,
// 1024 rows 14.3 -> 9.1, 64 rows x 37 choices 8.1 -> 4.3 (one launch in a
// captured sequence of 50).
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool finite_bits(float x) { return (__float_as_uint(x) & 0x7fffffffu) < 0x7f800000u; }
__device__ __forceinline__ bool sample_before(float a, uint32_t ai, float b, uint32_t bi) {
  return a > b || (a == b && ai < bi);
}
// Ascending key order = descending value order; -0 and +0 share a key (they
// compare equal, so their order is by index).
__device__ __forceinline__ uint32_t descending_key(float v) {
  const uint32_t b = __float_as_uint(v == 0.f ? 0.f : v);
  const uint32_t ascending = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
  return ~ascending;
}

__device__ __forceinline__ void write_sample(const ppk::RenyiArgs& a, uint32_t row, uint32_t token, uint32_t valid,
                                             uint32_t support) {
  a.out[row] = token;
  a.out[size_t(a.batch) + row] = valid;
  a.out[2 * size_t(a.batch) + row] = support;
}

// Inclusive prefix sum over the wave's lanes (DPP, no LDS).
__device__ __forceinline__ uint32_t wave_prefix(uint32_t v) {
  int x = int(v);
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);   // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);   // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);   // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);   // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return uint32_t(x);
}
// Lane 0 receives the sum over the wave in the halving order x[i] += x[i + o],
// o = 32, 16, ... 1 (the other lanes: partial sums).
__device__ __forceinline__ float halving_sum(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  x += dpp_f32<0x108>(x);  // row_shl:8
  x += dpp_f32<0x104>(x);
  x += dpp_f32<0x102>(x);
  x += dpp_f32<0x101>(x);
  return x;
}

__device__ __forceinline__ void renyi_sample_body(const ppk::RenyiArgs& a) {
  // Every float operation rounds on its own, as the reference kernel is built
  // (-ffp-contract=off, app/src/model/hip_kernel.rs:46) and as its host oracle
  // evaluates (app/src/inference/hip_sampling_reference.rs:73): the CFG value
  // u + cfg * (c - u) is a rounded product and then a rounded sum, never one
  // fused multiply-add, whose 1-ulp differences can reorder candidates.
#pragma clang fp contract(off)
  constexpr int T = ppk::kSamplerThreads;
  constexpr int PER = ppk::kSamplerMaxChoices / T;  // candidates per thread
  constexpr int BINS = 512;                         // value bins of the selection, BINS / 64 per lane
  constexpr uint32_t LIST = 64;                     // most candidates of the selected bin the fast path orders
  __shared__ float s_vals[ppk::kSamplerMaxChoices];
  __shared__ float s_sum[T], s_sum_a[T];
  __shared__ float s_wmax[T / 64], s_wmin[T / 64];
  __shared__ uint32_t s_wid[T / 64], s_wbad[T / 64];
  __shared__ __attribute__((aligned(16))) uint32_t s_bins[BINS + 64];
  __shared__ float s_list_v[LIST];
  __shared__ uint32_t s_list_i[LIST];
  __shared__ uint32_t s_listed;
  __shared__ uint32_t s_hist[256];
  __shared__ uint32_t s_wtotal[T / 64];
  __shared__ uint64_t s_ballot[PER][T / 64];
  __shared__ uint32_t s_state[4];  // selected bin / below of the radix passes

  const uint32_t row = blockIdx.x;
  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  // The whole head is requested first, beside the row's metadata: each
  // thread's columns (at most PER of each head, inside the row's raw logits
  // whatever the metadata say) before any is used, so the pass costs one
  // memory round trip instead of one or two per column.
  const float* c_row = a.raw + size_t(row) * a.guidance * a.choices;
  const bool guided = a.guidance == 2;
  float cv[PER], uv[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const uint32_t col = uint32_t(t) + uint32_t(k) * T;
    cv[k] = col < a.choices ? c_row[col] : 0.f;
    uv[k] = guided && col < a.choices ? c_row[a.choices + col] : 0.f;
  }
  const uint32_t start = a.bounds[2 * row];
  const uint32_t count = a.bounds[2 * row + 1];
  const float uniform = a.uniforms[row];
#pragma unroll
  for (int i = 0; i < BINS / T; ++i) s_bins[t + i * T] = 0;
  if (t == 0) s_listed = 0;
  // Every thread evaluates the same metadata, so these exits are uniform.
  if (!finite_bits(uniform) || uniform < 0.f || uniform >= 1.f || start >= a.choices || count == 0 ||
      count > a.choices - start) {
    if (t == 0) write_sample(a, row, a.token_offset + (start < a.choices ? start : 0u), 0, 1);
    return;
  }

  // Whole head, in column order: CFG combine and finiteness; legal values to
  // LDS; arg-max (the lowest index of the largest value) and minimum.
  float lmax = -INFINITY, lmin = INFINITY;
  uint32_t lid = 0xffffffffu, lbad = 0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const uint32_t col = uint32_t(t) + uint32_t(k) * T;
    if (col >= a.choices) continue;
    const float c = cv[k];
    float value = c;
    bool finite = finite_bits(c);
    if (guided) {
      const float u = uv[k];
      finite = finite && finite_bits(u);
      value = u + a.cfg * (c - u);
    }
    finite = finite && finite_bits(value);
    lbad |= finite ? 0u : 1u;
    if (!finite) value = 0.f;
    if (col >= start && col - start < count) {
      s_vals[col - start] = value;
      lmin = fminf(lmin, value);
      if (sample_before(value, col, lmax, lid)) {
        lmax = value;
        lid = col;
      }
    }
  }
  {
    const float wmax = wave_max(lmax);
    const float wmin = wave_reduce(lmin, [](float x, float y) { return fminf(x, y); });
    // The least index of the wave's maximum, with the indexes as floats (below 2^24: exact).
    const float id = wave_reduce(lmax == wmax && lid != 0xffffffffu ? float(lid) : 16777216.f,
                                 [](float x, float y) { return fminf(x, y); });
    const bool wbad = __any(lbad != 0);
    if (lane == 0) {
      s_wmax[wave] = wmax;
      s_wmin[wave] = wmin;
      s_wid[wave] = uint32_t(id);
      s_wbad[wave] = wbad ? 1u : 0u;
    }
  }
  __syncthreads();
  float maximum = s_wmax[0], minimum = s_wmin[0];
  uint32_t maximum_id = s_wid[0], bad = s_wbad[0];
#pragma unroll
  for (int w = 1; w < T / 64; ++w) {
    if (sample_before(s_wmax[w], s_wid[w], maximum, maximum_id)) {
      maximum = s_wmax[w];
      maximum_id = s_wid[w];
    }
    minimum = fminf(minimum, s_wmin[w]);
    bad |= s_wbad[w];
  }
  if (bad) {
    if (t == 0) write_sample(a, row, a.token_offset + start, 0, 1);
    return;
  }

  // Strided partial sums in candidate order, then the halving tree. The bins
  // of the selection are counted beside them: bin = (maximum - v) scaled to
  // BINS over the range or kSpan, whichever is less, a rounded subtraction and
  // a rounded product, so a larger value never has a higher bin. Values further
  // down than kSpan (masked ones, an outlier: weight below 2e-7 each) go to words
  // past the bins, spread by lane, that nothing reads: in the range they would stretch the
  // bins until nearly all values shared one, in the last bin they would queue
  // at its word (32 rows x 2048 with guidance 6.2 us, with one outlier 11.8, now
  // 6.3 both; in the last bin 7.5, with a branch around the count 6.5).
  constexpr float kSpan = 16.0f;
  const float range = maximum - minimum;
  const float last = float(range > kSpan ? BINS + lane : BINS - 1);
  const float bin_scale = float(BINS) / fminf(range, kSpan);
  const bool binned = range > 0.f && finite_bits(bin_scale);
  float vals[PER];
  uint32_t bins[PER];
  float sum = 0.f, sum_a = 0.f;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const uint32_t ci = uint32_t(t) + uint32_t(k) * T;
    vals[k] = ci < count ? s_vals[ci] : 0.f;
    bins[k] = 0xffffffffu;
    if (ci < count) {
      const float shifted = vals[k] - maximum;
      sum += expf(shifted);
      sum_a += expf(a.alpha * shifted);
      if (binned) {
        bins[k] = uint32_t(fminf((maximum - vals[k]) * bin_scale, last));
        atomicAdd(&s_bins[bins[k]], 1u);
      }
    }
  }
  s_sum[t] = sum;
  s_sum_a[t] = sum_a;
  __syncthreads();
  // Every wave adds the tree's 256 partials (128 and 64 apart from LDS, then
  // the halving steps across lanes, the same pairs in the same order) and
  // evaluates the support, instead of one wave for all behind two barriers.
  uint32_t support = 1, r = 0, invalid;
  {
    const float z = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(
        halving_sum((s_sum[lane] + s_sum[lane + 128]) + (s_sum[lane + 64] + s_sum[lane + 192])))));
    const float za = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(
        halving_sum((s_sum_a[lane] + s_sum_a[lane + 128]) + (s_sum_a[lane + 64] + s_sum_a[lane + 192])))));
    const float log_z = logf(z);
    const float log_za = logf(za);
    float correction = log_z - log_za;
    if (correction < 0.0f) correction = 0.0f;
    float entropy = log_z + correction / (a.alpha - 1.0f);
    invalid = !finite_bits(log_z) || !finite_bits(log_za) || !finite_bits(entropy);
    if (!invalid) {
      const float maximum_entropy = logf((float)count);
      if (entropy < 0.0f) entropy = 0.0f;
      if (entropy > maximum_entropy) entropy = maximum_entropy;
      const float rounded = expf(entropy) + 0.5f;
      support = (uint32_t)rounded;
      if (support < 1) support = 1;
      if (support > count) support = count;
      r = (uint32_t)(uniform * (float)support);
      if (r >= support) r = support - 1;
    }
  }
  support = __builtin_amdgcn_readfirstlane(support);
  r = __builtin_amdgcn_readfirstlane(r);
  if (__any(invalid != 0)) {
    if (t == 0) write_sample(a, row, a.token_offset + start, 0, 1);
    return;
  }
  if (r == 0) {
    if (t == 0) write_sample(a, row, a.token_offset + maximum_id, 1, support);
    return;
  }
  if (range == 0.f) {  // all candidates equal: ordered by index
    if (t == 0) write_sample(a, row, a.token_offset + start + r, 1, support);
    return;
  }

  // The bin that holds rank r (every wave finds it, from BINS / 64 bins per
  // lane and a prefix sum over the lanes); its few candidates go to a list and
  // are ordered by direct comparison. More than LIST candidates that are all
  // equal (heavy ties) are ordered by index below; other crowded bins, and a
  // rank among the values that are not counted, are left to the radix passes.
  uint32_t prefix = 0, pmask = 0;
  bool tied = false;
  if (binned) {
    constexpr int PL = BINS / 64;
    uint32_t h[PL], total = 0;
#pragma unroll
    for (int i = 0; i < PL; ++i) {
      h[i] = s_bins[lane * PL + i];
      total += h[i];
    }
    uint32_t below = wave_prefix(total) - total;
    const uint64_t here = __ballot(below <= r && r < below + total);
    uint32_t bin = 0, in_bin = 0;
    bool found = false;
#pragma unroll
    for (int i = 0; i < PL; ++i) {
      if (!found) {
        if (r < below + h[i]) {
          found = true;
          bin = uint32_t(lane * PL + i);
          in_bin = h[i];
        } else {
          below += h[i];
        }
      }
    }
    const int owner = here ? __builtin_ctzll(here) : 0;  // one lane at most
    bin = __builtin_amdgcn_readlane(bin, owner);
    in_bin = __builtin_amdgcn_readlane(in_bin, owner);
    below = __builtin_amdgcn_readlane(below, owner);
    if (here != 0 && in_bin <= LIST) {  // uniform
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        if (bins[k] == bin) {
          const uint32_t at = atomicAdd(&s_listed, 1u);
          s_list_v[at] = vals[k];
          s_list_i[at] = uint32_t(t) + uint32_t(k) * T;
        }
      }
      __syncthreads();
      if (wave != 0) return;
      const uint32_t mine = min(uint32_t(lane), in_bin - 1);
      const float v = s_list_v[mine];
      const uint32_t ci = s_list_i[mine];
      uint32_t rank = below;
      for (uint32_t i = 0; i < in_bin; ++i) {
        const float ov = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), int(i)));
        const uint32_t oi = __builtin_amdgcn_readlane(ci, int(i));
        rank += sample_before(ov, oi, v, ci) ? 1u : 0u;
      }
      if (uint32_t(lane) < in_bin && rank == r) write_sample(a, row, a.token_offset + start + ci, 1, support);
      return;
    }
    if (here != 0) {  // uniform
      float hi = -INFINITY, lo = INFINITY;
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        hi = bins[k] == bin ? fmaxf(hi, vals[k]) : hi;
        lo = bins[k] == bin ? fminf(lo, vals[k]) : lo;
      }
      hi = wave_max(hi);
      lo = wave_reduce(lo, [](float x, float y) { return fminf(x, y); });
      if (lane == 0) {  // last read before the sums' barrier
        s_wmax[wave] = hi;
        s_wmin[wave] = lo;
      }
      __syncthreads();
#pragma unroll
      for (int w = 0; w < T / 64; ++w) {
        hi = fmaxf(hi, s_wmax[w]);
        lo = fminf(lo, s_wmin[w]);
      }
      tied = hi == lo;
      if (tied) {
        prefix = descending_key(hi);
        r -= below;
      }
    }
  }

  // Radix select, 8 key bits per pass from the top: after four passes the
  // prefix is the selected value's key and r its rank among equal values.
  uint32_t keys[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) keys[k] = descending_key(vals[k]);
  for (int shift = tied ? -8 : 24; shift >= 0; shift -= 8) {
    s_hist[t] = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const uint32_t ci = uint32_t(t) + uint32_t(k) * T;
      if (ci < count && (keys[k] & pmask) == prefix) atomicAdd(&s_hist[(keys[k] >> shift) & 255u], 1u);
    }
    __syncthreads();
    const uint32_t h = s_hist[t];
    uint32_t incl = h;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(incl, o);
      if (lane >= o) incl += y;
    }
    if (lane == 63) s_wtotal[wave] = incl;
    __syncthreads();
    uint32_t below = incl - h;
    for (int w = 0; w < wave; ++w) below += s_wtotal[w];
    if (h > 0 && below <= r && r < below + h) {
      s_state[3] = uint32_t(t);
      s_hist[0] = below;  // every thread has read its own bin already
    }
    __syncthreads();
    const uint32_t bin = s_state[3];
    r -= s_hist[0];
    prefix |= bin << shift;
    pmask |= 255u << shift;
    __syncthreads();
  }

  // Among candidates with the selected key, the r-th by ascending index.
  // Candidate ci = t + 256 k: index order is (k, wave, lane) order. The
  // selection always names one candidate (r stays below the count of keys
  // matching the prefix); the record written first only keeps the row's
  // output defined should it not.
  if (t == 0) write_sample(a, row, a.token_offset + start, 0, 1);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const uint32_t ci = uint32_t(t) + uint32_t(k) * T;
    const uint64_t b = __ballot(ci < count && keys[k] == prefix);
    if (lane == 0) s_ballot[k][wave] = b;
  }
  __syncthreads();
  uint32_t before_k = 0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const uint32_t ci = uint32_t(t) + uint32_t(k) * T;
    if (ci < count && keys[k] == prefix) {
      uint32_t pos = before_k + uint32_t(__popcll(s_ballot[k][wave] & ((uint64_t(1) << lane) - 1)));
      for (int w = 0; w < wave; ++w) pos += uint32_t(__popcll(s_ballot[k][w]));
      if (pos == r) write_sample(a, row, a.token_offset + start + ci, 1, support);
    }
#pragma unroll
    for (int w = 0; w < T / 64; ++w) before_k += uint32_t(__popcll(s_ballot[k][w]));
  }
}

// ---------------------------------------------------------------------------
// Float-store append (the in-place slice_set / scatter_set of
// app/src/model/cache.rs:271-276,437-469): token records of K and V to their
// arena slots, UNIT bytes per thread and step, grid-stride. Slots at or past
// capacity are skipped (the host never plans them).
// ---------------------------------------------------------------------------
template <int UNIT>
struct UnitType;
template <>
struct UnitType<16> {
  using T = u4;
};
template <>
struct UnitType<4> {
  using T = uint32_t;
};
template <>
struct UnitType<2> {
  using T = uint16_t;
};

template <int UNIT>
__device__ __forceinline__ void scatter_body(const ppk::ScatterArgs& a) {
  using T = typename UnitType<UNIT>::T;
  const uint64_t per_tensor = a.rows * a.tokens * a.row_units;
  const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
  for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < 2 * per_tensor; i += stride) {
    const uint32_t tensor = i >= per_tensor ? 1u : 0u;
    const uint64_t j = i - (tensor ? per_tensor : 0);
    const uint64_t rt = j / a.row_units;
    const uint32_t u = uint32_t(j - rt * a.row_units);
    const uint64_t r = rt / a.tokens;
    const uint32_t t = uint32_t(rt - r * a.tokens);
    const uint64_t slot = uint64_t(a.past ? a.past[r / a.heads] : a.uniform_past) + t;
    if (slot >= a.capacity) continue;
    const T* src = reinterpret_cast<const T*>(a.src[tensor]);
    T* dst = reinterpret_cast<T*>(a.dst[tensor]);
    dst[(r * a.capacity + slot) * a.row_units + u] = src[rt * a.row_units + u];
  }
}

// ---------------------------------------------------------------------------
// Batched rectangle copy with zero fill (arena joins, growth and
// copy-on-write: every row of a new arena receives its committed prefix and
// zeros up to its capacity in one launch, instead of a memset of the whole
// arena plus one runtime copy per plane and sequence). Blocks stride over
// tiles of one row each, eight units in flight per thread.
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ void copy_rect(const ppk::Copy2D& c, uint32_t unit_bytes) {
  constexpr uint32_t ILP = 8;
  const uint32_t per_row = c.fill / unit_bytes;
  const uint32_t copy_cols = c.width / unit_bytes;
  if (per_row == 0) return;
  // Tiles of up to ILP * blockDim.x units of one row: a block finds its tile's
  // row and first column with one (block-uniform) division, and each lane's
  // columns follow by addition, so no unit pays an integer division.
  const uint32_t tile = min(per_row, ILP * blockDim.x);
  const uint32_t tiles_per_row = (per_row + tile - 1) / tile;
  const uint64_t tiles = uint64_t(c.height) * tiles_per_row;
  for (uint64_t t = blockIdx.x; t < tiles; t += gridDim.x) {
    const uint64_t row = t / tiles_per_row;
    const uint32_t col0 = uint32_t(t - row * tiles_per_row) * tile;
    const uint32_t end = min(col0 + tile, per_row);
    const T* src = reinterpret_cast<const T*>(c.src + row * c.spitch);
    T* dst = reinterpret_cast<T*>(c.dst + row * c.dpitch);
    T val[ILP];
#pragma unroll
    for (uint32_t k = 0; k < ILP; ++k) {
      const uint32_t col = col0 + k * blockDim.x + threadIdx.x;
      val[k] = T{};
      if (col < end && col < copy_cols) val[k] = __builtin_nontemporal_load(src + col);
    }
#pragma unroll
    for (uint32_t k = 0; k < ILP; ++k) {
      const uint32_t col = col0 + k * blockDim.x + threadIdx.x;
      if (col < end) dst[col] = val[k];
    }
  }
}

__device__ __forceinline__ void copy_batch_body(const ppk::CopyBatchArgs& a) {
  if (blockIdx.y >= a.n) return;
  const ppk::Copy2D& c = a.c[blockIdx.y];
  switch (c.unit) {  // uniform per block
    case 16: copy_rect<u4>(c, 16); break;
    case 4: copy_rect<uint32_t>(c, 4); break;
    case 2: copy_rect<uint16_t>(c, 2); break;
    default: copy_rect<uint8_t>(c, 1); break;
  }
}

}  // namespace

#define PPK_QUANTIZE(D)                                                                \
  extern "C" __global__ __launch_bounds__(256) void ppk_quantize_d##D(ppk::QuantizeArgs a) { \
    quantize_body<D>(a);                                                               \
  }
PPK_QUANTIZE(64)
PPK_QUANTIZE(128)
PPK_QUANTIZE(256)

extern "C" __global__ __launch_bounds__(256) void ppk_dequantize(ppk::DequantizeArgs a) { dequantize_body(a); }
// Streaming quantize: dense [rows, D] (ppk_quantize) and appends into arenas
// (ppk_quantize_append, KV arena writes), separate kernels so the dense path
// keeps its smaller register footprint.
#define PPK_QSTREAM(D)                                                                              \
  extern "C" __global__ __launch_bounds__(256) void ppk_quantize_dense_d##D(ppk::StreamQuantizeArgs a) {  \
    quantize_stream_dtype<D, false>(a);                                                             \
  }                                                                                                 \
  extern "C" __global__ __launch_bounds__(256) void ppk_quantize_append_d##D(ppk::StreamQuantizeArgs a) { \
    quantize_stream_dtype<D, true>(a);                                                              \
  }
PPK_QSTREAM(64)
PPK_QSTREAM(128)
PPK_QSTREAM(256)
#undef PPK_QSTREAM

// Blocks of up to 8 waves (the plan never makes larger int8 blocks): two
// waves per SIMD, up to 256 VGPRs each, a ring of kRing batches in flight.
// The late kernels wait for the row's length before their first batches; one
// kernel with both ways was 1-4 % slower on rows of one batch a wave (16 rows
// x 512 tokens at D = 64 4.45 us, now 4.38).
constexpr int kRing = 3;
#define PPK_ATTN(D)                                                                          \
  extern "C" __global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))    \
  void ppk_decode_d##D(ppk::DecodeArgs a) {                                                  \
    decode_body<D, false, kRing, true>(a);                                                   \
  }                                                                                          \
  extern "C" __global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))    \
  void ppk_decode_bf16h_d##D(ppk::DecodeArgs a) {                                            \
    decode_body<D, true, kRing, true>(a);                                                    \
  }                                                                                          \
  extern "C" __global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))    \
  void ppk_decode_late_d##D(ppk::DecodeArgs a) {                                             \
    decode_body<D, false, kRing, false>(a);                                                  \
  }                                                                                          \
  extern "C" __global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))    \
  void ppk_decode_late_bf16h_d##D(ppk::DecodeArgs a) {                                       \
    decode_body<D, true, kRing, false>(a);                                                   \
  }                                                                                          \
  extern "C" __global__ __launch_bounds__(64) void ppk_attn_merge_d##D(ppk::MergeArgs a) {   \
    attn_merge_body<D>(a);                                                                   \
  }
PPK_ATTN(64)
PPK_ATTN(128)
PPK_ATTN(256)

// Flat work list kernels: up to 256 VGPRs, i.e. 8 resident waves per CU (the host launches 8).
#define PPK_ATTN_FLAT(D)                                                                                \
  extern "C" __global__ __launch_bounds__(512) void ppk_decode_flat_d##D(ppk::DecodeFlatArgs a) {      \
    decode_flat_body<D, false>(a);                                                                      \
  }                                                                                                     \
  extern "C" __global__ __launch_bounds__(512) void ppk_decode_flat_bf16h_d##D(ppk::DecodeFlatArgs a) { \
    decode_flat_body<D, true>(a);                                                                       \
  }                                                                                                     \
  extern "C" __global__ __launch_bounds__(64) void ppk_attn_merge_flat_d##D(ppk::MergeFlatArgs a) {   \
    attn_merge_flat_body<D>(a);                                                                         \
  }
PPK_ATTN_FLAT(64)
PPK_ATTN_FLAT(128)
PPK_ATTN_FLAT(256)
#undef PPK_ATTN_FLAT

#define PPK_FLOAT_ATTN(D)                                                                        \
  extern "C" __global__ __launch_bounds__(1024) void ppk_fdecode_bf16_d##D(ppk::FloatDecodeArgs a) { \
    fdecode_body<D, true, false>(a);                                                             \
  }                                                                                              \
  extern "C" __global__ __launch_bounds__(1024) void ppk_fdecode_f32_d##D(ppk::FloatDecodeArgs a) {  \
    fdecode_body<D, false, false>(a);                                                            \
  }                                                                                              \
  extern "C" __global__ __launch_bounds__(1024) void ppk_fstep_bf16_d##D(ppk::FloatDecodeArgs a) {   \
    fdecode_body<D, true, true>(a);                                                              \
  }                                                                                              \
  extern "C" __global__ __launch_bounds__(1024) void ppk_fstep_f32_d##D(ppk::FloatDecodeArgs a) {    \
    fdecode_body<D, false, true>(a);                                                             \
  }                                                                                              \
  extern "C" __global__ __launch_bounds__(64) void ppk_fmerge_d##D(ppk::FloatMergeArgs a) {      \
    fmerge_body<D>(a);                                                                           \
  }
PPK_FLOAT_ATTN(64)
PPK_FLOAT_ATTN(128)
PPK_FLOAT_ATTN(256)

#define PPK_FLOAT_ATTN_FLAT(D)                                                                                 \
  extern "C" __global__ __launch_bounds__(512) void ppk_fdecode_flat_bf16_d##D(ppk::FloatDecodeFlatArgs a) { \
    fdecode_flat_body<D, true, false>(a);                                                                      \
  }                                                                                                            \
  extern "C" __global__ __launch_bounds__(512) void ppk_fdecode_flat_f32_d##D(ppk::FloatDecodeFlatArgs a) {  \
    fdecode_flat_body<D, false, false>(a);                                                                     \
  }                                                                                                            \
  extern "C" __global__ __launch_bounds__(512) void ppk_fstep_flat_bf16_d##D(ppk::FloatDecodeFlatArgs a) {   \
    fdecode_flat_body<D, true, true>(a);                                                                       \
  }                                                                                                            \
  extern "C" __global__ __launch_bounds__(512) void ppk_fstep_flat_f32_d##D(ppk::FloatDecodeFlatArgs a) {    \
    fdecode_flat_body<D, false, true>(a);                                                                      \
  }                                                                                                            \
  extern "C" __global__ __launch_bounds__(64) void ppk_fmerge_flat_d##D(ppk::FloatMergeFlatArgs a) {          \
    fmerge_flat_body<D>(a);                                                                                    \
  }
PPK_FLOAT_ATTN_FLAT(64)
PPK_FLOAT_ATTN_FLAT(128)
PPK_FLOAT_ATTN_FLAT(256)
#undef PPK_FLOAT_ATTN_FLAT

extern "C" __global__ __launch_bounds__(256) void ppk_renyi_sample(ppk::RenyiArgs a) { renyi_sample_body(a); }

extern "C" __global__ __launch_bounds__(256) void ppk_kv_scatter_u16(ppk::ScatterArgs a) { scatter_body<16>(a); }
extern "C" __global__ __launch_bounds__(256) void ppk_kv_scatter_u4(ppk::ScatterArgs a) { scatter_body<4>(a); }
extern "C" __global__ __launch_bounds__(256) void ppk_kv_scatter_u2(ppk::ScatterArgs a) { scatter_body<2>(a); }
extern "C" __global__ __launch_bounds__(256) void ppk_copy2d_batch(ppk::CopyBatchArgs a) { copy_batch_body(a); }
