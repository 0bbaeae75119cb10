// CDNA4 (gfx950) device templates used by the Enceladus HIP emitter.
//
// Every generated kernel includes this header. It provides:
//   - element conversions with the language's semantics (saturating float->int,
//     round-to-nearest-even bf16, C-style integer division that never traps);
//   - raw 1/2/4/8/16-byte vector moves for coalesced global and LDS access;
//   - wave64 cross-lane primitives (DPP row ops and ds_bpermute shuffles);
//   - MFMA wrappers for the gfx950 fp16/bf16/fp32 matrix instructions.
// The header is compiled by hiprtc; it uses only compiler builtins, no system headers.
#pragma once

typedef __INT8_TYPE__ int8_t;
typedef __UINT8_TYPE__ uint8_t;
typedef __INT16_TYPE__ int16_t;
typedef __UINT16_TYPE__ uint16_t;
typedef __INT32_TYPE__ int32_t;
typedef __UINT32_TYPE__ uint32_t;
typedef __INT64_TYPE__ int64_t;
typedef __UINT64_TYPE__ uint64_t;

#define EK_INLINE __device__ __attribute__((always_inline)) inline

// Device printf (tl.device_print); the HIP runtime services it through its hostcall buffer.
extern "C" __device__ int printf(const char*, ...);

namespace ek {

// ---------------------------------------------------------------------------
// bfloat16 storage type (bit pattern); arithmetic always goes through float.
// ---------------------------------------------------------------------------
struct bf16 {
  uint16_t x;
};

EK_INLINE float bits_f32(uint32_t u) { return __builtin_bit_cast(float, u); }
EK_INLINE uint32_t f32_bits(float f) { return __builtin_bit_cast(uint32_t, f); }

EK_INLINE float bf16_to_f32(bf16 h) { return bits_f32(((uint32_t)h.x) << 16); }
// fp32 -> bf16, round to nearest even (gfx950 converts in hardware: v_cvt_pk_bf16_f32).
EK_INLINE bf16 f32_to_bf16(float f) {
  return bf16{__builtin_bit_cast(uint16_t, (__bf16)f)};
}

// ---------------------------------------------------------------------------
// Conversions. `f32(x)` widens any element to the float compute type; `cvt<T>(x)`
// converts with the language's rules.
// ---------------------------------------------------------------------------
EK_INLINE float f32(float x) { return x; }
EK_INLINE float f32(_Float16 x) { return (float)x; }
EK_INLINE float f32(bf16 x) { return bf16_to_f32(x); }

template <typename T> struct int_limits;
template <> struct int_limits<int8_t> { static constexpr float lo = -128.f, hi = 127.f; };
template <> struct int_limits<uint8_t> { static constexpr float lo = 0.f, hi = 255.f; };
template <> struct int_limits<int16_t> { static constexpr float lo = -32768.f, hi = 32767.f; };
template <> struct int_limits<uint16_t> { static constexpr float lo = 0.f, hi = 65535.f; };

// float -> integer: truncate toward zero; NaN -> 0; out of range saturates (all widths
// except int64, which wraps modulo 2^64 and maps infinities to 0).
// v_cvt_i32_f32 / v_cvt_u32_f32 implement exactly that for 32 bits (the ISA: out-of-range
// values, infinities included, saturate and NaN converts to 0), so they are issued as is:
// one instruction instead of a NaN test and two clamps, which the compiler emits as nested
// branches. C++'s (int)x leaves out-of-range values undefined, hence the inline asm.
template <typename T> EK_INLINE T f2i(float x);
template <> EK_INLINE int32_t f2i<int32_t>(float x) {
  int32_t r;
  asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(x));
  return r;
}
template <> EK_INLINE uint32_t f2i<uint32_t>(float x) {
  uint32_t r;
  asm("v_cvt_u32_f32 %0, %1" : "=v"(r) : "v"(x));
  return r;
}
template <> EK_INLINE uint64_t f2i<uint64_t>(float x) {
  if (x != x || x <= 0.0f) return 0ull;
  if (x >= 18446744073709551616.0f) return ~0ull;
  return (uint64_t)x;
}
template <> EK_INLINE int64_t f2i<int64_t>(float x) {
  if (x != x || x == __builtin_inff() || x == -__builtin_inff()) return 0;
  float t = __builtin_truncf(x);
  float a = t < 0.f ? -t : t;
  if (a < 9223372036854775808.0f) return (int64_t)t;
  // |t| >= 2^63: t is a multiple of 2^40 at least; reduce modulo 2^64 exactly.
  double d = (double)t;
  double r = __builtin_fmod(d, 18446744073709551616.0);
  if (r >= 9223372036854775808.0) r -= 18446744073709551616.0;
  if (r < -9223372036854775808.0) r += 18446744073709551616.0;
  return (int64_t)r;
}
// 8/16-bit: the saturating 32-bit conversion, then a clamp (truncation commutes with it).
#define EK_SMALL_F2I(T)                                                       \
  template <> EK_INLINE T f2i<T>(float x) {                                   \
    const int32_t i = f2i<int32_t>(x);                                        \
    const int32_t lo = (int32_t)int_limits<T>::lo, hi = (int32_t)int_limits<T>::hi; \
    return (T)(i < lo ? lo : (i > hi ? hi : i));                              \
  }
EK_SMALL_F2I(int8_t)
EK_SMALL_F2I(uint8_t)
EK_SMALL_F2I(int16_t)
EK_SMALL_F2I(uint16_t)
#undef EK_SMALL_F2I
template <> EK_INLINE bool f2i<bool>(float x) { return x != 0.0f; }

template <typename To> struct Cvt {
  template <typename From> static EK_INLINE To from(From x) {
    if constexpr (__is_same(From, float) || __is_same(From, _Float16) || __is_same(From, bf16)) {
      return f2i<To>(f32(x));
    } else {
      return (To)x;
    }
  }
};
template <> struct Cvt<bool> {
  template <typename From> static EK_INLINE bool from(From x) {
    if constexpr (__is_same(From, bf16)) return (x.x & 0x7fffu) != 0;
    else return x != (From)0;
  }
};
template <> struct Cvt<float> {
  template <typename From> static EK_INLINE float from(From x) {
    if constexpr (__is_same(From, bf16) || __is_same(From, _Float16)) return f32(x);
    else return (float)x;
  }
};
template <> struct Cvt<_Float16> {
  template <typename From> static EK_INLINE _Float16 from(From x) {
    if constexpr (__is_same(From, bf16)) return (_Float16)f32(x);
    else if constexpr (__is_same(From, int64_t) || __is_same(From, uint64_t)) return (_Float16)(float)x;
    else return (_Float16)x;
  }
};
template <> struct Cvt<bf16> {
  template <typename From> static EK_INLINE bf16 from(From x) {
    if constexpr (__is_same(From, bf16)) return x;
    else if constexpr (__is_same(From, float)) return f32_to_bf16(x);
    else if constexpr (__is_same(From, _Float16)) return f32_to_bf16((float)x);
    else return f32_to_bf16((float)x);
  }
};
template <typename To, typename From> EK_INLINE To cvt(From x) { return Cvt<To>::from(x); }

// Round a float result to the storage type T (identity for non-half types).
template <typename T> EK_INLINE T rnd(float x) { return cvt<T>(x); }

// ---------------------------------------------------------------------------
// Integer arithmetic that never traps: x / 0 gives x, x % 0 gives 0 (matching the
// language's interpreter), and shifts by >= the width give 0 (or the sign fill).
// ---------------------------------------------------------------------------
template <typename T> EK_INLINE T idiv(T a, T b) { return b == (T)0 ? a : (T)(a / b); }
template <typename T> EK_INLINE T imod(T a, T b) { return b == (T)0 ? (T)0 : (T)(a % b); }
template <int N> struct uint_of;
template <> struct uint_of<1> { typedef uint8_t type; };
template <> struct uint_of<2> { typedef uint16_t type; };
template <> struct uint_of<4> { typedef uint32_t type; };
template <> struct uint_of<8> { typedef uint64_t type; };
// The left shift runs on the unsigned type of the same width, so bits shifted into or
// past the sign bit wrap instead of being undefined behaviour; a negative count (huge as
// an unsigned number) or one >= the width gives 0, as NumPy's left_shift does.
template <typename T> EK_INLINE T ishl(T a, T b) {
  typedef typename uint_of<sizeof(T)>::type U;
  return ((uint64_t)b >= sizeof(T) * 8) ? (T)0 : (T)(U)((U)a << b);
}
template <typename T> EK_INLINE T ishr(T a, T b) {
  if ((uint64_t)b >= sizeof(T) * 8) return (T)((T)-1 > (T)0 ? 0 : (a < (T)0 ? (T)-1 : (T)0));
  return (T)(a >> b);
}
EK_INLINE float fmodf_(float a, float b) { return __builtin_fmodf(a, b); }

// erf(x) by Abramowitz & Stegun, Handbook of Mathematical Functions, formula 7.1.26:
// erf(x) = 1 - (a1 t + a2 t^2 + a3 t^3 + a4 t^4 + a5 t^5) exp(-x^2), t = 1 / (1 + p x),
// x >= 0, extended as an odd function; |error| <= 1.5e-7. Branch-free, so it unrolls well
// in register-resident epilogues.
EK_INLINE float erf_as(float x) {
  const float ax = __builtin_fabsf(x);
  // v_rcp_f32 (1 ulp) instead of an IEEE division: t's rounding changes erf by < 1e-7
  const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(0.3275911f, ax, 1.0f));
  float poly = __builtin_fmaf(1.061405429f, t, -1.453152027f);
  poly = __builtin_fmaf(poly, t, 1.421413741f);
  poly = __builtin_fmaf(poly, t, -0.284496736f);
  poly = __builtin_fmaf(poly, t, 0.254829592f);
  poly *= t;
  const float y = 1.0f - poly * __builtin_amdgcn_exp2f(-ax * ax * 1.4426950408889634f);
  return __builtin_copysignf(y, x);
}

// 2^x with the hardware v_exp_f32 (1 ulp; results below 2^-126 flush to zero).
EK_INLINE float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// ---------------------------------------------------------------------------
// Raw vector moves. N is the byte count (1, 2, 4, 8 or 16).
// ---------------------------------------------------------------------------
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template <int N> struct raw_t;
template <> struct raw_t<1> { typedef uint8_t type; };
template <> struct raw_t<2> { typedef uint16_t type; };
template <> struct raw_t<4> { typedef uint32_t type; };
template <> struct raw_t<8> { typedef u32x2 type; };
template <> struct raw_t<16> { typedef u32x4 type; };

template <typename T, int V> EK_INLINE void vload(T* dst, const T* src) {
  typedef typename raw_t<sizeof(T) * V>::type R;
  R v = *reinterpret_cast<const R*>(src);
  __builtin_memcpy(dst, &v, sizeof(R));
}
// Streaming variants: non-temporal hint (data touched once; don't keep it in the caches).
template <typename T, int V> EK_INLINE void vload_nt(T* dst, const T* src) {
  typedef typename raw_t<sizeof(T) * V>::type R;
  R v = __builtin_nontemporal_load(reinterpret_cast<const R*>(src));
  __builtin_memcpy(dst, &v, sizeof(R));
}
template <typename T, int V> EK_INLINE void vstore_nt(T* dst, const T* src) {
  typedef typename raw_t<sizeof(T) * V>::type R;
  R v;
  __builtin_memcpy(&v, src, sizeof(R));
  __builtin_nontemporal_store(v, reinterpret_cast<R*>(dst));
}
template <typename T, int V> EK_INLINE void vstore(T* dst, const T* src) {
  typedef typename raw_t<sizeof(T) * V>::type R;
  R v;
  __builtin_memcpy(&v, src, sizeof(R));
  *reinterpret_cast<R*>(dst) = v;
}

// The same moves at element alignment, for global memory: gfx950 runs vector loads and
// stores at any alignment (the HSA queues' unaligned access mode, which hipcc's amdhsa
// target assumes), so a row that starts at an odd element still moves 16 bytes per lane in
// one instruction. Not for LDS, whose wide accesses need their alignment.
template <typename T, int V> struct raw_u {
  typedef typename raw_t<sizeof(T) * V>::type R;
  typedef R type __attribute__((aligned(sizeof(T))));
};
template <typename T, int V> EK_INLINE void vload_u(T* dst, const T* src) {
  const typename raw_u<T, V>::R v = *reinterpret_cast<const typename raw_u<T, V>::type*>(src);
  __builtin_memcpy(dst, &v, sizeof(v));
}
template <typename T, int V> EK_INLINE void vload_nt_u(T* dst, const T* src) {
  const typename raw_u<T, V>::R v =
      __builtin_nontemporal_load(reinterpret_cast<const typename raw_u<T, V>::type*>(src));
  __builtin_memcpy(dst, &v, sizeof(v));
}
template <typename T, int V> EK_INLINE void vstore_nt_u(T* dst, const T* src) {
  typename raw_u<T, V>::R v;
  __builtin_memcpy(&v, src, sizeof(v));
  __builtin_nontemporal_store(v, reinterpret_cast<typename raw_u<T, V>::type*>(dst));
}
template <typename T, int V> EK_INLINE void vstore_u(T* dst, const T* src) {
  typename raw_u<T, V>::R v;
  __builtin_memcpy(&v, src, sizeof(v));
  *reinterpret_cast<typename raw_u<T, V>::type*>(dst) = v;
}

// A vector read `s` elements early (s >= V: not selected at all), put back in place: element
// i is v[i + s], or o[i] past the vector's end. The vector is shifted as one integer, which
// keeps it in registers whatever `s` is.
template <int N> struct bits_of { typedef unsigned __int128 type; };
template <> struct bits_of<2> { typedef uint16_t type; };
template <> struct bits_of<4> { typedef uint32_t type; };
template <> struct bits_of<8> { typedef uint64_t type; };
template <typename T, int V> EK_INLINE void edge_shift(T* v, int s, const T* o) {
  typedef typename bits_of<sizeof(T) * V>::type U;
  static_assert(sizeof(U) == sizeof(T) * V, "vectors of 2 to 16 bytes");
  constexpr int B = sizeof(T) * 8;
  if (__builtin_amdgcn_ballot_w64(s > 0 && s < V) != 0) {
    U x, f;
    __builtin_memcpy(&x, v, sizeof(U));
    __builtin_memcpy(&f, o, sizeof(U));
    const int n = B * (s & (V - 1));
    const U sel = (U)((U)~(U)0 >> n);         // the V - s elements that were read
    x = (U)((x >> n) & sel) | (U)(f & (U)~sel);
    __builtin_memcpy(v, &x, sizeof(U));
  }
#pragma unroll
  for (int i = 0; i < V; ++i) v[i] = s >= V ? o[i] : v[i];
}

// The V elements that start s < V elements into `v` and go on, past its end, with the first
// ones of `w`.
template <typename T, int V> EK_INLINE void wrap_shift(T* v, int s, const T* w) {
  typedef typename bits_of<sizeof(T) * V>::type U;
  constexpr int B = sizeof(T) * 8;
  U x, y;
  __builtin_memcpy(&x, v, sizeof(U));
  __builtin_memcpy(&y, w, sizeof(U));
  if (s > 0) x = (U)(x >> (B * s)) | (U)(y << (B * (V - s)));
  __builtin_memcpy(v, &x, sizeof(U));
}

// ---------------------------------------------------------------------------
// Wave64 cross-lane moves.
// ---------------------------------------------------------------------------
EK_INLINE int lane_id() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

// Reads `v` from lane `src` (any lane of the wave); ds_bpermute.
EK_INLINE uint32_t shfl_u32(uint32_t v, int src) {
  return (uint32_t)__builtin_amdgcn_ds_bpermute(src << 2, (int)v);
}
template <typename T> EK_INLINE T shfl(T v, int src) {
  if constexpr (sizeof(T) == 8) {
    uint64_t u;
    __builtin_memcpy(&u, &v, 8);
    uint32_t lo = shfl_u32((uint32_t)u, src), hi = shfl_u32((uint32_t)(u >> 32), src);
    u = ((uint64_t)hi << 32) | lo;
    T r;
    __builtin_memcpy(&r, &u, 8);
    return r;
  } else {
    uint32_t u = 0;
    __builtin_memcpy(&u, &v, sizeof(T));
    u = shfl_u32(u, src);
    T r;
    __builtin_memcpy(&r, &u, sizeof(T));
    return r;
  }
}

// A 32-bit exchange with lane ^ MASK that stays in the VALU for every power of two
// (ds_bpermute, the general path, is an LDS round trip that the reductions would wait on):
// - 1, 2: one DPP quad permute ([1,0,3,2] = 0xB1, [2,3,0,1] = 0x4E);
// - 4: row_half_mirror (lane ^ 7), then quad_perm [3,2,1,0] = 0x1B (lane ^ 3);
// - 8: row_mirror (lane ^ 15), then row_half_mirror (lane ^ 7);
// - 16: v_permlane16_swap of the value with itself leaves rows (0,0,2,2) in the first
//   result and rows (1,1,3,3) in the second; a lane takes the other row of its pair;
// - 32: v_permlane32_swap likewise leaves halves (lo,lo) and (hi,hi).
template <int MASK> EK_INLINE uint32_t xor_lanes_u32(uint32_t u) {
  const int x = (int)u;
  if constexpr (MASK == 1 || MASK == 2) {
    return (uint32_t)__builtin_amdgcn_mov_dpp(x, MASK == 1 ? 0xB1 : 0x4E, 0xF, 0xF, false);
  } else if constexpr (MASK == 4) {
    const int t = __builtin_amdgcn_mov_dpp(x, 0x141, 0xF, 0xF, false);
    return (uint32_t)__builtin_amdgcn_mov_dpp(t, 0x1B, 0xF, 0xF, false);
  } else if constexpr (MASK == 8) {
    const int t = __builtin_amdgcn_mov_dpp(x, 0x140, 0xF, 0xF, false);
    return (uint32_t)__builtin_amdgcn_mov_dpp(t, 0x141, 0xF, 0xF, false);
  } else if constexpr (MASK == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return (lane_id() & 16) ? (uint32_t)r[0] : (uint32_t)r[1];
  } else if constexpr (MASK == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return (lane_id() & 32) ? (uint32_t)r[0] : (uint32_t)r[1];
  } else {
    return shfl_u32(u, lane_id() ^ MASK);
  }
}

// Exchange with lane ^ MASK, for values of up to 8 bytes (all lanes active).
template <int MASK, typename T> EK_INLINE T shfl_xor(T v) {
  if constexpr (sizeof(T) == 8) {
    uint64_t u;
    __builtin_memcpy(&u, &v, 8);
    const uint32_t lo = xor_lanes_u32<MASK>((uint32_t)u), hi = xor_lanes_u32<MASK>((uint32_t)(u >> 32));
    u = ((uint64_t)hi << 32) | lo;
    T r;
    __builtin_memcpy(&r, &u, 8);
    return r;
  } else {
    uint32_t u = 0;
    __builtin_memcpy(&u, &v, sizeof(T));
    u = xor_lanes_u32<MASK>(u);
    T r;
    __builtin_memcpy(&r, &u, sizeof(T));
    return r;
  }
}

// One step of a butterfly reduction over lanes: a and the value MASK lanes away combined, for
// values that lanes differing only in the bits below MASK already share. Any lane of the other
// group will then do, so 4 and 8 are one DPP mirror (lane ^ 7, lane ^ 15), which the compiler
// folds into the operation, and 16 and 32 combine the two results of a swap as they are
// (rows 0 and 1 for both, in the same order in every lane) instead of picking one by lane.
template <typename OP, int MASK, typename T> EK_INLINE T reduce_xor(T v) {
  if constexpr (sizeof(T) != 4) {
    return OP::template op<T>(v, shfl_xor<MASK>(v));
  } else {
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    if constexpr (MASK >= 16) {
      const auto r = [&] {
        if constexpr (MASK == 16) return __builtin_amdgcn_permlane16_swap(u, u, false, false);
        else return __builtin_amdgcn_permlane32_swap(u, u, false, false);
      }();
      return OP::template op<T>(__builtin_bit_cast(T, (uint32_t)r[0]),
                                __builtin_bit_cast(T, (uint32_t)r[1]));
    } else {
      constexpr int ctrl = MASK == 1 ? 0xB1 : MASK == 2 ? 0x4E : MASK == 4 ? 0x141 : 0x140;
      return OP::template op<T>(v, __builtin_bit_cast(T, (uint32_t)__builtin_amdgcn_update_dpp(
                                       0, (int)u, ctrl, 0xF, 0xF, true)));
    }
  }
}

// Inclusive prefix sum over lanes 0..63 of a 32-bit value with DPP moves: Kogge-Stone
// inside each 16-lane row (row_shr 1, 2, 4, 8), then row_bcast:15 carries row 0 into
// row 1 and row 2 into row 3, and row_bcast:31 carries lane 31 into rows 2 and 3. Lanes
// whose DPP source is out of range (or outside the row mask) add 0.
template <typename T> EK_INLINE T wave_prefix_sum(T v) {
  static_assert(sizeof(T) == 4, "32-bit values");
  int x = __builtin_bit_cast(int, v);
#define EK_SCAN_STEP(ctrl, rmask)                                                        \
  {                                                                                     \
    const int y = __builtin_amdgcn_update_dpp(0, x, ctrl, rmask, 0xF, false);           \
    x = __builtin_bit_cast(int, __builtin_bit_cast(T, x) + __builtin_bit_cast(T, y));  \
  }
  EK_SCAN_STEP(0x111, 0xF)   // row_shr:1
  EK_SCAN_STEP(0x112, 0xF)   // row_shr:2
  EK_SCAN_STEP(0x114, 0xF)   // row_shr:4
  EK_SCAN_STEP(0x118, 0xF)   // row_shr:8
  EK_SCAN_STEP(0x142, 0xA)   // row_bcast:15 into rows 1 and 3
  EK_SCAN_STEP(0x143, 0xC)   // row_bcast:31 into rows 2 and 3
#undef EK_SCAN_STEP
  return __builtin_bit_cast(T, x);
}

// ---------------------------------------------------------------------------
// Combine functions for reductions and scans.
// ---------------------------------------------------------------------------
struct Sum {
  template <typename T> static EK_INLINE T op(T a, T b) { return a + b; }
};
// Keeps the first operand: the element of a size-1 axis (split of a (2,) tile).
struct First {
  template <typename T> static EK_INLINE T op(T a, T) { return a; }
};
struct Max {
  template <typename T> static EK_INLINE T op(T a, T b) {
    if constexpr (__is_same(T, float)) return __builtin_fmaxf(a, b);
    else return a > b ? a : b;
  }
};
struct Min {
  template <typename T> static EK_INLINE T op(T a, T b) {
    if constexpr (__is_same(T, float)) return __builtin_fminf(a, b);
    else return a < b ? a : b;
  }
};

// ---------------------------------------------------------------------------
// MFMA wrappers (gfx950). Operand registers are passed as arrays of 2-byte elements;
// the accumulator as an array of floats. The array element order is the order of the
// instruction's per-lane operand registers.
// ---------------------------------------------------------------------------
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename V, typename T> EK_INLINE V pack(const T* p) {
  V v;
  __builtin_memcpy(&v, p, sizeof(V));
  return v;
}
template <typename V, typename T> EK_INLINE void unpack(T* p, V v) {
  __builtin_memcpy(p, &v, sizeof(V));
}
typedef int i32x16m __attribute__((ext_vector_type(16)));
typedef int i32x4m __attribute__((ext_vector_type(4)));

// D[32x32] += A[32x16] * B[16x32], fp16/bf16 inputs, 8 elements per lane.
EK_INLINE void mfma_32x32x16(float* acc, const _Float16* a, const _Float16* b) {
  f32x16 c = pack<f32x16>(acc);
  c = __builtin_amdgcn_mfma_f32_32x32x16_f16(pack<f16x8>(a), pack<f16x8>(b), c, 0, 0, 0);
  unpack(acc, c);
}
EK_INLINE void mfma_32x32x16(float* acc, const bf16* a, const bf16* b) {
  f32x16 c = pack<f32x16>(acc);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pack<bf16x8>(a), pack<bf16x8>(b), c, 0, 0, 0);
  unpack(acc, c);
}
// D[16x16] += A[16x32] * B[32x16], 8 elements per lane.
EK_INLINE void mfma_16x16x32(float* acc, const _Float16* a, const _Float16* b) {
  f32x4 c = pack<f32x4>(acc);
  c = __builtin_amdgcn_mfma_f32_16x16x32_f16(pack<f16x8>(a), pack<f16x8>(b), c, 0, 0, 0);
  unpack(acc, c);
}
EK_INLINE void mfma_16x16x32(float* acc, const bf16* a, const bf16* b) {
  f32x4 c = pack<f32x4>(acc);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pack<bf16x8>(a), pack<bf16x8>(b), c, 0, 0, 0);
  unpack(acc, c);
}
// D[32x32] += A[32x8] * B[8x32], 4 elements per lane.
EK_INLINE void mfma_32x32x8(float* acc, const _Float16* a, const _Float16* b) {
  f32x16 c = pack<f32x16>(acc);
  c = __builtin_amdgcn_mfma_f32_32x32x8f16(pack<f16x4>(a), pack<f16x4>(b), c, 0, 0, 0);
  unpack(acc, c);
}
EK_INLINE void mfma_32x32x8(float* acc, const bf16* a, const bf16* b) {
  f32x16 c = pack<f32x16>(acc);
  c = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(pack<s16x4>(a), pack<s16x4>(b), c, 0, 0, 0);
  unpack(acc, c);
}
// D[16x16] += A[16x16] * B[16x16], 4 elements per lane.
EK_INLINE void mfma_16x16x16(float* acc, const _Float16* a, const _Float16* b) {
  f32x4 c = pack<f32x4>(acc);
  c = __builtin_amdgcn_mfma_f32_16x16x16f16(pack<f16x4>(a), pack<f16x4>(b), c, 0, 0, 0);
  unpack(acc, c);
}
EK_INLINE void mfma_16x16x16(float* acc, const bf16* a, const bf16* b) {
  f32x4 c = pack<f32x4>(acc);
  c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(pack<s16x4>(a), pack<s16x4>(b), c, 0, 0, 0);
  unpack(acc, c);
}
// fp32 inputs: D[16x16] += A[16x4] * B[4x16], one element per lane.
EK_INLINE void mfma_16x16x4(float* acc, const float* a, const float* b) {
  f32x4 c = pack<f32x4>(acc);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[0], b[0], c, 0, 0, 0);
  unpack(acc, c);
}
// fp32 inputs: D[32x32] += A[32x2] * B[2x32], one element per lane.
EK_INLINE void mfma_32x32x2(float* acc, const float* a, const float* b) {
  f32x16 c = pack<f32x16>(acc);
  c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[0], b[0], c, 0, 0, 0);
  unpack(acc, c);
}
// int8 inputs, int32 accumulator; integer sums wrap modulo 2^32.
// D[32x32] += A[32x32] * B[32x32], 16 elements per lane (gfx950).
EK_INLINE void mfma_32x32x32(int32_t* acc, const int8_t* a, const int8_t* b) {
  i32x16m c = pack<i32x16m>(acc);
  c = __builtin_amdgcn_mfma_i32_32x32x32_i8(pack<i32x4m>(a), pack<i32x4m>(b), c, 0, 0, 0);
  unpack(acc, c);
}
// D[16x16] += A[16x64] * B[64x16], 16 elements per lane (gfx950).
EK_INLINE void mfma_16x16x64(int32_t* acc, const int8_t* a, const int8_t* b) {
  i32x4m c = pack<i32x4m>(acc);
  c = __builtin_amdgcn_mfma_i32_16x16x64_i8(pack<i32x4m>(a), pack<i32x4m>(b), c, 0, 0, 0);
  unpack(acc, c);
}
// D[32x32] += A[32x16] * B[16x32], 8 elements per lane.
EK_INLINE void mfma_32x32x16(int32_t* acc, const int8_t* a, const int8_t* b) {
  i32x16m c = pack<i32x16m>(acc);
  c = __builtin_amdgcn_mfma_i32_32x32x16_i8(pack<long>(a), pack<long>(b), c, 0, 0, 0);
  unpack(acc, c);
}
// D[16x16] += A[16x32] * B[32x16], 8 elements per lane.
EK_INLINE void mfma_16x16x32(int32_t* acc, const int8_t* a, const int8_t* b) {
  i32x4m c = pack<i32x4m>(acc);
  c = __builtin_amdgcn_mfma_i32_16x16x32_i8(pack<long>(a), pack<long>(b), c, 0, 0, 0);
  unpack(acc, c);
}


EK_INLINE uint32_t perm_lo(uint32_t lo_src, uint32_t hi_src) {
  return __builtin_amdgcn_perm(hi_src, lo_src, 0x05040100u);  // (lo16(lo_src), lo16(hi_src))
}
EK_INLINE uint32_t perm_hi(uint32_t lo_src, uint32_t hi_src) {
  return __builtin_amdgcn_perm(hi_src, lo_src, 0x07060302u);  // (hi16(lo_src), hi16(hi_src))
}

// r[j] holds 8 halves of row j (columns 0..7); o[i] receives column i (rows 0..7).
EK_INLINE void transpose8x8(const u32x4* r, u32x4* o) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int w = i >> 1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t a = r[2 * q][w], b = r[2 * q + 1][w];
      o[i][q] = (i & 1) ? perm_hi(a, b) : perm_lo(a, b);
    }
  }
}

EK_INLINE void transpose8x8(const u32x4* r, u32x4* o, int) { transpose8x8(r, o); }

// r[j] holds 4 halves of row j (columns 0..3); o[i] receives column i (rows 0..7).
EK_INLINE void transpose8x4(const u32x2* r, u32x4* o) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int w = i >> 1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t a = r[2 * q][w], b = r[2 * q + 1][w];
      o[i][q] = (i & 1) ? perm_hi(a, b) : perm_lo(a, b);
    }
  }
}

// Element offset in a staged LDS tile. Lines of 2^LENSH elements are packed 2^LSH to a row of
// PITCH elements; inside its row, a position's group of 2^CSH 8-element chunks is XOR-swizzled
// by ((row >> SA) ^ (row >> SB)) & MASK.
template <int PITCH, int MASK, int SA, int SB, int LSH, int LENSH, int CSH = 0>
EK_INLINE int swz(int line, int sp) {
  const int row = line >> LSH;
  const int vp = ((line & ((1 << LSH) - 1)) << LENSH) | sp;
  if constexpr (MASK == 0) {
    return row * PITCH + vp;
  } else {
    return row * PITCH + (vp ^ ((((row >> SA) ^ (row >> SB)) & MASK) << (3 + CSH)));
  }
}

// Raw buffer loads: the hardware range-checks each access against the resource size and
// returns zeros out of range, so edge tiles need no per-element predicates. Offsets are in
// bytes (< 2^31); a negative or too-large offset reads zeros.
EK_INLINE __amdgpu_buffer_rsrc_t buffer_rsrc(const void* base, uint32_t nbytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)nbytes,
                                           0x00020000);
}
EK_INLINE u32x4 buffer_load16(__amdgpu_buffer_rsrc_t r, int byte_off) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, byte_off, 0, 0));
}
EK_INLINE u32x2 buffer_load8(__amdgpu_buffer_rsrc_t r, int byte_off) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, byte_off, 0, 0));
}
constexpr int kOOB = 0x7ffffff0;  // an offset past any resource: loads read zeros

// ds_read_b64_tr_b16: in each group of 16 lanes, output lane L receives element L % 4 of the
// 8-byte LDS reads made by lanes 4t + L / 4, t = 0..3 (a 4x4 transpose of 16-bit elements).
template <typename T>
EK_INLINE void tr_read4(T* dst, const T* src) {
  typedef short v4s __attribute__((ext_vector_type(4)));
  const v4s v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) v4s*)(src));
  __builtin_memcpy(dst, &v, 8);
}

// tl.device_assert: the first failure claims word 0 and records the assert index and the
// program id (words 1..4); later failures leave the record alone.
EK_INLINE void assert_fail(uint32_t* buf, int index, int px, int py, int pz) {
  uint32_t expected = 0;
  if (__hip_atomic_compare_exchange_strong(buf, &expected, 1u, __ATOMIC_RELAXED,
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
    __hip_atomic_store(buf + 1, (uint32_t)index, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(buf + 2, (uint32_t)px, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(buf + 3, (uint32_t)py, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(buf + 4, (uint32_t)pz, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}
// Two's-complement wrapping add/sub/mul/neg for the language's signed 32/64-bit integers
// (signed overflow is undefined in C++).
EK_INLINE int32_t wadd(int32_t a, int32_t b) { return (int32_t)((uint32_t)a + (uint32_t)b); }
EK_INLINE int32_t wsub(int32_t a, int32_t b) { return (int32_t)((uint32_t)a - (uint32_t)b); }
EK_INLINE int32_t wmul(int32_t a, int32_t b) { return (int32_t)((uint32_t)a * (uint32_t)b); }
EK_INLINE int32_t wneg(int32_t a) { return (int32_t)(0u - (uint32_t)a); }
EK_INLINE int64_t wadd(int64_t a, int64_t b) { return (int64_t)((uint64_t)a + (uint64_t)b); }
EK_INLINE int64_t wsub(int64_t a, int64_t b) { return (int64_t)((uint64_t)a - (uint64_t)b); }
EK_INLINE int64_t wmul(int64_t a, int64_t b) { return (int64_t)((uint64_t)a * (uint64_t)b); }
EK_INLINE int64_t wneg(int64_t a) { return (int64_t)(0ull - (uint64_t)a); }

// Atomic read-modify-write as a compare-and-swap loop: `f(old)` gives the new value. Used for
// the updates without a native instruction: float max/min, value-compare CAS on floats, and
// every 8- and 16-bit element, which is updated inside its aligned 32-bit word (the CAS
// retries when a neighbour in the same word changed). Returns the old value.
template <int N> struct UBits;
template <> struct UBits<1> { typedef uint8_t type; };
template <> struct UBits<2> { typedef uint16_t type; };
template <> struct UBits<4> { typedef uint32_t type; };
template <typename T, typename F> EK_INLINE T atomic_update(T* p, F f) {
  static_assert(sizeof(T) == 1 || sizeof(T) == 2 || sizeof(T) == 4, "8/16/32-bit elements");
  if constexpr (sizeof(T) == 4) {
    uint32_t* w = reinterpret_cast<uint32_t*>(p);
    uint32_t o = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    while (true) {
      const T ov = __builtin_bit_cast(T, o);
      const uint32_t n = __builtin_bit_cast(uint32_t, (T)f(ov));
      if (n == o || __hip_atomic_compare_exchange_strong(w, &o, n, __ATOMIC_RELAXED,
                                                        __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT))
        return ov;
    }
  } else {
    typedef typename UBits<sizeof(T)>::type Bits;
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    uint32_t* w = reinterpret_cast<uint32_t*>(a & ~(uint64_t)3);
    const int sh = (int)(a & 3) * 8;
    const uint32_t m = (uint32_t)(Bits)~(Bits)0 << sh;
    uint32_t o = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    while (true) {
      const T ov = __builtin_bit_cast(T, (Bits)(o >> sh));
      const uint32_t n = (o & ~m) | ((uint32_t)__builtin_bit_cast(Bits, (T)f(ov)) << sh);
      if (n == o || __hip_atomic_compare_exchange_strong(w, &o, n, __ATOMIC_RELAXED,
                                                        __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT))
        return ov;
    }
  }
}

// tl.device_print: 16-bit floats print through float; everything else as itself.
template <typename T> EK_INLINE T f32_or_self(T x) { return x; }
EK_INLINE float f32_or_self(_Float16 x) { return (float)x; }
EK_INLINE float f32_or_self(bf16 x) { return bf16_to_f32(x); }

// Buffer resource as four SGPR words, for the inline-asm copy below.
typedef int i32x4 __attribute__((ext_vector_type(4)));
EK_INLINE i32x4 rsrc_words(const void* base, uint32_t nbytes) {
  const uint64_t b = (uint64_t)base;
  return i32x4{(int)(uint32_t)b, (int)((b >> 32) & 0xffff), (int)nbytes, 0x00020000};
}
// `rows` rows of `cols` 16-bit elements, `ld` elements apart (0, shorter than a row or negative
// too), under 2 GiB in all: the element offset of the lowest row (0, or the last one's where
// they descend), and the bytes from there to the end of the highest.
struct RowSpan {
  int low;
  uint32_t bytes;
  EK_INLINE RowSpan(int rows, int ld, int cols) {
    const int t = (int)((uint32_t)(rows - 1) * (uint32_t)ld);
    low = t < 0 ? t : 0;
    bytes = rows < 1 || cols < 1 ? 0u : ((uint32_t)(t - 2 * low) + (uint32_t)cols) * 2u;
  }
};
// LDS byte address of a pointer into __shared__ memory.
EK_INLINE uint32_t lds_addr(const void* p) {
  return (uint32_t)(uint64_t)(const __attribute__((address_space(3))) void*)p;
}
// One 16-byte-per-lane global -> LDS copy (buffer_load_dwordx4 ... lds): lane l's chunk lands
// at LDS byte `lds + 16 * l` (`lds` is wave-uniform). Issued from inline asm so the compiler
// does not order later LDS reads behind it: the caller waits with an explicit vmcnt.
EK_INLINE void dma16(i32x4 rsrc, uint32_t lds, int voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               ::"s"(lds), "v"(voff), "s"(rsrc) : "memory", "m0");
}

// ---------------------------------------------------------------------------
// Block GEMM loops for `for k in range(lo, hi, BK): acc = dot(A.load([m0, k]),
// B.load([k, n0]), acc)` with row-major 16-bit A [M, K] (lda) and B [K, N] (ldb).
//
// NT threads = WM x WN waves; each wave owns a (BM/WM) x (BN/WN) block of 32x32 MFMA tiles
// (v_mfma_f32_32x32x16_{f16,bf16}). The accumulator is held in the emitter's MFMA layout:
// acc[(tm * TN + tn) * 16 + j]. With TR the instruction computes each tile's transpose
// (B^T A^T, the same fragments in swapped slots), so a lane holds one row of C and 4
// consecutive columns per 4 registers instead of one column and 4 rows.
//
// GemmTile is one stage in LDS and the MFMAs on it: A [BM][BK] and B [BK][BN] row-major in
// 16-byte chunks. A fragments are 16-byte reads; B's k-major fragments come from
// ds_read_b64_tr_b16: in each group of 16 lanes, lane 4i + q reads 4 columns of k row i, and
// output lane L receives column L of the 4 rows. LDS swizzles (reads are served 256 bytes per
// pass): A chunk (row, kc) sits at row * KC + (kc ^ ((row >> ASH) & AMASK)); B chunk (k, nc)
// at k * NCB + (nc ^ (((k >> RSH) & RMASK) << 2)), which spreads the 4 rows a transpose read
// touches over the 4 64-byte quarters of a pass.
// ---------------------------------------------------------------------------
template <typename T, int BM, int BN, int BK, int WM, int WN, int NT, bool TR>
struct GemmTile {
  typedef uint16_t E;                                     // an element in LDS
  static constexpr int EC = 8;                            // elements per chunk
  static constexpr int TM = BM / WM / 32, TN = BN / WN / 32, TK = BK / 16;
  static constexpr int KC = BK / 8;                       // A chunks per row
  static constexpr int NCB = BN / 8;                      // B chunks per row
  static constexpr int A_ELEMS = BM * BK, STAGE = BM * BK + BK * BN;
  static constexpr int ASH = KC >= 16 ? 0 : (KC == 8 ? 1 : (KC == 4 ? 2 : 3));
  static constexpr int AMASK = (KC < 16 ? KC : 16) - 1;
  static constexpr int RP = BN >= 128 ? 1 : 128 / BN;     // B rows per 256 bytes
  static constexpr int RSH = RP == 1 ? 0 : (RP == 2 ? 1 : 2);
  static constexpr int RMASK = 4 / RP - 1;
  static_assert(TM >= 1 && TN >= 1 && TK >= 1, "tile too small for 32x32x16 MFMA");
  static_assert(WM * WN * 64 == NT, "warps must tile the block");
  static_assert(NCB >= 4 * (RMASK + 1), "B swizzle needs the row's chunks");

  static EK_INLINE int a_chunk(int row, int kc) { return row * KC + (kc ^ ((row >> ASH) & AMASK)); }
  static EK_INLINE int b_chunk(int k, int nc) { return k * NCB + (nc ^ (((k >> RSH) & RMASK) << 2)); }

  // One k slice: every A and B fragment read, then the TM x TN MFMAs.
  EK_INLINE void compute_kk(int kk, float* acc, const uint16_t* st, int lane, int wm, int wn) {
    typedef short v4s __attribute__((ext_vector_type(4)));
    const u32x4* sA = reinterpret_cast<const u32x4*>(st);
    const uint16_t* sB = st + A_ELEMS;
    const int r32 = lane & 31, h = lane >> 5;
    const int g = lane >> 4, ti = (lane >> 2) & 3, tq = lane & 3;
    T a[TM][8], b[TN][8];
    const int kc = kk * 2 + h;
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
      const u32x4 v = sA[a_chunk(wm * (BM / WM) + tm * 32 + r32, kc)];
      __builtin_memcpy(a[tm], &v, 16);
    }
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      const int n = wn * (BN / WN) + tn * 32 + 16 * (g & 1) + 4 * tq;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int k = kk * 16 + 8 * (g >> 1) + 4 * half + ti;
        const uint16_t* src = sB + b_chunk(k, n >> 3) * 8 + (n & 7);
        const v4s v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) v4s*)(src));
        __builtin_memcpy(&b[tn][4 * half], &v, 8);
      }
    }
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) {
        if constexpr (TR) mfma_32x32x16(&acc[(tm * TN + tn) * 16], b[tn], a[tm]);
        else mfma_32x32x16(&acc[(tm * TN + tn) * 16], a[tm], b[tn]);
      }
  }

  template <int KK0, int KK1>
  EK_INLINE void compute(float* acc, const uint16_t* st, int lane, int wm, int wn) {
#pragma unroll
    for (int kk = KK0; kk < KK1; ++kk) compute_kk(kk, acc, st, lane, wm, wn);
  }
};

// The same for fp32 operands: 16-byte chunks of 4 elements, v_mfma_f32_32x32x2_f32 (one element
// per lane: lanes 32..63 hold the odd k of a pair). A fragments are 16-byte reads, four k of a
// row at a time (both halves of the wave read the same chunk and pick their k); B's are one
// word per lane from two neighbouring rows, whose 128-byte runs the swizzle keeps in different
// halves of the banks. The pairs run in k order, as the dot's own lowering has them.
template <int BM, int BN, int BK, int WM, int WN, int NT, bool TR>
struct GemmTile<float, BM, BN, BK, WM, WN, NT, TR> {
  typedef float E;
  static constexpr int EC = 4;
  static constexpr int TM = BM / WM / 32, TN = BN / WN / 32, TK = BK / 4;
  static constexpr int KC = BK / 4, NCB = BN / 4;
  static constexpr int A_ELEMS = BM * BK, STAGE = BM * BK + BK * BN;
  static constexpr int ASH = KC >= 16 ? 0 : (KC == 8 ? 1 : 2);
  static constexpr int AMASK = (KC < 16 ? KC : 16) - 1;
  static constexpr int ODD = NCB >= 16 ? 8 : 0;
  static_assert(!TR, "fp32 dots keep the instruction's orientation");
  static_assert(TM >= 1 && TN >= 1 && KC >= 4, "tile too small for 32x32x2 MFMA");
  static_assert(WM * WN * 64 == NT, "warps must tile the block");

  static EK_INLINE int a_chunk(int row, int kc) { return row * KC + (kc ^ ((row >> ASH) & AMASK)); }
  static EK_INLINE int b_chunk(int k, int nc) { return k * NCB + (nc ^ ((k & 1) * ODD)); }

  template <int KK0, int KK1>
  EK_INLINE void compute(float* acc, const float* st, int lane, int wm, int wn) {
    const f32x4* sA = reinterpret_cast<const f32x4*>(st);
    const float* sB = st + A_ELEMS;
    const int r32 = lane & 31, h = lane >> 5;
#pragma unroll
    for (int q = KK0; q < KK1; ++q) {
      f32x4 a[TM];
      float b[2][TN];
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) a[tm] = sA[a_chunk(wm * (BM / WM) + tm * 32 + r32, q)];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) {
          const int n = wn * (BN / WN) + tn * 32 + r32;
          b[j][tn] = sB[b_chunk(q * 4 + 2 * j + h, n >> 2) * 4 + (n & 3)];
        }
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
          const float av = h ? a[tm][2 * j + 1] : a[tm][2 * j];
#pragma unroll
          for (int tn = 0; tn < TN; ++tn) mfma_32x32x2(&acc[(tm * TN + tn) * 16], &av, &b[j][tn]);
        }
    }
  }
};

// How a loop goes through its n steps: one after the other, or, where one workgroup takes the
// slices of a split k loop in turn (see split_reduce), in slices of `per` steps: at each slice's
// end the accumulator is added to the sum of those before and starts again from zero, so that
// the result has the bits of slices computed apart. A loop that can runs up to `end` and
// asks for `more` (fp16 64 x 4096 x 4096 at 64x64x128, captured: 22.7 us as one slice, 24.7
// in 4, 25.7 with a test in each step; 512 x 512 x 8192 at 128x128x64: 83.4 and 82.9 in 7; at
// 256x256x64, where accumulators and sums do not fit the registers, 145 and 174 in 7).
// Otherwise it calls `begin` before each step.
struct OneSlice {
  EK_INLINE int end(int, int n) { return n; }
  EK_INLINE bool more(int, int) { return false; }
  EK_INLINE void begin(int) {}
};
template <int R> struct SliceSum {
  float* acc;
  float sum[R];
  int per, next;
  EK_INLINE SliceSum(float* acc_, int per_) : acc(acc_), per(per_), next(per_) {
#pragma unroll
    for (int r = 0; r < R; ++r) sum[r] = 0.0f;
  }
  EK_INLINE void fold() {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      sum[r] += acc[r];
      acc[r] = 0.0f;
    }
  }
  EK_INLINE int end(int it, int n) { return Min::op<int>(next = it + per, n); }
  EK_INLINE bool more(int it, int n) {
    if (it == next) fold();
    return it < n;
  }
  EK_INLINE void begin(int it) {
    if (it == next) {
      fold();
      next += per;
    }
  }
  EK_INLINE void finish() {
    fold();
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = sum[r];
  }
};

// ---------------------------------------------------------------------------
// The loop for operands of any alignment and size, through registers: each thread loads its
// 16-byte chunks of the tile PD steps ahead (element-aligned vector loads) and writes the tile
// that has arrived to the other of two LDS stages, one barrier per step.
//
// What bounds it: with rows at odd element offsets there is no LDS DMA and no aligned chunk,
// so the loads' latency has to be covered from registers (PD steps of them) and each byte
// crosses the VGPRs. Edges cost no per-element loads: a chunk past the last row or column is
// read from the last row, or from the row's last 8 columns and shifted into place, so every
// address lies inside the operand; offsets are fixed before the loop (one set for the last k
// step, which may be ragged). Operands narrower than a chunk, and tiles that start before the
// operand, are read element by element.
// ---------------------------------------------------------------------------
template <typename T, int BM, int BN, int BK, int WM, int WN, int NT, bool BIG, bool TR = false>
struct GemmReg : GemmTile<T, BM, BN, BK, WM, WN, NT, TR> {
  typedef GemmTile<T, BM, BN, BK, WM, WN, NT, TR> G;
  using G::TK, G::KC, G::NCB, G::A_ELEMS, G::STAGE, G::EC;
  typedef typename G::E E;
  static constexpr int ES = sizeof(E);
  static constexpr int A_TOT = BM * KC, B_TOT = BK * NCB;
  static constexpr int A_CH = (A_TOT + NT - 1) / NT, B_CH = (B_TOT + NT - 1) / NT;
  static constexpr int CH = A_CH + B_CH;
  // k steps of loads in flight: about 32 registers' worth (64x64x32 tiles on 4 waves, bf16
  // 1000 x 3000 x 2000: 35.6 us at 4 steps, 38.9 at 1; 256x256x64 on 8 waves spills at 2)
  static constexpr int PD = CH <= 2 ? 4 : CH <= 4 ? 2 : 1;
  static constexpr int LDS_BYTES = 2 * STAGE * ES;
  // byte offsets from a tile's k origin: 32 bits, or 64 for operands of 2 GiB and more
  template <bool> struct off_of { typedef uint32_t type; };
  template <> struct off_of<true> { typedef int64_t type; };
  typedef typename off_of<BIG>::type Off;
  typedef typename raw_u<E, EC>::type chunk;

  u32x4 r[PD][CH];
  // Of each chunk, from a k step's first column less EC (A: a chunk moved back from a ragged
  // end starts up to EC - 1 columns before it) or first row (B), and there from the lowest of
  // the operand's (A) or the step's (B) rows, which is the last one where rows descend (a
  // negative row stride): 32-bit offsets are unsigned.
  Off off[CH], last[CH];    // of every k step, and of the last one
  int sh[CH], lsh[CH];      // elements to shift (EC and more: all zero), likewise

  static EK_INLINE int row_a(int i, int tid) { return (i * NT + tid) / KC; }
  static EK_INLINE int kc_a(int i, int tid) { return (i * NT + tid) % KC; }
  static EK_INLINE int row_b(int i, int tid) { return (i * NT + tid) / NCB; }
  static EK_INLINE int nc_b(int i, int tid) { return (i * NT + tid) % NCB; }
  // whether chunk i exists for this thread (always, when the tile fills the threads evenly)
  static EK_INLINE bool has(int i, int tid) {
    if (i < A_CH) return A_TOT % NT == 0 || i * NT + tid < A_TOT;
    return B_TOT % NT == 0 || (i - A_CH) * NT + tid < B_TOT;
  }

  EK_INLINE void plan(int lda, int ldb, int M, int N, int K, int m0, int n0, int klast, Off low_a,
                      Off low_b, int tid) {
#pragma unroll
    for (int i = 0; i < A_CH; ++i) {
      const int row = m0 + row_a(i, tid), rc = Min::op<int>(row, M - 1), c = kc_a(i, tid) * EC;
      const int cl = Min::op<int>(klast + c, K - EC) - klast;    // 1 - EC and more
      const Off at = (Off)rc * (Off)lda - low_a;
      off[i] = (at + (Off)(c + EC)) * ES;
      last[i] = (at + (Off)(cl + EC)) * ES;
      sh[i] = row < M ? 0 : EC;
      lsh[i] = row < M ? c - cl : EC;
    }
#pragma unroll
    for (int j = 0; j < B_CH; ++j) {
      const int i = A_CH + j, k = row_b(j, tid), gn = n0 + nc_b(j, tid) * EC;
      const int kl = Min::op<int>(klast + k, K - 1) - klast, nl = Min::op<int>(gn, N - EC);
      off[i] = ((Off)k * (Off)ldb - low_b + (Off)nl) * ES;
      last[i] = ((Off)kl * (Off)ldb - low_b + (Off)nl) * ES;
      sh[i] = gn - nl;
      lsh[i] = kl == k ? gn - nl : EC;
    }
  }

  EK_INLINE void load(int p, const char* a, const char* b, bool end, int tid) {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const char* q = (i < A_CH ? a : b) + (end ? last[i] : off[i]);
      if (has(i, tid)) r[p][i] = *reinterpret_cast<const chunk*>(q);
    }
  }

  EK_INLINE void put(int p, E* st, int tid) {
    u32x4* sA = reinterpret_cast<u32x4*>(st);
    u32x4* sB = reinterpret_cast<u32x4*>(st + A_ELEMS);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      if (!has(i, tid)) continue;
      if (i < A_CH) sA[G::a_chunk(row_a(i, tid), kc_a(i, tid))] = r[p][i];
      else sB[G::b_chunk(row_b(i - A_CH, tid), nc_b(i - A_CH, tid))] = r[p][i];
    }
  }

  EK_INLINE void shift(int p, bool end) {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int s = end ? lsh[i] : sh[i];
      unsigned __int128 x = __builtin_bit_cast(unsigned __int128, r[p][i]);
      x = s >= EC ? 0 : x >> (8 * ES * (s & (EC - 1)));
      r[p][i] = __builtin_bit_cast(u32x4, x);
    }
  }

  // One element of an operand [rows, cols], zero outside it.
  static EK_INLINE E elem(const T* P, int64_t ld, int rows, int cols, int i, int j) {
    if (i < 0 || i >= rows || j < 0 || j >= cols) return 0;
    return reinterpret_cast<const E*>(P)[i * ld + j];
  }

  // Runs the whole k loop: k = lo, lo + BK, ... < hi.
  template <typename At = OneSlice>
  EK_INLINE void run(float* acc, const T* A, int lda, const T* B, int ldb, int M, int N, int K,
                     int m0, int n0, int lo, int hi, char* smem, int tid, At&& at = At{}) {
    hi = Min::op<int>(hi, K);   // past K both operands are zero
    if (hi <= lo) return;
    const int niter = (int)(((int64_t)hi - lo + BK - 1) / BK);
    const int lane = tid & 63, warp = tid >> 6;
    const int wm = warp % WM, wn = warp / WM;
    E* sm = reinterpret_cast<E*>(smem);
    __syncthreads();  // earlier users of the LDS are done with it
    if (m0 < 0 || n0 < 0 || lo < 0 || M < 1 || N < EC || K < EC) {
      for (int it = 0; it < niter; ++it) {
        const int k = lo + it * BK;
        for (int c = tid; c < BM * BK; c += NT)
          sm[G::a_chunk(c / BK, (c % BK) / EC) * EC + c % EC] =
              elem(A, lda, M, K, m0 + c / BK, k + c % BK);
        for (int c = tid; c < BK * BN; c += NT)
          sm[A_ELEMS + G::b_chunk(c / BN, (c % BN) / EC) * EC + c % EC] =
              elem(B, ldb, K, N, k + c / BN, n0 + c % BN);
        __syncthreads();
        at.begin(it);
        G::template compute<0, TK>(acc, sm, lane, wm, wn);
        __syncthreads();
      }
      return;
    }
    const int klast = lo + (niter - 1) * BK;
    const bool edge = m0 + BM > M || n0 + BN > N, ragged = klast + BK > K;
    const int64_t low_a = lda < 0 ? (int64_t)(M - 1) * lda : 0;
    const int64_t low_b = ldb < 0 ? (int64_t)(Min::op<int>(BK, K) - 1) * ldb : 0;
    plan(lda, ldb, M, N, K, m0, n0, klast, (Off)low_a, (Off)low_b, tid);
    const char* a = reinterpret_cast<const char*>(A) + (low_a + lo - EC) * ES;
    const char* b = reinterpret_cast<const char*>(B) + ((int64_t)lo * ldb + low_b) * ES;
    const int64_t sa = BK * ES, sb = (int64_t)BK * ldb * ES;
#pragma unroll
    for (int p = 0; p < PD; ++p) {
      const int t = Min::op<int>(p, niter - 1);
      load(p, a + t * sa, b + t * sb, t == niter - 1, tid);
    }
    for (int it = 0, stop = PD == 1 ? at.end(0, niter) : niter;; stop = at.end(it, niter)) {
      for (; it < stop; it += PD) {
#pragma unroll
        for (int p = 0; p < PD; ++p) {
          const int t = it + p;
          if (t >= niter) break;
          const bool end = t == niter - 1;
          if (edge || (end && ragged)) shift(p, end);
          E* st = sm + (PD % 2 ? (t & 1) : (p & 1)) * STAGE;
          put(p, st, tid);
          // past the end: the last tile again, which nothing reads
          const int nx = Min::op<int>(t + PD, niter - 1);
          load(p, a + nx * sa, b + nx * sb, nx == niter - 1, tid);
          asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
          if constexpr (PD > 1) at.begin(t);
          G::template compute<0, TK>(acc, st, lane, wm, wn);
        }
      }
      if (PD > 1 || !at.more(it, niter)) break;
    }
    __syncthreads();
  }
};

// The same loop, named so in kernels whose operands' rows are known to start on 16 bytes (K or N,
// or the tile's origin, are no whole chunks): only the chunks moved at an edge are unaligned there.
template <typename T, int BM, int BN, int BK, int WM, int WN, int NT, bool BIG, bool TR = false>
using Gemm = GemmReg<T, BM, BN, BK, WM, WN, NT, BIG, TR>;

// ---------------------------------------------------------------------------
// GEMM main loop fed by LDS DMA: C[BM x BN] += A[BM x K] * B[K x BN], 16-bit row-major
// operands, fp32 accumulators in the 32x32x16 MFMA layout (GemmTile).
//
//  - Tiles move global -> LDS with buffer_load ... lds (16 bytes per lane, no VGPRs): the 64
//    lanes of one instruction fill 64 consecutive 16-byte LDS chunks, so each lane fetches
//    the global chunk that belongs at its LDS position under the swizzle below. Chunks past
//    the last column, and of rows of A past the last, are sent out of the buffer resource's
//    range and arrive as zeros (K and N are multiples of 8); rows of B past K lie outside it.
//    Row strides may be anything: 0, shorter than the row, negative.
//  - S stages in LDS; S - 1 tiles are in flight while one is computed. A stage is waited
//    for with an explicit vmcnt (this wave's copies) and a barrier (everyone's), which also
//    frees the stage consumed one step earlier for the next copy.
//  - A fragments are 16-byte LDS reads; B stays row-major in LDS and its k-major fragments
//    come from ds_read_b64_tr_b16: in each group of 16 lanes, lane 4i + q reads 4 columns of
//    k row i, and output lane L receives column L of the 4 rows.
//  - LDS swizzles (reads are served 256 bytes per pass): A chunk (row, kc) sits at
//    row * KC + (kc ^ ((row >> ASH) & AMASK)); B chunk (k, nc) at
//    k * NCB + (nc ^ (((k >> RSH) & RMASK) << 2)), which spreads the 4 rows a transpose
//    read touches over the 4 64-byte quarters of a pass.
// ---------------------------------------------------------------------------
template <typename T, int BM, int BN, int BK, int WM, int WN, int NT, int S, int SPLIT = 1,
          bool TR = false>
struct GemmDma : GemmTile<T, BM, BN, BK, WM, WN, NT, TR> {
  typedef GemmTile<T, BM, BN, BK, WM, WN, NT, TR> G;
  using G::TK, G::KC, G::NCB, G::A_ELEMS, G::STAGE, G::ASH, G::AMASK, G::RSH, G::RMASK;
  static constexpr int A_DMA = BM * KC / NT;              // copies per thread per stage
  static constexpr int B_DMA = BK * NCB / NT;
  static constexpr int D = A_DMA + B_DMA;
  static constexpr int LDS_BYTES = S * STAGE * 2;
  static_assert((BM * KC) % NT == 0 && (BK * NCB) % NT == 0, "tile/thread mismatch");
  static_assert(S >= 2 && (S - 2) * D <= 63, "vmcnt range");
  static_assert(SPLIT >= 0 && SPLIT <= TK, "copies issue after SPLIT of the TK k slices");

  // Per-thread copy plan, fixed for the whole loop: the global element offset of each chunk
  // relative to the k origin, from the operand's lowest row on. A chunk of a row of A outside it
  // has an offset past every resource at any k; one of a column of B, -1.
  static constexpr int kFar = 0x40000400;
  int a_off[A_DMA], b_off[B_DMA], a_kc[A_DMA];

  EK_INLINE void plan(int lda, int ldb, int M, int N, int m0, int n0, int low_a, int low_b,
                      int tid) {
#pragma unroll
    for (int i = 0; i < A_DMA; ++i) {
      const int p = i * NT + tid, row = p / KC;
      const int kc = (p % KC) ^ ((row >> ASH) & AMASK);
      a_kc[i] = kc * 8;
      a_off[i] = (unsigned)(m0 + row) < (unsigned)M ? (m0 + row) * lda - low_a + kc * 8 : kFar;
    }
#pragma unroll
    for (int i = 0; i < B_DMA; ++i) {
      const int p = i * NT + tid, k = p / NCB;
      const int nc = (p % NCB) ^ (((k >> RSH) & RMASK) << 2);
      const int gn = n0 + nc * 8;
      b_off[i] = (unsigned)gn < (unsigned)N ? k * ldb - low_b + gn : -1;
    }
  }

  static EK_INLINE int bytes(int elems) { return (int)((uint32_t)elems * 2u); }

  // Copies the k-th tile (k = first column of A / row of B) into the stage at LDS byte `st`.
  EK_INLINE void copy(i32x4 ra, i32x4 rb, int ldb, int K, int k, uint32_t st, int wave) {
    if (k + BK <= K) {
      // the whole k slice lies inside A: no per-chunk column test
#pragma unroll
      for (int i = 0; i < A_DMA; ++i) dma16(ra, st + (i * NT + wave * 64) * 16, bytes(a_off[i] + k));
    } else {
#pragma unroll
      for (int i = 0; i < A_DMA; ++i) {
        const int off = (k + a_kc[i] + 8 <= K) ? bytes(a_off[i] + k) : kOOB;
        dma16(ra, st + (i * NT + wave * 64) * 16, off);
      }
    }
#pragma unroll
    for (int i = 0; i < B_DMA; ++i) {
      const int off = b_off[i] >= 0 ? bytes(b_off[i] + k * ldb) : kOOB;
      dma16(rb, st + A_ELEMS * 2 + (i * NT + wave * 64) * 16, off);
    }
  }

  // The j-th of this thread's D copies of the k-th tile (j < A_DMA: A, else B).
  EK_INLINE void copy_one(int j, i32x4 ra, i32x4 rb, int ldb, int K, int k, uint32_t st,
                          int wave) {
    if (j < A_DMA) {
      const int off = (k + BK <= K || k + a_kc[j] + 8 <= K) ? bytes(a_off[j] + k) : kOOB;
      dma16(ra, st + (j * NT + wave * 64) * 16, off);
    } else {
      const int i = j - A_DMA;
      const int off = b_off[i] >= 0 ? bytes(b_off[i] + k * ldb) : kOOB;
      dma16(rb, st + A_ELEMS * 2 + (i * NT + wave * 64) * 16, off);
    }
  }

  // Runs the whole k loop: k = lo, lo + BK, ... < hi.
  template <typename At = OneSlice>
  EK_INLINE void run(float* acc, const T* A, int lda, const T* B, int ldb, int M, int N, int K,
                     int m0, int n0, int lo, int hi, char* smem, int tid, At&& at = At{}) {
    hi = Min::op<int>(hi, K);   // past K both operands are zero
    if (hi <= lo) return;
    const int niter = (hi - lo + BK - 1) / BK;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM;
    // Resources over the rows' elements and nothing else. Rows of B past K lie outside them
    // while rows do not overlap; where they do (also: coincide), or are so far apart that 32-bit
    // offsets past K wrap around, the address does not tell, and a ragged last step runs after
    // the loop on a stage cleared of them (fp16 64 x 4096 x 4096 + GELU: 14.0 us; 14.5 with a
    // test on each copy or a branch in each step).
    const RowSpan sa(M, lda, K), sb(K, ldb, N);
    const i32x4 ra = rsrc_words(A + sa.low, sa.bytes);
    const i32x4 rb = rsrc_words(B + sb.low, sb.bytes);
    const int klast = lo + (niter - 1) * BK;
    const int gap = ldb < 0 ? -ldb : ldb;
    const bool apart = klast + BK > K && (gap < N || gap > (1 << 30) / BK);
    const int nloop = niter - apart;
    uint16_t* s16 = reinterpret_cast<uint16_t*>(smem);
    const uint32_t l0 = lds_addr(smem);
    plan(lda, ldb, M, N, m0, n0, sa.low, sb.low, tid);
    __syncthreads();  // earlier users of the LDS are done with it
    // nothing loaded before the loop is outstanding, so the explicit vmcnt below counts
    // this loop's copies only
    __builtin_amdgcn_s_waitcnt(0x0F70);
#pragma unroll
    for (int s = 0; s < S - 1; ++s) copy(ra, rb, ldb, K, lo + s * BK, l0 + s * STAGE * 2, wave);
    for (int it = 0, stop = at.end(0, nloop);; stop = at.end(it, nloop)) {
      for (; it < stop; ++it) {
        // this wave's copies of stage `it` have landed (S - 2 younger stages may still fly),
        // its reads of the previous stage are complete; then everyone's are.
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((S - 2) * D) : "memory");
        // The first SPLIT k slices' fragment reads go out before any copy, so their latency
        // hides behind the copy issue instead of stalling the first MFMA; the copies of the
        // stage S - 1 ahead are then spread over the remaining slices, a share before each
        // slice's reads, so each share's issue overlaps the MFMAs already queued (as one block
        // the copies kept the wave from issuing for 500-800 cycles per k step).
        const uint16_t* cur = s16 + (it % S) * STAGE;
        G::template compute<0, SPLIT>(acc, cur, lane, wm, wn);
        if constexpr (SPLIT < TK) {
          constexpr int SL = TK - SPLIT, PER = (D + SL - 1) / SL;
          const int kn = lo + (it + S - 1) * BK;
          const uint32_t stn = l0 + ((it + S - 1) % S) * STAGE * 2;
#pragma unroll
          for (int q = 0; q < SL; ++q) {
#pragma unroll
            for (int j = q * PER; j < (q + 1) * PER && j < D; ++j)
              copy_one(j, ra, rb, ldb, K, kn, stn, wave);
            G::compute_kk(SPLIT + q, acc, cur, lane, wm, wn);
          }
        } else {
          copy(ra, rb, ldb, K, lo + (it + S - 1) * BK, l0 + ((it + S - 1) % S) * STAGE * 2, wave);
        }
      }
      if (!at.more(it, nloop)) break;
    }
    // drain the copies issued past the end before anyone reuses the LDS
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (__builtin_expect(apart, 0)) {
      uint16_t* const st = s16 + ((niter - 1) % S) * STAGE;
      u32x4* const rows = reinterpret_cast<u32x4*>(st + A_ELEMS);
      for (int p = Max::op<int>(K - klast, 0) * NCB + tid; p < BK * NCB; p += NT)
        rows[p] = u32x4{0, 0, 0, 0};
      __syncthreads();
#pragma unroll 1
      for (int kk = 0; kk < TK; ++kk) G::compute_kk(kk, acc, st, lane, wm, wn);
      __syncthreads();
    }
  }
};

// ---------------------------------------------------------------------------
// Split k loops. A grid with few tiles leaves most CUs idle while each workgroup walks the
// whole k range, one tile's latency after another; the launcher then starts ns = gridDim.z
// workgroups per tile, each on a slice of k. Every workgroup stores its accumulator (registers
// as they are, NT lanes side by side) to its row of the workspace and counts itself in; the
// last one of a tile adds all rows in slice order (so the sum does not depend on who is last),
// clears the tile's counter for the next launch and returns true: it runs the epilogue.
// Launches that find no workspace run one workgroup per tile, which walks the same slices in the
// same order (SliceSum): whether a launch had a workspace shows in its time, not in its bits.
//
// The partial rows go through relaxed agent-scope atomics, which write to and read from memory
// past the XCDs' private L2s; a vmcnt wait before the count makes sure that they are there. That
// costs the rows alone, where an agent-scope release or acquire fence writes back or drops
// a whole L2.
// ---------------------------------------------------------------------------
constexpr int kSplitCounters = 16384;     // words at the start of the workspace: one per tile

EK_INLINE int split_slice(int lo, int hi, int bk, int ns) {   // k extent of one slice
  const int steps = (hi - lo + bk - 1) / bk;
  return (steps + ns - 1) / ns * bk;
}

template <int R, int NT>
EK_INLINE bool split_reduce(float* acc, float* ws, char* smem, int tid) {
  constexpr int P = R / 2;                // pairs of accumulator registers: 8-byte accesses
  constexpr int U = R <= 16 ? 4 : R <= 64 ? 2 : 1;   // rows in flight while they are added
  static_assert(R % 2 == 0, "pairs of registers");
  const int ns = gridDim.z, tile = blockIdx.x + gridDim.x * blockIdx.y;
  uint32_t* count = reinterpret_cast<uint32_t*>(ws) + tile;
  uint64_t* rows = reinterpret_cast<uint64_t*>(ws + kSplitCounters) +
                   (int64_t)tile * ns * (P * NT) + tid;
  uint64_t* mine = rows + (int64_t)blockIdx.z * (P * NT);
#pragma unroll
  for (int r = 0; r < P; ++r) {
    uint64_t v;
    __builtin_memcpy(&v, &acc[2 * r], 8);
    __hip_atomic_store(mine + r * NT, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  uint32_t* last = reinterpret_cast<uint32_t*>(smem);
  __syncthreads();   // every lane's rows are in memory; the LDS is free
  if (tid == 0)
    *last = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
            (uint32_t)ns - 1;
  __syncthreads();
  if (*last == 0) return false;
  if (tid == 0) __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = 0.0f;
  for (int z = 0; z < ns; z += U) {
    uint64_t part[U][P];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int zr = z + u < ns ? z + u : ns - 1;
#pragma unroll
      for (int r = 0; r < P; ++r)
        part[u][r] = __hip_atomic_load(rows + (int64_t)zr * (P * NT) + r * NT, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (z + u >= ns) break;
#pragma unroll
      for (int r = 0; r < P; ++r) {
        float v[2];
        __builtin_memcpy(v, &part[u][r], 8);
        acc[2 * r] += v[0];
        acc[2 * r + 1] += v[1];
      }
    }
  }
  __syncthreads();   // `last` is read; the epilogue may use the LDS
  return true;
}

}  // namespace ek
