// device_io.h -- element I/O and wave reductions shared by this library's gfx950 kernels: eight-element vectors of bf16,
// fp16 or fp32 in and out of fp32 registers, at vector and at element alignment, and sums over lanes of a wave.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#ifndef LDR_F32_NT
#define LDR_F32_NT 1         // the reads' fp32 sources streamed non-temporally, as 16-bit ones
#endif
#ifndef LDR_NT
#define LDR_NT 1             // non-temporal loads for the streamed sources
#endif

namespace {

typedef uint16_t bf16_t;                // bf16 storage (raw bits)
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

// ---------------------------------------------------------------------------------------------------------------
// element I/O: 8 elements (one 16-byte bf16 or fp16 vector, or two fp32 float4) <-> 8 fp32 registers
// ---------------------------------------------------------------------------------------------------------------
template <typename T> struct IO;

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// bf16 <-> fp32: the upper 16 bits of the fp32 pattern; v_cvt_pk_bf16_f32 rounds to nearest even, NaN stays NaN
struct Bf16Cvt {
  static __device__ __forceinline__ void unpack2(uint32_t w, float& a, float& b) {
    a = __uint_as_float(w << 16);
    b = __uint_as_float(w & 0xffff0000u);
  }
  static __device__ __forceinline__ uint32_t pack2(float a, float b) {
    bf16x2_t v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, v);
  }
  static __device__ __forceinline__ float round(float x) { return (float)(__bf16)x; }
};
__device__ __forceinline__ uint32_t pack2(float a, float b) { return Bf16Cvt::pack2(a, b); }

// fp32 -> fp16 of the fp32 value: v_cvt_f16_f32 (round to nearest even; subnormals kept, overflow to inf). The empty
// asm holds x as an fp32 register value, so the compiler cannot fold the conversion into the operation that produced
// x (a v_fma_mixlo_f16 rounds the exact product or sum once, straight to fp16, which differs from rounding the fp32
// result in rare cases): every fp16 result is the fp32 result rounded, as torch's conversions round it.
__device__ __forceinline__ _Float16 to_f16(float x) {
  asm("" : "+v"(x));
  return (_Float16)x;
}

// fp16 <-> fp32: v_cvt_f32_f16 (exact) and to_f16
struct F16Cvt {
  static __device__ __forceinline__ void unpack2(uint32_t w, float& a, float& b) {
    a = (float)__builtin_bit_cast(_Float16, (uint16_t)(w & 0xffffu));
    b = (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16));
  }
  static __device__ __forceinline__ uint32_t pack2(float a, float b) {
    return (uint32_t)__builtin_bit_cast(uint16_t, to_f16(a)) |
           ((uint32_t)__builtin_bit_cast(uint16_t, to_f16(b)) << 16);
  }
  static __device__ __forceinline__ float round(float x) { return (float)to_f16(x); }
};

// 16-bit elements (bf16, fp16): one 16-byte vector of 8 elements; the sign is bit 15 of each half-word in both
template <typename T, typename Cvt> struct IO16 {
  struct Raw { uint4 u; };
  static __device__ __forceinline__ Raw raw(const T* p) { Raw r; r.u = *reinterpret_cast<const uint4*>(p); return r; }
  // non-temporal: for data read once per kernel and not again soon (the update stack, the output gradient)
  static __device__ __forceinline__ Raw raw_nt(const T* p) {
    Raw r;
#if LDR_NT
    const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
    r.u = make_uint4(v.x, v.y, v.z, v.w);
#else
    r.u = *reinterpret_cast<const uint4*>(p);
#endif
    return r;
  }
  static __device__ __forceinline__ Raw raw_str(const T* p) { return raw_nt(p); }   // the reads' source stream
  static __device__ __forceinline__ Raw zero() { Raw r; r.u = make_uint4(0u, 0u, 0u, 0u); return r; }
  static __device__ __forceinline__ void unpack(const Raw& r, float (&o)[8]) {
    Cvt::unpack2(r.u.x, o[0], o[1]); Cvt::unpack2(r.u.y, o[2], o[3]);
    Cvt::unpack2(r.u.z, o[4], o[5]); Cvt::unpack2(r.u.w, o[6], o[7]);
  }
  static __device__ __forceinline__ void load(const T* p, float (&o)[8]) { unpack(raw(p), o); }
  static __device__ __forceinline__ void store(T* p, const float (&o)[8]) {
    uint4 u;
    u.x = Cvt::pack2(o[0], o[1]); u.y = Cvt::pack2(o[2], o[3]);
    u.z = Cvt::pack2(o[4], o[5]); u.w = Cvt::pack2(o[6], o[7]);
    *reinterpret_cast<uint4*>(p) = u;
  }
  // non-temporal stores, for results not read again soon (the update gradients): they stream to HBM instead of
  // displacing the rows the next launches re-read from the caches
  static __device__ __forceinline__ void store_nt(T* p, const float (&o)[8]) {
    const u32x4 u{Cvt::pack2(o[0], o[1]), Cvt::pack2(o[2], o[3]), Cvt::pack2(o[4], o[5]), Cvt::pack2(o[6], o[7])};
    __builtin_nontemporal_store(u, reinterpret_cast<u32x4*>(p));
  }
  // stores -o (rounded): the sign bits of the rounded values flipped, exact (cached, and non-temporal)
  static __device__ __forceinline__ void store_neg(T* p, const float (&o)[8]) {
    uint4 u;
    u.x = Cvt::pack2(o[0], o[1]) ^ 0x80008000u; u.y = Cvt::pack2(o[2], o[3]) ^ 0x80008000u;
    u.z = Cvt::pack2(o[4], o[5]) ^ 0x80008000u; u.w = Cvt::pack2(o[6], o[7]) ^ 0x80008000u;
    *reinterpret_cast<uint4*>(p) = u;
  }
  static __device__ __forceinline__ void store_neg_nt(T* p, const float (&o)[8]) {
    const u32x4 u{Cvt::pack2(o[0], o[1]) ^ 0x80008000u, Cvt::pack2(o[2], o[3]) ^ 0x80008000u,
                  Cvt::pack2(o[4], o[5]) ^ 0x80008000u, Cvt::pack2(o[6], o[7]) ^ 0x80008000u};
    __builtin_nontemporal_store(u, reinterpret_cast<u32x4*>(p));
  }
  static __device__ __forceinline__ float round(float x) { return Cvt::round(x); }
};

template <> struct IO<bf16_t> : IO16<bf16_t, Bf16Cvt> {};
template <> struct IO<_Float16> : IO16<_Float16, F16Cvt> {};

template <> struct IO<float> {
  struct Raw { float4 a, b; };
  static __device__ __forceinline__ Raw raw(const float* p) {
    Raw r; r.a = reinterpret_cast<const float4*>(p)[0]; r.b = reinterpret_cast<const float4*>(p)[1]; return r;
  }
  static __device__ __forceinline__ Raw raw_nt(const float* p) { return raw(p); }
  // the reads' source stream: non-temporal (LDR_F32_NT; for the other kernels' fp32 rows the caches measured faster:
  // c4 fp32 read forward 15.5 -> 15.1 ms per pass, backward pass 1 and the update gradient 0.6-0.7 ms slower)
  static __device__ __forceinline__ Raw raw_str(const float* p) {
#if LDR_NT && LDR_F32_NT
    const u32x4 a = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
    const u32x4 b = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p) + 1);
    Raw r;
    r.a = make_float4(__uint_as_float(a.x), __uint_as_float(a.y), __uint_as_float(a.z), __uint_as_float(a.w));
    r.b = make_float4(__uint_as_float(b.x), __uint_as_float(b.y), __uint_as_float(b.z), __uint_as_float(b.w));
    return r;
#else
    return raw(p);
#endif
  }
  static __device__ __forceinline__ Raw zero() { Raw r; r.a = make_float4(0.f, 0.f, 0.f, 0.f); r.b = r.a; return r; }
  static __device__ __forceinline__ void unpack(const Raw& r, float (&o)[8]) {
    o[0] = r.a.x; o[1] = r.a.y; o[2] = r.a.z; o[3] = r.a.w; o[4] = r.b.x; o[5] = r.b.y; o[6] = r.b.z; o[7] = r.b.w;
  }
  static __device__ __forceinline__ void load(const float* p, float (&o)[8]) { unpack(raw(p), o); }
  static __device__ __forceinline__ void store(float* p, const float (&o)[8]) {
    reinterpret_cast<float4*>(p)[0] = make_float4(o[0], o[1], o[2], o[3]);
    reinterpret_cast<float4*>(p)[1] = make_float4(o[4], o[5], o[6], o[7]);
  }
  static __device__ __forceinline__ void store_nt(float* p, const float (&o)[8]) {
    __builtin_nontemporal_store(u32x4{__float_as_uint(o[0]), __float_as_uint(o[1]), __float_as_uint(o[2]),
                                      __float_as_uint(o[3])}, reinterpret_cast<u32x4*>(p));
    __builtin_nontemporal_store(u32x4{__float_as_uint(o[4]), __float_as_uint(o[5]), __float_as_uint(o[6]),
                                      __float_as_uint(o[7])}, reinterpret_cast<u32x4*>(p) + 1);
  }
  static __device__ __forceinline__ void store_neg(float* p, const float (&o)[8]) {
    reinterpret_cast<float4*>(p)[0] = make_float4(-o[0], -o[1], -o[2], -o[3]);
    reinterpret_cast<float4*>(p)[1] = make_float4(-o[4], -o[5], -o[6], -o[7]);
  }
  static __device__ __forceinline__ void store_neg_nt(float* p, const float (&o)[8]) {
    __builtin_nontemporal_store(u32x4{__float_as_uint(o[0]) ^ 0x80000000u, __float_as_uint(o[1]) ^ 0x80000000u,
                                      __float_as_uint(o[2]) ^ 0x80000000u, __float_as_uint(o[3]) ^ 0x80000000u},
                                reinterpret_cast<u32x4*>(p));
    __builtin_nontemporal_store(u32x4{__float_as_uint(o[4]) ^ 0x80000000u, __float_as_uint(o[5]) ^ 0x80000000u,
                                      __float_as_uint(o[6]) ^ 0x80000000u, __float_as_uint(o[7]) ^ 0x80000000u},
                                reinterpret_cast<u32x4*>(p) + 1);
  }
  static __device__ __forceinline__ float round(float x) { return x; }
};

__device__ __forceinline__ void load_f32x8(const float* p, float (&o)[8]) { IO<float>::load(p, o); }

// Reduction over an aligned group of g lanes of a wave (g a power of two <= 64) in registers, without the LDS
// crossbar: DPP (xor 1 and xor 2 inside quads, the 8- and 16-lane mirrors) and gfx950's row swaps
// (v_permlane16_swap, v_permlane32_swap), the smallest level first. At each level both operands already hold equal
// values across their halves, so every lane of the group ends with the same bits. All lanes of the wave must be
// active.
template <int CTRL>
__device__ __forceinline__ float dpp_f(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, false));
}
template <typename Op>
__device__ __forceinline__ float lanes_reduce(float x, int g, Op op) {
  if (g >= 2) x = op(x, dpp_f<0xB1>(x));    // quad_perm [1, 0, 3, 2]
  if (g >= 4) x = op(x, dpp_f<0x4E>(x));    // quad_perm [2, 3, 0, 1]
  if (g >= 8) x = op(x, dpp_f<0x141>(x));   // row_half_mirror
  if (g >= 16) x = op(x, dpp_f<0x140>(x));  // row_mirror
  if (g >= 32) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto sw = __builtin_amdgcn_permlane16_swap(u, u, false, false);   // rows (0, 0, 2, 2) and (1, 1, 3, 3)
    x = op(__builtin_bit_cast(float, (unsigned)sw[0]), __builtin_bit_cast(float, (unsigned)sw[1]));
  }
  if (g >= 64) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto sw = __builtin_amdgcn_permlane32_swap(u, u, false, false);   // lower half twice, upper half twice
    x = op(__builtin_bit_cast(float, (unsigned)sw[0]), __builtin_bit_cast(float, (unsigned)sw[1]));
  }
  return x;
}
struct AddOp { __device__ __forceinline__ float operator()(float a, float b) const { return a + b; } };
struct MaxOp { __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); } };


// one element at element alignment
__device__ __forceinline__ float ld1(const bf16_t* p) { return __uint_as_float((uint32_t)*p << 16); }
__device__ __forceinline__ float ld1(const float* p) { return *p; }
__device__ __forceinline__ float ld1(const _Float16* p) { return (float)*p; }
__device__ __forceinline__ void st1(bf16_t* p, float v) { *p = __builtin_bit_cast(bf16_t, (__bf16)v); }
__device__ __forceinline__ void st1(float* p, float v) { *p = v; }
__device__ __forceinline__ void st1(_Float16* p, float v) { *p = to_f16(v); }

// wave_lds_sync: the lanes of one wave meet around LDS (no barrier: the wave's LDS operations are in order)
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// eight elements at element alignment: global loads take any alignment (one that crosses a cache line costs a second
// line, not a second instruction)
typedef unsigned int u32x4_u16 __attribute__((ext_vector_type(4), aligned(2), may_alias));
typedef unsigned int u32x4_u32 __attribute__((ext_vector_type(4), aligned(4), may_alias));

template <typename T> struct UIO {   // 16-bit elements: one 16-byte vector at 2-byte alignment
  typedef typename IO<T>::Raw Raw;
  struct Mask { uint4 m; };
  static __device__ __forceinline__ Raw put(u32x4 v) { Raw r; r.u = make_uint4(v.x, v.y, v.z, v.w); return r; }
  static __device__ __forceinline__ Raw raw(const T* p) { return put(*reinterpret_cast<const u32x4_u16*>(p)); }
  static __device__ __forceinline__ Raw raw_nt(const T* p) {
    return put(__builtin_nontemporal_load(reinterpret_cast<const u32x4_u16*>(p)));
  }
  static __device__ __forceinline__ Mask mask(int skip) {   // zero for the first `skip` elements
    auto word = [&](int w) -> unsigned {
      return (2 * w >= skip ? 0xffffu : 0u) | (2 * w + 1 >= skip ? 0xffff0000u : 0u);
    };
    return Mask{make_uint4(word(0), word(1), word(2), word(3))};
  }
  static __device__ __forceinline__ Raw masked(Raw r, const Mask& m) {
    r.u.x &= m.m.x; r.u.y &= m.m.y; r.u.z &= m.m.z; r.u.w &= m.m.w;
    return r;
  }
  static __device__ __forceinline__ void store(T* p, const float (&o)[8]) {
    typedef typename std::conditional<std::is_same<T, bf16_t>::value, Bf16Cvt, F16Cvt>::type Cvt;
    *reinterpret_cast<u32x4_u16*>(p) = u32x4{Cvt::pack2(o[0], o[1]), Cvt::pack2(o[2], o[3]), Cvt::pack2(o[4], o[5]),
                                             Cvt::pack2(o[6], o[7])};
  }
};

template <> struct UIO<float> {      // fp32 elements: two 16-byte vectors at 4-byte alignment
  typedef IO<float>::Raw Raw;
  struct Mask { uint4 a, b; };
  static __device__ __forceinline__ Raw put(u32x4 a, u32x4 b) {
    Raw r;
    r.a = make_float4(__uint_as_float(a.x), __uint_as_float(a.y), __uint_as_float(a.z), __uint_as_float(a.w));
    r.b = make_float4(__uint_as_float(b.x), __uint_as_float(b.y), __uint_as_float(b.z), __uint_as_float(b.w));
    return r;
  }
  static __device__ __forceinline__ Raw raw(const float* p) {
    const u32x4_u32* q = reinterpret_cast<const u32x4_u32*>(p);
    return put(q[0], q[1]);
  }
  static __device__ __forceinline__ Raw raw_nt(const float* p) {
    const u32x4_u32* q = reinterpret_cast<const u32x4_u32*>(p);
    return put(__builtin_nontemporal_load(q), __builtin_nontemporal_load(q + 1));
  }
  static __device__ __forceinline__ Mask mask(int skip) {
    auto word = [&](int k) -> unsigned { return k >= skip ? 0xffffffffu : 0u; };
    return Mask{make_uint4(word(0), word(1), word(2), word(3)), make_uint4(word(4), word(5), word(6), word(7))};
  }
  static __device__ __forceinline__ float and_f(float x, unsigned m) { return __uint_as_float(__float_as_uint(x) & m); }
  static __device__ __forceinline__ Raw masked(Raw r, const Mask& m) {
    r.a = make_float4(and_f(r.a.x, m.a.x), and_f(r.a.y, m.a.y), and_f(r.a.z, m.a.z), and_f(r.a.w, m.a.w));
    r.b = make_float4(and_f(r.b.x, m.b.x), and_f(r.b.y, m.b.y), and_f(r.b.z, m.b.z), and_f(r.b.w, m.b.w));
    return r;
  }
  static __device__ __forceinline__ void store(float* p, const float (&o)[8]) {
    u32x4_u32* q = reinterpret_cast<u32x4_u32*>(p);
    q[0] = u32x4{__float_as_uint(o[0]), __float_as_uint(o[1]), __float_as_uint(o[2]), __float_as_uint(o[3])};
    q[1] = u32x4{__float_as_uint(o[4]), __float_as_uint(o[5]), __float_as_uint(o[6]), __float_as_uint(o[7])};
  }
};

}  // namespace
