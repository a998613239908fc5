// Device functors: the load / reduce / store customisation of the schedule.
//
// The reference expresses these as GLSL macros (NVPRO_PYRAMID_TYPE, _LOAD,
// _REDUCE, _REDUCE2, _REDUCE4, _LOAD_REDUCE4, _STORE, nvpro_pyramid.glsl:27-120)
// and ships one set, sRGBA8 (srgba8_mipmap_preamble.glsl:19-128).  Here each set
// is a struct of static device functions; the kernels are templates over it.
//
//   Raw                  storage texel (what a level holds in memory)
//   Val                  NVPRO_PYRAMID_TYPE: the value reductions operate on
//   Tables               per-workgroup LDS tables (may be empty)
//   fill<BS>(t, scale)   workgroup-cooperative set-up by BS threads; `scale`
//                        premultiplies decoded values (0.25 for the 2x2 box)
//   DualTables,          tables serving load<true> (times 0.25) and
//   fillDual<BS>(t)      load<false> (times 1) alike
//   load<PRE>(t, raw)    NVPRO_PYRAMID_LOAD: Raw -> Val (times 0.25 if PRE)
//   store(t, v)          NVPRO_PYRAMID_STORE: Val -> Raw
//   add, mul, reduce3    the arithmetic REDUCE, REDUCE2 and REDUCE4 are built
//                        from (box, reduce2, reduce3 below)
//   Acc, first3, next3,  reduce3 tap by tap: done3(next3(w2, v2, next3(w1, v1,
//   done3                first3(w0, v0)))) is reduce3(w0, v0, w1, v1, w2, v2)
//   Chan, chanRaw,       one channel of a Val (a Val is four in memory order), of a
//   chanStore, chanLoad  Raw, and NVPRO_PYRAMID_STORE / _LOAD of channel c alone
//   kPrescale            whether load<true> then box<true> equals box<false>
//                        of plain loads bit for bit (exact scaling by 0.25)
//
// Every FP32 operation is written out; the library is compiled with
// -ffp-contract=off so none is fused behind our back.
#pragma once

#include <stdint.h>

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "srgb_tables.inc"

namespace nvpro_pyramid {

static __constant__ __attribute__((aligned(16))) uint32_t gSrgbDecode[256]                    = {NVPRO_SRGB_DECODE_BITS};
static __constant__ __attribute__((aligned(16))) uint32_t gSrgbEncode[NVPRO_SRGB_ENC_BUCKETS] = {NVPRO_SRGB_ENCODE_BUCKETS};

__device__ __forceinline__ float4 f4add(float4 a, float4 b)
{
  return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}
__device__ __forceinline__ float4 f4mul(float4 a, float s)
{
  return make_float4(a.x * s, a.y * s, a.z * s, a.w * s);
}

// NVPRO_PYRAMID_REDUCE of srgba8_mipmap_preamble.glsl:24-25, a0*v0 + a1*v1 + a2*v2,
// with the contraction fixed as fma(a2, v2, fma(a1, v1, a0 * v0)).
__device__ __forceinline__ float fma3(float w0, float v0, float w1, float v1, float w2, float v2)
{
  return __builtin_fmaf(w2, v2, __builtin_fmaf(w1, v1, w0 * v0));
}

// Round an FP32 value to binary16 (nearest even) after it has been rounded to
// FP32.  The empty asm keeps the compiler from merging the producing FMA and the
// conversion into one mixed-precision instruction (v_fma_mixlo_f16), which
// would round once instead of twice.
__device__ __forceinline__ __half toHalf(float f)
{
  __asm__ volatile("" : "+v"(f));
  return __float2half_rn(f);
}
__device__ __forceinline__ float4 fma3(float w0, float4 v0, float w1, float4 v1, float w2, float4 v2)
{
  return make_float4(fma3(w0, v0.x, w1, v1.x, w2, v2.x), fma3(w0, v0.y, w1, v1.y, w2, v2.y),
                     fma3(w0, v0.z, w1, v1.z, w2, v2.z), fma3(w0, v0.w, w1, v1.w, w2, v2.w));
}

// FP32 arithmetic on float4 values, shared by the FP32 functors.
struct Fp32Arith
{
  using Val                          = float4;
  static constexpr bool kPrescale    = true;
  __device__ static Val add(Val a, Val b) { return f4add(a, b); }
  __device__ static Val mul(Val a, float s) { return f4mul(a, s); }
  __device__ static Val reduce3(float w0, Val v0, float w1, Val v1, float w2, Val v2)
  {
    return fma3(w0, v0, w1, v1, w2, v2);
  }
  using Chan = float;
  using Acc  = float4;
  __device__ static Acc first3(float w, Val v) { return f4mul(v, w); }
  __device__ static Acc next3(float w, Val v, Acc a)
  {
    return make_float4(__builtin_fmaf(w, v.x, a.x), __builtin_fmaf(w, v.y, a.y), __builtin_fmaf(w, v.z, a.z),
                       __builtin_fmaf(w, v.w, a.w));
  }
  __device__ static Val done3(Acc a) { return a; }
};

// NVPRO_PYRAMID_REDUCE2 of srgba8_mipmap_preamble.glsl:35: 0.5 * (v0 + v1).
template <class F>
__device__ __forceinline__ typename F::Val reduce2(typename F::Val v0, typename F::Val v1)
{
  return F::mul(F::add(v0, v1), 0.5f);
}

// NVPRO_PYRAMID_REDUCE4 of srgba8_mipmap_preamble.glsl:37-38,
// 0.25 * ((v00 + v01) + (v10 + v11)).  The reference passes the four quadrants
// of a 2x2 square in one of two orders (nvpro_pyramid.glsl:179-188 vs
// :364-392); `order` selects which pairs are added first:
//   order 0: (UL + LL) + (UR + LR)      order 1: (UL + UR) + (LL + LR)
// PRE: the inputs were already multiplied by 0.25 (exactly), so the sum is the
// result.
template <class F, bool PRE>
__device__ __forceinline__ typename F::Val box(typename F::Val ul, typename F::Val ur, typename F::Val ll,
                                               typename F::Val lr, int order)
{
  const typename F::Val s =
      order == 0 ? F::add(F::add(ul, ll), F::add(ur, lr)) : F::add(F::add(ul, ur), F::add(ll, lr));
  return PRE ? s : F::mul(s, 0.25f);
}

// Summation order of relative level r of a fast dispatch filling `count` levels
// (nvpro_pyramid.glsl:272-532): LOAD_REDUCE4 and the 6-level in-thread stage use
// order 0, the subgroup-shuffle stages order 1, the shared-memory stages order 0.
__host__ __device__ __forceinline__ int fastOrder(uint32_t count, uint32_t r)
{
  if(r == 1u)
    return 0;
  if(count <= 3u)
    return 1;
  if(count == 6u)
    return (r == 3u || r == 4u) ? 1 : 0;
  return r <= 3u ? 1 : 0;
}

// ---------------------------------------------------------------------------
// sRGBA8: srgba8_mipmap_preamble.glsl:19-128 with exact conversions.
// ---------------------------------------------------------------------------
struct Srgba8 : Fp32Arith
{
  using Raw                        = uint32_t;
  static constexpr uint32_t kBytes = 4;

  // Alpha is carried in code units: the reference decodes the UNORM code as
  // c / 255 and encodes uint(a * 255 + 0.5) (preamble:125), a linear map whose
  // scale commutes with every reduction, so the value here is c itself (times
  // the fill scale) and the encode is floor(a + 0.5).  Box filters of codes are
  // then exact in FP32 (a 2x2 sum of 4^k codes stays below 2^24), and every
  // .5 tie rounds up as exact arithmetic does.
  //
  // LDS tables: the decoded value of every RGB code (times the fill scale) and
  // the encode buckets.
  struct __attribute__((aligned(16))) Tables
  {
    float dec[256];
    // Code at the bucket's start << 16 | 0x10000 - the low 16 bits of the float
    // where it steps up (srgb_tables.inc with its low half complemented).
    uint32_t enc[NVPRO_SRGB_ENC_BUCKETS];
  };
  static_assert(NVPRO_SRGB_ENC_BUCKETS % 4u == 0u, "16-byte table loads");
  static_assert(23u - NVPRO_SRGB_ENC_MANT_BITS == 16u, "the floats of a bucket differ in their low 16 bits");

  // The fill in two halves, so that a kernel can issue its own loads between
  // the table's and the wait for them.  No branches: a conditional load would
  // end a block that the scheduler cannot cross.  Threads past the tables' end
  // load and store words of other threads again, each its own (one word from
  // many lanes would serialise the LDS write).
  template <int BS>
  struct TableLoads
  {
    static constexpr int kEnc = (NVPRO_SRGB_ENC_BUCKETS / 4 + BS - 1) / BS;
    uint4 e[kEnc], d;
  };
  template <int BS>
  __device__ static uint32_t encWord(int k)
  {
    constexpr uint32_t N = NVPRO_SRGB_ENC_BUCKETS / 4u;
    static_assert(BS <= 3 * N, "at most two words past the table's end");
    uint32_t i = threadIdx.x + k * BS;
    i          = i < N ? i : i - N;
    return i < N ? i : i - N;
  }
  template <int BS>
  __device__ static void fillLoad(TableLoads<BS>& r)
  {
#pragma unroll
    for(int k = 0; k < TableLoads<BS>::kEnc; ++k)
      r.e[k] = reinterpret_cast<const uint4*>(gSrgbEncode)[encWord<BS>(k)];
    r.d = reinterpret_cast<const uint4*>(gSrgbDecode)[threadIdx.x & 63u];
  }
  template <int BS>
  __device__ static void fillStore(Tables& t, const TableLoads<BS>& r, float scale)
  {
    reinterpret_cast<float4*>(t.dec)[threadIdx.x & 63u] =
        make_float4(__uint_as_float(r.d.x) * scale, __uint_as_float(r.d.y) * scale, __uint_as_float(r.d.z) * scale,
                    __uint_as_float(r.d.w) * scale);
#pragma unroll
    for(int k = 0; k < TableLoads<BS>::kEnc; ++k)
      reinterpret_cast<uint4*>(t.enc)[encWord<BS>(k)] =
          make_uint4(r.e[k].x ^ 0xffffu, r.e[k].y ^ 0xffffu, r.e[k].z ^ 0xffffu, r.e[k].w ^ 0xffffu);
  }
  template <int BS>
  __device__ static void fill(Tables& t, float scale)
  {
    // 16-byte loads, every global load issued before any LDS store.
    constexpr int kEnc = (NVPRO_SRGB_ENC_BUCKETS / 4 + BS - 1) / BS;
    const uint4* genc = reinterpret_cast<const uint4*>(gSrgbEncode);
    uint4 e[kEnc];
#pragma unroll
    for(int k = 0; k < kEnc; ++k)
    {
      const uint32_t i = threadIdx.x + k * BS;
      e[k] = i < NVPRO_SRGB_ENC_BUCKETS / 4u ? genc[i] : make_uint4(0, 0, 0, 0);
    }
    const uint4 d = threadIdx.x < 64u ? reinterpret_cast<const uint4*>(gSrgbDecode)[threadIdx.x] : make_uint4(0, 0, 0, 0);
    if(threadIdx.x < 64u)
      reinterpret_cast<float4*>(t.dec)[threadIdx.x] =
          make_float4(__uint_as_float(d.x) * scale, __uint_as_float(d.y) * scale, __uint_as_float(d.z) * scale,
                      __uint_as_float(d.w) * scale);
#pragma unroll
    for(int k = 0; k < kEnc; ++k)
    {
      const uint32_t i = threadIdx.x + k * BS;
      if(i < NVPRO_SRGB_ENC_BUCKETS / 4u)
      {
        // Keeps the compiler from moving the complement up to each load, which
        // would wait for every load before issuing the next.
        __asm__ volatile("" : "+v"(e[k].x), "+v"(e[k].y), "+v"(e[k].z), "+v"(e[k].w));
        reinterpret_cast<uint4*>(t.enc)[i] =
            make_uint4(e[k].x ^ 0xffffu, e[k].y ^ 0xffffu, e[k].z ^ 0xffffu, e[k].w ^ 0xffffu);
      }
    }
  }

  // Tables for kernels that run premultiplied (fast) and plain (general, tail)
  // loads alike: the unscaled tables, with load<true> multiplying by 0.25 after
  // the lookup.  Scaling by 0.25 is exact for every decoded value (none is
  // subnormal), so this equals the lookup in a table filled at scale 0.25, bit
  // for bit, and the LDS holds one set of tables instead of two.
  struct DualTables : Tables
  {
  };

  template <int BS>
  __device__ static void fillDual(DualTables& t)
  {
    fill<BS>(t, 1.0f);
  }

  // texelFetch of the sRGB sampler (preamble:21-22): sRGB decode of RGB by table
  // lookup; alpha in code units (see Tables).  With plain Tables, PRE says the
  // tables were filled at 0.25 (the fast pipeline) and alpha gets the same
  // exact scale; plain loads (tables filled at 1) take the code as it is.
  template <bool PRE>
  __device__ static float4 load(const Tables& t, uint32_t texel)
  {
    const float a = (float)(texel >> 24) * (PRE ? 0.25f : 1.0f);
    return make_float4(t.dec[texel & 0xffu], t.dec[(texel >> 8) & 0xffu], t.dec[(texel >> 16) & 0xffu], a);
  }
  template <bool PRE>
  __device__ static float4 load(const DualTables& t, uint32_t texel)
  {
    const float4 v = load<false>(static_cast<const Tables&>(t), texel);
    return PRE ? f4mul(v, 0.25f) : v;
  }

  // srgbFromLinear (preamble:110-121), exact: x is clamped to [2^-13, 1) (every
  // smaller value, and NaN, encodes to 0, every larger one to 255); the bucket
  // of its exponent and top mantissa bits holds the code at the bucket start
  // and, complemented, where in the bucket the code steps up: adding the
  // float's low 16 bits carries into the code exactly from the step on.  The
  // code is in bits 16-23 of the result, the bits above are 0.  With the byte
  // permutes of store() 16 VALU instructions a texel instead of 27 (compare,
  // add with carry and shifts per channel): 255x127 chain 10.98 -> 10.67 us,
  // 4095x2047 29.6 -> 29.3, 512-texture batch 807 -> 795.
  __device__ static uint32_t encodeHigh(const Tables& t, float x)
  {
    const uint32_t b = __float_as_uint(__builtin_amdgcn_fmed3f(x, 0x1p-13f, 0x1.fffffep-1f));
    // Byte offset of the bucket, 4 * (high half - first bucket's), in one
    // instruction (the compiler takes two).
    uint32_t off;
    __asm__("v_mad_u32_u16 %0, %1, 4, %2 op_sel:[1,0,0,0]"
            : "=v"(off)
            : "v"(b), "s"(0u - 4u * (NVPRO_SRGB_ENC_MIN_EXP << NVPRO_SRGB_ENC_MANT_BITS)));
    const uint32_t e = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(t.enc) + off);
    return e + (b & 0xffffu);
  }
  __device__ static uint32_t encodeChannel(const Tables& t, float x) { return encodeHigh(t, x) >> 16; }

  using ChanRaw = uint8_t;
  __device__ static ChanRaw chanStore(const Tables& t, float v, uint32_t c)
  {
    const uint32_t rgb = encodeChannel(t, v);
    const uint32_t a   = (uint32_t)__builtin_amdgcn_fmed3f(v + 0.5f, 0.0f, 255.0f);
    return (ChanRaw)(c == 3u ? a : rgb);
  }
  __device__ static float chanLoad(const Tables& t, ChanRaw q, uint32_t c) { return c == 3u ? (float)q : t.dec[q]; }

  // srgbFromLinearVec (preamble:123-128); alpha (code units) = floor(a + 0.5)
  // clamped to [0, 255].  Byte selectors of v_perm_b32: 0-3 the second
  // operand's bytes, 4-7 the first's, 12 zero.
  __device__ static uint32_t store(const Tables& t, float4 v)
  {
    const uint32_t a = (uint32_t)__builtin_amdgcn_fmed3f(v.w + 0.5f, 0.0f, 255.0f);
    const uint32_t r = encodeHigh(t, v.x), g = encodeHigh(t, v.y), b = encodeHigh(t, v.z);
    return __builtin_amdgcn_perm(g, r, 0x0c0c0602u) | __builtin_amdgcn_perm(a, b, 0x04020c0cu);
  }
};

// ---------------------------------------------------------------------------
// RGBA32F: linear float4 texels, identity load and store.
// ---------------------------------------------------------------------------
struct Rgba32f : Fp32Arith
{
  struct __attribute__((aligned(4))) Raw
  {
    float x, y, z, w;
  };
  static constexpr uint32_t kBytes = 16;
  struct Tables
  {
    int unused;
  };
  using DualTables = Tables;
  template <int BS>
  struct TableLoads
  {
  };
  template <int BS>
  __device__ static void fillLoad(TableLoads<BS>&)
  {
  }
  template <int BS>
  __device__ static void fillStore(Tables&, const TableLoads<BS>&, float)
  {
  }
  template <int BS>
  __device__ static void fill(Tables&, float)
  {
  }
  template <int BS>
  __device__ static void fillDual(Tables&)
  {
  }
  template <bool PRE>
  __device__ static float4 load(const Tables&, Raw t)
  {
    float4 v = make_float4(t.x, t.y, t.z, t.w);
    return PRE ? f4mul(v, 0.25f) : v;
  }
  __device__ static Raw store(const Tables&, float4 v)
  {
    return Raw{v.x, v.y, v.z, v.w};
  }
  using ChanRaw = float;
  __device__ static ChanRaw chanStore(const Tables&, float v, uint32_t) { return v; }
  __device__ static float chanLoad(const Tables&, ChanRaw q, uint32_t) { return q; }
};

// ---------------------------------------------------------------------------
// RGBA16F: linear half4 texels; FP32 arithmetic, round-to-nearest-even on store.
// ---------------------------------------------------------------------------
struct Rgba16f : Fp32Arith
{
  struct __attribute__((aligned(4))) Raw
  {
    uint32_t lo, hi;  // (r | g << 16), (b | a << 16) as IEEE half bits
  };
  static constexpr uint32_t kBytes = 8;
  struct Tables
  {
    int unused;
  };
  using DualTables = Tables;
  template <int BS>
  struct TableLoads
  {
  };
  template <int BS>
  __device__ static void fillLoad(TableLoads<BS>&)
  {
  }
  template <int BS>
  __device__ static void fillStore(Tables&, const TableLoads<BS>&, float)
  {
  }
  template <int BS>
  __device__ static void fill(Tables&, float)
  {
  }
  template <int BS>
  __device__ static void fillDual(Tables&)
  {
  }
  __device__ static float h2f(uint32_t bits) { return __half2float(__ushort_as_half((unsigned short)bits)); }
  __device__ static uint32_t f2h(float f) { return __half_as_ushort(toHalf(f)); }
  template <bool PRE>
  __device__ static float4 load(const Tables&, Raw t)
  {
    float4 v = make_float4(h2f(t.lo & 0xffffu), h2f(t.lo >> 16), h2f(t.hi & 0xffffu), h2f(t.hi >> 16));
    return PRE ? f4mul(v, 0.25f) : v;
  }
  __device__ static Raw store(const Tables&, float4 v)
  {
    return Raw{f2h(v.x) | f2h(v.y) << 16, f2h(v.z) | f2h(v.w) << 16};
  }
  using ChanRaw = uint16_t;
  __device__ static ChanRaw chanStore(const Tables&, float v, uint32_t) { return (ChanRaw)f2h(v); }
  __device__ static float chanLoad(const Tables&, ChanRaw q, uint32_t) { return h2f(q); }
};

// ---------------------------------------------------------------------------
// RGBA16F with PACKED_FP16 arithmetic: 2x2 boxes and 2-tap reductions run in
// binary16 on (r,g) and (b,a) pairs (v_pk_add_f16 / v_pk_mul_f16); 3-tap
// reductions widen to FP32 for the weights and round the result to binary16.
// ---------------------------------------------------------------------------
struct Rgba16fPacked
{
  using Raw                        = Rgba16f::Raw;
  static constexpr uint32_t kBytes = 8;
  // Scaling a binary16 subnormal by 0.25 can round, so no premultiplied loads.
  static constexpr bool kPrescale = false;
  struct Val
  {
    __half2 rg, ba;
  };
  using Tables     = Rgba16f::Tables;
  using DualTables = Tables;
  template <int BS>
  struct TableLoads
  {
  };
  template <int BS>
  __device__ static void fillLoad(TableLoads<BS>&)
  {
  }
  template <int BS>
  __device__ static void fillStore(Tables&, const TableLoads<BS>&, float)
  {
  }
  template <int BS>
  __device__ static void fill(Tables&, float)
  {
  }
  template <int BS>
  __device__ static void fillDual(Tables&)
  {
  }
  template <bool PRE>
  __device__ static Val load(const Tables&, Raw t)
  {
    static_assert(!PRE, "binary16 values are not premultiplied");
    return Val{__builtin_bit_cast(__half2, t.lo), __builtin_bit_cast(__half2, t.hi)};
  }
  __device__ static Raw store(const Tables&, Val v)
  {
    return Raw{__builtin_bit_cast(uint32_t, v.rg), __builtin_bit_cast(uint32_t, v.ba)};
  }
  __device__ static Val add(Val a, Val b) { return Val{__hadd2(a.rg, b.rg), __hadd2(a.ba, b.ba)}; }
  __device__ static Val mul(Val a, float s)
  {
    const __half2 k = __float2half2_rn(s);  // 0.25 and 0.5 are exact in binary16
    return Val{__hmul2(a.rg, k), __hmul2(a.ba, k)};
  }
  using Chan    = _Float16;
  using ChanRaw = _Float16;
  __device__ static ChanRaw chanStore(const Tables&, Chan v, uint32_t) { return v; }
  __device__ static Chan chanLoad(const Tables&, ChanRaw q, uint32_t) { return q; }
  using Acc = float4;
  __device__ static float4 widen(Val v)
  {
    const float2 rg = __half22float2(v.rg), ba = __half22float2(v.ba);
    return make_float4(rg.x, rg.y, ba.x, ba.y);
  }
  __device__ static Acc first3(float w, Val v) { return Fp32Arith::first3(w, widen(v)); }
  __device__ static Acc next3(float w, Val v, Acc a) { return Fp32Arith::next3(w, widen(v), a); }
  __device__ static Val done3(Acc a)
  {
    return Val{__halves2half2(toHalf(a.x), toHalf(a.y)), __halves2half2(toHalf(a.z), toHalf(a.w))};
  }
  __device__ static Val reduce3(float w0, Val v0, float w1, Val v1, float w2, Val v2)
  {
    const float2 a0 = __half22float2(v0.rg), a1 = __half22float2(v1.rg), a2 = __half22float2(v2.rg);
    const float2 b0 = __half22float2(v0.ba), b1 = __half22float2(v1.ba), b2 = __half22float2(v2.ba);
    return Val{__halves2half2(toHalf(fma3(w0, a0.x, w1, a1.x, w2, a2.x)), toHalf(fma3(w0, a0.y, w1, a1.y, w2, a2.y))),
               __halves2half2(toHalf(fma3(w0, b0.x, w1, b1.x, w2, b2.x)), toHalf(fma3(w0, b0.y, w1, b1.y, w2, b2.y)))};
  }
};

// One channel of F as a value of its own: the same operations, in the same
// arithmetic, as F's on that channel.
template <class Chan>
struct ChannelArith;
template <>
struct ChannelArith<float>
{
  using Val = float;
  __device__ static Val add(Val a, Val b) { return a + b; }
  __device__ static Val mul(Val a, float s) { return a * s; }
  __device__ static Val reduce3(float w0, Val v0, float w1, Val v1, float w2, Val v2)
  {
    return fma3(w0, v0, w1, v1, w2, v2);
  }
};
template <>
struct ChannelArith<_Float16>
{
  using Val = _Float16;
  __device__ static Val add(Val a, Val b) { return a + b; }
  __device__ static Val mul(Val a, float s) { return a * (_Float16)s; }
  __device__ static Val reduce3(float w0, Val v0, float w1, Val v1, float w2, Val v2)
  {
    return __builtin_bit_cast(_Float16, toHalf(fma3(w0, (float)v0, w1, (float)v1, w2, (float)v2)));
  }
};

}  // namespace nvpro_pyramid
