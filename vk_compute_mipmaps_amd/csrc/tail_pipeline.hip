// Tail kernel: the small remainder of a plan in one workgroup.
//
// Once a plan reaches small levels, one kernel per step only buys launch
// latency: this one runs every remaining step, fast and general alike.  The
// first source level is loaded and decoded into LDS once; every level is then
// computed from LDS, stored to memory and kept in LDS for the next one; at a
// step boundary the value kept is the decode of the stored texel, exactly what
// the next dispatch would load.  The arithmetic per channel is that of the
// per-step bodies (fast: box with the reference's order; general:
// reduceStoreSample_), so results do not depend on which kernel ran a step.
//
// What bounds it is one workgroup's latency: a chain of memory and LDS round
// trips and of instructions on one compute unit.  So in levels of up to 256
// texels a thread computes one channel of a texel (a quarter of the
// instructions on the chain, four times the lanes, of which small levels leave
// most idle), everything a level needs beside the values comes ready from the
// host in kernel-argument memory, the source is read in one round while the
// tables are on their way, with arguments that are in registers at the start,
// and once a level fits one wave that wave goes on alone, without barriers.
// Cycles from the start for the five levels under 63x31 (medians): tables and
// source here 2500, decoded 3700, then 2100 for 465 texels, 1400 for 105, and
// 1100-1250 for each of 21, 3 and 1, most of it about a hundred dependent
// instructions and three LDS round trips; the stores complete 640 later.  The
// texel-per-thread tail that read its first level's windows from memory took
// 7.2 us a launch, this one 5.4: 255x127 chain 10.4 -> 8.9 us, 4095x2047 27.9
// -> 26.6.
#include "groups.hpp"

namespace nvpro_pyramid {

constexpr int kTailBS = 1024;

// A first output level of kTailMaxTexels texels has no more levels than this.
constexpr uint32_t kTailLevels = 11;
static_assert(kTailMaxTexels == 1u << (kTailLevels - 1u), "levels of a tail");

struct TailLevel
{
  uint8_t* dst;
  uint32_t pitch, width, texels;
  uint32_t inverse;    // texel / width is texel * inverse >> 20, exact below 2^20 / width
  uint32_t srcWidth;
  uint32_t mode;       // TailMode
  uint32_t requantise; // the last level of its step
  Axis3 ax, ay;
};
// What a level computes: a fast step's box in one of the two orders, or a
// general step's kernel by its sizes (a side of 1 leaves a row or a column).
enum TailMode : uint32_t
{
  kTail33, kTail22, kTail32, kTail23, kTailRow3, kTailRow2, kTailColumn3, kTailColumn2, kTailBox0, kTailBox1
};
static uint32_t tailMode(bool fast, int order, int kx, int ky)
{
  if(fast)
    return order == 0 ? kTailBox0 : kTailBox1;
  if(ky == 1)
    return kx == 3 ? kTailRow3 : kTailRow2;
  if(kx == 1)
    return ky == 3 ? kTailColumn3 : kTailColumn2;
  return kx == 3 ? (ky == 3 ? kTail33 : kTail32) : (ky == 3 ? kTail23 : kTail22);
}
struct TailArgs
{
  uint32_t count, pad;
  TailLevel lv[kTailLevels];
};
// The first source level: the kernel's leading arguments, which the hardware
// loads into scalar registers ahead of the kernel (build.py's
// kernarg-preload-count), so that the source's loads wait for no argument.
struct TailSource
{
  const uint8_t* base;
  uint32_t pitch, width, texels;
  uint32_t inverse;  // texel / width is the high word of texel * inverse
};

template <class F>
constexpr size_t kTailValuesAt = (sizeof(typename F::Tables) + 15u) / 16u * 16u;

// Dynamic LDS: the tables, then the values of the source, of the first output
// level and of the second (later levels take turns in the last two).
template <class F>
static size_t tailSharedBytes(const TailSource& src, const TailArgs& a)
{
  const size_t values = src.texels + a.lv[0].texels + (a.count > 1u ? a.lv[1].texels : 0u);
  return kTailValuesAt<F> + values * sizeof(typename F::Val);
}

// Level l of the arguments (the last one past the end), all its words in one
// scalar load round here.
__device__ __forceinline__ TailLevel tailLevel(const TailArgs& a, uint32_t l)
{
  TailLevel q = a.lv[l < kTailLevels ? l : kTailLevels - 1u];
  __asm__ volatile("" : "+s"(q.dst), "+s"(q.pitch), "+s"(q.width), "+s"(q.texels), "+s"(q.inverse), "+s"(q.srcWidth));
  __asm__ volatile("" : "+s"(q.mode), "+s"(q.requantise), "+s"(q.ax.nf), "+s"(q.ax.rcp), "+s"(q.ay.nf), "+s"(q.ay.rcp));
  return q;
}

// Texel (x, y) of level q, whose window's value at (column j, row r) at(j, r)
// returns: the per-step bodies' arithmetic, one straight path per kind of level.
template <class F, class At>
__device__ __forceinline__ typename F::Val tailSample(At at, const TailLevel& q, uint32_t x, uint32_t y)
{
  // Odd sides most of the time, and one comparison ahead of the others.
  if(__builtin_expect(q.mode == kTail33, 1))
    return generalSample<F>(at, 3, 3, q.ax, q.ay, x, y);
  switch(q.mode)
  {
    case kTailBox0: return box<F, false>(at(0, 0), at(1, 0), at(0, 1), at(1, 1), 0);
    case kTailBox1: return box<F, false>(at(0, 0), at(1, 0), at(0, 1), at(1, 1), 1);
    case kTailRow3: return horizontalTap<F>(weights3(q.ax, x), 3, at(0, 0), at(1, 0), at(2, 0));
    case kTailRow2: return reduce2<F>(at(0, 0), at(1, 0));
    case kTailColumn3: return verticalTap<F>(weights3(q.ay, y), 3, at(0, 0), at(0, 1), at(0, 2));
    case kTailColumn2: return reduce2<F>(at(0, 0), at(0, 1));
    case kTail32: return generalSample<F>(at, 3, 2, q.ax, q.ay, x, y);
    case kTail23: return generalSample<F>(at, 2, 3, q.ax, q.ay, x, y);
    default: return generalSample<F>(at, 2, 2, q.ax, q.ay, x, y);
  }
}

template <class F>
__global__ void __launch_bounds__(kTailBS) tailKernel(const uint8_t* srcBase, uint32_t srcPitch,
                                                      uint32_t srcWidth, uint32_t srcTexels,
                                                      uint32_t srcInverse, TailArgs a)
{
  using V    = typename F::Val;
  using Chan = typename F::Chan;
  using C    = ChannelArith<Chan>;
  using Raw  = typename F::Raw;
  using Q    = typename F::ChanRaw;
  static_assert(sizeof(V) == 4u * sizeof(Chan) && 4u * sizeof(Q) == F::kBytes, "a value is four channels");
  extern __shared__ __align__(16) unsigned char shared[];
  typename F::Tables& tab = *reinterpret_cast<typename F::Tables*>(shared);
  V* const values         = reinterpret_cast<V*>(shared + kTailValuesAt<F>);
  typename F::template TableLoads<kTailBS> tables;
  F::template fillLoad<kTailBS>(tables);
  // The source, two texels a thread in flight at a time.
  constexpr uint32_t AHEAD = 2;
  auto sourceLoad          = [&](uint32_t base, Raw(&r)[AHEAD]) {
#pragma unroll
    for(uint32_t k = 0; k < AHEAD; ++k)
    {
      uint32_t i       = base + k * kTailBS + threadIdx.x;
      i                = i < srcTexels ? i : srcTexels - 1u;
      const uint32_t y = srcWidth == 1u ? i : __umulhi(i, srcInverse), x = i - y * srcWidth;
      r[k]             = loadTexel<F>(srcBase + (uint64_t)y * srcPitch + x * F::kBytes);
    }
  };
  Raw raw[AHEAD], more[AHEAD];
  sourceLoad(0u, raw);
  if(srcTexels > AHEAD * kTailBS)
    sourceLoad(AHEAD * kTailBS, more);
  // Every line of the level table into the scalar cache, as prefetchLevels
  // does, behind the vector loads in flight.
  const uint32_t count = a.count;
  uint32_t lines       = 0;
#pragma unroll
  for(uint32_t k = 0; k < sizeof(TailArgs) / 64u; ++k)
    lines ^= reinterpret_cast<const uint32_t*>(&a)[16u * k + 8u];
  TailLevel q = tailLevel(a, 0u);
  levelsReady(lines);
  F::template fillStore<kTailBS>(tab, tables, 1.0f);
  __syncthreads();
  for(uint32_t base = 0; base < srcTexels; base += AHEAD * kTailBS)
  {
    V v[AHEAD];
#pragma unroll
    for(uint32_t k = 0; k < AHEAD; ++k)
      v[k] = F::template load<false>(tab, raw[k]);
#pragma unroll
    for(uint32_t k = 0; k < AHEAD; ++k)
    {
      const uint32_t i = base + k * kTailBS + threadIdx.x;
      if(i < srcTexels)
        values[i] = v[k];
      raw[k] = more[k];
    }
    if(base + 2u * AHEAD * kTailBS < srcTexels)
      sourceLoad(base + 2u * AHEAD * kTailBS, more);
  }
  __syncthreads();

  const V* src = values;
  V* dst       = values + srcTexels;
  V* other     = dst + q.texels;
  for(uint32_t l = 0; l < count; ++l)
  {
    const uint32_t n = 4u * q.texels;
    const bool alone = n <= 64u;
    if(alone && threadIdx.x >= 64u)
      return;  // levels only get smaller: the first wave finishes them
    if(n > kTailBS)
      for(uint32_t t = threadIdx.x; t < q.texels; t += kTailBS)
      {
        const uint32_t y = __umul24(t, q.inverse) >> 20, x = t - __umul24(y, q.width);
        const V* s = src + __umul24(2u * y, q.srcWidth) + 2u * x;
        auto at    = [&](int j, int r) { return s[(uint32_t)r * q.srcWidth + (uint32_t)j]; };
        const V v      = tailSample<F>(at, q, x, y);
        const Raw code = F::store(tab, v);
        storeTexel<F>(q.dst + (uint64_t)y * q.pitch + x * F::kBytes, code);
        dst[t] = q.requantise ? F::template load<false>(tab, code) : v;
      }
    else if(threadIdx.x < n)
    {
      const uint32_t c = threadIdx.x & 3u, t = threadIdx.x >> 2;
      const uint32_t y = __umul24(t, q.inverse) >> 20, x = t - __umul24(y, q.width);
      const Chan* s = reinterpret_cast<const Chan*>(src + __umul24(2u * y, q.srcWidth) + 2u * x) + c;
      auto at       = [&](int j, int r) { return s[4u * ((uint32_t)r * q.srcWidth + (uint32_t)j)]; };
      const Chan v  = tailSample<C>(at, q, x, y);
      const Q code  = F::chanStore(tab, v, c);
      reinterpret_cast<Q*>(q.dst + (uint64_t)y * q.pitch + x * F::kBytes)[c] = code;
      reinterpret_cast<Chan*>(dst)[threadIdx.x] = q.requantise ? F::chanLoad(tab, code, c) : v;
    }
    // The next level's words, while the others catch up.
    q = tailLevel(a, l + 1u);
    if(alone)
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // one wave's LDS accesses stay in order
    else
      __syncthreads();
    V* const next = other;
    src           = dst;
    other         = dst;
    dst           = next;
  }
}

static TailSource tailSource(const ImageDesc& img, const TailPlan& plan)
{
  const LevelDesc& l = img.lv[plan.steps[0].inputLevel];
  return TailSource{img.base + l.offset, l.pitch, l.width, l.width * l.height,
                    (uint32_t)((0x100000000ull + l.width - 1u) / l.width)};
}

static TailArgs tailArgs(const ImageDesc& img, const TailPlan& plan)
{
  TailArgs a{};
  for(uint32_t s = 0; s < plan.count; ++s)
    for(uint32_t r = 1; r <= plan.steps[s].levelCount; ++r)
    {
      const LevelDesc &sl = img.lv[plan.steps[s].inputLevel + r - 1u], &dl = img.lv[plan.steps[s].inputLevel + r];
      const bool fast     = plan.steps[s].pipeline == NVPRO_PYRAMID_PIPELINE_FAST;
      TailLevel& q        = a.lv[a.count++];
      q.dst               = img.base + dl.offset;
      q.pitch             = dl.pitch;
      q.width             = dl.width;
      q.texels            = dl.width * dl.height;
      q.inverse           = ((1u << 20) + dl.width - 1u) / dl.width;
      q.srcWidth          = sl.width;
      q.mode = tailMode(fast, fastOrder(plan.steps[s].levelCount, r), kernelSize(sl.width), kernelSize(sl.height));
      q.requantise        = r == plan.steps[s].levelCount ? 1u : 0u;
      q.ax                = axis3(dl.width);
      q.ay                = axis3(dl.height);
    }
  return a;
}

template <class F>
static hipError_t launchTailTyped(hipStream_t stream, const TailSource& src, const TailArgs& args)
{
  hipLaunchKernelGGL((tailKernel<F>), dim3(1), dim3(kTailBS), tailSharedBytes<F>(src, args), stream, src.base,
                     src.pitch, src.width, src.texels, src.inverse, args);
  return hipGetLastError();
}

hipError_t launchTail(hipStream_t stream, const ImageDesc& img, const TailPlan& plan)
{
  uint32_t levels = 0;
  for(uint32_t s = 0; s < plan.count; ++s)
    levels += plan.steps[s].levelCount;
  if(plan.count == 0u || levels > kTailLevels || firstOutputTexels(img, plan.steps[0].inputLevel) > kTailMaxTexels)
    return hipErrorInvalidValue;
  const TailSource src = tailSource(img, plan);
  const TailArgs args  = tailArgs(img, plan);
  switch(img.format)
  {
    case NVPRO_PYRAMID_FORMAT_SRGBA8:
      return launchTailTyped<Srgba8>(stream, src, args);
    case NVPRO_PYRAMID_FORMAT_RGBA16F:
      return img.arithmetic == NVPRO_PYRAMID_ARITH_PACKED_FP16 ? launchTailTyped<Rgba16fPacked>(stream, src, args)
                                                               : launchTailTyped<Rgba16f>(stream, src, args);
    case NVPRO_PYRAMID_FORMAT_RGBA32F:
      return launchTailTyped<Rgba32f>(stream, src, args);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace nvpro_pyramid
