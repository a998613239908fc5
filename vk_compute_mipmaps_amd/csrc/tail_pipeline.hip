// Tail kernel: the small remainder of a plan in one workgroup, and small runs
// of steps before it in one launch of tiles.
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
//
// Tiles (TILED): steps of a few levels, too large for one workgroup but small
// enough that each launch is one tile's latency, run in one launch instead of
// one each.  A workgroup computes a tile of the last of the levels and, above
// it, the windows the tile needs: twice its size and one more texel a level, so
// four levels read 79x47 texels for 64x32 and compute the texels shared with a
// neighbour twice; each texel is stored by the workgroup that owns it.  RGBA16F
// 4095x2047, whose four levels under 1023x511 were two steps: 34.0 -> 31.5 us a
// chain; RGBA32F 2002x1234: 25.8 -> 23.7.  Two or four times as many smaller
// tiles, and the tail in the last workgroup of the same launch, were slower
// (RGBA16F 33.1, 33.3 us): more windows overlap, and a launch costs less than
// arriving and reading the levels back.
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
  uint32_t sides, own; // of a tile: the level's width | height << 16, and the same of what the tile owns
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
  uint32_t inverse;     // texel / width is the high word of texel * inverse
  uint32_t sides, own;  // as TailLevel's
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
  __asm__ volatile("" : "+s"(q.sides), "+s"(q.own));
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

// Where a level's window lies: its first texel, and how many of its columns
// and rows are in the level and which of those this workgroup stores.
struct TailPlace
{
  uint32_t x0, y0, width, height, ownWidth, ownHeight;
};
template <bool TILED>
__device__ __forceinline__ TailPlace tailPlace(uint32_t sides, uint32_t own)
{
  TailPlace p{};
  if constexpr(TILED)
  {
    p.x0        = blockIdx.x * (own & 0xffffu);
    p.y0        = blockIdx.y * (own >> 16);
    p.width     = (sides & 0xffffu) - p.x0;
    p.height    = (sides >> 16) - p.y0;
    p.ownWidth  = blockIdx.x + 1u < gridDim.x ? own & 0xffffu : p.width;
    p.ownHeight = blockIdx.y + 1u < gridDim.y ? own >> 16 : p.height;
  }
  return p;
}

template <class F, bool TILED>
__global__ void __launch_bounds__(kTailBS) tailKernel(const uint8_t* srcBase, uint32_t srcPitch,
                                                      uint32_t srcWidth, uint32_t srcTexels,
                                                      uint32_t srcInverse, uint32_t srcSides, uint32_t srcOwn,
                                                      TailArgs a)
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
  const TailPlace from     = tailPlace<TILED>(srcSides, srcOwn);
  auto sourceLoad          = [&](uint32_t base, Raw(&r)[AHEAD]) {
#pragma unroll
    for(uint32_t k = 0; k < AHEAD; ++k)
    {
      uint32_t i       = base + k * kTailBS + threadIdx.x;
      i                = i < srcTexels ? i : srcTexels - 1u;
      uint32_t y = srcWidth == 1u ? i : __umulhi(i, srcInverse), x = i - y * srcWidth;
      if constexpr(TILED)
      {
        x = from.x0 + (x < from.width ? x : from.width - 1u);
        y = from.y0 + (y < from.height ? y : from.height - 1u);
      }
      r[k] = loadTexel<F>(srcBase + (uint64_t)y * srcPitch + x * F::kBytes);
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
    const TailPlace p = tailPlace<TILED>(q.sides, q.own);
    if(alone && threadIdx.x >= 64u)
      return;  // levels only get smaller: the first wave finishes them
    if(n > kTailBS)
      for(uint32_t t = threadIdx.x; t < q.texels; t += kTailBS)
      {
        const uint32_t y = __umul24(t, q.inverse) >> 20, x = t - __umul24(y, q.width);
        const V* s = src + __umul24(2u * y, q.srcWidth) + 2u * x;
        auto at    = [&](int j, int r) { return s[(uint32_t)r * q.srcWidth + (uint32_t)j]; };
        const uint32_t gx = TILED ? p.x0 + (x < p.width ? x : p.width - 1u) : x;
        const uint32_t gy = TILED ? p.y0 + (y < p.height ? y : p.height - 1u) : y;
        const V v         = tailSample<F>(at, q, gx, gy);
        const Raw code    = F::store(tab, v);
        if(!TILED || (x < p.ownWidth && y < p.ownHeight))
          storeTexel<F>(q.dst + (uint64_t)gy * q.pitch + gx * F::kBytes, code);
        dst[t] = q.requantise ? F::template load<false>(tab, code) : v;
      }
    else if(threadIdx.x < n)
    {
      const uint32_t c = threadIdx.x & 3u, t = threadIdx.x >> 2;
      const uint32_t y = __umul24(t, q.inverse) >> 20, x = t - __umul24(y, q.width);
      const Chan* s = reinterpret_cast<const Chan*>(src + __umul24(2u * y, q.srcWidth) + 2u * x) + c;
      auto at       = [&](int j, int r) { return s[4u * ((uint32_t)r * q.srcWidth + (uint32_t)j)]; };
      const uint32_t gx = TILED ? p.x0 + (x < p.width ? x : p.width - 1u) : x;
      const uint32_t gy = TILED ? p.y0 + (y < p.height ? y : p.height - 1u) : y;
      const Chan v      = tailSample<C>(at, q, gx, gy);
      const Q code      = F::chanStore(tab, v, c);
      if(!TILED || (x < p.ownWidth && y < p.ownHeight))
        reinterpret_cast<Q*>(q.dst + (uint64_t)gy * q.pitch + gx * F::kBytes)[c] = code;
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

// Tiles of tileX x tileY texels of the plan's last level (0: one workgroup for
// the whole levels).  A tile's window in the level `shift` levels above that
// one: (tile << shift) texels it owns and the 2^shift - 1 that they need beside
// (a window of 3 starts at twice the index), cut at the level's edge; the last
// tile owns the texels beyond the last window too.
static uint32_t tileWindow(uint32_t tile, uint32_t shift)
{
  return (tile << shift) + (1u << shift) - 1u;
}

static TailSource tailSource(const ImageDesc& img, const TailPlan& plan, uint32_t levels, uint32_t tileX,
                             uint32_t tileY)
{
  const LevelDesc& l = img.lv[plan.steps[0].inputLevel];
  const uint32_t w = tileX ? tileWindow(tileX, levels) : l.width, h = tileY ? tileWindow(tileY, levels) : l.height;
  return TailSource{img.base + l.offset, l.pitch, w, w * h, (uint32_t)((0x100000000ull + w - 1u) / w),
                    l.width | l.height << 16, tileX << levels | tileY << (levels + 16u)};
}

static TailArgs tailArgs(const ImageDesc& img, const TailPlan& plan, uint32_t levels, uint32_t tileX, uint32_t tileY)
{
  TailArgs a{};
  uint32_t srcWidth = tileX ? tileWindow(tileX, levels) : img.lv[plan.steps[0].inputLevel].width;
  for(uint32_t s = 0; s < plan.count; ++s)
    for(uint32_t r = 1; r <= plan.steps[s].levelCount; ++r)
    {
      const LevelDesc &sl = img.lv[plan.steps[s].inputLevel + r - 1u], &dl = img.lv[plan.steps[s].inputLevel + r];
      const bool fast     = plan.steps[s].pipeline == NVPRO_PYRAMID_PIPELINE_FAST;
      TailLevel& q        = a.lv[a.count++];
      const uint32_t left = levels - a.count;
      q.dst               = img.base + dl.offset;
      q.pitch             = dl.pitch;
      q.width             = tileX ? tileWindow(tileX, left) : dl.width;
      q.texels            = q.width * (tileY ? tileWindow(tileY, left) : dl.height);
      q.inverse           = ((1u << 20) + q.width - 1u) / q.width;
      q.srcWidth          = srcWidth;
      q.mode = tailMode(fast, fastOrder(plan.steps[s].levelCount, r), kernelSize(sl.width), kernelSize(sl.height));
      q.requantise = r == plan.steps[s].levelCount ? 1u : 0u;
      q.ax         = axis3(dl.width);
      q.ay         = axis3(dl.height);
      q.sides      = dl.width | dl.height << 16;
      q.own        = tileX << left | tileY << (left + 16u);
      srcWidth     = q.width;
    }
  return a;
}

template <class F>
static hipError_t launchTailTyped(hipStream_t stream, const TailSource& src, const TailArgs& args, dim3 tiles)
{
  if(args.lv[0].own)
    hipLaunchKernelGGL((tailKernel<F, true>), tiles, dim3(kTailBS), tailSharedBytes<F>(src, args), stream, src.base,
                       src.pitch, src.width, src.texels, src.inverse, src.sides, src.own, args);
  else
    hipLaunchKernelGGL((tailKernel<F, false>), dim3(1), dim3(kTailBS), tailSharedBytes<F>(src, args), stream,
                       src.base, src.pitch, src.width, src.texels, src.inverse, src.sides, src.own, args);
  return hipGetLastError();
}

static hipError_t launchTailTiles(hipStream_t stream, const ImageDesc& img, const TailPlan& plan, uint32_t levels,
                                  uint32_t tileX, uint32_t tileY)
{
  const TailStep& last = plan.steps[plan.count - 1u];
  const LevelDesc& d   = img.lv[last.inputLevel + last.levelCount];
  const dim3 tiles     = tileX ? dim3((d.width + tileX - 1u) / tileX, (d.height + tileY - 1u) / tileY) : dim3(1);
  const TailSource src = tailSource(img, plan, levels, tileX, tileY);
  const TailArgs args  = tailArgs(img, plan, levels, tileX, tileY);
  switch(img.format)
  {
    case NVPRO_PYRAMID_FORMAT_SRGBA8:
      return launchTailTyped<Srgba8>(stream, src, args, tiles);
    case NVPRO_PYRAMID_FORMAT_RGBA16F:
      return img.arithmetic == NVPRO_PYRAMID_ARITH_PACKED_FP16
                 ? launchTailTyped<Rgba16fPacked>(stream, src, args, tiles)
                 : launchTailTyped<Rgba16f>(stream, src, args, tiles);
    case NVPRO_PYRAMID_FORMAT_RGBA32F:
      return launchTailTyped<Rgba32f>(stream, src, args, tiles);
    default:
      return hipErrorInvalidValue;
  }
}

static uint32_t tailLevels(const TailPlan& plan)
{
  uint32_t levels = 0;
  for(uint32_t s = 0; s < plan.count; ++s)
    levels += plan.steps[s].levelCount;
  return levels;
}

hipError_t launchTail(hipStream_t stream, const ImageDesc& img, const TailPlan& plan)
{
  const uint32_t levels = tailLevels(plan);
  if(plan.count == 0u || levels > kTailLevels || firstOutputTexels(img, plan.steps[0].inputLevel) > kTailMaxTexels)
    return hipErrorInvalidValue;
  return launchTailTiles(stream, img, plan, levels, 0u, 0u);
}

// The steps (from steps[0] on, two at least or 0) that one launch of tiles runs,
// and the tile: the smallest of which there is at most one per compute unit.
// With more, each unit has several to run one after the other, and steps of one
// launch each, which read and compute every texel once, are as quick (1023x1023
// sRGBA8 in 256 tiles of 4x4: 16.2 -> 14.9 us a chain; two tiles a unit: 19.3).
// Where the second step could be in the tail, tiles save no launch: they pay
// while its first level is more than one pass of the tail's workgroup by
// channels (255x127 sRGBA8, 465 texels: 9.0 -> 8.6 us, 257x257, 1024 texels:
// 8.2 -> 7.5; 127x127, 225 texels: 8.05 -> 8.4).  sRGBA8 steps that the general
// pipeline begins keep one launch each before the tail, the number that the
// dispatch's interface states.
uint32_t tileSteps(const ImageDesc& img, const NvproPyramidStep* steps, uint32_t count, uint32_t* tileX,
                   uint32_t* tileY)
{
  uint32_t n = 0, levels = 0;
  while(n < count && levels + steps[n].levelCount <= kTileLevels
        && (n == 0u || steps[n].inputLevel == steps[n - 1u].inputLevel + steps[n - 1u].levelCount))
    levels += steps[n++].levelCount;
  if(n < 2u)
    return 0u;
  const uint64_t second = firstOutputTexels(img, steps[1].inputLevel);
  const bool oneEach =
      img.format == NVPRO_PYRAMID_FORMAT_SRGBA8 && steps[0].pipeline == NVPRO_PYRAMID_PIPELINE_GENERAL;
  if(second > kTailMaxTexels ? oneEach : 4u * second <= kTailBS)
    return 0u;
  const LevelDesc& d = img.lv[steps[0].inputLevel + levels];
  uint32_t x = 1, y = 1;
  while((uint64_t)((d.width + x - 1u) / x) * ((d.height + y - 1u) / y) > deviceComputeUnits())
  {
    if(y == kTileSide)
      return 0u;
    (x <= y ? x : y) *= 2u;
  }
  *tileX = x;
  *tileY = y;
  return n;
}

hipError_t launchTiles(hipStream_t stream, const ImageDesc& img, const TailPlan& plan, uint32_t tileX, uint32_t tileY)
{
  const uint32_t levels = tailLevels(plan);
  if(plan.count == 0u || levels > kTileLevels || tileX == 0u || tileX > kTileSide || tileY == 0u || tileY > kTileSide)
    return hipErrorInvalidValue;
  return launchTailTiles(stream, img, plan, levels, tileX, tileY);
}

}  // namespace nvpro_pyramid
