// Fast pipeline kernels (nvpro_pyramid.glsl:209-534) for gfx950, wave64: one
// launch per fast step, or per two when the second is a single group or a
// small tail.  The group body (fastGroup) is in groups.hpp.
//
// Workgroups are persistent (the LDS tables are filled once, then the
// workgroup loops over tile groups) and small enough in registers for eight
// waves per SIMD, so the hardware overlaps one wave's loads with another's
// arithmetic (four for 16-byte texels, whose 4x4 block alone takes 64
// registers).
#include <map>
#include <mutex>

#include "groups.hpp"

namespace nvpro_pyramid {

// The arrival counters of fused launches: zero when the code object is loaded,
// and every fused launch leaves its block zeroed, so no memset is ever needed.
// Per device, this array is the only device memory the dispatch path uses
// besides the caller's image.
static __device__ __align__(256) uint32_t gFusedCounters[kFusedSlots * kArriveWords];

uint32_t* fusedCounterBlock(uint32_t slot)
{
  static std::mutex lock;
  static std::map<int, uint32_t*> base;  // by device
  int device = 0;
  if(slot >= kFusedSlots || hipGetDevice(&device) != hipSuccess)
  {
    (void)hipGetLastError();
    return nullptr;
  }
  std::lock_guard<std::mutex> guard(lock);
  auto it = base.find(device);
  if(it == base.end())
  {
    uint32_t* p = nullptr;
    if(hipGetSymbolAddress((void**)&p, HIP_SYMBOL(gFusedCounters)) != hipSuccess)
    {
      (void)hipGetLastError();
      p = nullptr;
    }
    it = base.emplace(device, p).first;
  }
  return it->second ? it->second + (size_t)slot * kArriveWords : nullptr;
}

template <class F, int COUNT, bool CONT>
struct FastShared
{
  typename F::Tables tab;
  typename F::Val level2[(FastGeom<COUNT>::UPPER || CONT) ? kGroupBS : 1];
};

// A fused launch (CONT): the step's last level is stored coherently, and the
// last workgroup to finish (arriveLast) then runs `next`, a fast step of one
// group with the tables it already holds, or a tail plan with its ping-pong in
// the level-2 scratch and the tables refilled at the unscaled decode the tail's
// bodies load with.
static_assert(2u * kFastTailTexels <= (uint32_t)kGroupBS, "tail ping-pong fits the level-2 scratch");

// The groups of a step that this workgroup has, as both kernels below run them.
// The first group's loads are issued behind the tables', so that one memory
// round trip covers both.  NT: the input loads carry the non-temporal hint.
// Returns how many groups it ran.
template <class F, int COUNT, bool CONT, bool NT>
__device__ __forceinline__ uint32_t fastGroups(FastShared<F, COUNT, CONT>& sh, const uint8_t* src, uint32_t pitch,
                                               const FastTilesInverse<COUNT>& tiles, uint32_t blocks,
                                               const FastOut<COUNT, true>& out, uint32_t lines)
{
  constexpr bool STRIP     = COUNT == 6;
  constexpr bool TABLES    = F::kBytes == 4u;  // the other formats have none to overlap, and no registers to spare
  const uint32_t numGroups = (tiles.count + FastGeom<COUNT>::TILES_PER_WG - 1u) / FastGeom<COUNT>::TILES_PER_WG;
  typename F::template TableLoads<kGroupBS> tables;
  F::template fillLoad<kGroupBS>(tables);
  FastWindow<F, COUNT> w;
  uint32_t g = blockIdx.x, iter = 0;
  // The successor's index arithmetic is not to be shared with this: it would be
  // held in registers, or spilled, over the whole loop.
  uint32_t thread = threadIdx.x;
  __asm__ volatile("" : "+v"(thread));
  if constexpr(TABLES)
    fastLoad<F, COUNT, STRIP, NT>(src, pitch, tiles, g, thread, w);
  out.ready();
  F::template fillStore<kGroupBS>(sh.tab, tables, F::kPrescale ? 0.25f : 1.0f);
  __syncthreads();
  levelsReady(lines);
  for(;;)
  {
    if constexpr(!TABLES)
      fastLoad<F, COUNT, STRIP, NT>(src, pitch, tiles, g, thread, w);
    fastCompute<F, COUNT, CONT, STRIP>(sh.tab, sh.level2, out, tiles, g, iter, thread, w);
    g += blocks;
    ++iter;
    if(g >= numGroups)
      return iter;
    if constexpr(TABLES)
      fastLoad<F, COUNT, STRIP, NT>(src, pitch, tiles, g, thread, w);
  }
}

// The leading scalar arguments are in registers at the start (build.py's
// kernarg-preload-count), so that the first loads wait for no argument, and all
// of them are 96 bytes: a launch with more than that costs the host another
// 0.7 us.  With both, chains of 256^2, 1024^2 and 2560x1440 sRGBA8 went from
// 6.4, 8.2 and 16.2 us to 6.2, 7.2 and 13.3.
template <class F, int COUNT, bool NT>
__global__ void __launch_bounds__(kGroupBS) __attribute__((amdgpu_waves_per_eu(F::kBytes > 8u ? 4 : 8, 8)))
fastPipelineKernel(const uint8_t* src, uint32_t pitch, uint32_t numTiles, uint32_t tilesInverse, uint16_t tilesX,
                   uint16_t blocks, FastOut<COUNT, true> out)
{
  __shared__ FastShared<F, COUNT, false> sh;
  fastGroups<F, COUNT, false, NT>(sh, src, pitch, FastTilesInverse<COUNT>(tilesX, numTiles, tilesInverse), blocks, out, 0u);
}

// The same and then, in the last workgroup, the successor (a NextStep's fields).
template <class F, int COUNT, bool NT>
__global__ void __launch_bounds__(kGroupBS) __attribute__((amdgpu_waves_per_eu(F::kBytes > 8u ? 4 : 8, 8)))
fastFusedKernel(const uint8_t* src, uint32_t pitch, uint32_t numTiles, uint32_t tilesInverse, uint16_t tilesX,
                uint16_t blocks, uint32_t* arrive, uint32_t nextKind, uint32_t nextLevel, uint32_t nextCount,
                uint32_t nextTilesX, uint32_t nextTiles, FastOut<COUNT, true> out, ImageDesc img, TailPlan tail)
{
  __shared__ FastShared<F, COUNT, true> sh;
  const uint32_t lines = prefetchLevels(img);
  const FastTilesInverse<COUNT> tiles(tilesX, numTiles, tilesInverse);
  const uint32_t iter = fastGroups<F, COUNT, true, NT>(sh, src, pitch, tiles, blocks, out, lines);
  if(!arriveLast(arrive, blocks, reinterpret_cast<uint32_t*>(sh.level2)))
    return;
  if(nextKind == kNextTail)
  {
    if(F::kPrescale)
    {
      F::template fill<kGroupBS>(sh.tab, 1.0f);
      __syncthreads();
    }
    tailRun<F, false>(sh.tab, sh.level2, sh.level2 + kFastTailTexels, img, tail);
    return;
  }
  switch(nextCount)
  {
    case 1: fastGroup<F, 1>(sh.tab, sh.level2, img, nextLevel, nextTilesX, nextTiles, 0u, iter); break;
    case 2: fastGroup<F, 2>(sh.tab, sh.level2, img, nextLevel, nextTilesX, nextTiles, 0u, iter); break;
    case 3: fastGroup<F, 3>(sh.tab, sh.level2, img, nextLevel, nextTilesX, nextTiles, 0u, iter); break;
    case 4: fastGroup<F, 4>(sh.tab, sh.level2, img, nextLevel, nextTilesX, nextTiles, 0u, iter); break;
    case 5: fastGroup<F, 5>(sh.tab, sh.level2, img, nextLevel, nextTilesX, nextTiles, 0u, iter); break;
    case 6: fastGroup<F, 6>(sh.tab, sh.level2, img, nextLevel, nextTilesX, nextTiles, 0u, iter); break;
    default: break;
  }
}

// Whether a fast step of `groups` groups loads its input with the non-temporal
// hint: sRGBA8 steps of more than one group and up to 64 per compute unit (an
// input of up to 256 MiB), whose input then leaves the caches to the levels
// being written.  Measured on MI355X, us per chain over images that are not in
// any cache, without and with: 1920x1080 13.3 and 12.9, 2048^2 11.5 and 11.1,
// 4096^2 25.0 and 22.7, 8192x4096 47.0 and 41.4, 8192^2 (64 groups) 88 and 74;
// beyond, 10240^2 122 and 127, 16384^2 304 and 324.  Wider texels are slower
// with it at every size (RGBA16F 8192^2 140 and 152, RGBA32F 4096^2 69 and 95).
bool fastInputStreams(uint32_t format, uint64_t groups)
{
  const uint64_t cus = deviceComputeUnits();
  return format == NVPRO_PYRAMID_FORMAT_SRGBA8 && groups > cus && groups <= 64u * cus;
}

template <class F, int COUNT>
static void launchFastCount(hipStream_t stream, const ImageDesc& img, uint32_t inLevel, uint32_t wgPerCU,
                            const NextStep* next, const TailPlan* tail)
{
  const LevelDesc& in     = img.lv[inLevel];
  const uint32_t tilesX   = in.width >> COUNT, tilesY = in.height >> COUNT;
  const uint64_t groups   = fastGroupCount(in.width, in.height, COUNT);
  const uint64_t cap      = min((uint64_t)deviceComputeUnits() * wgPerCU, (uint64_t)0xffffu);
  const uint32_t blocks   = (uint32_t)(groups < cap ? groups : cap);
  const dim3 grid(blocks), wg(kGroupBS);
  const uint32_t inverse  = FastTilesInverse<COUNT>::inverseOf(tilesX);
  FastOut<COUNT, true> out;
  for(int r = 0; r < COUNT; ++r)
  {
    out.base[r]  = img.base + img.lv[inLevel + 1u + (uint32_t)r].offset;
    out.pitch[r] = img.lv[inLevel + 1u + (uint32_t)r].pitch;
  }
  constexpr bool NT = F::kBytes == 4u;
  const bool nt     = fastInputStreams(img.format, groups);
  auto launch       = [&](auto kernel, auto... more) {
    hipLaunchKernelGGL(kernel, grid, wg, 0, stream, img.base + in.offset, in.pitch, tilesX * tilesY, inverse,
                       (uint16_t)tilesX, (uint16_t)blocks, more...);
  };
  if(next)
    launch(nt ? fastFusedKernel<F, COUNT, NT> : fastFusedKernel<F, COUNT, false>, next->arrive, next->kind,
           next->inLevel, next->count, next->tilesX, next->numTiles, out, img, tail ? *tail : TailPlan{});
  else
    launch(nt ? fastPipelineKernel<F, COUNT, NT> : fastPipelineKernel<F, COUNT, false>, out);
}

template <class F>
static hipError_t launchFastTyped(hipStream_t stream, const ImageDesc& img, uint32_t inLevel, uint32_t count,
                                  uint32_t wgPerCU, const NextStep* next, const TailPlan* tail)
{
  switch(count)
  {
    case 1: launchFastCount<F, 1>(stream, img, inLevel, wgPerCU, next, tail); break;
    case 2: launchFastCount<F, 2>(stream, img, inLevel, wgPerCU, next, tail); break;
    case 3: launchFastCount<F, 3>(stream, img, inLevel, wgPerCU, next, tail); break;
    case 4: launchFastCount<F, 4>(stream, img, inLevel, wgPerCU, next, tail); break;
    case 5: launchFastCount<F, 5>(stream, img, inLevel, wgPerCU, next, tail); break;
    case 6: launchFastCount<F, 6>(stream, img, inLevel, wgPerCU, next, tail); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launchFast(hipStream_t stream, const ImageDesc& img, uint32_t inLevel, uint32_t count, uint32_t wgPerCU,
                      const NextStep* next, const TailPlan* tail)
{
  if(next && (!next->arrive || (next->kind == kNextFast && (next->count < 1u || next->count > 6u)) ||
              (next->kind == kNextTail && (!tail || tail->count == 0u || tail->count > NVPRO_PYRAMID_MAX_LEVELS)) ||
              (next->kind != kNextFast && next->kind != kNextTail)))
    return hipErrorInvalidValue;
  switch(img.format)
  {
    case NVPRO_PYRAMID_FORMAT_SRGBA8:
      return launchFastTyped<Srgba8>(stream, img, inLevel, count, wgPerCU, next, tail);
    case NVPRO_PYRAMID_FORMAT_RGBA16F:
      return img.arithmetic == NVPRO_PYRAMID_ARITH_PACKED_FP16
                 ? launchFastTyped<Rgba16fPacked>(stream, img, inLevel, count, wgPerCU, next, tail)
                 : launchFastTyped<Rgba16f>(stream, img, inLevel, count, wgPerCU, next, tail);
    case NVPRO_PYRAMID_FORMAT_RGBA32F:
      return launchFastTyped<Rgba32f>(stream, img, inLevel, count, wgPerCU, next, tail);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace nvpro_pyramid
