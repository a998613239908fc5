// General pipeline kernels (nvpro_pyramid.glsl:536-884) for gfx950: one launch
// per general step of 1 or 2 levels.  The group bodies (generalOneGroup,
// generalTwoGroup) are in groups.hpp.  Also the per-step executor.
#include <stdlib.h>

#include "groups.hpp"

namespace nvpro_pyramid {

template <class F>
struct ThinShared
{
  typename F::Tables tab;
  typename F::Val mid[gen2MidTexels<F, true>()];
};

template <class F>
__global__ void __launch_bounds__(kGroupBS) generalOneLevelKernel(ImageDesc img, uint32_t inLevel, uint32_t groups)
{
  __shared__ typename F::Tables tab;
  const uint32_t lines = prefetchLevels(img);
  F::template fill<kGroupBS>(tab, 1.0f);
  __syncthreads();
  levelsReady(lines);
  for(uint32_t g = blockIdx.x; g < groups; g += gridDim.x)
    generalOneGroup<F>(tab, img, inLevel, g);
}

// Thin tiles, one per workgroup (the grid is numTiles): straight-line code.
// The window's loads are issued behind the tables', one memory round trip for
// both (2002x1234 RGBA32F chain 23.6 -> 23.2 us, 801x401 sRGBA8 14.7 -> 14.1).
// KX, KY: the first level's kernel sizes, or 0 (read from the image).
template <class F, int KX, int KY>
__global__ void __launch_bounds__(kGroupBS) thinTwoLevelKernel(ImageDesc img, uint32_t inLevel, uint32_t tilesX,
                                                             uint32_t numTiles)
{
  __shared__ ThinShared<F> sh;
  if(blockIdx.x >= numTiles)  // the same for the whole workgroup
    return;
  typename F::template TableLoads<kGroupBS> tables;
  F::template fillLoad<kGroupBS>(tables);
  const uint32_t lines = prefetchLevels(img);
  Gen2Window<F, true> w;
  gen2Load<F, KX, KY, true>(img, inLevel, tilesX, blockIdx.x, w);
  F::template fillStore<kGroupBS>(sh.tab, tables, 1.0f);
  __syncthreads();
  levelsReady(lines);
  gen2Compute<F, false, KX, KY, true>(sh.tab, sh.mid, img, inLevel, tilesX, blockIdx.x, w);
}

// One strip group per workgroup, strips of a row of groups side by side, in the
// order of xcdContiguous: neighbouring groups share cache lines at their
// borders, and groups in flight together read one region of memory (4095^2 and
// 8191^2, memory accesses alone: 20.9 -> 19.2 and 73 -> 66 us).  The tables'
// loads are issued first and the window's behind them, so that one memory round
// trip covers both (4095x2047 15.9 -> 14.3 us, 8191^2 86 -> 78).
using StripWide = StripGeom<8, 1>;

template <class F>
struct StripShared
{
  typename F::Tables tab;
  typename F::Val border[StripWide::BORDER];
};

template <class F, int KX, int KY>
__global__ void __launch_bounds__(StripWide::BS) __attribute__((amdgpu_waves_per_eu(4, 8)))
stripKernel(StripStep step, uint32_t strips, uint32_t stripsInverse)
{
  constexpr int BS = StripWide::BS;
  __shared__ StripShared<F> sh;
  typename F::template TableLoads<BS> tables;
  F::template fillLoad<BS>(tables);
  const uint32_t unit  = xcdContiguous(blockIdx.x, gridDim.x);
  const uint32_t block = strips == 1u ? unit : __umulhi(unit, stripsInverse);  // unit / strips
  const StripLane L    = stripLane<StripWide>(step, unit - block * strips, block);
  StripWindow<F, StripWide, KY> w;
  stripLoad<F, StripWide, KY>(step, L, w);
  F::template fillStore<BS>(sh.tab, tables, 1.0f);
  __syncthreads();
  stripMoved<F, StripWide, KY>(step, L, w);
  stripCompute<F, StripWide, KX, KY>(sh.tab, sh.border, step, L, w);
}

// Workgroups of `kernel` that are resident on one compute unit at once.
template <class K>
static uint32_t residentPerCU(K kernel, int threads)
{
  int n = 0;
  if(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, threads, 0) != hipSuccess || n <= 0)
    n = 1;
  return (uint32_t)n;
}

// A step with at most two thin tiles per compute unit runs thin tiles: its time
// is then one tile's latency, and a thin tile's lanes run less serial work than
// a strip's.  A larger one runs strips, which decode and load less at the
// borders (us per G(0,2), thin and strips; sRGBA8: 801x401, 238 thin tiles, 4.4
// and 4.6; 1001x501, 378 tiles, 4.9 and 4.6, but after a larger step, whose
// output is in the caches, thin: 2047x1023 chains 18.7 and 19.5; 1201x701, 590 tiles, 5.5 and 4.9; 2002x1234
// 8.05 and 6.5; RGBA16F 4.3 and 4.4, 4.8 and 4.4, 5.6 and 4.9, 9.1 and 8.4).
// 16-byte texels run thin tiles while they all fit on the GPU at once (RGBA32F
// 1001x501 5.7 and 6.5, 2002x1234 14.3 and 15.4; in between, 1501x1001, 10.3 and
// 8.9).  A step with a first-level side of 1 always runs
// thin tiles (a 65535-texel side has 529 of them).  The environment variable
// NVPRO_PYRAMID_THIN=1 / =0 forces thin tiles / strips where both apply (the
// bytes are the same either way).
template <class F, int KX, int KY>
static void launchTwoLevel(hipStream_t stream, const ImageDesc& img, uint32_t inLevel)
{
  static const uint32_t perCU = F::kBytes > 8u ? residentPerCU(thinTwoLevelKernel<F, KX, KY>, kGroupBS) : 2u;
  const LevelDesc& d          = img.lv[inLevel + 2u];
  uint32_t thinX              = 0;
  const uint32_t numThin = generalGroupCount(d.width, d.height, 2u, F::kBytes, &thinX, true);
  const char* force      = getenv("NVPRO_PYRAMID_THIN");
  const bool thin        = force && (force[0] == '0' || force[0] == '1')
                               ? force[0] == '1'
                               : (uint64_t)numThin <= (uint64_t)deviceComputeUnits() * perCU;
  if constexpr(KX != 0 && KY != 0)
    if(!thin && stripsApply(img, inLevel))
    {
      const uint32_t strips  = stripCount(d.width), rows = StripWide::rows(img.lv[inLevel + 1u].height);
      const uint32_t blocks  = (d.height + rows - 1u) / rows;
      const uint32_t inverse = (uint32_t)((0x100000000ull + strips - 1u) / strips);
      hipLaunchKernelGGL((stripKernel<F, KX, KY>), dim3(strips * blocks), dim3(StripWide::BS), 0, stream,
                         stripStep(img, inLevel), strips, inverse);
      return;
    }
  hipLaunchKernelGGL((thinTwoLevelKernel<F, KX, KY>), dim3(numThin), dim3(kGroupBS), 0, stream, img, inLevel, thinX,
                     numThin);
}

template <class F>
static hipError_t launchGeneralTyped(hipStream_t stream, const ImageDesc& img, uint32_t inLevel, uint32_t count)
{
  if(count == 1u)
  {
    static const uint32_t oneFit = residentPerCU(generalOneLevelKernel<F>, kGroupBS);
    const LevelDesc& d           = img.lv[inLevel + 1u];
    uint32_t unused              = 0;
    const uint64_t want          = generalGroupCount(d.width, d.height, 1u, F::kBytes, &unused);
    const uint64_t cap    = (uint64_t)deviceComputeUnits() * oneFit;
    const uint32_t blocks = (uint32_t)(want < cap ? want : cap);
    hipLaunchKernelGGL((generalOneLevelKernel<F>), dim3(blocks ? blocks : 1), dim3(kGroupBS), 0, stream, img,
                       inLevel, (uint32_t)want);
    return hipGetLastError();
  }
  // Two levels: the kernel specialised for the first level's kernel sizes.
  const int kx = kernelSize(img.lv[inLevel].width), ky = kernelSize(img.lv[inLevel].height);
  if(kx == 3 && ky == 3)
    launchTwoLevel<F, 3, 3>(stream, img, inLevel);
  else if(kx == 2 && ky == 2)
    launchTwoLevel<F, 2, 2>(stream, img, inLevel);
  else if(kx == 3 && ky == 2)
    launchTwoLevel<F, 3, 2>(stream, img, inLevel);
  else if(kx == 2 && ky == 3)
    launchTwoLevel<F, 2, 3>(stream, img, inLevel);
  else
    launchTwoLevel<F, 0, 0>(stream, img, inLevel);
  return hipGetLastError();
}

hipError_t launchGeneral(hipStream_t stream, const ImageDesc& img, uint32_t inLevel, uint32_t count)
{
  switch(img.format)
  {
    case NVPRO_PYRAMID_FORMAT_SRGBA8:
      return launchGeneralTyped<Srgba8>(stream, img, inLevel, count);
    case NVPRO_PYRAMID_FORMAT_RGBA16F:
      return img.arithmetic == NVPRO_PYRAMID_ARITH_PACKED_FP16
                 ? launchGeneralTyped<Rgba16fPacked>(stream, img, inLevel, count)
                 : launchGeneralTyped<Rgba16f>(stream, img, inLevel, count);
    case NVPRO_PYRAMID_FORMAT_RGBA32F:
      return launchGeneralTyped<Rgba32f>(stream, img, inLevel, count);
    default:
      return hipErrorInvalidValue;
  }
}

uint32_t deviceComputeUnits()
{
  static uint32_t cached[64] = {};
  int dev = 0;
  if(hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64)
    return 256u;
  if(cached[dev] == 0u)
  {
    int cus = 0;
    if(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      cus = 256;
    cached[dev] = (uint32_t)cus;
  }
  return cached[dev];
}

static TailPlan tailFrom(const NvproPyramidStep* steps, uint32_t first, uint32_t count)
{
  TailPlan plan{};
  for(uint32_t k = first; k < count && plan.count < NVPRO_PYRAMID_MAX_LEVELS; ++k)
    plan.steps[plan.count++] = TailStep{steps[k].pipeline, steps[k].inputLevel, steps[k].levelCount, 0u};
  return plan;
}

static uint64_t firstOutput(const ImageDesc& img, const NvproPyramidStep& s)
{
  const LevelDesc& first = img.lv[s.inputLevel + 1u];
  return (uint64_t)first.width * first.height;
}

// Whether each of the steps from `first` on starts at the level the one before
// it ends with, as the dispatcher loop's own steps do (a custom dispatcher may
// record others): a tail hands its levels on without reading them back.
static bool consecutive(const NvproPyramidStep* steps, uint32_t first, uint32_t count)
{
  for(uint32_t k = first; k + 1u < count; ++k)
    if(steps[k + 1u].inputLevel != steps[k].inputLevel + steps[k].levelCount)
      return false;
  return true;
}

// Persistent workgroups per compute unit of a fast step (at most 8 fit):
// fewer than fit leave fewer waves to hide latency behind, but the rows that
// are read at one time, which lie far apart in a large image, are fewer too.
// Measured on MI355X, us per chain over images that are not in any cache:
// sRGBA8 with the input loads of fastInputStreams, 5 against 8 and 4: 4096^2
// (16 groups per unit) 22.7, 23.0, 23.4; 5120^2 34.1, 35.2, 34.0; 6144^2 45.2,
// 44.7, 43.8; 8192^2 (64) 73.8, 75.5, 74.5; without them, 4 against 8:
// 10240^2 123 and 132, 16384^2 (256) 323 and 345 (with 2: 350; with 3, 298 to
// 307 against 4's 298 to 323 by where the images lie in memory).  Texels of 8
// and 16 bytes, 2 against 8: RGBA16F 3072^2 24.9 and 27.0, 4096^2 37.9 and
// 38.7, 12288x8192 209 and 220; RGBA32F 4096^2 69.3 and 71.4.
static uint32_t fastWorkgroupsPerCU(const ImageDesc& img, uint64_t groups)
{
  if(img.format != NVPRO_PYRAMID_FORMAT_SRGBA8)
    return 2u;
  return fastInputStreams(img.format, groups) || groups <= deviceComputeUnits() ? 5u : 4u;
}

static uint32_t fastWorkgroupsPerCU(const ImageDesc& img, const NvproPyramidStep& s)
{
  const LevelDesc& in = img.lv[s.inputLevel];
  return fastWorkgroupsPerCU(img, fastGroupCount(in.width, in.height, s.levelCount));
}

// Whether fusing a successor into fast step s pays, by the step's workgroups
// (measured on MI355X, sRGBA8): a small grid counts at one arrival counter and
// gains the successor's launch and start-up (4 workgroups with a one-texel
// tail: 8.7 -> 7.2 us); a large grid also skips waiting for its own end of
// kernel, the write-back of everything it stored (2048 workgroups of 4096^2
// with F(6,6): 28.1 -> 26.5 us per chain); in between, two arrival counts and
// the continuation cost what they save (256 workgroups of 1024^2 with F(6,4):
// 7.4 -> 8.2 us).
static bool fusionPays(const ImageDesc& img, const NvproPyramidStep& s)
{
  const LevelDesc& in   = img.lv[s.inputLevel];
  const uint64_t groups = fastGroupCount(in.width, in.height, s.levelCount);
  const uint64_t cap    = (uint64_t)fastWorkgroupsPerCU(img, groups) * deviceComputeUnits();
  const uint64_t blocks = groups < cap ? groups : cap;
  return blocks <= kArriveLeaves || blocks >= 4ull * deviceComputeUnits();
}

hipError_t executePlan(hipStream_t stream, const ImageDesc& img, const NvproPyramidStep* steps, uint32_t count,
                       uint32_t* arrive, uint32_t* launches)
{
  *launches = 0;
  for(uint32_t i = 0; i < count; ++i, ++*launches)
  {
    const NvproPyramidStep& s = steps[i];
    // The one-workgroup tail pays off when it saves launches: with a single step
    // left, that step's own kernel is as quick.
    if(firstOutput(img, s) <= kTailMaxTexels && count - i >= 2u && consecutive(steps, i, count))
    {
      ++*launches;
      return launchTail(stream, img, tailFrom(steps, i, count));
    }
    const bool fast = s.pipeline == NVPRO_PYRAMID_PIPELINE_FAST;
    if(arrive && i + 1u < count && fast && fusionPays(img, s))
    {
      // Fusion: the successor runs in this launch's last workgroup, saving a
      // launch and the second kernel's start-up (tables, first loads).  It has to
      // read this step's last level, the only one stored for other workgroups to
      // see, and a tail's steps each the one before's.
      const NvproPyramidStep& n = steps[i + 1u];
      const LevelDesc& nin      = img.lv[n.inputLevel];
      if(n.pipeline == NVPRO_PYRAMID_PIPELINE_FAST && fastGroupCount(nin.width, nin.height, n.levelCount) == 1u
         && consecutive(steps, i, i + 2u))
      {
        const uint32_t tilesX = nin.width >> n.levelCount, tilesY = nin.height >> n.levelCount;
        const NextStep next{arrive, kNextFast, n.inputLevel, n.levelCount, tilesX, tilesX * tilesY};
        if(hipError_t e = launchFast(stream, img, s.inputLevel, s.levelCount, fastWorkgroupsPerCU(img, s), &next))
          return e;
        ++i;
        continue;
      }
      // A tail small enough for the fast kernel's scratch.  (A general step
      // followed by a tail measured no faster fused: the tail's first level
      // then takes several passes of a 256-thread workgroup, where the tail
      // kernel takes one pass of 1024 threads.)
      if(firstOutput(img, n) <= kFastTailTexels && consecutive(steps, i, count))
      {
        const TailPlan tail = tailFrom(steps, i + 1u, count);
        const NextStep next{arrive, kNextTail, 0u, 0u, 0u, 0u};
        ++*launches;
        return launchFast(stream, img, s.inputLevel, s.levelCount, fastWorkgroupsPerCU(img, s), &next, &tail);
      }
    }
    uint32_t tileX = 0, tileY = 0;
    if(const uint32_t n = tileSteps(img, steps + i, count - i, &tileX, &tileY))
    {
      if(hipError_t e = launchTiles(stream, img, tailFrom(steps, i, i + n), tileX, tileY))
        return e;
      i += n - 1u;
      continue;
    }
    hipError_t e = fast ? launchFast(stream, img, s.inputLevel, s.levelCount, fastWorkgroupsPerCU(img, s))
                        : launchGeneral(stream, img, s.inputLevel, s.levelCount);
    if(e != hipSuccess)
      return e;
  }
  return hipSuccess;
}

}  // namespace nvpro_pyramid
