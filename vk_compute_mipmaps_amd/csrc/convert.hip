// Level-0 conversion on the device: premultiplied alpha.
//
// The reference premultiplies while staging a file on the host
// (include/scoped_image.hpp:233-252): alpha = a / 255, rgb = srgbFromLinear(
// linearFromSrgb(c) * alpha), alpha byte unchanged.  Here the same formula runs
// on level 0 in device memory, with the functors' exact conversions (the FP32
// rounding of the exact sRGB decode; the exact encode) in place of the host's
// powf.
//
// A byte in and a byte out per byte of the level: bound by memory once a thread
// moves four texels an access.  Workgroups take segments of a row, so that the
// only division is one of scalars per segment; narrow rows with padding have a
// kernel of their own, below.  (A thread per texel with a 64-bit division each
// was bound by those: 3840x2160 sRGBA8, level 0 in the caches, 18.3 us; now 13.7.
// One access in flight a thread 14.1, four 13.9.)
#include "kernel_common.hpp"

namespace nvpro_pyramid {

struct PremultiplySrgba8 : Srgba8
{
  __device__ static Raw texel(const Tables& tab, Raw c)
  {
    const float4 v   = load<false>(tab, c);  // linear RGB
    const float a    = (float)(c >> 24) * (1.0f / 255.0f);
    const uint32_t r = encodeHigh(tab, v.x * a), g = encodeHigh(tab, v.y * a), b = encodeHigh(tab, v.z * a);
    // Bytes: the codes in bits 16-23 of r, g and b, and c's alpha.
    return __builtin_amdgcn_perm(g, r, 0x0c0c0602u) | __builtin_amdgcn_perm(c, b, 0x07020c0cu);
  }
};

// rgb * a in FP32, rounded to binary16; alpha unchanged.
struct PremultiplyRgba16f : Rgba16f
{
  __device__ static Raw texel(const Tables&, Raw q)
  {
    const float a    = h2f(q.hi >> 16);
    const uint32_t r = f2h(h2f(q.lo & 0xffffu) * a), g = f2h(h2f(q.lo >> 16) * a), b = f2h(h2f(q.hi & 0xffffu) * a);
    return Raw{r | g << 16, b | (q.hi & 0xffff0000u)};
  }
};

// Texels a thread moves per access, and accesses it has in flight.
constexpr uint32_t kPremultiplyBS = 256, kPremultiplyPer = 4, kPremultiplyAhead = 2;
constexpr uint32_t kPremultiplySegment = kPremultiplyBS * kPremultiplyPer * kPremultiplyAhead;

// `units` segments of kPremultiplySegment texels (the last of a row shorter), `segments` to a row.
template <class P>
__global__ void __launch_bounds__(kPremultiplyBS) premultiplyKernel(uint8_t* base, uint64_t width, uint32_t pitch,
                                                                   uint64_t segments, uint64_t units)
{
  using Raw              = typename P::Raw;
  constexpr uint32_t PER = kPremultiplyPer, AHEAD = kPremultiplyAhead;
  __shared__ typename P::Tables tab;
  P::template fill<kPremultiplyBS>(tab, 1.0f);
  __syncthreads();
  for(uint64_t u = blockIdx.x; u < units; u += gridDim.x)
  {
    const uint64_t y = units >> 32 ? u / segments : (uint32_t)u / (uint32_t)segments;  // 32 bits for any level that fits memory
    const uint64_t x0   = (u - y * segments) * kPremultiplySegment;
    uint8_t* const row  = base + y * pitch;
    const uint64_t lane = threadIdx.x * PER;
    if(x0 + kPremultiplySegment <= width)  // the same for the whole workgroup
    {
      uint8_t* const p = row + (x0 + lane) * P::kBytes;
      Raw t[AHEAD][PER];
#pragma unroll
      for(uint32_t a = 0; a < AHEAD; ++a)
        loadRow<P, PER>(p + a * kPremultiplyBS * PER * P::kBytes, t[a]);
#pragma unroll
      for(uint32_t a = 0; a < AHEAD; ++a)
      {
#pragma unroll
        for(uint32_t k = 0; k < PER; ++k)
          t[a][k] = P::texel(tab, t[a][k]);
        storeRow<P, PER>(p + a * kPremultiplyBS * PER * P::kBytes, t[a]);
      }
    }
    else
      for(uint64_t x = x0 + threadIdx.x; x < width; x += kPremultiplyBS)
        storeTexel<P>(row + x * P::kBytes, P::texel(tab, loadTexel<P>(row + x * P::kBytes)));
  }
}

// Narrow rows longer than the level: a segment's workgroup has little to do in a
// row of them, so here a workgroup takes units of `rows` rows, as many as there
// are whole ones in kNarrowAhead texels a thread, a texel per lane and access,
// all loads of a unit in flight at once.  A texel's row in the unit is
// t / width = t * inverse >> 20, exact while t * width < 2^20.  (Level 0 in the
// caches, us a call with a segment a row and with units: sRGBA8 64x16384 10.1 and
// 4.0, 16x65535 32.8 and 4.0, 300x9000 8.6 and 5.7, RGBA16F 64x16384 9.2 and 3.9;
// calls this small come every 4 us at best.  Wider rows fill their segments better
// and would leave more of a unit idle: 700x5000 7.6 with segments, and a thread
// per texel with a division each, 9.4.)
constexpr uint32_t kNarrowMost = 512, kNarrowAhead = 8;
static_assert(kNarrowAhead * kPremultiplyBS * kNarrowMost <= 1u << 20, "exact rows");

template <class P>
__global__ void __launch_bounds__(kPremultiplyBS) premultiplyNarrowKernel(uint8_t* base, uint32_t width, uint32_t height,
                                                                         uint32_t pitch, uint32_t inverse,
                                                                         uint32_t rows, uint32_t units)
{
  __shared__ typename P::Tables tab;
  P::template fill<kPremultiplyBS>(tab, 1.0f);
  __syncthreads();
  for(uint32_t u = blockIdx.x; u < units; u += gridDim.x)
  {
    const uint32_t first = u * rows;
    const uint32_t count = height - first < rows ? height - first : rows;
    uint8_t* p[kNarrowAhead];
    bool own[kNarrowAhead];
    typename P::Raw t[kNarrowAhead];
#pragma unroll
    for(uint32_t a = 0; a < kNarrowAhead; ++a)
    {
      // No branch around the loads: past the unit its last row's texels, unused.
      const uint32_t i = a * kPremultiplyBS + threadIdx.x, r = __umul24(i, inverse) >> 20;
      own[a] = r < count;
      p[a]   = base + (uint64_t)(first + (own[a] ? r : count - 1u)) * pitch + (i - __umul24(r, width)) * P::kBytes;
      t[a] = loadTexel<P>(p[a]);
    }
#pragma unroll
    for(uint32_t a = 0; a < kNarrowAhead; ++a)
      if(own[a])
        storeTexel<P>(p[a], P::texel(tab, t[a]));
  }
}

template <class P>
static void launchPremultiply(hipStream_t stream, uint8_t* base, uint32_t imageWidth, uint32_t imageHeight, uint32_t pitch)
{
  // Rows without padding are one long row.
  const bool tight   = pitch == (uint64_t)imageWidth * P::kBytes;
  const uint64_t cap = deviceComputeUnits() * 8u;
  if(!tight && imageWidth <= kNarrowMost)
  {
    const uint32_t rows    = kNarrowAhead * kPremultiplyBS / imageWidth;
    const uint32_t units   = imageHeight / rows + (imageHeight % rows ? 1u : 0u);
    const uint32_t inverse = ((1u << 20) + imageWidth - 1u) / imageWidth;
    const uint32_t grid    = (uint32_t)(units < cap ? units : cap);
    hipLaunchKernelGGL((premultiplyNarrowKernel<P>), dim3(grid), dim3(kPremultiplyBS), 0, stream, base, imageWidth,
                       imageHeight, pitch, inverse, rows, units);
    return;
  }
  const uint64_t width    = (uint64_t)imageWidth * (tight ? imageHeight : 1u);
  const uint64_t segments = (width + kPremultiplySegment - 1u) / kPremultiplySegment;
  const uint64_t units    = segments * (tight ? 1u : imageHeight);
  const uint32_t grid     = (uint32_t)(units < cap ? units : cap);
  hipLaunchKernelGGL((premultiplyKernel<P>), dim3(grid), dim3(kPremultiplyBS), 0, stream, base, width, pitch, segments,
                     units);
}

}  // namespace nvpro_pyramid

using namespace nvpro_pyramid;

extern "C" int nvproPyramidPremultiplyAlpha(hipStream_t stream, uint32_t format, const NvproPyramidImage* image)
{
  const char* who = "nvproPyramidPremultiplyAlpha";
  if(!image || !image->data)
    return hostFail(hipErrorInvalidValue, "%s: null image", who);
  if(format != NVPRO_PYRAMID_FORMAT_SRGBA8 && format != NVPRO_PYRAMID_FORMAT_RGBA16F)
    return hostFail(hipErrorInvalidValue, "%s: format %u not supported", who, format);
  if(image->width == 0 || image->height == 0)
    return hostFail(hipErrorInvalidValue, "%s: zero image size", who);
  const uint32_t bpt   = nvproPyramidBytesPerTexel(format);
  const uint64_t pitch = image->rowPitches ? image->rowPitches[0] : (uint64_t)image->width * bpt;
  const uint64_t off   = image->levelOffsets ? image->levelOffsets[0] : 0u;
  if(pitch < (uint64_t)image->width * bpt || pitch > 0xffffffffull || pitch % bpt != 0 ||
     (((uintptr_t)image->data + off) % bpt) != 0)
    return hostFail(hipErrorInvalidValue, "%s: level 0 layout not aligned to %u bytes", who, bpt);
  uint8_t* base = (uint8_t*)image->data + off;
  if(format == NVPRO_PYRAMID_FORMAT_SRGBA8)
    launchPremultiply<PremultiplySrgba8>(stream, base, image->width, image->height, (uint32_t)pitch);
  else
    launchPremultiply<PremultiplyRgba16f>(stream, base, image->width, image->height, (uint32_t)pitch);
  hipError_t e = hipGetLastError();
  if(e != hipSuccess)
    return hostFail(e, "%s: launch failed: %s", who, hipGetErrorString(e));
  return 0;
}
