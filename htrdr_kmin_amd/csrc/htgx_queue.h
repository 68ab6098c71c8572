/*
 * The chunk queue of the persistent solvers and the merge of its results.
 *
 * A chunk is up to K consecutive realisations of one pixel. Chunks are handed
 * out by atomic counters, one per XCD over a contiguous range of 8x8 tiles
 * (pixels of a tile in Morton order, src/core/htrdr_draw_map.c:301-319), so
 * that the wavefronts of an XCD trace neighbouring pixels and share its L2; an
 * XCD whose range is empty takes chunks from the others. Every chunk writes a
 * partial accumulator of its own and the merge folds them per pixel in chunk
 * order, so a map does not depend on the schedule.
 *
 * A map may have several planes (the channels of a CIE XYZ image) that follow
 * each other in the queue: one launch, so that the longest walks of a plane,
 * which end alone, overlap with the others.
 *
 * The queue is any struct with the fields width, height, ntx, K, nsub, planes,
 * plane_tiles (tiles of a plane), ntiles (of all), xcd_tiles and counters.
 */
#ifndef HTGX_QUEUE_H
#define HTGX_QUEUE_H

#include "htgx.h"

#include <hip/hip_runtime.h>

#include <math.h>

namespace {

constexpr int kXcds = 8;

/* Chunks for the lanes with `need', from this XCD's tile range, else from the
 * others: one atomic per wavefront and range, the lanes sharing what it
 * reserved in lane order. `tried' counts the ranges the wavefront has found
 * empty; it does not ask them again. Returns false for a lane that finds no
 * chunk left anywhere. The whole wavefront calls this together. */
template<class Q>
__device__ __forceinline__ bool fetch_chunks(const Q& P, uint32_t xcd, uint32_t* tried, bool need,
                                             uint32_t* chunk)
{
  const uint32_t per_tile = P.nsub * 64u;
  bool got = false;
  uint64_t mask = __ballot(need);
  while(mask && *tried < (uint32_t)kXcds) {
    const uint32_t x = (xcd + *tried) % (uint32_t)kXcds;
    const uint32_t t0 = min(x * P.xcd_tiles, P.ntiles), t1 = min(t0 + P.xcd_tiles, P.ntiles);
    const uint32_t n = (t1 - t0) * per_tile;
    if(n) {
      const int leader = __ffsll((unsigned long long)mask) - 1;
      uint32_t c = 0;
      if((int)(threadIdx.x & 63u) == leader) c = atomicAdd(P.counters + x, (uint32_t)__popcll(mask));
      c = (uint32_t)__builtin_amdgcn_readlane((int)c, leader) +
          (uint32_t)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                              __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
      if(need && !got && c < n) { *chunk = t0 * per_tile + c; got = true; }
    }
    mask = __ballot(need && !got);
    if(mask) ++*tried;
  }
  return got;
}

/* Pixel, slice and plane of a chunk; false if the pixel lies outside the image */
template<class Q>
__device__ __forceinline__ bool chunk_pixel(const Q& P, uint32_t c, uint32_t* pixel, uint32_t* sub,
                                            uint32_t* plane)
{
  const uint32_t m = c & 63u, rest = c >> 6;
  const uint32_t tt = rest / P.nsub, t = tt % P.plane_tiles;
  *sub = rest % P.nsub;
  *plane = tt / P.plane_tiles;
  const uint32_t x = (t % P.ntx) * 8u + ((m & 1u) | ((m >> 1) & 2u) | ((m >> 2) & 4u));
  const uint32_t y = (t / P.ntx) * 8u + (((m >> 1) & 1u) | ((m >> 2) & 2u) | ((m >> 3) & 4u));
  *pixel = y * P.width + x;
  return x < P.width && y < P.height;
}

/* Neumaier compensated accumulation */
__device__ __forceinline__ void neumaier(double& sum, double& c, double x)
{
  const double t = sum + x;
  if(fabs(sum) >= fabs(x)) c += (sum - t) + x;
  else c += (x - t) + sum;
  sum = t;
}

/* Fold the chunks of pixel i (of all planes), in chunk order, into its
 * accumulator */
template<class Q>
__device__ __forceinline__ void
merge_pixel(const Q& P, htgx_mc_accum* accum, uint32_t i)
{
  const uint32_t npix = P.width * P.height, p = i % npix, nsub = P.nsub;
  const uint32_t x = p % P.width, y = p / P.width;
  const uint32_t t = (i / npix) * P.plane_tiles + (y / 8u) * P.ntx + (x / 8u);
  const uint32_t ix = x & 7u, iy = y & 7u;
  const uint32_t m = (ix & 1u) | ((iy & 1u) << 1) | ((ix & 2u) << 1) | ((iy & 2u) << 2)
                   | ((ix & 4u) << 2) | ((iy & 4u) << 3);
  htgx_mc_accum a = accum[i];
  for(uint32_t s = 0; s < nsub; ++s) {
    const htgx_mc_accum q = P.partials[((size_t)t * nsub + s) * 64u + m];
    neumaier(a.sum, a.sum_c, q.sum);
    a.sum_c += q.sum_c;
    neumaier(a.sum2, a.sum2_c, q.sum2);
    a.sum2_c += q.sum2_c;
    a.tsum += q.tsum;
    a.tsum2 += q.tsum2;
    a.n += q.n;
    a.nfail += q.nfail;
  }
  accum[i] = a;
}

template<class Q>
__global__ void __launch_bounds__(256)
merge_chunks_kernel(Q P, htgx_mc_accum* accum)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i < P.width * P.height * P.planes) merge_pixel(P, accum, i);
}

/* The queue's sizes for a map of width x height pixels */
template<class Q>
inline void set_queue_size(Q& P, uint32_t width, uint32_t height, uint32_t planes)
{
  P.width = width;
  P.height = height;
  P.ntx = (width + 7) / 8;
  P.planes = planes;
  P.plane_tiles = P.ntx * ((height + 7) / 8);
  P.ntiles = P.plane_tiles * planes;
  P.xcd_tiles = (P.ntiles + kXcds - 1) / kXcds;
}

__global__ void
zero_u32_kernel(unsigned int* p, uint32_t n)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i < n) p[i] = 0u;
}

__global__ void
zero_u64_kernel(unsigned long long* p, uint32_t n)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i < n) p[i] = 0ull;
}

__device__ __forceinline__ uint64_t wave_sum64(uint64_t v)
{
  for(int off = 32; off > 0; off >>= 1) v += (uint64_t)__shfl_xor((unsigned long long)v, off, 64);
  return v;
}

/* Pointers to constant memory (the kernel argument segment, or a table in
 * device memory that no kernel writes while it is read), and scalar loads
 * through them; the host compilation pass, which only needs the declaration,
 * gets an empty value */
template<class T>
using KPtr = const __attribute__((address_space(4))) T*;

template<class T>
__device__ __forceinline__ T kload(KPtr<T> p)
{
#if defined(__HIP_DEVICE_COMPILE__)
  return *p;
#else
  (void)p;
  return T{};
#endif
}

/* A wavefront's copy of constants into LDS, whole dwords */
template<class T>
__device__ __forceinline__ void copy_to_lds(KPtr<T> src, T* dst)
{
  static_assert(sizeof(T) % 4 == 0, "copied by dwords");
  for(uint32_t i = threadIdx.x & 63u; i < sizeof(T) / 4; i += 64u)
    ((uint32_t*)dst)[i] = kload((KPtr<uint32_t>)src + i);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

} /* namespace */

#endif /* HTGX_QUEUE_H */
