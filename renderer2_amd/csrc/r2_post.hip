// Post-process of a rendered frame (rt::Raytracer::renderFrame after the spp
// loop, raytracer/raytracer.cu:53-127,192-206): global log-average tonemapping
// c / (c + k), gamma and bytes.  The column and row sums run in the same order
// as the reference kernels (one thread per column over the rows, then one
// thread over the columns); log / exp / pow are the double-evaluated forms of
// r2_detmath.hpp so that the result does not depend on the device library.
#include "r2_internal.hpp"
#include "r2_detmath.hpp"
#include <algorithm>
#include <cfloat>

namespace {

using namespace r2;

// a + q[0] + q[1] + ... in that order, n values of LDS (16-byte aligned).  The chain
// of additions is the bound: the next 32 values are read while 32 are added, so that
// no addition waits for LDS (read four by four as they were needed, 1920 values took
// 24 us, 29 cycles an addition).
__device__ __forceinline__ float add_in_order(float a, const float* q, int n) {
  const float4* q4 = reinterpret_cast<const float4*>(q);
  int r = 0;
  if (n >= 32) {
    float4 v[8], u[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = q4[j];
    for (; r + 32 <= n; r += 32) {
      const int nx = r + 64 <= n ? r / 4 + 8 : 0;  // the last round reads the first values again
#pragma unroll
      for (int j = 0; j < 8; ++j) u[j] = q4[nx + j];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        a += v[j].x;
        a += v[j].y;
        a += v[j].z;
        a += v[j].w;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = u[j];
    }
  }
  for (; r < n; ++r) a += q[r];
  return a;
}

// avg[x] = sum_y log(r + g + b + FLT_MIN) / (W H 3)  (computeGlobalTonemapping1)
//
// A column's terms are added one after another (the reference's order), but they
// do not depend on each other: a block takes kTmCols columns, its waves 1.. compute
// the terms of kTmRows rows into LDS while wave 0 adds those of the kTmRows rows
// before, one column per lane, four terms per LDS read.  What bounds it is the
// chain of h additions (about 3 us for 1080) behind the double-evaluated logs of
// one chunk; with one thread per column it was the load, log and addition of every
// row in turn: 81 us for 1920 x 1080, now 14 us.  8 columns per block give 240
// blocks at 1920 (fewer columns would cut a row's 96 bytes below a line).  Frames wider
// than kTmBlocks blocks take several turns of the grid: a launch holds fewer than 2^32
// threads, and a frame may have 2^28 columns.
constexpr int kTmCols = 8, kTmRows = 512, kTmThreads = 1024, kTmBlocks = 65536;
constexpr int kTmStride = kTmRows + 4;  // columns 4 banks apart, 16-byte aligned
__global__ __launch_bounds__(kTmThreads) void k_tm_columns(const float* __restrict__ hdr, int w, int h,
                                                           float* __restrict__ avg) {
  __shared__ __align__(16) float term[2][kTmCols * kTmStride];
  const float divisor = (float)(h * w * 3);
  const int nchunk = (h + kTmRows - 1) / kTmRows;
  const int t = (int)threadIdx.x - 64;
  for (int x0 = (int)blockIdx.x * kTmCols; x0 < w; x0 += (int)gridDim.x * kTmCols) {
    float a = 0.f;
    for (int c = 0; c <= nchunk; ++c) {
      if (t >= 0) {
        const int y0 = c * kTmRows, rows = min(kTmRows, h - y0);  // rows <= 0 past the last chunk
        for (int i = t; i < rows * kTmCols; i += kTmThreads - 64) {
          const int col = i % kTmCols, r = i / kTmCols, x = x0 + col;
          if (x < w) {
            const float* p = hdr + 3 * ((size_t)(y0 + r) * w + x);
            term[c & 1][col * kTmStride + r] = det_logf(p[0] + p[1] + p[2] + FLT_MIN) / divisor;
          }
        }
      } else if (c > 0 && threadIdx.x < kTmCols) {
        const int rows = min(kTmRows, h - (c - 1) * kTmRows);
        a = add_in_order(a, term[(c - 1) & 1] + threadIdx.x * kTmStride, rows);
      }
      __syncthreads();
    }
    if (threadIdx.x < kTmCols && x0 + (int)threadIdx.x < w) avg[x0 + threadIdx.x] = a;
  }
}

// k = exp(sum_x avg[x]) - W H FLT_MIN  (computeGlobalTonemapping2): one chain of w
// additions, staged through LDS by the whole block (reading each column sum from
// memory in the chain took 510 us for 1920 columns, now 10 us)
constexpr int kTmFactorThreads = 1024;
__global__ __launch_bounds__(kTmFactorThreads) void k_tm_factor(const float* __restrict__ avg, int w, int h,
                                                                float* __restrict__ factor) {
  __shared__ __align__(16) float s[kTmFactorThreads];
  float r = 0.f;
  for (int x0 = 0; x0 < w; x0 += kTmFactorThreads) {
    const int n = min(kTmFactorThreads, w - x0);
    if ((int)threadIdx.x < n) s[threadIdx.x] = avg[x0 + threadIdx.x];
    __syncthreads();
    if (threadIdx.x == 0) r = add_in_order(r, s, n);
    __syncthreads();
  }
  if (threadIdx.x == 0) *factor = det_expf(r) - (float)(w * h) * FLT_MIN;
}

// applyTonemapping, correctGamma, fillByteFrame.  Bound by the double-evaluated
// power (26 us at 1920 x 1080, 11 us of which the memory needs); a thread takes four
// values, so that the frame moves in 16-byte loads and stores and the bytes in whole
// words where the pointers are aligned for it (kVec).
template <bool kVec>
__global__ void k_tm_apply(const float* __restrict__ hdr, size_t n3, const float* __restrict__ factor, float inv_gamma,
                           float* __restrict__ ldr, uint8_t* __restrict__ bytes) {
  const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (i >= n3) return;
  const float k = *factor;
  const int n = n3 - i < 4 ? (int)(n3 - i) : 4;
  float c[4] = {0.f, 0.f, 0.f, 0.f}, t[4];
  uint8_t b[4];
  if (kVec && n == 4) {
    const float4 v = *reinterpret_cast<const float4*>(hdr + i);
    c[0] = v.x; c[1] = v.y; c[2] = v.z; c[3] = v.w;
  } else {
    for (int j = 0; j < n; ++j) c[j] = hdr[i + j];
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    t[j] = det_powf(c[j] / (c[j] + k), inv_gamma);
    b[j] = (uint8_t)roundf(t[j] * 255.0f);
  }
  if (kVec && n == 4) {
    if (ldr) *reinterpret_cast<float4*>(ldr + i) = make_float4(t[0], t[1], t[2], t[3]);
    if (bytes) *reinterpret_cast<uchar4*>(bytes + i) = make_uchar4(b[0], b[1], b[2], b[3]);
  } else {
    for (int j = 0; j < n; ++j) {
      if (ldr) ldr[i + j] = t[j];
      if (bytes) bytes[i + j] = b[j];
    }
  }
}

}  // namespace

extern "C" int r2_postprocess(r2_ctx* ctx, const float* hdr, int32_t w, int32_t h, float gamma, float* ldr,
                              uint8_t* bytes, int32_t on_device) {
  if (!ctx || !hdr || w <= 0 || h <= 0 || !(gamma > 0.f)) return R2_ERR_INVALID;
  if ((int64_t)w * h > (1ll << 28)) return r2host::fail(ctx, R2_ERR_UNSUPPORTED, "postprocess: frame too large");
  hipStream_t st = ctx->stream;
  const size_t n3 = (size_t)w * h * 3;
  void* buf = nullptr;
  // scratch: column sums, factor, and (host mode) the frame in and out
  const size_t need = sizeof(float) * ((size_t)w + 64) + (on_device ? 0 : n3 * (4 + 4 + 1) + 512);
  if (r2host::pool_get(ctx, 23, need, &buf) != hipSuccess)
    return r2host::fail(ctx, R2_ERR_OOM, "postprocess: scratch");
  float* avg = (float*)buf;
  float* factor = avg + w;
  const float* d_hdr = hdr;
  float* d_ldr = ldr;
  uint8_t* d_bytes = bytes;
  if (!on_device) {
    // each array 16-byte aligned (the 512 spare bytes cover the rounding)
    const size_t n3p = (n3 + 3) & ~(size_t)3;
    float* in = (float*)(((uintptr_t)(factor + 64) + 15) & ~(uintptr_t)15);
    float* outf = in + n3p;
    uint8_t* outb = (uint8_t*)(outf + n3p);
    R2_HIP(ctx, hipMemcpyAsync(in, hdr, n3 * 4, hipMemcpyHostToDevice, st));
    d_hdr = in;
    d_ldr = ldr ? outf : nullptr;
    d_bytes = bytes ? outb : nullptr;
  }
  hipLaunchKernelGGL(k_tm_columns, dim3(std::min((w + kTmCols - 1) / kTmCols, kTmBlocks)), dim3(kTmThreads), 0, st, d_hdr, w, h, avg);
  hipLaunchKernelGGL(k_tm_factor, dim3(1), dim3(kTmFactorThreads), 0, st, avg, w, h, factor);
  const dim3 ablk((unsigned)((n3 + 1023) / 1024));
  const bool vec = (((uintptr_t)d_hdr | (uintptr_t)d_ldr) & 15) == 0 && ((uintptr_t)d_bytes & 3) == 0;
  if (vec)
    hipLaunchKernelGGL(k_tm_apply<true>, ablk, dim3(256), 0, st, d_hdr, n3, factor, 1.f / gamma, d_ldr, d_bytes);
  else
    hipLaunchKernelGGL(k_tm_apply<false>, ablk, dim3(256), 0, st, d_hdr, n3, factor, 1.f / gamma, d_ldr, d_bytes);
  R2_HIP(ctx, hipGetLastError());
  if (!on_device) {
    if (ldr) R2_HIP(ctx, hipMemcpyAsync(ldr, d_ldr, n3 * 4, hipMemcpyDeviceToHost, st));
    if (bytes) R2_HIP(ctx, hipMemcpyAsync(bytes, d_bytes, n3, hipMemcpyDeviceToHost, st));
  }
  R2_HIP(ctx, hipStreamSynchronize(st));
  return R2_OK;
}
