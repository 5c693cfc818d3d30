// Phase-retrieval transfer function over many reconstructions, on the
// device: the computation of the reference's prtf() (src/_spimage_prtf.py:
// 17-101) with sp_image_superimpose (src/image_util.c:2973-3005),
// sp_image_phase_match (:3160-3186) and the unnormalised forward transform.
//
// Each reconstruction after the first is aligned against the running sum
// of the aligned ones, so the loop over reconstructions is sequential, and at
// 256 x 256 a step is bound by its launches (about 3 us each).  What does not
// depend on the running sum stays out of the loop: the spectra of the
// magnitudes before it, the transforms of the aligned reconstructions and
// their unit phasors after it, for many reconstructions a launch.  A step
// is the sum's transform, both products, both inverse transforms in one
// launch a pass, the argmax, the gather that shifts and reflects (each of its
// work-groups repeats the small decision; it also takes the phase match's
// partial sums) and the phase match: 8 launches instead of 19 (32
// reconstructions of 256 x 256: 3.3 -> 2.2 ms, of which 1.0 ms are kernels and
// most of the rest the copies from and to pageable memory; uploading behind
// the loop on a second stream made it 2.5 ms).  There is no host round trip
// inside the loop.
#include <limits.h>
#include <math.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "engine.h"
#include "sp_prtf.h"

namespace spx {
namespace {

constexpr int kThreads = 256;

inline dim3 grid_for(long n) {
  long b = (n + kThreads - 1) / kThreads;
  if (b > 2048) b = 2048;
  if (b < 1) b = 1;
  return dim3((unsigned)b);
}

#define PRTF_STRIDE(i, n) \
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < (n); i += (long)gridDim.x * blockDim.x)

// |in| as a real complex value (sp_image_dephase, src/image_util.c:1035-1042)
__global__ void k_magnitude(const float2* in, float2* out, long n) {
  PRTF_STRIDE(i, n) out[i] = make_float2(cabsf_ref(in[i]), 0.f);
}

// corr = A conj(B) (sp_image_cross_correlate, src/image_util.c:1356-1358) and,
// with conv, A B behind it (sp_image_convolute, :1524-1526)
__global__ void k_corr_conv(const float2* A, const float2* B, float2* out, long n, int conv) {
  PRTF_STRIDE(i, n) {
    const float2 a = A[i], b = B[i];
    out[i] = make_float2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
    if (conv) out[n + i] = make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
  }
}

// larger magnitude wins; equal magnitudes go to the lower index, so the
// result is the first maximum in raster order (sp_c3matrix_max,
// include/spimage/linear_alg.h:1974-1988)
__device__ __forceinline__ void keep_best(float& v, int& i, float v2, int i2) {
  if (v2 > v || (v2 == v && i2 < i)) {
    v = v2;
    i = i2;
  }
}

// grid (parts, arrays)
__global__ __launch_bounds__(kThreads) void k_argmax_part(const float2* c, long n, float* pv, int* pi) {
  c += blockIdx.y * n;
  pv += blockIdx.y * gridDim.x;
  pi += blockIdx.y * gridDim.x;
  float v = -1.f;
  int idx = INT_MAX;
  PRTF_STRIDE(i, n) keep_best(v, idx, cabsf_ref(c[i]), (int)i);
  for (int off = 32; off > 0; off >>= 1) {
    const float v2 = __shfl_xor(v, off, 64);
    const int i2 = __shfl_xor(idx, off, 64);
    keep_best(v, idx, v2, i2);
  }
  __shared__ float sv[kThreads / 64];
  __shared__ int si[kThreads / 64];
  if ((threadIdx.x & 63) == 0) {
    sv[threadIdx.x >> 6] = v;
    si[threadIdx.x >> 6] = idx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < kThreads / 64; ++k) keep_best(v, idx, sv[k], si[k]);
    pv[blockIdx.x] = v;
    pi[blockIdx.x] = idx;
  }
}

// The superposition decision (src/image_util.c:2983-3004): the shift is the
// coordinates of the correlation peak, or of the convolution peak plus one
// when that is strictly larger, which also reflects.  Every thread of the
// work-group gets {x, y, z, reflect} from the partial maxima (of the
// convolution behind those of the correlation).
__device__ __forceinline__ int4 decide(const float* pv, const int* pi, int nparts, int enantio, int nx, int ny) {
  // (value, index) pairs under keep_best form a total order, so any order of
  // reduction finds the same first maximum as a scan in raster order
  __shared__ float sv[2][kThreads / 64];
  __shared__ int si[2][kThreads / 64];
  const int tid = threadIdx.x;
  float v[2] = {-1.f, -1.f};
  int i[2] = {INT_MAX, INT_MAX};
  for (int k = tid; k < nparts; k += kThreads) {
    keep_best(v[0], i[0], pv[k], pi[k]);
    if (enantio) keep_best(v[1], i[1], pv[nparts + k], pi[nparts + k]);
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    for (int off = 32; off > 0; off >>= 1) {
      const float v2 = __shfl_xor(v[q], off, 64);
      const int i2 = __shfl_xor(i[q], off, 64);
      keep_best(v[q], i[q], v2, i2);
    }
    if ((tid & 63) == 0) {
      sv[q][tid >> 6] = v[q];
      si[q][tid >> 6] = i[q];
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 2; ++q)
    for (int k = 0; k < kThreads / 64; ++k) keep_best(v[q], i[q], sv[q][k], si[q][k]);
  const int add = enantio && v[1] > v[0] ? 1 : 0;
  const int idx = i[add];
  return make_int4(idx % nx + add, (idx / nx) % ny + add, idx / (nx * ny) + add, add);
}

__device__ __forceinline__ int pmod(int v, int m) { return ((v % m) + m) % m; }

// out(q) = reflect(img)(q - d), mout(q) = mask(q - d), cyclic
// (sp_image_translate with SP_TRANSLATE_WRAP_AROUND, src/image_util.c:3188-
// 3215, after sp_image_reflect(.., SP_ORIGO), :161-175, which moves the
// image but not the mask).  In 3-D the reflection leaves the middle plane
// of an odd number of planes in place, as the reference's in-place swap loop
// does (src/image_util.c:290-306).
// Also counts the pixels outside the aligned mask (src/_spimage_prtf.py:72-73)
// where the reconstruction has a mask (has_mask), and sums over pixels
// |a|^2 exp(i (arg a - arg b)), a the running sum and b the aligned image
// (sp_image_phase_match with weighted = 2, src/image_util.c:3160-3177), in
// double, one partial per work-group.
__global__ __launch_bounds__(kThreads) void k_align(const float2* img, const int* mask, float2* out, int* mout, float* cnt,
                                                    const int* has_mask, const float2* avg, int nx, int ny, int nz,
                                                    const float* pv, const int* pi, int nparts, int enantio,
                                                    double2* part) {
  const int4 dec = decide(pv, pi, nparts, enantio, nx, ny);
  const bool count = mask && *has_mask;
  const long n = (long)nx * ny * nz;
  double sx = 0.0, sy = 0.0;
  PRTF_STRIDE(q, n) {
    const int x = (int)(q % nx);
    const long r = q / nx;
    const int y = (int)(r % ny), z = (int)(r / ny);
    const int px = pmod(x - dec.x, nx), py = pmod(y - dec.y, ny), pz = pmod(z - dec.z, nz);
    const long p = ((long)pz * ny + py) * nx + px;
    const int mv = mask ? mask[p] : 0;
    if (mout) mout[q] = mv;
    if (count && mv == 0) cnt[q] += 1.f;
    long s = p;
    if (dec.w && !(nz > 1 && (nz & 1) && pz == nz / 2)) s = ((long)(nz - 1 - pz) * ny + (ny - 1 - py)) * nx + (nx - 1 - px);
    const float2 av = avg[q], bv = img[s];
    out[q] = bv;
    const float ang = atan2f(av.y, av.x) - atan2f(bv.y, bv.x);
    const double m = (double)(av.y * av.y + av.x * av.x);
    double sn, cs;
    sincos((double)ang, &sn, &cs);
    sx += cs * m;
    sy += sn * m;
  }
  for (int off = 32; off > 0; off >>= 1) {
    sx += __shfl_xor(sx, off, 64);
    sy += __shfl_xor(sy, off, 64);
  }
  __shared__ double s[2][kThreads / 64];
  if ((threadIdx.x & 63) == 0) {
    s[0][threadIdx.x >> 6] = sx;
    s[1][threadIdx.x >> 6] = sy;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < kThreads / 64; ++k) {
      sx += s[0][k];
      sy += s[1][k];
    }
    part[blockIdx.x] = make_double2(sx, sy);
  }
}

// b = |b| exp(i (arg b + phi)), phi the angle of the summed partials
// (src/image_util.c:3178-3184)
// also adds the result to the running sum avg (the k_add_c64 step)
__global__ __launch_bounds__(kThreads) void k_phase_apply(const float2* b, float2* out, float2* avg, long n,
                                                          const double2* part, int nparts) {
  // every block sums the partials in the same fixed order
  __shared__ double sx[kThreads], sy[kThreads];
  const int tid = threadIdx.x;
  double x = 0.0, y = 0.0;
  for (int k = tid; k < nparts; k += kThreads) {
    x += part[k].x;
    y += part[k].y;
  }
  sx[tid] = x;
  sy[tid] = y;
  __syncthreads();
  for (int off = kThreads / 2; off > 0; off >>= 1) {
    if (tid < off) {
      sx[tid] += sx[tid + off];
      sy[tid] += sy[tid + off];
    }
    __syncthreads();
  }
  const float phi = (float)atan2(sy[0], sx[0]);
  PRTF_STRIDE(i, n) {
    const float2 v = b[i];
    const float ang = atan2f(v.y, v.x) + phi;
    const double m = (double)cabsf_ref(v);
    double sn, cs;
    sincos((double)ang, &sn, &cs);
    const float2 r = make_float2((float)(cs * m), (float)(sn * m));
    out[i] = r;
    avg[i] = make_float2(avg[i].x + r.x, avg[i].y + r.y);
  }
}

// avg += imgs[0] + imgs[1] + ..., in that order; cnt counts the pixels outside
// the masks of those that have one (src/_spimage_prtf.py:72-73)
__global__ void k_add_all(float2* avg, const float2* imgs, const int* masks, const int* has_mask, float* cnt, long n,
                          int count) {
  PRTF_STRIDE(i, n) {
    float2 a = avg[i];
    float c = cnt[i];
    for (int r = 0; r < count; ++r) {
      const float2 b = imgs[r * n + i];
      a = make_float2(a.x + b.x, a.y + b.y);
      if (masks && has_mask[r] && masks[r * n + i] == 0) c += 1.f;
    }
    avg[i] = a;
    cnt[i] = c;
  }
}

// running sum of F / |F| where F != 0, and a count of the zeros
// (src/_spimage_prtf.py:80-86), over `count` transforms in their order
__global__ void k_unit_accum(const float2* F, float2* sum, int* zeros, long n, int count, int first) {
  PRTF_STRIDE(i, n) {
    float2 s = first ? make_float2(0.f, 0.f) : sum[i];
    int z = first ? 0 : zeros[i];
    for (int r = 0; r < count; ++r) {
      const float2 f = F[r * n + i];
      float2 u = make_float2(0.f, 0.f);
      if (f.x != 0.f || f.y != 0.f) {
        const float m = hypotf(f.x, f.y);
        u = make_float2(f.x / m, f.y / m);
      } else {
        ++z;
      }
      s = first && r == 0 ? u : make_float2(s.x + u.x, s.y + u.y);
    }
    sum[i] = s;
    zeros[i] = z;
  }
}

// has[r] = the sum of mask r is positive, one work-group per reconstruction
// (the masks whose pixels count; a translation keeps the sum)
__global__ __launch_bounds__(1024) void k_has_mask(const int* masks, long n, int* has) {
  const int* m = masks + blockIdx.x * n;
  long long t = 0;
  if (n % 4 == 0) {  // every mask starts on 16 bytes
    const int4* m4 = reinterpret_cast<const int4*>(m);
    for (long i = threadIdx.x; i < n / 4; i += 1024) {
      const int4 v = m4[i];
      t += ((long long)v.x + v.y) + ((long long)v.z + v.w);
    }
  } else {
    for (long i = threadIdx.x; i < n; i += 1024) t += m[i];
  }
  __shared__ long long s[1024];
  s[threadIdx.x] = t;
  __syncthreads();
  for (int off = 512; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) s[threadIdx.x] += s[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) has[blockIdx.x] = s[0] > 0;
}

// |sum / n|, zero where any transform was zero (src/_spimage_prtf.py:91-94)
__global__ void k_prtf_final(const float2* sum, const int* zeros, float* out, long n, float nimg) {
  PRTF_STRIDE(i, n) {
    const float2 s = make_float2(sum[i].x / nimg, sum[i].y / nimg);
    out[i] = zeros[i] > 0 ? 0.f : cabsf_ref(s);
  }
}

__global__ void k_fill_f32(float* p, long n, float v) { PRTF_STRIDE(i, n) p[i] = v; }

// spectra kept at once, in elements: launches of this size fill the chip
constexpr long kSpectra = 1L << 22;

// device buffers of one call, released on every path
struct Buffers {
  std::vector<void*> ptrs;
  hipStream_t s = nullptr;
  ~Buffers() {
    if (s) (void)hipStreamSynchronize(s);
    for (void* p : ptrs) (void)hipFree(p);
    if (s) (void)hipStreamDestroy(s);
  }
  template <class T>
  int alloc(T** p, size_t count) {
    *p = nullptr;
    if (hipMalloc(p, sizeof(T) * (count ? count : 1)) != hipSuccess) {
      set_error("spx_prtf: device allocation of %zu bytes failed", sizeof(T) * count);
      return -20;
    }
    ptrs.push_back(*p);
    return 0;
  }
};

int prtf_impl(const float* images, const int* masks, int nx, int ny, int nz, int n, int translate, int enantio,
              float* prtf, float* super_image, float* aligned, int* aligned_masks, float* mask_count) {
  if (!images || !prtf || n < 1 || nx < 1 || ny < 1 || nz < 1) {
    set_error("spx_prtf: images, prtf, n >= 1 and positive sizes are required");
    return -1;
  }
  if (!device_available()) {
    set_error("no HIP device available");
    return -10;
  }
  Shape sh;
  if (int rc = make_shape(nx, ny, nz, 1, &sh)) return rc;
  const long N = (long)nx * ny * nz;
  Buffers b;
  SPX_HIP(hipStreamCreateWithFlags(&b.s, hipStreamNonBlocking));
  hipStream_t s = b.s;
  const int nparts = (int)grid_for(N).x;
  // spectra of this many reconstructions at a time
  const int chunk = (int)std::max(1L, std::min((long)n, kSpectra / N));
  float2 *imgs = nullptr, *avg = nullptr, *t1 = nullptr, *cc = nullptr, *spec = nullptr, *sum = nullptr;
  int *msk = nullptr, *amsk = nullptr, *has = nullptr, *zeros = nullptr, *pi = nullptr;
  float *cnt = nullptr, *pv = nullptr;
  double2* ph = nullptr;
  if (b.alloc(&imgs, (size_t)n * N) || b.alloc(&spec, (size_t)chunk * N) || b.alloc(&avg, N) || b.alloc(&t1, N) ||
      b.alloc(&cc, 2 * N) || b.alloc(&sum, N) || b.alloc(&zeros, N) || b.alloc(&cnt, N) || b.alloc(&pv, 2 * nparts) ||
      b.alloc(&pi, 2 * nparts) || b.alloc(&ph, nparts))
    return -20;
  if (masks && (b.alloc(&msk, (size_t)n * N) || b.alloc(&has, n))) return -20;
  if (masks && aligned_masks && translate && b.alloc(&amsk, (size_t)n * N)) return -20;
  const dim3 g = grid_for(N), blk(kThreads);
  SPX_HIP(hipMemcpyAsync(imgs, images, sizeof(float2) * n * N, hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(k_fill_f32, g, blk, 0, s, cnt, N, 0.f);
  SPX_HIP(hipMemcpyAsync(avg, imgs, sizeof(float2) * N, hipMemcpyDeviceToDevice, s));
  if (masks) {
    SPX_HIP(hipMemcpyAsync(msk, masks, sizeof(int) * n * N, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_has_mask, dim3(n), dim3(1024), 0, s, msk, N, has);
    if (amsk) SPX_HIP(hipMemcpyAsync(amsk, msk, sizeof(int) * N, hipMemcpyDeviceToDevice, s));
  }
  // the magnitudes are taken in the transforms' x pass
  auto abs_fft = [&](const Shape& shp, const float2* in, float2* out) {
    if (shp.ex) {
      enqueue_abs_fft(shp, in, out, s);
    } else {
      hipLaunchKernelGGL(k_magnitude, grid_for(N * shp.nrec), blk, 0, s, in, out, N * shp.nrec);
      enqueue_fft(shp, out, out, -1, s);
    }
  };
  if (translate) {
    const Shape pair = shape_of_many(sh, enantio ? 2 : 1);
    for (int i = 1; i < n; ++i) {
      const int k = (i - 1) % chunk;
      if (k == 0) abs_fft(shape_of_many(sh, std::min(chunk, n - i)), imgs + (long)i * N, spec);
      float2* img = imgs + (long)i * N;
      const int* im = msk ? msk + (long)i * N : nullptr;
      abs_fft(sh, avg, t1);
      hipLaunchKernelGGL(k_corr_conv, g, blk, 0, s, t1, spec + (long)k * N, cc, N, enantio ? 1 : 0);
      enqueue_fft(pair, cc, cc, +1, s);
      hipLaunchKernelGGL(k_argmax_part, dim3(g.x, enantio ? 2 : 1), blk, 0, s, cc, N, pv, pi);
      hipLaunchKernelGGL(k_align, g, blk, 0, s, img, im, t1, amsk ? amsk + (long)i * N : nullptr, cnt, has + i, avg, nx, ny,
                         nz, pv, pi, nparts, enantio ? 1 : 0, ph);
      // the aligned, phase-matched reconstruction replaces the input in
      // place and joins the running sum
      hipLaunchKernelGGL(k_phase_apply, g, blk, 0, s, t1, img, avg, N, ph, nparts);
    }
  } else if (n > 1) {
    hipLaunchKernelGGL(k_add_all, g, blk, 0, s, avg, imgs + N, msk ? msk + N : nullptr, has + 1, cnt, N, n - 1);
  }
  for (int i = 0; i < n; i += chunk) {
    const int m = std::min(chunk, n - i);
    enqueue_fft(shape_of_many(sh, m), imgs + (long)i * N, spec, -1, s);
    hipLaunchKernelGGL(k_unit_accum, g, blk, 0, s, spec, sum, zeros, N, m, i == 0 ? 1 : 0);
  }
  float* dprtf = reinterpret_cast<float*>(t1);
  hipLaunchKernelGGL(k_prtf_final, g, blk, 0, s, sum, zeros, dprtf, N, (float)n);
  SPX_HIP(hipGetLastError());
  if (int rc = download_d2h(prtf, dprtf, sizeof(float) * N, s)) return rc;
  if (super_image)
    if (int rc = download_d2h(super_image, avg, sizeof(float2) * N, s)) return rc;
  if (aligned) SPX_HIP(hipMemcpyAsync(aligned, imgs, sizeof(float2) * n * N, hipMemcpyDeviceToHost, s));
  if (aligned_masks) {
    if (msk) SPX_HIP(hipMemcpyAsync(aligned_masks, amsk ? amsk : msk, sizeof(int) * n * N, hipMemcpyDeviceToHost, s));
    else memset(aligned_masks, 0, sizeof(int) * n * N);
  }
  if (mask_count)
    if (int rc = download_d2h(mask_count, cnt, sizeof(float) * N, s)) return rc;
  SPX_HIP(hipStreamSynchronize(s));
  return 0;
}

}  // namespace
}  // namespace spx

extern "C" int spx_prtf(const float* images, const int* masks, int nx, int ny, int nz, int n, int translate,
                        int enantio, float* prtf, float* super_image, float* aligned, int* aligned_masks,
                        float* mask_count) {
  return spx::prtf_impl(images, masks, nx, ny, nz, n, translate, enantio, prtf, super_image, aligned, aligned_masks,
                        mask_count);
}
