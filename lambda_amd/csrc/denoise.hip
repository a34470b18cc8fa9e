// Film denoiser: the project's replacement for the OIDN filter of Denoise::SetData/Process
// (Denoise.cpp:13-67), which takes the colour image with albedo and normal auxiliary images.
// OIDN's trained network is not available, so the filter is the edge-avoiding A-Trous wavelet
// transform (Dammertz, Sewtz, Hanika, Lensch 2010): `iterations` passes of the 5x5 B3-spline
// kernel h = [1/16, 1/4, 3/8, 1/4, 1/16] (x) itself with taps 2^i pixels apart, each tap weighted
// by exp(-|dc|^2 / sc_i^2) exp(-|dn|^2 / sn^2) exp(-|da|^2 / sa^2) (colour, normal, albedo
// differences to the centre pixel; sc_i = sc 2^-i, a sigma of 0 drops that term). With an albedo
// image and `demodulate`, the filter runs on colour / albedo and multiplies the albedo back
// (Schied et al. 2017), so texture detail is not blurred. Each pass is an HBM-bound stencil:
// 16 B written per pixel, its 25 taps x 48 B read mostly from cache.
#include "host.h"

using namespace lgpu;

namespace {

constexpr float kAlbedoEps = 1e-3f;  // albedo channels below it are not divided out

__device__ inline float Demod(float c, float a) { return a > kAlbedoEps ? c / a : c; }
__device__ inline float Remod(float c, float a) { return a > kAlbedoEps ? c * a : c; }

__device__ inline float4 Mean(const double *sum, const uint32_t *count, uint32_t i) {
  const uint32_t c = count[i];
  const double inv = c ? 1.0 / (double)c : 0.0;
  return make_float4((float)(sum[3 * (size_t)i] * inv), (float)(sum[3 * (size_t)i + 1] * inv),
                     (float)(sum[3 * (size_t)i + 2] * inv), 0.f);
}
// The films' means; with `demod` the colour's is divided by the albedo's. asum, nsum: null without one.
__global__ void k_dn_prepare(const double *csum, const uint32_t *ccount, const double *asum, const uint32_t *acount,
                             const double *nsum, const uint32_t *ncount, uint32_t demod, float4 *cout, float4 *aout,
                             float4 *nout, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float4 v = Mean(csum, ccount, i);
  if (asum) {
    const float4 al = Mean(asum, acount, i);
    aout[i] = al;
    if (demod) v = make_float4(Demod(v.x, al.x), Demod(v.y, al.y), Demod(v.z, al.z), 0.f);
  }
  if (nsum) nout[i] = Mean(nsum, ncount, i);
  cout[i] = v;
}

struct AtrousParams {
  uint32_t w, h, step;
  float invSc2, invSn2, invSa2;  // 1 / sigma^2 of this pass, 0 = term off
  uint32_t hasN, hasA, remod;
};

__device__ inline float Dist2(float4 a, float4 b) {
  const float x = a.x - b.x, y = a.y - b.y, z = a.z - b.z;
  return x * x + y * y + z * z;
}

// One A-Trous pass; taps outside the image are skipped (the weights renormalise). A thread takes kRows
// pixels of a column, `step` rows apart: their taps fall on the same kRows + 4 rows, so a tap is loaded
// once for all of them: 45 loads a pixel with two rows instead of 75. Bound by the latency of those loads,
// the more so the fewer waves the image gives: the five taps of a row are loaded together (outside the
// image from its edge, unused). Denoise call of five passes with both guides, against one pixel a thread and
// one load at a time: 1920 x 1080 1.95 -> 0.47 ms, 640 x 480 340 -> 119 us, 135 x 95 120 -> 58 us; with four
// rows and one load at a time 1080p took 0.50 ms, but 135 x 95 215 us.
// Taps reach each pixel in row-major order, whatever kRows is. kFilm: the last pass writes the film
// (sums with counts of 1, the albedo multiplied back).
template <int kRows, bool kFilm>
__global__ void __launch_bounds__(256) k_dn_atrous(const float4 *__restrict__ cin, const float4 *__restrict__ alb,
                                                   const float4 *__restrict__ nrm, AtrousParams p, float4 *__restrict__ cout,
                                                   double *__restrict__ sum, uint32_t *__restrict__ count) {
  const int s = (int)p.step, w = (int)p.w, h = (int)p.h;
  const uint32_t across = (p.w + 63) / 64;  // blocks: 64 columns by 4 row groups, row by row
  const int x = blockIdx.x % across * 64 + threadIdx.x % 64, group = blockIdx.x / across * 4 + threadIdx.x / 64;
  const int y0 = (group / s) * (kRows * s) + group % s;  // rows y0, y0 + s, ...
  if (x >= w || y0 >= h) return;
  float4 cp[kRows], np[kRows], ap[kRows];
  float sx[kRows], sy[kRows], sz[kRows], sw[kRows];
#pragma unroll
  for (int k = 0; k < kRows; ++k) {
    const size_t pi = (size_t)min(y0 + k * s, h - 1) * w + x;  // a row past the image is not written
    cp[k] = cin[pi];
    np[k] = p.hasN ? nrm[pi] : make_float4(0.f, 0.f, 0.f, 0.f);
    ap[k] = p.hasA ? alb[pi] : make_float4(0.f, 0.f, 0.f, 0.f);
    sx[k] = sy[k] = sz[k] = sw[k] = 0.f;
  }
#pragma unroll
  for (int r = -2; r < kRows + 2; ++r) {
    const int qy = y0 + r * s;
    if (qy < 0 || qy >= h) continue;
    float4 cq[5], nq[5], aq[5];
#pragma unroll
    for (int dx = -2; dx <= 2; ++dx) {
      const size_t qi = (size_t)qy * w + min(max(x + dx * s, 0), w - 1);
      cq[dx + 2] = cin[qi];
      nq[dx + 2] = p.hasN ? nrm[qi] : make_float4(0.f, 0.f, 0.f, 0.f);
      aq[dx + 2] = p.hasA ? alb[qi] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int dx = -2; dx <= 2; ++dx) {
      const int qx = x + dx * s;
      if (qx < 0 || qx >= w) continue;
      const float kx = dx == 0 ? 0.375f : (dx == 1 || dx == -1 ? 0.25f : 0.0625f);
      const float4 c = cq[dx + 2];
#pragma unroll
      for (int k = 0; k < kRows; ++k) {
        const int dy = r - k;
        if (dy < -2 || dy > 2) continue;
        const float ky = dy == 0 ? 0.375f : (dy == 1 || dy == -1 ? 0.25f : 0.0625f);
        float e = Dist2(c, cp[k]) * p.invSc2;
        if (p.hasN) e += Dist2(nq[dx + 2], np[k]) * p.invSn2;
        if (p.hasA) e += Dist2(aq[dx + 2], ap[k]) * p.invSa2;
        const float wt = kx * ky * expf(-e);
        sx[k] += wt * c.x; sy[k] += wt * c.y; sz[k] += wt * c.z; sw[k] += wt;
      }
    }
  }
#pragma unroll
  for (int k = 0; k < kRows; ++k) {
    const int y = y0 + k * s;
    if (y >= h) break;
    const size_t pi = (size_t)y * w + x;
    // the centre tap has weight 9/64, so sw > 0
    float4 v = make_float4(sx[k] / sw[k], sy[k] / sw[k], sz[k] / sw[k], 0.f);
    if (kFilm) {
      if (p.remod) v = make_float4(Remod(v.x, ap[k].x), Remod(v.y, ap[k].y), Remod(v.z, ap[k].z), 0.f);
      sum[3 * pi] = v.x; sum[3 * pi + 1] = v.y; sum[3 * pi + 2] = v.z;
      count[pi] = 1u;
    } else {
      cout[pi] = v;
    }
  }
}

// Images up to this many pixels take one row a thread, for more waves, larger ones two, for fewer loads:
// 480 x 270 72 and 82 us, 640 x 480 both 118, 800 x 600 175 and 151, 1920 x 1080 559 and 468.
constexpr uint32_t kOneRow = 1u << 18;

template <int kRows>
void LaunchPass(hipStream_t st, const AtrousParams &p, const float4 *src, const float4 *alb, const float4 *nrm, float4 *dst,
                bool last, lgpu_film out) {
  const uint64_t span = (uint64_t)kRows * p.step, groups = (p.h + span - 1) / span * p.step;
  const dim3 g((uint32_t)((p.w + 63) / 64 * ((groups + 3) / 4)));  // one dimension: the second holds 65,535 blocks
  if (last)
    hipLaunchKernelGGL((k_dn_atrous<kRows, true>), g, dim3(256), 0, st, src, alb, nrm, p, nullptr, out->sum.as<double>(),
                       out->count.as<uint32_t>());
  else
    hipLaunchKernelGGL((k_dn_atrous<kRows, false>), g, dim3(256), 0, st, src, alb, nrm, p, dst, nullptr, nullptr);
}

}  // namespace

extern "C" {

lgpu_status lgpu_film_denoise(lgpu_film colour, lgpu_film albedo, lgpu_film normal, const lgpu_denoise_desc *d,
                              lgpu_film out) {
  if (!colour || !out || !d) return Fail(LGPU_ERR_INVALID_ARGUMENT, "film_denoise: null colour, output or descriptor");
  for (lgpu_film f : {albedo, normal, out}) {
    if (!f) continue;
    if (f->dev != colour->dev) return Fail(LGPU_ERR_INVALID_ARGUMENT, "film_denoise: films on different devices");
    if (f->width != colour->width || f->height != colour->height)
      return Fail(LGPU_ERR_INVALID_ARGUMENT, "film_denoise: films of different sizes");
  }
  if (d->iterations == 0 || d->iterations > 12) return Fail(LGPU_ERR_INVALID_ARGUMENT, "film_denoise: iterations must be 1..12");
  for (float s : {d->sigma_colour, d->sigma_normal, d->sigma_albedo})
    if (!(s >= 0.f) || !std::isfinite(s)) return Fail(LGPU_ERR_INVALID_ARGUMENT, "film_denoise: sigmas must be finite and >= 0");
  const uint32_t w = colour->width, h = colour->height, n = w * h;
  if (!n) return LGPU_OK;
  std::lock_guard<std::mutex> lk(colour->dev->mu);
  LGPU_HIP(hipSetDevice(colour->dev->device));
  (void)hipGetLastError();
  const hipStream_t st = colour->dev->stream;
  WorkUse use{colour->dev};
  DevBuf &ca = colour->dev->work[0], &cb = colour->dev->work[1], &ab = colour->dev->work[2], &nb = colour->dev->work[3];
  LGPU_HIP(ca.alloc(16ull * n));
  LGPU_HIP(cb.alloc(16ull * n));
  const dim3 g1((n + 255) / 256), b1(256);
  const bool demod = albedo && d->demodulate;
  if (albedo) LGPU_HIP(ab.alloc(16ull * n));
  if (normal) LGPU_HIP(nb.alloc(16ull * n));
  hipLaunchKernelGGL(k_dn_prepare, g1, b1, 0, st, colour->sum.as<double>(), colour->count.as<uint32_t>(),
                     albedo ? albedo->sum.as<double>() : nullptr, albedo ? albedo->count.as<uint32_t>() : nullptr,
                     normal ? normal->sum.as<double>() : nullptr, normal ? normal->count.as<uint32_t>() : nullptr,
                     demod ? 1u : 0u, ca.as<float4>(), ab.as<float4>(), nb.as<float4>(), n);
  float4 *src = ca.as<float4>(), *dst = cb.as<float4>();
  for (uint32_t i = 0; i < d->iterations; ++i) {
    AtrousParams p;
    p.w = w; p.h = h; p.step = 1u << i;
    const float sc = d->sigma_colour * std::ldexp(1.f, -(int)i);
    p.invSc2 = sc > 0.f ? 1.f / (sc * sc) : 0.f;
    p.invSn2 = d->sigma_normal > 0.f ? 1.f / (d->sigma_normal * d->sigma_normal) : 0.f;
    p.invSa2 = d->sigma_albedo > 0.f ? 1.f / (d->sigma_albedo * d->sigma_albedo) : 0.f;
    p.hasN = normal ? 1u : 0u;
    p.hasA = albedo ? 1u : 0u;
    p.remod = demod ? 1u : 0u;
    const bool last = i + 1 == d->iterations;
    const float4 *a4 = albedo ? ab.as<float4>() : nullptr, *n4 = normal ? nb.as<float4>() : nullptr;
    if (n <= kOneRow) LaunchPass<1>(st, p, src, a4, n4, dst, last, out);
    else LaunchPass<2>(st, p, src, a4, n4, dst, last, out);
    std::swap(src, dst);
  }
  const hipError_t le = hipGetLastError();
  const hipError_t se = hipStreamSynchronize(st);  // before the buffers are used by another call
  LGPU_HIP(le);
  LGPU_HIP(se);
  use.ok = true;
  return LGPU_OK;
}

}  // extern "C"
