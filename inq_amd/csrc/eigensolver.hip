// eigensolver.hip -- the per-state passes of the steepest-descent
// eigensolver and of the Teter-Payne-Allan preconditioner on band-major sphere
// states [nst][npw].
//
// Every pass is bound by HBM, so a step reads and writes each block as few times
// as its dependencies allow, and a pass ends with the per-state sums that the
// next one needs:
//
//   energy    (H phi, phi), (phi, phi)                         before the first step
//   residual  r = H phi - (e / Re n) phi  (steepest_descent.hpp:37-49), with the
//             preconditioner's sums of r
//   tpa       r(G) *= K((1/2)|G|^2 / <T>)  (preconditioner.hpp:31-58)
//   cross     (r, r), (phi, r), (r, H r), (phi, H r)            after H r
//   update    lambda from the six state overlaps, phi += lambda r and
//             H phi += lambda H r  (steepest_descent.hpp:53-83), with the energy
//             sums of the next step
//
// One work-group takes 4096 points of one state: it adds the previous pass's
// partial sums of its state itself (in chunk order, FP64) instead of waiting for
// a kernel that does, and leaves its own, so sums do not depend on the launch.
// The overlaps are those of operations::overlap_diagonal
// (src/operations/overlap_diagonal.hpp:25-60).  128 states x 67691, complex64, per
// step: ten launches and 290 us with separate dot, combine and lambda kernels, four
// launches and 175 us now (a pass moves 138-414 MB: 23-69 us at 6 TB/s).
#include "internal.hpp"

#include <algorithm>

#if defined(__HIP_DEVICE_COMPILE__)
#define GAS __attribute__((address_space(1)))
#else
#define GAS
#endif

namespace inqx {

namespace {

template <typename T> __device__ __forceinline__ const GAS T *sgp(const T *p) { return (const GAS T *)p; }
template <typename T> __device__ __forceinline__ GAS T *sgw(T *p) { return (GAS T *)p; }

constexpr int kChunk = 4096;
constexpr int kThreads = 256;

// state and points of a work-group
struct SdItem {
  int s, c;
  long p0, p1;
};
__device__ __forceinline__ SdItem sd_item(long K, int nch) {
  SdItem it;
  it.s = blockIdx.x / nch;
  it.c = blockIdx.x - it.s * nch;
  it.p0 = (long)it.c * kChunk;
  it.p1 = it.p0 + kChunk < K ? it.p0 + kChunk : K;
  return it;
}

// acc[0..N) summed over the work-group into part[(s nch + c) N + k], in a fixed order
template <int N>
__device__ __forceinline__ void sd_store_sums(double (&acc)[N], double *part, const SdItem &it, int nch) {
  __shared__ double red[kThreads / 64][N];
#pragma unroll
  for (int k = 0; k < N; ++k) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc[k] += __shfl_xor(acc[k], off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][k] = acc[k];
  }
  __syncthreads();
  if ((int)threadIdx.x < N) {
    double t = red[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < kThreads / 64; ++w) t += red[w][threadIdx.x];
    sgw(part)[((size_t)it.s * nch + it.c) * N + threadIdx.x] = t;
  }
}

// the sums of one state over its chunks, in chunk order, on every thread
template <int N> __device__ __forceinline__ void sd_load_sums(double (&out)[N], const double *part, int s, int nch) {
  __shared__ double tot[N];
  if ((int)threadIdx.x < N) {
    const GAS double *q = sgp(part) + (size_t)s * nch * N + threadIdx.x;
    double t = 0.0;
#pragma unroll 4
    for (int c = 0; c < nch; ++c) t += q[(size_t)c * N];
    tot[threadIdx.x] = t;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < N; ++k) out[k] = tot[k];
}

// += conj(x) y in FP64
template <typename C> __device__ __forceinline__ void dot_add(double &re, double &im, const C &x, const C &y) {
  re += (double)x.x * y.x + (double)x.y * y.y;
  im += (double)x.x * y.y - (double)x.y * y.x;
}

// sums {(H phi, phi), (phi, phi)}
template <typename T>
__global__ void __launch_bounds__(kThreads) k_sd_energy(const cplx<T> *phi, const cplx<T> *hphi, long K, int nch,
                                                        double *part) {
  using C = cplx<T>;
  const SdItem it = sd_item(K, nch);
  const GAS C *f = sgp(phi) + (size_t)it.s * K, *h = sgp(hphi) + (size_t)it.s * K;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
  for (long p = it.p0 + threadIdx.x; p < it.p1; p += kThreads) {
    const C x = f[p], y = h[p];
    dot_add(acc[0], acc[1], y, x);
    dot_add(acc[2], acc[3], x, x);
  }
  sd_store_sums(acc, part, it, nch);
}

// sums {sum g2h |r|^2, sum |r|^2}
template <typename T>
__global__ void __launch_bounds__(kThreads) k_tpa_sums(const cplx<T> *res, const double *g2h, long K, int nch,
                                                       double *part) {
  using C = cplx<T>;
  const SdItem it = sd_item(K, nch);
  const GAS C *r = sgp(res) + (size_t)it.s * K;
  double acc[2] = {0.0, 0.0};
#pragma unroll 4
  for (long p = it.p0 + threadIdx.x; p < it.p1; p += kThreads) {
    const C v = r[p];
    const double n2 = (double)v.x * v.x + (double)v.y * v.y;
    acc[0] += sgp(g2h)[p] * n2;
    acc[1] += n2;
  }
  sd_store_sums(acc, part, it, nch);
}

// r = hphi - (e / Re n) phi with (e, n) the energy sums times vol; TPA: the
// preconditioner's sums of r
template <typename T, bool TPA>
__global__ void __launch_bounds__(kThreads) k_sd_residual(const cplx<T> *__restrict__ phi,
                                                          const cplx<T> *__restrict__ hphi, cplx<T> *__restrict__ res,
                                                          long K, int nch, const double *part_e, double vol,
                                                          const double *__restrict__ g2h, double *part_k) {
  using C = cplx<T>;
  const SdItem it = sd_item(K, nch);
  double en[4];
  sd_load_sums(en, part_e, it.s, nch);
  const double nr = vol * en[2];
  const T er = (T)(vol * en[0] / nr), ei = (T)(vol * en[1] / nr);
  const GAS C *f = sgp(phi) + (size_t)it.s * K, *h = sgp(hphi) + (size_t)it.s * K;
  GAS C *r = sgw(res) + (size_t)it.s * K;
  double acc[2] = {0.0, 0.0};
#pragma unroll 8
  for (long p = it.p0 + threadIdx.x; p < it.p1; p += kThreads) {
    const C x = f[p], y = h[p];
    const C v{y.x - (er * x.x - ei * x.y), y.y - (er * x.y + ei * x.x)};
    r[p] = v;
    if constexpr (TPA) {
      const double n2 = (double)v.x * v.x + (double)v.y * v.y;
      acc[0] += sgp(g2h)[p] * n2;
      acc[1] += n2;
    }
  }
  if constexpr (TPA) sd_store_sums(acc, part_k, it, nch);
}

__device__ __forceinline__ double tpa_k(double x) {
  const double num = ((8.0 * x + 12.0) * x + 18.0) * x + 27.0;
  const double den = (((16.0 * x + 8.0) * x + 12.0) * x + 18.0) * x + 27.0;
  return num / den;
}

// r(G) *= K(g2h(G) / <T>), <T> = sum g2h |r|^2 / sum |r|^2
template <typename T>
__global__ void __launch_bounds__(kThreads) k_tpa_scale(cplx<T> *__restrict__ res,
                                                        const double *__restrict__ g2h, long K, int nch,
                                                        const double *part_k) {
  using C = cplx<T>;
  const SdItem it = sd_item(K, nch);
  double kn[2];
  sd_load_sums(kn, part_k, it.s, nch);
  const double kin = kn[0] / kn[1];
  GAS C *r = sgw(res) + (size_t)it.s * K;
#pragma unroll 4
  for (long p = it.p0 + threadIdx.x; p < it.p1; p += kThreads) {
    const T f = (T)tpa_k(sgp(g2h)[p] / kin);
    C v = r[p];
    v.x *= f;
    v.y *= f;
    r[p] = v;
  }
}

// sums {(r, r), (phi, r), (r, H r), (phi, H r)}
template <typename T>
__global__ void __launch_bounds__(kThreads) k_sd_cross(const cplx<T> *phi, const cplx<T> *res, const cplx<T> *hres,
                                                       long K, int nch, double *part) {
  using C = cplx<T>;
  const SdItem it = sd_item(K, nch);
  const GAS C *f = sgp(phi) + (size_t)it.s * K, *r = sgp(res) + (size_t)it.s * K, *h = sgp(hres) + (size_t)it.s * K;
  double acc[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) acc[k] = 0.0;
#pragma unroll 8
  for (long p = it.p0 + threadIdx.x; p < it.p1; p += kThreads) {
    const C x = f[p], y = r[p], z = h[p];
    dot_add(acc[0], acc[1], y, y);
    dot_add(acc[2], acc[3], x, y);
    dot_add(acc[4], acc[5], y, z);
    dot_add(acc[6], acc[7], x, z);
  }
  sd_store_sums(acc, part, it, nch);
}

__device__ __forceinline__ void cmul_d(double ar, double ai, double br, double bi, double &cr, double &ci) {
  cr = ar * br - ai * bi;
  ci = ar * bi + ai * br;
}

// lambda of a state from m0..m3 = (r,r), (phi,r), (r,Hr), (phi,Hr) and m4, m5 = (Hphi,phi), (phi,phi)
__device__ __forceinline__ double sd_lambda(const double (&m03)[8], const double (&m45)[4], double vol) {
  double m[6][2];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    m[k][0] = vol * m03[2 * k];
    m[k][1] = vol * m03[2 * k + 1];
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    m[4 + k][0] = vol * m45[2 * k];
    m[4 + k][1] = vol * m45[2 * k + 1];
  }
  double x, y, u, v;
  cmul_d(m[0][0], m[0][1], m[3][0], m[3][1], x, y);
  cmul_d(m[2][0], m[2][1], m[1][0], m[1][1], u, v);
  const double ca = x - u;
  cmul_d(m[5][0], m[5][1], m[2][0], m[2][1], x, y);
  cmul_d(m[4][0], m[4][1], m[0][0], m[0][1], u, v);
  const double cb = x - u;
  cmul_d(m[4][0], m[4][1], m[1][0], m[1][1], x, y);
  cmul_d(m[3][0], m[3][1], m[5][0], m[5][1], u, v);
  const double cc = x - u;
  const double den = cb + sqrt(cb * cb - 4.0 * ca * cc);
  return fabs(den) < 1e-15 ? 0.0 : 2.0 * cc / den;
}

// phi += lambda r; with hphi, hphi += lambda hr and the energy sums of the result
// (part_out: not part_e, which other work-groups of the state still read)
template <typename T>
__global__ void __launch_bounds__(kThreads) k_sd_update(cplx<T> *__restrict__ phi, cplx<T> *__restrict__ hphi,
                                                        const cplx<T> *__restrict__ res,
                                                        const cplx<T> *__restrict__ hres, long K, int nch,
                                                        const double *part_m, const double *part_e, double vol,
                                                        double *part_out) {
  using C = cplx<T>;
  const SdItem it = sd_item(K, nch);
  double m03[8], m45[4];
  sd_load_sums(m03, part_m, it.s, nch);
  sd_load_sums(m45, part_e, it.s, nch);
  const T l = (T)sd_lambda(m03, m45, vol);
  const size_t o = (size_t)it.s * K;
  GAS C *f = sgw(phi) + o;
  const GAS C *r = sgp(res) + o;
  if (!hphi) {
#pragma unroll 4
    for (long p = it.p0 + threadIdx.x; p < it.p1; p += kThreads) {
      const C y = r[p];
      C x = f[p];
      x.x += l * y.x;
      x.y += l * y.y;
      f[p] = x;
    }
    return;
  }
  GAS C *h = sgw(hphi) + o;
  const GAS C *hr = sgp(hres) + o;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
  for (long p = it.p0 + threadIdx.x; p < it.p1; p += kThreads) {
    const C y = r[p], z = hr[p];
    C x = f[p], w = h[p];
    x.x += l * y.x;
    x.y += l * y.y;
    w.x += l * z.x;
    w.y += l * z.y;
    f[p] = x;
    h[p] = w;
    dot_add(acc[0], acc[1], w, x);
    dot_add(acc[2], acc[3], x, x);
  }
  sd_store_sums(acc, part_out, it, nch);
}

}  // namespace

int sd_chunks(long K) { return (int)((K + kChunk - 1) / kChunk); }

// KERNEL(ARGS) for the precision T over one work-group per (state, chunk)
#define SD_LAUNCH(NAME, KERNEL, ...)                                                                      \
  do {                                                                                                    \
    const int nch = sd_chunks(K);                                                                         \
    ProfScope ps(cx, NAME);                                                                               \
    const dim3 grid((unsigned)(nst * nch));                                                               \
    if (prec == INQX_FP64) {                                                                              \
      using T = double;                                                                                   \
      hipLaunchKernelGGL((KERNEL), grid, dim3(kThreads), 0, cx.stream, __VA_ARGS__);                      \
    } else {                                                                                              \
      using T = float;                                                                                    \
      hipLaunchKernelGGL((KERNEL), grid, dim3(kThreads), 0, cx.stream, __VA_ARGS__);                      \
    }                                                                                                     \
    INQX_HIP(hipGetLastError());                                                                          \
  } while (0)

void launch_sd_energy(Ctx &cx, int prec, int nst, long K, const void *phi, const void *hphi, double *part) {
  SD_LAUNCH("sd_energy", k_sd_energy<T>, (const cplx<T> *)phi, (const cplx<T> *)hphi, K, nch, part);
}
void launch_tpa_sums(Ctx &cx, int prec, int nst, long K, const void *res, const double *g2h, double *part) {
  SD_LAUNCH("tpa_sums", k_tpa_sums<T>, (const cplx<T> *)res, g2h, K, nch, part);
}
void launch_sd_residual(Ctx &cx, int prec, int nst, long K, const void *phi, const void *hphi, void *res,
                        const double *part_e, double vol, const double *g2h, double *part_k) {
  if (g2h)
    SD_LAUNCH("sd_residual", (k_sd_residual<T, true>), (const cplx<T> *)phi, (const cplx<T> *)hphi, (cplx<T> *)res, K,
              nch, part_e, vol, g2h, part_k);
  else
    SD_LAUNCH("sd_residual", (k_sd_residual<T, false>), (const cplx<T> *)phi, (const cplx<T> *)hphi, (cplx<T> *)res, K,
              nch, part_e, vol, g2h, part_k);
}
void launch_tpa_scale(Ctx &cx, int prec, int nst, long K, void *res, const double *g2h, const double *part_k) {
  SD_LAUNCH("tpa_scale", k_tpa_scale<T>, (cplx<T> *)res, g2h, K, nch, part_k);
}
void launch_sd_cross(Ctx &cx, int prec, int nst, long K, const void *phi, const void *res, const void *hres,
                     double *part) {
  SD_LAUNCH("sd_cross", k_sd_cross<T>, (const cplx<T> *)phi, (const cplx<T> *)res, (const cplx<T> *)hres, K, nch, part);
}
void launch_sd_update(Ctx &cx, int prec, int nst, long K, void *phi, void *hphi, const void *res, const void *hres,
                      const double *part_m, const double *part_e, double vol, double *part_out) {
  SD_LAUNCH("sd_update", k_sd_update<T>, (cplx<T> *)phi, (cplx<T> *)hphi, (const cplx<T> *)res, (const cplx<T> *)hres, K,
            nch, part_m, part_e, vol, part_out);
}

}  // namespace inqx
