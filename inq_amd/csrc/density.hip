// density.hip -- spin density of sphere states: den += sum_i occ_i |phi_i(r)|^2
// (observables::density::calculate_add, src/observables/density.hpp:24-38).
//
// The inverse transform along i0 and the sum over states are one pass.  Writing
// the real-space states out and summing them in a second kernel moved each of
// them twice, 1.1 GB for 96 states at 72^3 complex128, and kept nst N complex
// values of scratch; here a wave keeps the running sums of its lines in registers
// while it walks a range of states, and only one double per point and range is
// written.  What bounds it is the latency of one state's loads and butterflies
// per wave, with two or three waves per SIMD.
// 96 states, 72^3 complex128: 188 + 132 -> 96 + 7 us.
#include "plane_common.hpp"

#include <algorithm>

namespace inqx {
namespace {

// a quarter line per lane where the length allows it: values and sums of a lane
// then take 3 N0 / 4 doubles at most, so two or more waves fit a SIMD up to 128 points
template <int N0> constexpr int den_lanes() { return N0 % 4 == 0 ? 4 : 2; }

// waves the ranges of states are cut for: three per SIMD
constexpr int kDenWavesPerCu = 12;

// part[g][N] = sum over the states of range g (per states each, in order) of
// occ |phi|^2; t1 are the plane slots of k_plane_inverse, scale = 1/N
template <typename T, int N0>
__global__ void __launch_bounds__(256) k_line_density(const cplx<T> *t1, int m_lo, int nslot, int n12, int ntile,
                                                      int nst, int per, T scale, const double *occ, double *part) {
  using C = cplx<T>;
  constexpr int S = den_lanes<N0>(), LPW = 64 / S, M = N0 / S, UP = (N0 + 1) / 2;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int item = (int)blockIdx.x * 4 + wave, g = item / ntile, tile = item - g * ntile;
  const int s0 = g * per, s1 = min(s0 + per, nst);
  if (s0 >= nst) return;  // wave-uniform, no barrier follows
  const int q = lane / LPW;
  const int L = tile * LPW + lane % LPW, Lc = L < n12 ? L : n12 - 1;
  const unsigned pl = (unsigned)(n12 * sizeof(C)), vl = (unsigned)(Lc * sizeof(C)), vq = vl + (unsigned)q * pl;
  double acc[M];
#pragma unroll
  for (int k = 0; k < M; ++k) acc[k] = 0.0;
  for (int s = s0; s < s1; ++s) {
    const auto rs = make_rsrc(t1 + (size_t)s * nslot * n12, (unsigned)nslot * pl);
    const double o = gp(occ)[s];
    // the slot offsets of the line's values are not kept across states: 150 SGPRs
    // of them spill to lanes of VGPRs
    int lo = m_lo;
    asm volatile("" : "+s"(lo));
    C v[M];
#pragma unroll
    for (int n = 0; n < M; ++n) {  // i0 = S n + q in slot sym(i0) - m_lo, zero where the line has no slot
      const bool straddle = S * n < UP && S * n + S > UP;  // both ends of the symmetric range
      const int b = (S * n >= UP ? S * n - N0 : S * n) - lo;  // slot of part 0
      C x{0, 0};
      if (!straddle && b >= 0 && b + S <= nslot) {
        bload(rs, vq, (unsigned)b * pl, x);
      } else if (straddle || (b + S > 0 && b < nslot)) {
        const int j = b + q - (S * n < UP && S * n + q >= UP ? N0 : 0);
        bload(rs, (unsigned)j < (unsigned)nslot ? vl + (unsigned)j * pl : kOOB, 0u, x);
      }
      v[n] = x;
    }
    line_dit<N0, +1, C, S, true>(v, q);
#pragma unroll
    for (int k = 0; k < M; ++k) {
      const double re = (double)(v[k].x * scale), im = (double)(v[k].y * scale);
      acc[k] += o * (re * re + im * im);
    }
  }
  if (L >= n12) return;
  GAS double *out = gw(part) + (size_t)g * N0 * n12 + (size_t)line_out_q<N0, S>(q) * n12 + L;
#pragma unroll
  for (int k = 0; k < M; ++k) out[(size_t)line_out_j<N0, S>(k) * n12] = acc[k];
}

__global__ void __launch_bounds__(256) k_density_sum(const double *part, int ng, long N, int ncomp, int ispin,
                                                     double *den) {
  const long p = (long)blockIdx.x * 256 + threadIdx.x;
  if (p >= N) return;
  double acc = 0.0;
#pragma unroll 4
  for (int g = 0; g < ng; ++g) acc += gp(part)[(size_t)g * N + p];
  gw(den)[p * ncomp + ispin] += acc;
}

struct OccChunk {
  double v[256];
};
__global__ void __launch_bounds__(256) k_put_occ(OccChunk c, int n, double *out) {
  if ((int)threadIdx.x < n) gw(out)[threadIdx.x] = c.v[threadIdx.x];
}

}  // namespace

// occupations from the host as kernel arguments: no staging copy to wait for
void launch_put_occ(Ctx &cx, const double *occ, int nst, double *dev) {
  for (int s0 = 0; s0 < nst; s0 += 256) {
    OccChunk c;
    const int n = std::min(256, nst - s0);
    std::copy(occ + s0, occ + s0 + n, c.v);
    std::fill(c.v + n, c.v + 256, 0.0);
    hipLaunchKernelGGL(k_put_occ, dim3(1), dim3(256), 0, cx.stream, c, n, dev + s0);
    INQX_HIP(hipGetLastError());
  }
}

template <typename T>
void launch_line_density(inqx_ham_s *h, const Basis &B, int nst, const DensityOut &o) {
  Ctx &cx = h->ctx->c;
  const Grid &g = h->g;
  const int prec = std::is_same<T, double>::value ? INQX_FP64 : INQX_FP32, n12 = g.n[1] * g.n[2];
  const int lpw = g.n[0] % 4 == 0 ? 16 : 32, ntile = (n12 + lpw - 1) / lpw;
  // ranges of states: as many as keep the chip's waves busy, each at least one state
  const int want = std::max(1, std::min(nst, cx.num_cu * kDenWavesPerCu / ntile));
  const int per = (nst + want - 1) / want, ng = (nst + per - 1) / per;
  o.work->ensure(sizeof(double) * (size_t)ng * g.N);
  double *part = o.work->as<double>();
  {
    ProfScope ps(cx, prec == INQX_FP64 ? "line_density_f64" : "line_density_f32");
    const dim3 grid((unsigned)((ntile * (long)ng + 3) / 4));
    switch (g.n[0]) {
#define CASE(S)                                                                                                  \
  case S:                                                                                                        \
    hipLaunchKernelGGL((k_line_density<T, S>), grid, dim3(256), 0, cx.stream, B.t1[prec].as<cplx<T>>(), B.m_lo, \
                       B.nslot, n12, ntile, nst, per, (T)(1.0 / (double)g.N), o.occ, part);                     \
    break;
      INQX_SIZES(CASE)
#undef CASE
      default:
        INQX_CHECK(false, INQX_ERR_UNSUPPORTED, "grid size not built for the sphere path");
    }
    INQX_HIP(hipGetLastError());
  }
  ProfScope ps(cx, "density_sum");
  hipLaunchKernelGGL(k_density_sum, dim3((unsigned)((g.N + 255) / 256)), dim3(256), 0, cx.stream, part, ng, g.N,
                     o.ncomp, o.ispin, o.den);
  INQX_HIP(hipGetLastError());
}
template void launch_line_density<double>(inqx_ham_s *, const Basis &, int, const DensityOut &);
template void launch_line_density<float>(inqx_ham_s *, const Basis &, int, const DensityOut &);

}  // namespace inqx
