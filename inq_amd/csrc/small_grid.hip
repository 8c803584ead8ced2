// small_grid.hip -- H|psi> on G-sphere blocks whose whole real-space cube fits
// one work-group's LDS (24^3 complex64, 20^3 complex128): one launch, one
// work-group per state.
//
// The five passes of ham_kernels.hip move a state's planes through memory five
// times, 0.7 GB for the 1536 states of 128 blocks at 24^3, and each pass waits
// for the one before over the whole grid.  Here a state is read once, all
// transforms, the potential and the projectors run on its cube in LDS, and the
// result is written once; the projections of one state need no other state's.
// What bounds it is the LDS and VALU work of one state per CU: about 21 us.
// 128 blocks x 12 states at 24^3 complex64: 234 -> 130 us; 16 states at
// 20^3 complex128: 39 -> 25 us.
//
// Layout in LDS: C u[n0][n1][n2 + 1], FFT index order in every direction; the odd
// row stride keeps the row transforms (a row per lane) free of bank conflicts.
// Each transform takes a whole line per lane in registers.
#include "plane_common.hpp"

#include <algorithm>

namespace inqx {
namespace {

// (28 is left out: its radix-7 stage spills)
#define INQX_SMALL_SIZES(X) X(12) X(16) X(18) X(20) X(24) X(30) X(32)

// 768 threads (168 VGPRs) for complex64 and 512 (256) for complex128: a line of
// 32 values per lane and its twiddled copies fit without spilling
template <typename T> constexpr int small_threads() { return sizeof(T) == 4 ? 768 : 512; }

struct SmallDev {
  int n0, n1, n2, n12, s1, s2;  // s2 = n2 + 1, s1 = n1 s2: strides in LDS
  int natoms, wpg;              // KB groups, waves per group in the projection
  int part_off, dp_off;         // bytes: projection sums [group][part][kMaxNlm] (re, im) double, D P [group][kMaxNlm]
  const int *g_row;             // [natoms + 1] first row (of 64 records) of a group
  const int *g_off;             // LDS offset of a record's point, -1: padding
  const void *g_b;              // projector values, 4 per record
  const void *g_item;           // rows of the projectors, by class (KBTables)
  const int *g_class;           // [classes + 1] first item
  int classes;
  const double *coeff;          // [natoms][kMaxNlm][kCoeffCols]
  const int *group_sib;
  double kb_scale;
};

enum { kRows = 0, kCols = 1, kLines = 2 };

template <typename T, int N, int SIGN, typename F>
__device__ __forceinline__ void transform_lines(cplx<T> *u, int stride, int count, F off) {
  using C = cplx<T>;
  for (int i = threadIdx.x; i < count; i += small_threads<T>()) {
    C *p = u + off(i);
    C v[N];
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = p[k * stride];
    fft_line<N, SIGN, C>::run(v);
#pragma unroll
    for (int k = 0; k < N; ++k) p[k * stride] = v[k];
  }
}

template <typename T, int SIGN, typename F>
__device__ __forceinline__ void transform_any(cplx<T> *u, int n, int stride, int count, F off) {
  switch (n) {  // uniform
#define CASE(S)                                              \
  case S:                                                    \
    transform_lines<T, S, SIGN>(u, stride, count, off);      \
    break;
    INQX_SMALL_SIZES(CASE)
#undef CASE
  }
}

template <typename T>
__global__ void __launch_bounds__(small_threads<T>()) k_small_apply(const SphereBlock<T> *blocks, const int *items,
                                                                    SmallDev d, T c1r, T c1i, T c2r, T c2i) {
  using C = cplx<T>;
  constexpr int NT = small_threads<T>(), NW = NT / 64;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  C *u = reinterpret_cast<C *>(smem_raw);
  double *part = reinterpret_cast<double *>(smem_raw + d.part_off);
  C *dpl = reinterpret_cast<C *>(smem_raw + d.dp_off);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const float rn2 = 1.0f / (float)d.n2;
  const V2<int> it = ld2<int>(items, blockIdx.x);
  const SphereBlock<T> B = blocks[__builtin_amdgcn_readfirstlane(it.x)];
  const int s = __builtin_amdgcn_readfirstlane(it.y), npw = B.npw;
  const GAS C *psi = gp(B.psi) + (size_t)s * npw;
  const GAS int *po = gp(B.cube_off);
  // the first points of the sphere (LDS offset, value, kinetic factor), loaded while
  // the cube is cleared and kept for the gather: with one work-group per CU no other
  // one hides a load's latency (a work-group that loops over states and loads the
  // next one early spills: 58 registers at 768 threads)
  constexpr int PF = 3;
  int fo[PF];
  T fx[PF], fy[PF], fk[PF];
  const int row0 = gp(B.cube_rows)[min(tid, B.ncube_rows - 1)];
#pragma unroll
  for (int k = 0; k < PF; ++k) {
    const int i = min(tid + k * NT, npw - 1);
    fo[k] = po[i];
    const C v = psi[i];
    fx[k] = v.x;
    fy[k] = v.y;
    fk[k] = gp(B.kin)[i];
  }
  const int nvec = (d.n0 * d.s1 * (int)sizeof(C) + 15) / 16;
  for (int i = tid; i < nvec; i += NT) reinterpret_cast<float4 *>(smem_raw)[i] = float4{0.f, 0.f, 0.f, 0.f};
  __syncthreads();
#pragma unroll
  for (int q = 0; q < PF; ++q)
    if (tid + q * NT < npw) u[fo[q]] = C{fx[q], fy[q]};
  for (int i = tid + PF * NT; i < npw; i += NT) u[po[i]] = psi[i];
  __syncthreads();

  // lines of the three kinds: the sphere's rows along i2, the columns along i1 of
  // the planes that hold sphere points, every line along i0
  auto stage = [&](auto sign, int kind) {
    constexpr int SIGN = decltype(sign)::value;
    const int count = kind == kRows ? B.ncube_rows : kind == kCols ? B.nslot * d.n2 : d.n12;
    const int n = kind == kRows ? d.n2 : kind == kCols ? d.n1 : d.n0;
    const int stride = kind == kRows ? 1 : kind == kCols ? d.s2 : d.s1;
    transform_any<T, SIGN>(u, n, stride, count, [&](int i) {
      if (kind == kRows) return i == tid ? row0 : gp(B.cube_rows)[i];
      const int q = div_rcp(i, d.n2, rn2), z = i - q * d.n2;
      if (kind == kLines) return q * d.s2 + z;
      const int m = B.m_lo + q;
      return (m < 0 ? m + d.n0 : m) * d.s1 + z;
    });
    __syncthreads();
  };
  for (int k = kRows; k <= kLines; ++k) stage(std::integral_constant<int, 1>{}, k);

  if (d.natoms > 0) {
    // P of group g: wave (g, p) sums the rows p, p + wpg, ... of the group's records,
    // in the working precision per lane and in FP64 over the lanes
    for (int w = wave; w < d.natoms * d.wpg; w += NW) {
      const int g = w / d.wpg, p = w - g * d.wpg;
      const int r0 = gp(d.g_row)[g], r1 = gp(d.g_row)[g + 1];
      T a[2 * kMaxNlm];
#pragma unroll
      for (int l = 0; l < 2 * kMaxNlm; ++l) a[l] = 0;
#pragma unroll 4
      for (int r = r0 + p; r < r1; r += d.wpg) {
        const int e = 64 * r + lane;
        const V4<T> bt = ld4<T>(d.g_b, e);
        const int o = gp(d.g_off)[e];
        C x = u[max(o, 0)];
        x.x = o < 0 ? (T)0 : x.x;
        x.y = o < 0 ? (T)0 : x.y;
        if (!B.gamma) x = cmul(x, gp(B.sgph)[e]);
        a[0] += bt.x * x.x; a[1] += bt.x * x.y;
        a[2] += bt.y * x.x; a[3] += bt.y * x.y;
        a[4] += bt.z * x.x; a[5] += bt.z * x.y;
        a[6] += bt.w * x.x; a[7] += bt.w * x.y;
      }
      // eight sums over 64 lanes: a lane hands on half of its values per step, so
      // that lanes 8 l .. 8 l + 7 end with value l (10 exchanges instead of 48)
      double t[8];
#pragma unroll
      for (int l = 0; l < 8; ++l) t[l] = (double)a[l];
#pragma unroll
      for (int l = 0; l < 4; ++l) {
        swap32(t[l], t[l + 4]);
        t[l] += t[l + 4];
      }
#pragma unroll
      for (int l = 0; l < 2; ++l) {
        swap16(t[l], t[l + 2]);
        t[l] += t[l + 2];
      }
      const bool b8 = (lane & 8) != 0;
      double y = b8 ? t[1] : t[0];
      y += __shfl_xor(b8 ? t[0] : t[1], 8, 64);
      y += __shfl_xor(y, 4, 64);
      y += __shfl_xor(y, 2, 64);
      y += __shfl_xor(y, 1, 64);
      if ((lane & 7) == 0) part[w * 2 * kMaxNlm + (lane >> 3)] = y;
    }
    __syncthreads();
    // D P of every group from the sums of its projector's groups (from the last wave
    // down: the first ones have the most lines below)
    for (int i = NT - 1 - tid; i < d.natoms * kMaxNlm; i += NT) {
      const int g = i / kMaxNlm;
      const V2<int> sb = ld2<int>(d.group_sib, g);
      const GAS double *D = gp(d.coeff) + (size_t)i * kCoeffCols;
      double dr = 0.0, di = 0.0;
      for (int q = 0; q < sb.y; ++q)
        for (int m = 0; m < kMaxNlm; ++m) {
          double pr = 0.0, pi = 0.0;
          for (int p = 0; p < d.wpg; ++p) {
            const double *x = part + ((sb.x + q) * d.wpg + p) * 2 * kMaxNlm + 2 * m;
            pr += x[0];
            pi += x[1];
          }
          dr += D[q * kMaxNlm + m] * pr;
          di += D[q * kMaxNlm + m] * pi;
        }
      dpl[i] = C{(T)(dr * d.kb_scale), (T)(di * d.kb_scale)};
    }
  }
  // V/N on every point (a line along i0 per lane: V is read in rows of lanes)
  for (int i = tid; i < d.n12; i += NT) {
    const int y = div_rcp(i, d.n2, rn2);
    C *p = u + y * d.s2 + (i - y * d.n2);
    const GAS T *v = gp(B.vloc) + i;
#pragma unroll 12
    for (int k = 0; k < d.n0; ++k) {
      const T vv = v[k * d.n12];
      p[k * d.s1].x *= vv;
      p[k * d.s1].y *= vv;
    }
  }
  __syncthreads();
  // + exp(-ik.r) beta D P: a row of a projector per wave; projectors of one class
  // share no point, and the classes follow one another, so no sum depends on timing
  for (int c = 0; c < d.classes; ++c) {
    const int w1 = gp(d.g_class)[c + 1];
#pragma unroll 2
    for (int w = gp(d.g_class)[c] + wave; w < w1; w += NW) {
      const V4<int> item = ld4<int>(d.g_item, w);  // row, first group, groups, rows between groups
      const int e = 64 * item.x + lane, o = gp(d.g_off)[e];
      C ph{1, 0}, t{0, 0};
      if (!B.gamma) ph = gp(B.sgph)[e];
      for (int q = 0; q < item.z; ++q) {
        const V4<T> bt = ld4<T>(d.g_b, e + 64 * q * item.w);
        const C *p = dpl + (item.y + q) * kMaxNlm;
        t.x += bt.x * p[0].x + bt.y * p[1].x + bt.z * p[2].x + bt.w * p[3].x;
        t.y += bt.x * p[0].y + bt.y * p[1].y + bt.z * p[2].y + bt.w * p[3].y;
      }
      if (o >= 0) u[o] = cadd(u[o], cmul(t, C{ph.x, -ph.y}));
    }
    __syncthreads();
  }
  for (int k = kLines; k >= kRows; --k) stage(std::integral_constant<int, -1>{}, k);

  // the sphere, + 1/2|G+k|^2 psi, into H psi and the Taylor accumulators
  const GatherBufs R = gather_bufs(B, s, 0, 1, npw);
  auto finish = [&](int i, int at, C c, T kv) {
    const unsigned o = (unsigned)(i * (int)sizeof(C));
    C out = u[at];
    out.x += kv * c.x;
    out.y += kv * c.y;
    if (B.write_h) bstore(R.h, o, 0u, out);
    if (B.acc1) acc_update<T>(R.a1, o, B.acc_wide != 0, c1r, c1i, out);
    if (B.acc2) acc_update<T>(R.a2, o, B.acc_wide != 0, c2r, c2i, out);
  };
#pragma unroll
  for (int q = 0; q < PF; ++q)
    if (tid + q * NT < npw) finish(tid + q * NT, fo[q], C{fx[q], fy[q]}, fk[q]);
#pragma unroll 2
  for (int i = tid + PF * NT; i < npw; i += NT) finish(i, po[i], psi[i], gp(B.kin)[i]);
}

bool small_length(int n) {
  switch (n) {
#define CASE(S) case S:
    INQX_SMALL_SIZES(CASE)
#undef CASE
    return true;
    default: return false;
  }
}

constexpr int kLdsBytes = 160 * 1024;
int small_waves(int prec) { return (prec == INQX_FP64 ? small_threads<double>() : small_threads<float>()) / 64; }
// waves that share a group's records
int small_wpg(int prec, int natoms) { return std::max(1, small_waves(prec) / std::max(1, natoms)); }
size_t cube_bytes(const int *n, int prec) {
  return (prec == INQX_FP64 ? 16 : 8) * (size_t)n[0] * n[1] * (n[2] + 1);
}
size_t part_bytes(int prec, int natoms) { return 2 * kMaxNlm * sizeof(double) * (size_t)natoms * small_wpg(prec, natoms); }

}  // namespace

// the lengths are built and the cube, the projection sums and D P fit the LDS
bool small_grid_fits(const int *n, int prec, int natoms) {
  return small_length(n[0]) && small_length(n[1]) && small_length(n[2]) &&
         cube_bytes(n, prec) + 16 + part_bytes(prec, natoms) +
                 (prec == INQX_FP64 ? 16 : 8) * (size_t)kMaxNlm * natoms <=
             (size_t)kLdsBytes;
}

template <typename T>
void launch_small_apply(inqx_ham_s *h, const SphereBlock<T> *blk, const int *items, int total, bool has_kb,
                        const double *cf) {
  const int prec = std::is_same<T, double>::value ? INQX_FP64 : INQX_FP32;
  Ctx &cx = h->ctx->c;
  const Grid &g = h->g;
  const KBTables &kb = h->kb;
  SmallDev d;
  d.n0 = g.n[0];
  d.n1 = g.n[1];
  d.n2 = g.n[2];
  d.n12 = g.n[1] * g.n[2];
  d.s2 = g.n[2] + 1;
  d.s1 = g.n[1] * d.s2;
  d.natoms = has_kb ? kb.natoms : 0;
  d.wpg = small_wpg(prec, d.natoms);
  d.part_off = (int)((cube_bytes(g.n, prec) + 15) / 16 * 16);
  d.dp_off = d.part_off + (int)part_bytes(prec, d.natoms);
  const int lds = d.dp_off + (int)sizeof(cplx<T>) * kMaxNlm * d.natoms;
  INQX_CHECK(lds <= kLdsBytes, INQX_ERR_UNSUPPORTED, "the cube does not fit the LDS");
  d.g_row = kb.sg_row;
  d.g_off = kb.sg_off;
  d.g_b = prec == INQX_FP64 ? kb.sg_b64 : kb.sg_b32;
  d.g_item = kb.sg_item;
  d.g_class = kb.sg_class;
  d.classes = has_kb ? kb.sg_classes : 0;
  d.coeff = kb.coeff.as<double>();
  d.group_sib = kb.group_sib.as<int>();
  d.kb_scale = (g.vol / (double)g.N) / (double)g.N;
  static DeviceOnce once;
  if (!once.test_and_set(cx.device))
    INQX_HIP(hipFuncSetAttribute((const void *)k_small_apply<T>, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes));
  ProfScope ps(cx, prec == INQX_FP64 ? "small_apply_f64" : "small_apply_f32");
  hipLaunchKernelGGL(k_small_apply<T>, dim3(total), dim3(small_threads<T>()), lds, cx.stream, blk, items, d, (T)cf[0],
                     (T)cf[1], (T)cf[2], (T)cf[3]);
  INQX_HIP(hipGetLastError());
}

template void launch_small_apply<float>(inqx_ham_s *, const SphereBlock<float> *, const int *, int, bool,
                                        const double *);
template void launch_small_apply<double>(inqx_ham_s *, const SphereBlock<double> *, const int *, int, bool,
                                         const double *);

}  // namespace inqx
