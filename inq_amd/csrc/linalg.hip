// linalg.hip -- contractions over band-major sphere states on MFMA, and the
// FP64 small-matrix steps of orthogonalisation.
//
//   overlap   S = vol * A^H B   (operations::overlap, src/operations/overlap.hpp:26-41)
//             A [n1][K], B [n2][K] complex; split-K over K with
//             matrix-core products of the complex values' real and imaginary parts;
//             partial tiles are reduced in FP64 in a fixed order.
//   rotate    Out = M C (+ beta Out): C [n][K] complex, M [n][n] complex
//             (operations::rotate, src/operations/rotate.hpp:26-156) on the matrix
//             cores; half of it, in place, for a triangular M.
//   cholesky  FP64 lower Cholesky S = L L^H, upper zeroed (matrix::cholesky,
//             src/matrix/cholesky.hpp:28-100), blocked in 32-wide panels.
//   trinv     FP64 inverse of a lower-triangular matrix (matrix::invert_triangular,
//             src/matrix/invert_triangular.hpp:20-50), 32x32 tiles merged by doubling.
//
// MFMA lane layouts (CDNA4), checked against numpy by tests/test_gpu_linalg.py: 16x16x4
// lane l supplies A[l%16][l/16] and B[l/16][l%16] and receives column l%16 of D in
// its four accumulators; the accumulator-to-row map differs between the f32 and f64
// forms (mm_t::row).
#include "internal.hpp"

#include <algorithm>
#include <cstring>
#include <type_traits>

#if defined(__HIP_DEVICE_COMPILE__)
#define GAS __attribute__((address_space(1)))
#else
#define GAS
#endif

namespace inqx {

template <typename T> __device__ __forceinline__ const GAS T *lgp(const T *p) { return (const GAS T *)p; }
template <typename T> __device__ __forceinline__ GAS T *lgw(T *p) { return (GAS T *)p; }

typedef float floatx4 __attribute__((ext_vector_type(4)));
struct alignas(16) V4f {
  float x, y, z, w;
};
typedef double doublex4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef double doublex2 __attribute__((ext_vector_type(2)));

template <typename T> struct mfma_t;
template <> struct mfma_t<float> {
  using pair = floatx2;
};
template <> struct mfma_t<double> {
  using pair = doublex2;
};
template <typename T> struct Vec16;  // 16 bytes of values
template <> struct Vec16<float> {
  typedef floatx4 type;
};
template <> struct Vec16<double> {
  typedef doublex2 type;
};

// ------------------------------------------------------------------------ matrix-core blocks
// Both contractions run 64 x 64 output tiles on four waves, each wave a 32 x 32
// complex block of 2 x 2 16x16x4 products (eight independent accumulators per
// wave keep the matrix cores at 153 of 157 TFLOP/s FP32 and 67 TFLOP/s FP64 in a
// register-only loop; two 32x32x2 accumulators reach 140).  A stage
// is kStage bytes (128) of complex values along the contraction per row.  Any
// order of the contraction index is the same sum, so a lane takes contiguous
// complex values of its row (16-byte LDS reads) and uses real and imaginary
// parts in separate steps: no operand is stored twice or sign-flipped in memory.
constexpr int kMT = 64;                          // output tile edge
constexpr int kStageBytes = 128;                 // of one row, per stage
constexpr int kRowStride = kStageBytes + 16;     // LDS row stride: 16 rows of 16-byte reads cover all banks
template <typename T> constexpr int kStage = kStageBytes / (2 * (int)sizeof(T));  // complex values: 16 or 8

// 16 bytes of complex values, and the same at the alignment of one complex value
// (rows of an odd count of complex64 values start at 8 bytes)
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
template <typename T> struct chunk16;
template <> struct chunk16<float> {
  typedef uintx4 type __attribute__((aligned(8)));
};
template <> struct chunk16<double> {
  typedef uintx4 type;
};
template <typename T> __device__ __forceinline__ uintx4 load16(const GAS cplx<T> *p) {
  return *(const GAS typename chunk16<T>::type *)p;
}
// the first m complex values at p, zero after them
template <typename T> __device__ __forceinline__ uintx4 load16_part(const GAS cplx<T> *p, long m) {
  constexpr int W = (int)sizeof(cplx<T>) / 4;
  uintx4 v{};
#pragma unroll
  for (int q = 0; q < 4 / W; ++q)
    if (q < m)
#pragma unroll
      for (int i = 0; i < W; ++i) v[W * q + i] = ((const GAS unsigned *)(p + q))[i];
  return v;
}

template <typename T> struct mm_t;
template <> struct mm_t<float> {
  typedef floatx4 acc;
  static __device__ __forceinline__ acc run(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int i) { return 4 * (lane >> 4) + i; }
};
template <> struct mm_t<double> {
  typedef doublex4 acc;
  static __device__ __forceinline__ acc run(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int i) { return (lane >> 4) + 4 * i; }
};

// the wave's 32 x 32 complex block as 2 x 2 sub-tiles; value r = 8 x + 4 y + i is
// accumulator i of sub-tile (x, y), at row(lane, r), col(lane, r)
template <typename T> struct Block {
  using M = mm_t<T>;
  static constexpr int kAcc = 16;
  static constexpr int CL = kStage<T> / 4;           // complex values per lane and stage: 4 or 2
  static constexpr int W = 2 * (int)sizeof(T) * CL;  // their bytes: 32
  typename M::acc re[2][2] = {}, im[2][2] = {};
  struct Frag {
    T v[2][2 * CL];
  };
  static __device__ __forceinline__ int row(int lane, int r) { return 16 * (r >> 3) + M::row(lane, r & 3); }
  static __device__ __forceinline__ int col(int lane, int r) { return 16 * ((r >> 2) & 1) + (lane & 15); }
  __device__ __forceinline__ T vr(int r) const { return re[r >> 3][(r >> 2) & 1][r & 3]; }
  __device__ __forceinline__ T vi(int r) const { return im[r >> 3][(r >> 2) & 1][r & 3]; }
  // rows of an LDS tile [row][kStage complex]
  static __device__ __forceinline__ Frag rows(const unsigned char *tile, int lane) {
    using V = typename Vec16<T>::type;
    constexpr int PV = 16 / (int)sizeof(T);
    Frag f;
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const V *p = reinterpret_cast<const V *>(tile + (16 * x + (lane & 15)) * kRowStride + (lane >> 4) * W);
#pragma unroll
      for (int u = 0; u < W / 16; ++u) {
        const V q = p[u];
#pragma unroll
        for (int i = 0; i < PV; ++i) f.v[x][PV * u + i] = q[i];
      }
    }
    return f;
  }
  // columns c0 .. c0 + 31 of an LDS tile [kStage][64 complex]
  static __device__ __forceinline__ Frag cols(const unsigned char *tile, int c0, int lane) {
    using P = typename mfma_t<T>::pair;
    Frag f;
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const P *p = reinterpret_cast<const P *>(tile) + (lane >> 4) * CL * kMT + c0 + 16 * x + (lane & 15);
#pragma unroll
      for (int u = 0; u < CL; ++u) {
        const P q = p[u * kMT];
        f.v[x][2 * u] = q.x;
        f.v[x][2 * u + 1] = q.y;
      }
    }
    return f;
  }
  // += conj(a) b over the stage (CONJ) or a b; eight independent sums follow one another
  template <bool CONJ> __device__ __forceinline__ void mac(const Frag &a, const Frag &b) {
#pragma unroll
    for (int u = 0; u < CL; ++u) {
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) {
          re[x][y] = M::run(a.v[x][2 * u], b.v[y][2 * u], re[x][y]);
          im[x][y] = M::run(a.v[x][2 * u], b.v[y][2 * u + 1], im[x][y]);
        }
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) {
          const T ai = a.v[x][2 * u + 1];
          re[x][y] = M::run(CONJ ? ai : -ai, b.v[y][2 * u + 1], re[x][y]);
          im[x][y] = M::run(CONJ ? -ai : ai, b.v[y][2 * u], im[x][y]);
        }
    }
  }
};

// Work-groups are dealt round-robin to the 8 XCDs; renumber so that each XCD runs
// a contiguous range, whose neighbours read the same rows through the same L2.
__device__ __forceinline__ int xcd_logical(int b, int G) {
  const int xq = G / 8, xr = G % 8, x = b % 8;
  return (x < xr ? x * (xq + 1) : xr * (xq + 1) + (x - xr) * xq) + b / 8;
}

// ------------------------------------------------------------------------ overlap
// S = vol A^H B split over K: a work-group sums one chunk of K for one 64 x 64
// tile.  The grid is sized to run as one round of equal work-groups (up to four
// per CU), so none waits for a last partial round.  FP32 products accumulate over
// at most `run` complex values before they are added in FP64 (WIDE: chunks
// longer than that keep FP64 sums in registers and write FP64 partial tiles).
// HERM (A and B the same states): only the tiles on and below the diagonal.
// Measured, before -> now: 432 states x 228487 with themselves, complex64, 3.38 ->
// 1.87 ms (112 TFLOP/s over the products done); 128 x 67691 93 -> 67 us complex64,
// two different blocks of it in complex128 176 -> 166 us (53 of 67 TFLOP/s).
constexpr int kOvRunMin = 128, kOvRunMax = 1024;  // complex values per FP32 accumulation
constexpr int kOvRunSplit = 1024;   // the contractions of all tiles are cut in so many runs between the two
constexpr int kOvChunkMin = 128;    // complex values per work-group at least
constexpr int kOvChunkGood = 256;   // enough stages to hide a work-group's start and end

struct OvPlan {
  int tiles_i, tiles_j, tiles;  // tiles: all, or those on and below the diagonal
  int nchunk;
  long chunk;  // complex values, a multiple of the stage
  int run;     // complex64: complex values per FP32 accumulation, a multiple of the stage
  bool wide;   // complex64: FP64 sums within a chunk
};
// work-groups per CU in the one round: what the registers hold
static int overlap_slots(bool f64, bool wide) { return f64 || wide ? 3 : 4; }
static OvPlan overlap_plan(int n1, int n2, long K, bool herm, int cus, bool f64) {
  OvPlan p;
  p.tiles_i = (n1 + kMT - 1) / kMT;
  p.tiles_j = (n2 + kMT - 1) / kMT;
  const int all = p.tiles_i * p.tiles_j;
  p.tiles = herm ? p.tiles_i * (p.tiles_i + 1) / 2 : all;
  const int stage = f64 ? kStage<double> : kStage<float>;
  const auto stages = [&](long c) { return (c + stage - 1) / stage * stage; };
  // The rounding of an FP32 sum grows with its length, so the length does not follow
  // the launch shape below: small contractions end after 128 values, the longest
  // after 1024 (error of a norm over 30000 values: 1.5e-8 rms with 128, 4.3e-8 with 368)
  const long want_run = (kOvRunSplit + all - 1) / all;
  p.run = (int)stages(std::min<long>(kOvRunMax, std::max<long>(kOvRunMin, (K + want_run - 1) / want_run)));
  for (int m = 4; m >= 1; --m) {
    const long want = std::max<long>(1, (long)m * cus / p.tiles);
    p.chunk = stages(std::max<long>((K + want - 1) / want, kOvChunkMin));
    p.wide = !f64 && p.chunk > p.run;
    if (m > overlap_slots(f64, p.wide)) continue;
    if (p.chunk >= kOvChunkGood) break;
  }
  p.nchunk = (int)((K + p.chunk - 1) / p.chunk);
  return p;
}

// tile t of the list on and below the diagonal
__device__ __forceinline__ void lower_tile(int t, int &ti, int &tj) {
  int i = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
  while ((i + 1) * (i + 2) / 2 <= t) ++i;
  while (i * (i + 1) / 2 > t) --i;
  ti = i;
  tj = t - i * (i + 1) / 2;
}

template <typename T, typename P, bool WIDE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WIDE || sizeof(T) == 8 ? 3 : 4)))
k_overlap_partial(const T *A, const T *B, int n1, int n2, long K, int tiles,
                                                         int tiles_j, int herm, long chunk, int run,
                                                         P *partial) {
  constexpr int KC = kStage<T>, CV = 16 / (2 * (int)sizeof(T)), kTile = kMT * kRowStride;
  __shared__ __align__(16) unsigned char sm[2][2][kTile];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int id = xcd_logical(blockIdx.x, gridDim.x);
  const int c = id / tiles, t = id - c * tiles;
  int ti, tj;
  if (herm) {
    lower_tile(t, ti, tj);
  } else {
    ti = t / tiles_j;
    tj = t - ti * tiles_j;
  }
  const int i0 = ti * kMT, j0 = tj * kMT, wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  const long k0 = (long)c * chunk, k1 = min(k0 + chunk, K);
  // this thread's 16 bytes of rows lr and lr + 32 of both tiles, chunk lc (rows past
  // the last state repeat it: their outputs are not used).  The pipelined loop runs
  // over whole stages with plain loads; the last chunk's odd stage follows it
  const int lr = tid >> 3, lc = tid & 7;
  const GAS cplx<T> *pa[2], *pb[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    pa[h] = (const GAS cplx<T> *)lgp(A) + (long)min(i0 + 32 * h + lr, n1 - 1) * K + lc * CV;
    pb[h] = (const GAS cplx<T> *)lgp(B) + (long)min(j0 + 32 * h + lr, n2 - 1) * K + lc * CV;
  }
  uintx4 ra[2], rb[2];
  auto load = [&](long k) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      ra[h] = load16<T>(pa[h] + k);
      rb[h] = load16<T>(pb[h] + k);
    }
  };
  auto store = [&](int b) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      *reinterpret_cast<uintx4 *>(&sm[b][0][(32 * h + lr) * kRowStride + 16 * lc]) = ra[h];
      *reinterpret_cast<uintx4 *>(&sm[b][1][(32 * h + lr) * kRowStride + 16 * lc]) = rb[h];
    }
  };
  Block<T> acc;
  double wre[WIDE ? 16 : 1] = {}, wim[WIDE ? 16 : 1] = {};
  auto mac = [&](int b) {
    const auto a = Block<T>::rows(&sm[b][0][wr * kRowStride], lane);
    const auto c = Block<T>::rows(&sm[b][1][wc * kRowStride], lane);
    acc.template mac<true>(a, c);
  };
  auto widen = [&]() {
    if constexpr (WIDE) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        wre[r] += (double)acc.vr(r);
        wim[r] += (double)acc.vi(r);
      }
      acc = Block<T>();
    }
  };
  const long kw = k0 + (k1 - k0) / KC * KC;  // end of the whole stages
  int buf = 0, summed = 0;
  if (k0 < kw) {
    load(k0);
    store(0);
    __syncthreads();
  }
  for (long k = k0; k < kw; k += KC) {
    const bool more = k + KC < kw;
    if (more) load(k + KC);
    mac(buf);
    if (WIDE && (summed += KC) >= run) {
      summed = 0;
      widen();
    }
    buf ^= 1;
    if (more) store(buf);
    __syncthreads();
  }
  if (kw < k1) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      ra[h] = load16_part<T>(pa[h] + kw, k1 - kw - lc * CV);
      rb[h] = load16_part<T>(pb[h] + kw, k1 - kw - lc * CV);
    }
    store(buf);
    __syncthreads();
    mac(buf);
  }
  widen();
  GAS P *out = lgw(partial) + (long)id * kMT * kMT * 2;
#pragma unroll
  for (int r = 0; r < Block<T>::kAcc; ++r) {
    const int e = (wr + Block<T>::row(lane, r)) * kMT + wc + Block<T>::col(lane, r);
    out[2 * e] = WIDE ? (P)wre[WIDE ? r : 0] : (P)acc.vr(r);
    out[2 * e + 1] = WIDE ? (P)wim[WIDE ? r : 0] : (P)acc.vi(r);
  }
}

// S[i][j] = vol * sum_chunks partial in FP64, in a fixed order: work-group = one
// 64-wide row of one output tile; lane group g (of 4) sums chunks g, g+4, g+8, ...
// in ascending order, and the four group sums are added g = 0..3.  herm: the
// tiles below the diagonal also give S[j][i], the conjugate.
constexpr int kOvRedGroups = 4;
template <typename P>
__global__ void __launch_bounds__(256) k_overlap_reduce(const P *partial, int n1, int n2, int tiles, int tiles_j,
                                                        int herm, int nchunk, double vol, double *S) {
  using P2 = typename mfma_t<P>::pair;
  __shared__ double red[kOvRedGroups][kMT][2];
  const int jj = threadIdx.x & (kMT - 1), g = threadIdx.x >> 6;
  const int ii = blockIdx.x % kMT, tile = blockIdx.x / kMT;
  int ti, tj;
  if (herm) {
    lower_tile(tile, ti, tj);
  } else {
    ti = tile / tiles_j;
    tj = tile - ti * tiles_j;
  }
  const long tile_stride = (long)tiles * kMT * kMT;  // P2 per chunk
  const GAS P2 *p = (const GAS P2 *)lgp(partial) + (long)tile * kMT * kMT + ii * kMT + jj;
  double sr = 0.0, si = 0.0;
#pragma unroll 8
  for (int c = g; c < nchunk; c += kOvRedGroups) {
    const P2 v = p[(long)c * tile_stride];
    sr += (double)v.x;
    si += (double)v.y;
  }
  red[g][jj][0] = sr;
  red[g][jj][1] = si;
  __syncthreads();
  const int i = ti * kMT + ii, j = tj * kMT + jj;
  if (g == 0 && i < n1 && j < n2) {
    double tr = red[0][jj][0], tim = red[0][jj][1];
#pragma unroll
    for (int q = 1; q < kOvRedGroups; ++q) {
      tr += red[q][jj][0];
      tim += red[q][jj][1];
    }
    GAS double *Sg = lgw(S);
    Sg[2 * ((long)i * n2 + j)] = vol * tr;
    Sg[2 * ((long)i * n2 + j) + 1] = vol * tim;
    if (herm && ti != tj) {
      Sg[2 * ((long)j * n2 + i)] = vol * tr;
      Sg[2 * ((long)j * n2 + i) + 1] = -vol * tim;
    }
  }
}

// ------------------------------------------------------------------------ rotate
// operand matrix M [nr_pad][ld] complex in T, rows padded to a multiple of 64 and
// ld to a multiple of 16, the padding zero
// mode 0: M = conj(R) (Phi <- Phi R^H);  mode 1: M = alpha R^T (5-argument rotate,
// R is [nc][nr]); mode 2: M = R
template <typename T>
__global__ void k_rot_prep(const double *R, int nr, int nc, int mode, double ar, double ai, int nr_pad, int ld,
                           cplx<T> *M) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long)nr_pad * ld) return;
  const int i = (int)(idx / ld), j = (int)(idx - (long)i * ld);
  double mr = 0.0, mi = 0.0;
  if (i < nr && j < nc) {
    if (mode == 1) {
      const double rr = R[2 * ((long)j * nr + i)], ri = R[2 * ((long)j * nr + i) + 1];
      mr = ar * rr - ai * ri;
      mi = ar * ri + ai * rr;
    } else {
      mr = R[2 * ((long)i * nc + j)];
      mi = R[2 * ((long)i * nc + j) + 1];
      if (mode == 0) mi = -mi;
    }
  }
  M[idx] = cplx<T>{(T)mr, (T)mi};
}

// Out[i][p] = sum_j M[i][j] C[j][p] (+ beta Out[i][p]), i < nr, j < nc; a 64 x 64
// tile per work-group, or, with `lower` (M lower triangular), every row tile of
// one column block, the last rows first: row tile i reads rows j < i0 + 64 only, so
// Out may be C itself (a tile's rows are read by that tile and later rows alone,
// which are done), half of the products are left out and no copy follows.
// Measured, before -> now: triangular 432 x 228487 complex64, 3.09 ms and a 0.30 ms
// copy -> 1.84 ms; 128 x 67691 94 + 27 -> 78 us; the full complex128 product with
// beta = 1 of 128 x 67691 250 -> 198 us.
template <typename T>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 3 : 4)))
k_rotate(const cplx<T> *Mm, int ld, const cplx<T> *Cm, int nr, int nc, long K,
                                                cplx<T> *Out, double br, double bi, int tiles_i, int lower,
                                                const int *info) {
  using C = cplx<T>;
  constexpr int KC = kStage<T>, CV = 16 / (int)sizeof(C);
  constexpr int kA = kMT * kRowStride, kB = KC * kMT * (int)sizeof(C);
  __shared__ __align__(16) unsigned char sm[2][kA + kB];
  if (info && *info != 0) return;  // the factorisation that gave M failed
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int id = xcd_logical(blockIdx.x, gridDim.x);
  const int tp = lower ? id : id / tiles_i;
  const long p0 = (long)tp * kMT;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  const GAS C *Mg = lgp(Mm);
  const GAS C *Cg = lgp(Cm);
  const int mr = tid >> 3, mc = tid & 7;              // M loads: rows mr, mr + 32, 16-byte chunk mc
  constexpr int CPR = kMT / CV, RPP = 256 / CPR;      // C loads: chunks per row, rows per pass
  const int cr = tid / CPR, cc = (tid % CPR) * CV;
  const bool full = p0 + kMT <= K;                    // uniform
  for (int ti = lower ? tiles_i - 1 : id - tp * tiles_i; ti >= 0; --ti) {
    const int i0 = ti * kMT;
    const int jend = lower ? min(nc, i0 + kMT) : nc;
    Block<T> acc;
    auto sweep = [&](auto whole) {
      uintx4 ra[2], rb[KC / RPP];
      auto load = [&](int j) {
#pragma unroll
        for (int h = 0; h < 2; ++h)  // rows and columns of M are padded: no check
          ra[h] = *(const GAS uintx4 *)(Mg + (long)(i0 + 32 * h + mr) * ld + j + mc * CV);
#pragma unroll
        for (int h = 0; h < KC / RPP; ++h) {  // rows past the last repeat it and are cleared below
          const GAS C *p = Cg + (long)min(j + RPP * h + cr, nc - 1) * K + p0 + cc;
          if constexpr (decltype(whole)::value) rb[h] = load16<T>(p);
          else rb[h] = load16_part<T>(p, K - p0 - cc);
        }
      };
      auto store = [&](int b, int j) {
#pragma unroll
        for (int h = 0; h < 2; ++h) *reinterpret_cast<uintx4 *>(&sm[b][(32 * h + mr) * kRowStride + 16 * mc]) = ra[h];
#pragma unroll
        for (int h = 0; h < KC / RPP; ++h) {
          const uintx4 zero{};
          *reinterpret_cast<uintx4 *>(&sm[b][kA + ((RPP * h + cr) * kMT + cc) * (int)sizeof(C)]) =
              j + RPP * h + cr < nc ? rb[h] : zero;
        }
      };
      load(0);
      store(0, 0);
      __syncthreads();
      int buf = 0;
      for (int j = 0; j < jend; j += KC) {
        const bool more = j + KC < jend;
        if (more) load(j + KC);
        const auto a = Block<T>::rows(&sm[buf][wr * kRowStride], lane);
        const auto b = Block<T>::cols(&sm[buf][kA], wc, lane);
        acc.template mac<false>(a, b);
        buf ^= 1;
        if (more) store(buf, j + KC);
        __syncthreads();
      }
    };
    if (full) sweep(std::true_type{});
    else sweep(std::false_type{});
    GAS C *Og = lgw(Out);
    const bool beta = (br != 0.0 || bi != 0.0);
#pragma unroll
    for (int r = 0; r < Block<T>::kAcc; ++r) {
      const int i = i0 + wr + Block<T>::row(lane, r);
      const long p = p0 + wc + Block<T>::col(lane, r);
      if (i < nr && p < K) {
        C o{acc.vr(r), acc.vi(r)};
        if (beta) {
          const C qv = Og[(long)i * K + p];
          o.x += (T)(br * (double)qv.x - bi * (double)qv.y);
          o.y += (T)(br * (double)qv.y + bi * (double)qv.x);
        }
        Og[(long)i * K + p] = o;
      }
    }
    if (!lower) break;
  }
}

// ------------------------------------------------------------------------ Cholesky / inverse (FP64)
// Blocked in 32 x 32 tiles; every read of a value another work-group wrote
// happens in a later launch.  Both are chains of dependent steps far below any
// bandwidth or matrix-core limit, so what counts is the number of launches and
// the length of each one's longest work-group.
//
// Cholesky S = L L^H in place (lower; the strict upper triangle is zeroed):
//   k_chol_first   factors the first diagonal tile
//   k_chol_step    panel c0, one work-group per tile (i, j) of the trailing lower
//                  triangle: L_i = S_i L_dd^{-H} and L_j (each tile recomputes its
//                  two panel tiles by substitution instead of waiting for a panel
//                  launch), S_ij -= L_i L_j^H on the matrix cores; the work-group
//                  of the first tile then factors it, the next diagonal tile.  The
//                  panel's tiles are read by many work-groups, so L_i goes as L_i^H
//                  to the unused upper tile (c0, i)
//   k_chol_finish  moves the panels from the upper to the lower triangle
// One launch per panel instead of three, and tiles of 32 also for the small
// blocks: n = 128 150 -> 83 us, n = 432 690 -> 290 us.  Up to n = 64 one work-group
// did it in one launch before; two launches without k_chol_finish, and a last tile
// that takes the steps of its rows only: n = 33 42 us then, 44 now, n = 40 48
// and 44, n = 64 69 and 54.
// info[0] = 0 or the first non-positive leading minor (LAPACK convention); the first
// launch writes it, and every later launch returns at once when it is set.
constexpr int kChB = 32;
typedef double2 ctile[kChB][kChB + 1];

__device__ __forceinline__ double2 dmulc(double2 a, double2 b) {  // a conj(b)
  return double2{a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y};
}

// tile (i0, j0) of an n x n row-major complex matrix, zero outside it (256 threads)
__device__ __forceinline__ void load_ctile(ctile &t, const double *S, int n, int i0, int j0) {
  const GAS double2 *g = (const GAS double2 *)lgp(S);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int e = threadIdx.x + 256 * u, r = e >> 5, c = e & 31;
    double2 v{0.0, 0.0};
    if (i0 + r < n && j0 + c < n) v = g[(long)(i0 + r) * n + j0 + c];
    t[r][c] = v;
  }
}

// the 32 x 32 product of two tiles, wave w taking the 16 x 16 sub-tile (w >> 1, w & 1):
// += A B (B a tile [k][col]), or A conj(B)^T with CONJT (B a tile [col][k])
template <bool CONJT>
__device__ __forceinline__ void ctile_mac(const ctile &A, const ctile &B, int lane, int wave, doublex4 &re,
                                          doublex4 &im) {
  const int i = 16 * (wave >> 1) + (lane & 15), j = 16 * (wave & 1) + (lane & 15), q = lane >> 4;
#pragma unroll
  for (int k = 0; k < kChB; k += 4) {
    const double2 a = A[i][k + q], b = CONJT ? B[j][k + q] : B[k + q][j];
    const double bi = CONJT ? -b.y : b.y;
    re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, re, 0, 0, 0);
    im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, bi, im, 0, 0, 0);
    re = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.y, bi, re, 0, 0, 0);
    im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.x, im, 0, 0, 0);
  }
}
__device__ __forceinline__ int ctile_row(int lane, int wave, int i) { return 16 * (wave >> 1) + mm_t<double>::row(lane, i); }
__device__ __forceinline__ int ctile_col(int lane, int wave) { return 16 * (wave & 1) + (lane & 15); }

// factors the diagonal tile D (b valid rows, the rest identity) in one wave without
// barriers: lane (row r, half h) keeps the columns 2 q + h of its row in registers,
// column j goes through LDS (in order within the wave), and the update uses 1 / d;
// the scaling by 1 / sqrt(d) follows for all columns at once.  Writes L into S.
// STEPS >= b columns are factored.
template <int STEPS>
__device__ __forceinline__ void factor_tile(const ctile &D, double2 (&col)[2][2 * kChB], double *S, int n, int c0,
                                            int *info, bool first) {
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int b = min(kChB, n - c0);
  double2 a[kChB / 2];
#pragma unroll
  for (int q = 0; q < kChB / 2; ++q) {
    const int k = 2 * q + h;
    a[q] = D[r][k];
    if (r >= b) a[q] = double2{r == k ? 1.0 : 0.0, 0.0};
  }
  double dr = 1.0;  // this row's pivot
  int bad = 0;
#pragma unroll
  for (int j = 0; j < STEPS; ++j) {
    col[j & 1][h == (j & 1) ? r : r + kChB] = a[j >> 1];  // the other half's value is not used
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const double2 me = col[j & 1][r];
    const double d = col[j & 1][j].x;
    bad = !(d > 0.0) && bad == 0 ? c0 + j + 1 : bad;
    dr = r == j ? d : dr;
    const double rd = 1.0 / d;
    const double2 f{me.x * rd, me.y * rd};
    __builtin_amdgcn_sched_barrier(0);  // one step's values in registers at a time
#pragma unroll
    for (int q = 0; q < STEPS / 2; ++q)
      if (2 * q + 1 > j) {  // k = 2 q + h > j, but for k = j on half 0, whose value is final
        const double2 g{2 * q > j || h == 1 ? f.x : 0.0, 2 * q > j || h == 1 ? f.y : 0.0};
        const double2 p = dmulc(g, col[j & 1][2 * q + h]);
        a[q].x -= p.x;
        a[q].y -= p.y;
      }
    __builtin_amdgcn_sched_barrier(0);
  }
  if (bad) {  // uniform
    if (lane == 0) info[0] = bad;
    return;
  }
  if (first && lane == 0) info[0] = 0;
  const double l = sqrt(dr);
  if (h == 0) col[0][r] = double2{1.0 / l, l};
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  GAS double2 *g = (GAS double2 *)lgw(S);
  if (r < b)
#pragma unroll
    for (int q = 0; q < kChB / 2; ++q) {
      const int k = 2 * q + h;
      if (k <= r) {
        const double2 s = col[0][k];
        g[(long)(c0 + r) * n + c0 + k] = k == r ? double2{s.y, 0.0} : double2{a[q].x * s.x, a[q].y * s.x};
      }
    }
}

__global__ void __launch_bounds__(256) k_chol_first(double *S, int n, int *info) {
  __shared__ ctile D;
  __shared__ double2 col[2][2 * kChB];
  load_ctile(D, S, n, 0, 0);
  __syncthreads();
  if (threadIdx.x >= 64) return;
  if (n <= 8) factor_tile<8>(D, col, S, n, 0, info, true);
  else if (n <= 16) factor_tile<16>(D, col, S, n, 0, info, true);
  else factor_tile<kChB>(D, col, S, n, 0, info, true);
  if (n > kChB) return;
  for (int e = threadIdx.x; e < n * n; e += 64) {  // one tile: the whole upper triangle
    const int i = e / n, j = e - i * n;
    if (j > i) ((GAS double2 *)lgw(S))[e] = double2{0.0, 0.0};
  }
}

// x <- x L_dd^{-H} of one panel tile, eight lanes per row (columns c + 8 q): once
// x_j is final it goes to its row's lanes and x_k -= x_j conj(L_dd[k][j]) for k > j
__device__ __forceinline__ void panel_step(double2 (&x)[4], const ctile &Lk, const double *rd, int j, int c, int lane) {
  const int q = j >> 3, own = j & 7;
  double2 v{x[q].x * rd[j], x[q].y * rd[j]};
  v.x = __shfl(v.x, (lane & 56) | own, 64);
  v.y = __shfl(v.y, (lane & 56) | own, 64);
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    if (p < q) continue;
    const double2 t = dmulc(v, Lk[c + 8 * p][j]);
    const bool later = p > q || c > own;
    x[p].x = later ? x[p].x - t.x : x[p].x;
    x[p].y = later ? x[p].y - t.y : x[p].y;
  }
  if (c == own) x[q] = v;
}

// whole: the matrix has two panels, so this work-group is the only one; it leaves L in
// place instead of k_chol_finish
__global__ void __launch_bounds__(256) k_chol_step(double *S, int n, int c0, int whole, int *info) {
  __shared__ ctile Lk, Li, Lj;
  __shared__ double rd[kChB];
  __shared__ double2 col[2][2 * kChB];
  if (info[0] != 0) return;
  int ti, tj;
  lower_tile(blockIdx.x, ti, tj);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int i0 = c0 + kChB * (ti + 1), j0 = c0 + kChB * (tj + 1);
  load_ctile(Lk, S, n, c0, c0);
  load_ctile(Li, S, n, i0, c0);
  if (ti != tj) load_ctile(Lj, S, n, j0, c0);
  if (tid < kChB) rd[tid] = 1.0 / S[2 * ((long)(c0 + tid) * n + c0 + tid)];
  __syncthreads();
  const int r = tid >> 3, c = tid & 7;
  double2 xi[4], xj[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    xi[q] = Li[r][c + 8 * q];
    xj[q] = Lj[r][c + 8 * q];
  }
  if (ti != tj) {
#pragma unroll
    for (int j = 0; j < kChB; ++j) {
      panel_step(xi, Lk, rd, j, c, lane);
      panel_step(xj, Lk, rd, j, c, lane);
    }
  } else {
#pragma unroll
    for (int j = 0; j < kChB; ++j) panel_step(xi, Lk, rd, j, c, lane);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {  // every lane writes the values it read itself
    Li[r][c + 8 * q] = xi[q];
    if (ti != tj) Lj[r][c + 8 * q] = xj[q];
  }
  __syncthreads();
  GAS double2 *g = (GAS double2 *)lgw(S);
  if (whole) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = tid + 256 * u, k = e >> 5, m = e & 31;
      const double2 zero{0.0, 0.0};
      if (i0 + k < n) g[(long)(i0 + k) * n + c0 + m] = Li[k][m];
      if (i0 + m < n) g[(long)(c0 + k) * n + i0 + m] = zero;
      if (m > k) g[(long)(c0 + k) * n + c0 + m] = zero;
      if (m > k && i0 + m < n) g[(long)(i0 + k) * n + i0 + m] = zero;
    }
  } else if (tj == 0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {  // L_i^H to the upper tile (c0, i0)
      const int e = tid + 256 * u, k = e >> 5, m = e & 31;
      if (i0 + m < n) g[(long)(c0 + k) * n + i0 + m] = double2{Li[m][k].x, -Li[m][k].y};
    }
  }
  doublex4 re{}, im{};
  if (ti != tj) ctile_mac<true>(Li, Lj, lane, wave, re, im);
  else ctile_mac<true>(Li, Li, lane, wave, re, im);
  const bool next = blockIdx.x == 0;  // the next diagonal tile: factored below
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int a = ctile_row(lane, wave, i), b = ctile_col(lane, wave);
    if (i0 + a < n && j0 + b <= i0 + a) {
      const long o = (long)(i0 + a) * n + j0 + b;
      double2 s = g[o];
      s.x -= re[i];
      s.y -= im[i];
      if (next) Lj[a][b] = s;  // (ti == tj: Lj is free)
      else g[o] = s;
    } else if (next) {
      Lj[a][b] = double2{0.0, 0.0};
    }
  }
  if (!next) return;
  __syncthreads();
  if (tid >= 64) return;
  if (n - i0 <= 8) factor_tile<8>(Lj, col, S, n, i0, info, false);
  else if (n - i0 <= 16) factor_tile<16>(Lj, col, S, n, i0, info, false);
  else factor_tile<kChB>(Lj, col, S, n, i0, info, false);
}

__global__ void __launch_bounds__(256) k_chol_finish(double *S, int n, const int *info) {
  __shared__ ctile t;
  if (info[0] != 0) return;
  int ti, tj;
  lower_tile(blockIdx.x, ti, tj);
  const int i0 = kChB * ti, j0 = kChB * tj;
  GAS double2 *g = (GAS double2 *)lgw(S);
  if (ti != tj) {
    load_ctile(t, S, n, j0, i0);
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int e = threadIdx.x + 256 * u, r = e >> 5, c = e & 31;
    if (ti != tj) {
      if (i0 + r < n) g[(long)(i0 + r) * n + j0 + c] = double2{t[c][r].x, -t[c][r].y};
      if (i0 + c < n) g[(long)(j0 + r) * n + i0 + c] = double2{0.0, 0.0};
    } else if (c > r && i0 + c < n) {
      g[(long)(i0 + r) * n + i0 + c] = double2{0.0, 0.0};
    }
  }
}

// X = L^{-1} for lower-triangular L: the 32 x 32 diagonal tiles, then pairs of
// neighbouring inverted blocks of 32, 64, 128, ... rows are merged,
// X_21 = -X_22 (L_21 X_11), all pairs in parallel: 2 launches per doubling
// instead of one per block row (n = 128 79 -> 44 us, n = 432 550 -> 105 us).
//   k_trinv_diag   one wave per diagonal tile: lane (column c, half h) keeps the
//                  rows 2 q + h of its column of X; tiles above the diagonal zeroed
//   k_trinv_merge  one 32 x 32 tile of T = L_21 X_11 or of X_21 = -X_22 T
// the inverse of the diagonal tile of b <= STEPS rows at r0, in one wave
template <int STEPS>
__device__ __forceinline__ void invert_tile(ctile &t, double2 (&id)[kChB], const GAS double2 *lg, GAS double2 *g, int n,
                                            int r0, int b) {
  const int lane = threadIdx.x;
#pragma unroll 4
  for (int u = 0; u < STEPS / 2; ++u) {
    const int e = lane + 64 * u, i = e >> 5, j = e & 31;
    double2 v{i == j ? 1.0 : 0.0, 0.0};  // identity past the last row
    if (i < b && j <= i) v = lg[(long)(r0 + i) * n + r0 + j];
    t[i][j] = v;
  }
  __syncthreads();
  if (lane < STEPS) {
    const double2 l = t[lane][lane];
    const double m = 1.0 / (l.x * l.x + l.y * l.y);
    id[lane] = double2{l.x * m, -l.y * m};
  }
  __syncthreads();
  const int c = lane & 31, h = lane >> 5;
  double2 x[STEPS / 2];
#pragma unroll
  for (int q = 0; q < STEPS / 2; ++q) x[q] = double2{2 * q + h == c ? 1.0 : 0.0, 0.0};
  // forward substitution, a column of the inverse per lane pair
#pragma unroll
  for (int j = 0; j < STEPS; ++j) {
    __builtin_amdgcn_sched_barrier(0);  // one step's values in registers at a time
    const double2 w = id[j], y = x[j >> 1];
    double2 v{y.x * w.x - y.y * w.y, y.x * w.y + y.y * w.x};  // right on half j & 1
    double2 lo = v, hi = v;
    swap32(lo.x, hi.x);
    swap32(lo.y, hi.y);
    v = (j & 1) ? hi : lo;
    x[j >> 1].x = h == (j & 1) ? v.x : x[j >> 1].x;
    x[j >> 1].y = h == (j & 1) ? v.y : x[j >> 1].y;
#pragma unroll
    for (int q = 0; q < STEPS / 2; ++q)
      if (2 * q + 1 > j) {
        const double2 l = t[2 * q + h][j], g{2 * q > j || h == 1 ? v.x : 0.0, 2 * q > j || h == 1 ? v.y : 0.0};
        x[q].x -= l.x * g.x - l.y * g.y;
        x[q].y -= l.x * g.y + l.y * g.x;
      }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int q = 0; q < STEPS / 2; ++q) t[2 * q + h][c] = x[q];  // its column, read by no other lane's steps now
  __syncthreads();
#pragma unroll 4
  for (int u = 0; u < STEPS / 2; ++u) {
    const int e = lane + 64 * u, i = e >> 5, j = e & 31;
    if (i < b && j < b) g[(long)(r0 + i) * n + r0 + j] = j <= i ? t[i][j] : double2{0.0, 0.0};
  }
}

// X = L^{-1}: the diagonal tiles; tiles above the diagonal zeroed
__global__ void __launch_bounds__(64) k_trinv_diag(const double *L, int n, double *X) {
  __shared__ ctile t;
  __shared__ double2 id[kChB];  // 1 / L[i][i]
  const int bi = blockIdx.y, bj = blockIdx.x, lane = threadIdx.x;
  const int r0 = bi * kChB, q0 = bj * kChB;
  GAS double2 *g = (GAS double2 *)lgw(X);
  const GAS double2 *lg = (const GAS double2 *)lgp(L);
  if (bj < bi) return;
  if (bj > bi) {
    for (int e = lane; e < kChB * kChB; e += 64) {
      const int i = e >> 5, j = e & 31;
      if (q0 + j < n) g[(long)(r0 + i) * n + q0 + j] = double2{0.0, 0.0};
    }
    return;
  }
  const int b = min(kChB, n - r0);
  if (b <= 2) invert_tile<2>(t, id, lg, g, n, r0, b);
  else if (b <= 8) invert_tile<8>(t, id, lg, g, n, r0, b);
  else if (b <= 16) invert_tile<16>(t, id, lg, g, n, r0, b);
  else invert_tile<kChB>(t, id, lg, g, n, r0, b);
}

// pair blockIdx.z of blocks of `blk` rows; tile (blockIdx.y, blockIdx.x) of its
// lower-left block.  second = 0: T = L_21 X_11; 1: X_21 = -X_22 T
__global__ void __launch_bounds__(256) k_trinv_merge(const double *L, int n, double *X, double *T, int blk, int second) {
  __shared__ ctile A, B;
  const int base = 2 * blk * blockIdx.z, i0 = base + blk + kChB * blockIdx.y, j0 = base + kChB * blockIdx.x;
  if (i0 >= n) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const double *Am = second ? X : L, *Bm = second ? T : X;
  const int k0 = second ? base + blk : j0;              // X_11 is zero above its diagonal,
  const int k1 = second ? i0 + kChB : base + blk;       // X_22 right of its own
  doublex4 re{}, im{};
  for (int k = k0; k < k1; k += kChB) {
    if (k != k0) __syncthreads();
    load_ctile(A, Am, n, i0, k);
    load_ctile(B, Bm, n, k, j0);
    __syncthreads();
    ctile_mac<false>(A, B, lane, wave, re, im);
  }
  GAS double2 *g = (GAS double2 *)lgw(second ? X : T);
  const double s = second ? -1.0 : 1.0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int a = i0 + ctile_row(lane, wave, i), b = j0 + ctile_col(lane, wave);
    if (a < n) g[(long)a * n + b] = double2{s * re[i], s * im[i]};
  }
}

// ------------------------------------------------------------------------ HBM copy (calibration)
// plain 16-byte-per-lane device copy: the STREAM-style bandwidth reference and
// the known-size kernel that calibrates the FETCH_SIZE / WRITE_SIZE counters
// one 16-byte element per thread and no loop: the fastest plain copy form
// measured on MI355X (6.1 TB/s for 2 GiB; a grid-stride loop over 8192
// work-groups reached 4.6 TB/s, several elements per thread less)
__global__ void __launch_bounds__(256) k_stream_copy(const V4f *src, V4f *dst, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

// ------------------------------------------------------------------------ host launchers
void launch_overlap(Ctx &cx, int prec, int n1, int n2, long K, const void *A, const void *B, double vol, double *S,
                    DevMem &partial) {
  const bool herm = A == B && n1 == n2;
  const bool f64 = prec == INQX_FP64;
  const OvPlan p = overlap_plan(n1, n2, K, herm, cx.num_cu, f64);
  const size_t es = f64 || p.wide ? 8 : 4;
  partial.ensure(es * (size_t)p.nchunk * p.tiles * kMT * kMT * 2);
  const long grid = (long)p.nchunk * p.tiles;
  INQX_CHECK(grid <= INT32_MAX / kMT, INQX_ERR_ARG, "overlap: too many tiles");
  const dim3 g((unsigned)grid), gr((unsigned)(p.tiles * kMT));
  const int h = herm ? 1 : 0;
  {
    ProfScope ps(cx, f64 ? "overlap_mfma_f64" : "overlap_mfma_f32");
    if (f64)
      hipLaunchKernelGGL((k_overlap_partial<double, double, false>), g, dim3(256), 0, cx.stream, (const double *)A,
                         (const double *)B, n1, n2, K, p.tiles, p.tiles_j, h, p.chunk, p.run, partial.as<double>());
    else if (p.wide)
      hipLaunchKernelGGL((k_overlap_partial<float, double, true>), g, dim3(256), 0, cx.stream, (const float *)A,
                         (const float *)B, n1, n2, K, p.tiles, p.tiles_j, h, p.chunk, p.run, partial.as<double>());
    else
      hipLaunchKernelGGL((k_overlap_partial<float, float, false>), g, dim3(256), 0, cx.stream, (const float *)A,
                         (const float *)B, n1, n2, K, p.tiles, p.tiles_j, h, p.chunk, p.run, partial.as<float>());
  }
  INQX_HIP(hipGetLastError());
  ProfScope ps(cx, f64 ? "overlap_reduce_f64" : "overlap_reduce_f32");
  if (es == 8)
    hipLaunchKernelGGL(k_overlap_reduce<double>, gr, dim3(256), 0, cx.stream, partial.as<double>(), n1, n2, p.tiles,
                       p.tiles_j, h, p.nchunk, vol, S);
  else
    hipLaunchKernelGGL(k_overlap_reduce<float>, gr, dim3(256), 0, cx.stream, partial.as<float>(), n1, n2, p.tiles,
                       p.tiles_j, h, p.nchunk, vol, S);
  INQX_HIP(hipGetLastError());
}

void launch_rotate(Ctx &cx, int prec, int nr, int nc, long K, const double *R, int mode, double ar, double ai,
                   const void *Cm, void *Out, double br, double bi, DevMem &ops, bool lower, const int *info) {
  INQX_CHECK(mode == 1 || nr == nc, INQX_ERR_ARG, "rotate: modes 0 and 2 need a square matrix");
  INQX_CHECK(!lower || nr == nc, INQX_ERR_ARG, "rotate: a triangular matrix is square");
  const size_t es = prec == INQX_FP64 ? 8 : 4;
  const long tiles_p = (K + kMT - 1) / kMT;
  const int tiles_i = (nr + kMT - 1) / kMT;
  const int nr_pad = tiles_i * kMT, ld = (nc + 15) / 16 * 16;
  ops.ensure(2 * es * (size_t)nr_pad * ld);
  const int gprep = (int)(((size_t)nr_pad * ld + 255) / 256);
  const long grid = lower ? tiles_p : tiles_p * tiles_i;
  INQX_CHECK(grid <= INT32_MAX, INQX_ERR_ARG, "rotate: too many tiles");
  if (prec == INQX_FP64) {
    cplx<double> *M = ops.as<cplx<double>>();
    hipLaunchKernelGGL(k_rot_prep<double>, dim3(gprep), dim3(256), 0, cx.stream, R, nr, nc, mode, ar, ai, nr_pad, ld, M);
    INQX_HIP(hipGetLastError());
    ProfScope ps(cx, "rotate_mfma_f64");
    hipLaunchKernelGGL(k_rotate<double>, dim3((unsigned)grid), dim3(256), 0, cx.stream, M, ld, (const cplx<double> *)Cm,
                       nr, nc, K, (cplx<double> *)Out, br, bi, tiles_i, lower ? 1 : 0, info);
  } else {
    cplx<float> *M = ops.as<cplx<float>>();
    hipLaunchKernelGGL(k_rot_prep<float>, dim3(gprep), dim3(256), 0, cx.stream, R, nr, nc, mode, ar, ai, nr_pad, ld, M);
    INQX_HIP(hipGetLastError());
    ProfScope ps(cx, "rotate_mfma_f32");
    hipLaunchKernelGGL(k_rotate<float>, dim3((unsigned)grid), dim3(256), 0, cx.stream, M, ld, (const cplx<float> *)Cm,
                       nr, nc, K, (cplx<float> *)Out, br, bi, tiles_i, lower ? 1 : 0, info);
  }
  INQX_HIP(hipGetLastError());
}

// zero fill with vector stores (no memset node when a caller captures the stream)
__global__ void __launch_bounds__(256) k_fill_zero(V4f *p, long n16, unsigned char *tail, int ntail) {
  const long stride = (long)gridDim.x * blockDim.x;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride) p[i] = V4f{0.f, 0.f, 0.f, 0.f};
  if (blockIdx.x == 0 && (int)threadIdx.x < ntail) tail[threadIdx.x] = 0;
}

// ------------------------------------------------------------------------ overlap_diagonal
// per state: sum conj(phi1) phi2 and sum |phi2|^2 in FP64 (one work-group per
// state, fixed reduction order); out = vol * value, or value / norm
template <typename T>
__global__ void __launch_bounds__(256) k_overlap_diag(const cplx<T> *A, const cplx<T> *B, long K, double vol,
                                                     int normalized, double *out) {
  __shared__ double red[3][256];
  const int tid = threadIdx.x, s = blockIdx.x;
  const GAS cplx<T> *a = lgp(A) + (size_t)s * K;
  const GAS cplx<T> *b = lgp(B) + (size_t)s * K;
  double vr = 0.0, vi = 0.0, nn = 0.0;
  for (long p = tid; p < K; p += 256) {
    const cplx<T> x = a[p], y = b[p];
    vr += (double)x.x * y.x + (double)x.y * y.y;
    vi += (double)x.x * y.y - (double)x.y * y.x;
    nn += (double)y.x * y.x + (double)y.y * y.y;
  }
  red[0][tid] = vr;
  red[1][tid] = vi;
  red[2][tid] = nn;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (tid < w)
      for (int c = 0; c < 3; ++c) red[c][tid] += red[c][tid + w];
    __syncthreads();
  }
  if (tid == 0) {
    GAS double *o = lgw(out) + 2 * (size_t)s;
    if (normalized) {
      o[0] = red[0][0] / red[2][0];
      o[1] = red[1][0] / red[2][0];
    } else {
      o[0] = vol * red[0][0];
      o[1] = vol * red[1][0];
    }
  }
}

void launch_overlap_diagonal(Ctx &cx, int prec, int n, long K, double vol, const void *A, const void *B,
                             int normalized, double *out) {
  ProfScope ps(cx, "overlap_diagonal");
  if (prec == INQX_FP64)
    hipLaunchKernelGGL(k_overlap_diag<double>, dim3(n), dim3(256), 0, cx.stream, (const cplx<double> *)A,
                       (const cplx<double> *)B, K, vol, normalized, out);
  else
    hipLaunchKernelGGL(k_overlap_diag<float>, dim3(n), dim3(256), 0, cx.stream, (const cplx<float> *)A,
                       (const cplx<float> *)B, K, vol, normalized, out);
  INQX_HIP(hipGetLastError());
}

// ------------------------------------------------------------------------ randomize
// operations::randomize (src/operations/randomize.hpp:48-70): value (ip, ist)
// comes from pcg32 (64-bit LCG, XSH-RR output of the pre-step state) seeded
// with bump(seed + inc) and advanced by (ip nst + ist) samples (jump-ahead,
// Brown 1994); U = 2 r / 2^32 - 1, real part first
constexpr uint64_t kPcgMult = 6364136223846793005ULL;
constexpr uint64_t kPcgInc = 1442695040888963407ULL;

__device__ __forceinline__ uint64_t pcg_jump(uint64_t state, uint64_t delta) {
  uint64_t cm = kPcgMult, cp = kPcgInc, am = 1, ap = 0;
  while (delta > 0) {
    if (delta & 1) {
      am *= cm;
      ap = ap * cm + cp;
    }
    cp = (cm + 1) * cp;
    cm *= cm;
    delta >>= 1;
  }
  return am * state + ap;
}

__device__ __forceinline__ double pcg_uniform(uint64_t s) {
  const uint32_t rot = (uint32_t)(s >> 59);
  const uint32_t x = (uint32_t)(((s >> 18) ^ s) >> 27);
  const uint32_t r = (x >> rot) | (x << ((32u - rot) & 31u));
  return 2.0 * (double)r / 4294967296.0 - 1.0;
}

__global__ void __launch_bounds__(256) k_randomize(long npoints, int nst, uint64_t start, int type, int layout,
                                                   void *out) {
  const long total = npoints * nst;
  const int per = type == 2 ? 1 : 2;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (long)gridDim.x * blockDim.x) {
    const long ip = idx / nst;
    const int ist = (int)(idx - ip * nst);
    uint64_t st = pcg_jump(start, (uint64_t)idx * per);
    const double re = pcg_uniform(st);
    double im = 0.0;
    if (per == 2) im = pcg_uniform(st * kPcgMult + kPcgInc);
    const long o = layout == 0 ? (long)ist * npoints + ip : idx;
    if (type == INQX_FP64) {
      lgw((double *)out)[2 * o] = re;
      lgw((double *)out)[2 * o + 1] = im;
    } else if (type == INQX_FP32) {
      lgw((float *)out)[2 * o] = (float)re;
      lgw((float *)out)[2 * o + 1] = (float)im;
    } else {
      lgw((double *)out)[o] = re;
    }
  }
}

void launch_randomize(Ctx &cx, int type, long npoints, int nst, int index, int layout, void *out) {
  const uint64_t seed = (uint64_t)npoints * (uint64_t)nst + (uint64_t)index;
  const uint64_t start = (seed + kPcgInc) * kPcgMult + kPcgInc;
  const long total = npoints * nst;
  const int grid = (int)std::max<long>(1, std::min<long>((total + 255) / 256, (long)cx.num_cu * 32));
  ProfScope ps(cx, "randomize");
  hipLaunchKernelGGL(k_randomize, dim3(grid), dim3(256), 0, cx.stream, npoints, nst, start, type, layout, out);
  INQX_HIP(hipGetLastError());
}

void launch_fill_zero(Ctx &cx, void *p, size_t bytes) {
  if (bytes == 0) return;
  const long n16 = (long)(bytes / 16);
  const int ntail = (int)(bytes - 16 * (size_t)n16);
  const int grid = (int)std::max<long>(1, std::min<long>((n16 + 255) / 256, (long)cx.num_cu * 16));
  hipLaunchKernelGGL(k_fill_zero, dim3(grid), dim3(256), 0, cx.stream, (V4f *)p, n16,
                     (unsigned char *)p + 16 * (size_t)n16, ntail);
  INQX_HIP(hipGetLastError());
}

void launch_cholesky(Ctx &cx, int n, double *S, int *info) {
  ProfScope ps(cx, "cholesky_f64");
  const int nb = (n + kChB - 1) / kChB;
  hipLaunchKernelGGL(k_chol_first, dim3(1), dim3(256), 0, cx.stream, S, n, info);
  INQX_HIP(hipGetLastError());
  if (nb == 1) return;
  for (int b = 0; b + 1 < nb; ++b) {
    const int m = nb - 1 - b;  // tile rows of the trailing triangle
    hipLaunchKernelGGL(k_chol_step, dim3(m * (m + 1) / 2), dim3(256), 0, cx.stream, S, n, kChB * b, nb == 2 ? 1 : 0,
                       info);
    INQX_HIP(hipGetLastError());
  }
  if (nb == 2) return;
  hipLaunchKernelGGL(k_chol_finish, dim3(nb * (nb + 1) / 2), dim3(256), 0, cx.stream, S, n, (const int *)info);
  INQX_HIP(hipGetLastError());
}

void launch_stream_copy(Ctx &cx, const void *src, void *dst, size_t bytes) {
  const long n = (long)(bytes / 16);
  INQX_CHECK((n + 255) / 256 <= INT32_MAX, INQX_ERR_ARG, "stream copy too long");
  const int grid = (int)((n + 255) / 256);
  if (grid == 0) return;
  ProfScope ps(cx, "stream_copy");
  hipLaunchKernelGGL(k_stream_copy, dim3(grid), dim3(256), 0, cx.stream, (const V4f *)src, (V4f *)dst, n);
  INQX_HIP(hipGetLastError());
}

void launch_trinv(Ctx &cx, int n, const double *L, double *X, DevMem &work) {
  const int nb = (n + kChB - 1) / kChB;
  if (nb > 1) work.ensure(16 * (size_t)n * n);
  double *T = work.as<double>();
  ProfScope ps(cx, "trinv_f64");
  hipLaunchKernelGGL(k_trinv_diag, dim3(nb, nb), dim3(64), 0, cx.stream, L, n, X);
  INQX_HIP(hipGetLastError());
  for (int blk = kChB; blk < n; blk *= 2) {
    const dim3 grid(blk / kChB, blk / kChB, (n + 2 * blk - 1) / (2 * blk));
    for (int second = 0; second < 2; ++second) {
      hipLaunchKernelGGL(k_trinv_merge, grid, dim3(256), 0, cx.stream, L, n, X, T, blk, second);
      INQX_HIP(hipGetLastError());
    }
  }
}

}  // namespace inqx
