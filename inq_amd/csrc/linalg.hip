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
//             src/matrix/invert_triangular.hpp:20-50), blocked by 32x32 block rows.
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
// at most kOvRun complex values before they are added in FP64 (WIDE: chunks
// longer than that keep FP64 sums in registers and write FP64 partial tiles).
// HERM (A and B the same states): only the tiles on and below the diagonal.
// Measured, before -> now: 432 states x 228487 with themselves, complex64, 3.38 ->
// 1.87 ms (112 TFLOP/s over the products done); 128 x 67691 93 -> 67 us complex64,
// two different blocks of it in complex128 176 -> 166 us (53 of 67 TFLOP/s).
constexpr int kOvRun = 1024;        // complex values per FP32 accumulation
constexpr int kOvChunkMin = 128;    // complex values per work-group at least
constexpr int kOvChunkGood = 256;   // enough stages to hide a work-group's start and end

struct OvPlan {
  int tiles_i, tiles_j, tiles;  // tiles: all, or those on and below the diagonal
  int nchunk;
  long chunk;  // complex values, a multiple of the stage
};
// work-groups per CU in the one round: what the registers hold
static int overlap_slots(bool f64, bool wide) { return f64 || wide ? 3 : 4; }
static OvPlan overlap_plan(int n1, int n2, long K, bool herm, int cus, bool f64) {
  OvPlan p;
  p.tiles_i = (n1 + kMT - 1) / kMT;
  p.tiles_j = (n2 + kMT - 1) / kMT;
  p.tiles = herm ? p.tiles_i * (p.tiles_i + 1) / 2 : p.tiles_i * p.tiles_j;
  const int stage = f64 ? kStage<double> : kStage<float>;
  for (int m = 4; m >= 1; --m) {
    const long want = std::max<long>(1, (long)m * cus / p.tiles);
    if (m > overlap_slots(f64, K > want * kOvRun)) continue;
    long c = std::max<long>((K + want - 1) / want, kOvChunkMin);
    p.chunk = (c + stage - 1) / stage * stage;
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
                                                         int tiles_j, int herm, long chunk, P *partial) {
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
  int buf = 0, run = 0;
  if (k0 < kw) {
    load(k0);
    store(0);
    __syncthreads();
  }
  for (long k = k0; k < kw; k += KC) {
    const bool more = k + KC < kw;
    if (more) load(k + KC);
    mac(buf);
    if (WIDE && (run += KC) >= kOvRun) {
      run = 0;
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
// Blocked in 32-wide panels, one launch per step so that every read of a value
// another work-group wrote happens in a later launch.
//
// Cholesky S = L L^H in place (lower; the strict upper triangle is zeroed), per panel c0:
//   k_chol_diag    factor the diagonal block (already updated by earlier panels) in LDS
//   k_chol_panel   rows below: L[i][c0+j] = (S[i][c0+j] - sum_{k<j} L[i][c0+k] conj(L_dd[j][k])) / L_dd[j][j]
//   k_chol_update  S[i][j] -= sum_k L[i][c0+k] conj(L[j][c0+k]) on the lower trailing matrix
// info[0] = 0 or the first non-positive leading minor (LAPACK convention); the first
// diagonal launch writes it, and every later launch returns at once when it is set.
constexpr int kChB = 32;

// right-looking in LDS with one barrier per column: every lane reads the same pivot d,
// column j (scaled by 1/sqrt(d)) goes straight to S, and the lanes update the lower
// block right of column j from the unscaled column (column j is not written in step j)
__global__ void __launch_bounds__(256) k_chol_diag(double *S, int n, int c0, int *info) {
  __shared__ double Dr[kChB][kChB + 1], Di[kChB][kChB + 1];
  const int tid = threadIdx.x;
  if (c0 > 0 && info[0] != 0) return;
  const int b = min(kChB, n - c0);
  for (int e = tid; e < kChB * kChB; e += 256) {
    const int i = e / kChB, j = e - i * kChB;
    double vr = 0.0, vi = 0.0;
    if (i < b && j <= i) {
      vr = S[2 * ((long)(c0 + i) * n + c0 + j)];
      vi = S[2 * ((long)(c0 + i) * n + c0 + j) + 1];
    }
    Dr[i][j] = vr;
    Di[i][j] = vi;
  }
  __syncthreads();
  int bad = 0;
  for (int j = 0; j < b; ++j) {
    const double d = Dr[j][j];
    if (!(d > 0.0)) {
      bad = c0 + j + 1;
      break;
    }
    const double ljj = sqrt(d), rl = 1.0 / ljj;
    if (tid < b - j) {
      const int i = j + tid;
      const long o = 2 * ((long)(c0 + i) * n + c0 + j);
      S[o] = tid == 0 ? ljj : Dr[i][j] * rl;
      S[o + 1] = tid == 0 ? 0.0 : Di[i][j] * rl;
    }
    const double rd = rl * rl;  // L[i][j] conj(L[k][j]) = D[i][j] conj(D[k][j]) / d
#pragma unroll
    for (int e = tid; e < kChB * kChB; e += 256) {
      const int i = e / kChB, k = e - i * kChB;
      if (k > j && k <= i && i < b) {
        const double ar = Dr[i][j] * rd, ai = Di[i][j] * rd, br = Dr[k][j], bi = Di[k][j];
        Dr[i][k] -= ar * br + ai * bi;
        Di[i][k] -= ai * br - ar * bi;
      }
    }
    __syncthreads();
  }
  if (bad) {
    if (tid == 0) info[0] = bad;
    return;
  }
  if (c0 == 0 && tid == 0) info[0] = 0;
  for (int e = tid; e < b * b; e += 256) {  // upper part of the diagonal block
    const int i = e / b, j = e - i * b;
    if (j > i) {
      S[2 * ((long)(c0 + i) * n + c0 + j)] = 0.0;
      S[2 * ((long)(c0 + i) * n + c0 + j) + 1] = 0.0;
    }
  }
  // rows of this panel right of the diagonal block are upper triangle: zero
  const int w = n - c0 - b;
  for (int e = tid; e < b * w; e += 256) {
    const int i = e / w, j = e - i * w;
    S[2 * ((long)(c0 + i) * n + c0 + b + j)] = 0.0;
    S[2 * ((long)(c0 + i) * n + c0 + b + j) + 1] = 0.0;
  }
}

// n <= kCholSmall: the whole factorisation in one work-group, the lower triangle
// packed in LDS (row i at i(i+1)/2, n(n+1)/2 x 16 bytes <= 132 KB).  Right-looking
// with one barrier per column: the lanes update the trailing lower triangle from
// the unscaled column j, then, after the barrier, scale column j while the next
// column's update (which reads column j + 1 and writes columns > j + 1) runs.
constexpr int kCholSmall = 128;
__global__ void __launch_bounds__(1024) k_chol_small(double *S, int n, int *info) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double2 *T = reinterpret_cast<double2 *>(smem_raw);
  const int tid = threadIdx.x, ty = tid >> 5, tx = tid & 31;
  for (int i = ty; i < n; i += 32)
    for (int k = tx; k <= i; k += 32) T[i * (i + 1) / 2 + k] = double2{S[2 * ((long)i * n + k)], S[2 * ((long)i * n + k) + 1]};
  __syncthreads();
  int bad = 0;
  for (int j = 0; j < n; ++j) {
    const double d = T[j * (j + 1) / 2 + j].x;
    if (!(d > 0.0)) {
      bad = j + 1;
      break;
    }
    const double rd = 1.0 / d;
    for (int i = j + 1 + ty; i < n; i += 32) {
      const double2 a = T[i * (i + 1) / 2 + j];
      const double ar = a.x * rd, ai = a.y * rd;
      for (int k = j + 1 + tx; k <= i; k += 32) {  // L[i][j] conj(L[k][j]) = D[i][j] conj(D[k][j]) / d
        const double2 b = T[k * (k + 1) / 2 + j];
        double2 &t = T[i * (i + 1) / 2 + k];
        t.x -= ar * b.x + ai * b.y;
        t.y -= ai * b.x - ar * b.y;
      }
    }
    __syncthreads();
    if (tid < n - j) {
      const int i = j + tid;
      double2 &c = T[i * (i + 1) / 2 + j];
      const double ljj = sqrt(d);
      if (tid == 0) {
        c = double2{ljj, 0.0};
      } else {
        const double rl = 1.0 / ljj;
        c.x *= rl;
        c.y *= rl;
      }
    }
  }
  __syncthreads();
  if (tid == 0) info[0] = bad;
  if (bad) return;
  for (int e = tid; e < n * n; e += 1024) {
    const int i = e / n, k = e - i * n;
    const double2 v = k <= i ? T[i * (i + 1) / 2 + k] : double2{0.0, 0.0};
    S[2 * (long)e] = v.x;
    S[2 * (long)e + 1] = v.y;
  }
}

// one lane per row i >= c0 + 32 (launched only when such rows exist, so the panel is 32 wide)
__global__ void __launch_bounds__(256) k_chol_panel(double *S, int n, int c0, const int *info) {
  __shared__ double Lr[kChB][kChB + 1], Li[kChB][kChB + 1], rdiag[kChB];
  if (info[0] != 0) return;
  for (int e = threadIdx.x; e < kChB * kChB; e += 256) {
    const int i = e / kChB, j = e - i * kChB;
    Lr[i][j] = j <= i ? S[2 * ((long)(c0 + i) * n + c0 + j)] : 0.0;
    Li[i][j] = j <= i ? S[2 * ((long)(c0 + i) * n + c0 + j) + 1] : 0.0;
  }
  if (threadIdx.x < kChB) rdiag[threadIdx.x] = 1.0 / S[2 * ((long)(c0 + threadIdx.x) * n + c0 + threadIdx.x)];
  __syncthreads();
  const int i = c0 + kChB + blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  double *row = S + 2 * ((long)i * n + c0);
  double xr[kChB], xi[kChB];
#pragma unroll
  for (int j = 0; j < kChB; ++j) {
    xr[j] = row[2 * j];
    xi[j] = row[2 * j + 1];
  }
  // right-looking: once x_j is final, x_m -= x_j conj(L_dd[m][j]) for every m > j
  // (independent updates, short dependency chains)
#pragma unroll
  for (int j = 0; j < kChB; ++j) {
    xr[j] *= rdiag[j];
    xi[j] *= rdiag[j];
#pragma unroll
    for (int m = j + 1; m < kChB; ++m) {
      xr[m] -= xr[j] * Lr[m][j] + xi[j] * Li[m][j];
      xi[m] -= xi[j] * Lr[m][j] - xr[j] * Li[m][j];
    }
  }
#pragma unroll
  for (int j = 0; j < kChB; ++j) {
    row[2 * j] = xr[j];
    row[2 * j + 1] = xi[j];
  }
}

// 32x32 output tile (ti, tj), tj <= ti, of the trailing matrix starting at c0 + 32;
// lane: row tid / 8, columns tid % 8 + 8 q
__global__ void __launch_bounds__(256) k_chol_update(double *S, int n, int c0, const int *info) {
  __shared__ double Ar[kChB][kChB + 1], Ai[kChB][kChB + 1], Br[kChB][kChB + 1], Bi[kChB][kChB + 1];
  const int ti = blockIdx.y, tj = blockIdx.x;
  if (tj > ti || info[0] != 0) return;
  const int r0 = c0 + kChB, i0 = r0 + ti * kChB, j0 = r0 + tj * kChB;
  for (int e = threadIdx.x; e < kChB * kChB; e += 256) {
    const int r = e / kChB, k = e - r * kChB;
    const bool ia = i0 + r < n, jb = j0 + r < n;
    Ar[r][k] = ia ? S[2 * ((long)(i0 + r) * n + c0 + k)] : 0.0;
    Ai[r][k] = ia ? S[2 * ((long)(i0 + r) * n + c0 + k) + 1] : 0.0;
    Br[r][k] = jb ? S[2 * ((long)(j0 + r) * n + c0 + k)] : 0.0;
    Bi[r][k] = jb ? S[2 * ((long)(j0 + r) * n + c0 + k) + 1] : 0.0;
  }
  __syncthreads();
  const int r = threadIdx.x >> 3, cb = threadIdx.x & 7, i = i0 + r;
  double sr[4] = {0, 0, 0, 0}, si[4] = {0, 0, 0, 0};
#pragma unroll 8
  for (int k = 0; k < kChB; ++k) {  // A[r][k] conj(B[c][k]); out-of-range rows are zero
    const double ar = Ar[r][k], ai = Ai[r][k];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = cb + 8 * q;
      sr[q] += ar * Br[c][k] + ai * Bi[c][k];
      si[q] += ai * Br[c][k] - ar * Bi[c][k];
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int j = j0 + cb + 8 * q;
    if (i < n && j <= i) {
      S[2 * ((long)i * n + j)] -= sr[q];
      S[2 * ((long)i * n + j) + 1] -= si[q];
    }
  }
}

// X = L^{-1} for lower-triangular L (complex double), blocked in 32x32 blocks:
//   k_trinv_diag  X_bb = L_bb^{-1} (one lane per column, forward substitution in LDS),
//                 blocks above the diagonal zeroed
//   k_trinv_row   block row r, one work-group per block column jb < r:
//                 X_r,jb = -X_rr sum_{k=jb}^{r-1} L_rk X_k,jb  (every X read was written
//                 by an earlier launch)
__global__ void __launch_bounds__(256) k_trinv_diag(const double *L, int n, double *X) {
  __shared__ double Lr[kChB][kChB + 1], Li[kChB][kChB + 1], Xr[kChB][kChB + 1], Xi[kChB][kChB + 1];
  const int bi = blockIdx.y, bj = blockIdx.x, tid = threadIdx.x;
  const int r0 = bi * kChB, q0 = bj * kChB;
  const int b = min(kChB, n - r0), bc = min(kChB, n - q0);
  if (bj > bi) {
    for (int e = tid; e < b * bc; e += 256) {
      const int i = e / bc, j = e - i * bc;
      X[2 * ((long)(r0 + i) * n + q0 + j)] = 0.0;
      X[2 * ((long)(r0 + i) * n + q0 + j) + 1] = 0.0;
    }
    return;
  }
  if (bj < bi) return;
  for (int e = tid; e < kChB * kChB; e += 256) {
    const int i = e / kChB, j = e - i * kChB;
    const bool in = i < b && j <= i;
    Lr[i][j] = in ? L[2 * ((long)(r0 + i) * n + r0 + j)] : 0.0;
    Li[i][j] = in ? L[2 * ((long)(r0 + i) * n + r0 + j) + 1] : 0.0;
    Xr[i][j] = 0.0;
    Xi[i][j] = 0.0;
  }
  __shared__ double Ir[kChB], Ii[kChB];  // 1 / L[i][i]
  if (tid < b) {
    const double lr = L[2 * ((long)(r0 + tid) * n + r0 + tid)], li = L[2 * ((long)(r0 + tid) * n + r0 + tid) + 1];
    const double rd = 1.0 / (lr * lr + li * li);
    Ir[tid] = lr * rd;
    Ii[tid] = -li * rd;
  }
  __syncthreads();
  const int c = tid;
  if (c < b) {
    Xr[c][c] = Ir[c];
    Xi[c][c] = Ii[c];
    for (int i = c + 1; i < b; ++i) {
      double sr = 0.0, si = 0.0;
      for (int k = c; k < i; ++k) {
        sr += Lr[i][k] * Xr[k][c] - Li[i][k] * Xi[k][c];
        si += Lr[i][k] * Xi[k][c] + Li[i][k] * Xr[k][c];
      }
      Xr[i][c] = -(sr * Ir[i] - si * Ii[i]);  // -(s / l)
      Xi[i][c] = -(sr * Ii[i] + si * Ir[i]);
    }
  }
  __syncthreads();
  for (int e = tid; e < b * b; e += 256) {
    const int i = e / b, j = e - i * b;
    X[2 * ((long)(r0 + i) * n + r0 + j)] = Xr[i][j];
    X[2 * ((long)(r0 + i) * n + r0 + j) + 1] = Xi[i][j];
  }
}

__global__ void __launch_bounds__(256) k_trinv_row(const double *L, int n, int r, double *X) {
  __shared__ double Ar[kChB][kChB + 1], Ai[kChB][kChB + 1], Br[kChB][kChB + 1], Bi[kChB][kChB + 1];
  const int jb = blockIdx.x, tid = threadIdx.x;
  const int r0 = r * kChB, q0 = jb * kChB;
  const int row = tid >> 3, cb = tid & 7;
  double tr[4] = {0, 0, 0, 0}, tim[4] = {0, 0, 0, 0};
  // the next k block's L and X values are loaded into registers during the products
  double par[4], pai[4], pbr[4], pbi[4];
  auto fetch = [&](int k) {
    const int k0 = k * kChB;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = tid + 256 * u, a = e / kChB, m = e - a * kChB;
      const bool la = r0 + a < n && k0 + m < n, xb = k0 + a < n && q0 + m < n;
      par[u] = la ? L[2 * ((long)(r0 + a) * n + k0 + m)] : 0.0;
      pai[u] = la ? L[2 * ((long)(r0 + a) * n + k0 + m) + 1] : 0.0;
      pbr[u] = xb ? X[2 * ((long)(k0 + a) * n + q0 + m)] : 0.0;
      pbi[u] = xb ? X[2 * ((long)(k0 + a) * n + q0 + m) + 1] : 0.0;
    }
  };
  fetch(jb);
  for (int k = jb; k < r; ++k) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = tid + 256 * u, a = e / kChB, m = e - a * kChB;
      Ar[a][m] = par[u];
      Ai[a][m] = pai[u];
      Br[a][m] = pbr[u];
      Bi[a][m] = pbi[u];
    }
    __syncthreads();
    if (k + 1 < r) fetch(k + 1);
#pragma unroll 8
    for (int m = 0; m < kChB; ++m) {
      const double ar = Ar[row][m], ai = Ai[row][m];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int c = cb + 8 * q;
        tr[q] += ar * Br[m][c] - ai * Bi[m][c];
        tim[q] += ar * Bi[m][c] + ai * Br[m][c];
      }
    }
    __syncthreads();
  }
  // Y = -X_rr T: T to LDS (B), X_rr to LDS (A)
  for (int e = tid; e < kChB * kChB; e += 256) {
    const int a = e / kChB, m = e - a * kChB;
    const bool xa = r0 + a < n && r0 + m < n;
    Ar[a][m] = xa ? X[2 * ((long)(r0 + a) * n + r0 + m)] : 0.0;
    Ai[a][m] = xa ? X[2 * ((long)(r0 + a) * n + r0 + m) + 1] : 0.0;
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    Br[row][cb + 8 * q] = tr[q];
    Bi[row][cb + 8 * q] = tim[q];
  }
  __syncthreads();
  double yr[4] = {0, 0, 0, 0}, yi[4] = {0, 0, 0, 0};
#pragma unroll 8
  for (int m = 0; m < kChB; ++m) {
    const double ar = Ar[row][m], ai = Ai[row][m];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = cb + 8 * q;
      yr[q] += ar * Br[m][c] - ai * Bi[m][c];
      yi[q] += ar * Bi[m][c] + ai * Br[m][c];
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int c = cb + 8 * q;
    if (r0 + row < n && q0 + c < n) {
      X[2 * ((long)(r0 + row) * n + q0 + c)] = -yr[q];
      X[2 * ((long)(r0 + row) * n + q0 + c) + 1] = -yi[q];
    }
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
  const bool wide = !f64 && p.chunk > kOvRun;  // FP64 partial tiles of FP32 products
  const size_t es = f64 || wide ? 8 : 4;
  partial.ensure(es * (size_t)p.nchunk * p.tiles * kMT * kMT * 2);
  const long grid = (long)p.nchunk * p.tiles;
  INQX_CHECK(grid <= INT32_MAX / kMT, INQX_ERR_ARG, "overlap: too many tiles");
  const dim3 g((unsigned)grid), gr((unsigned)(p.tiles * kMT));
  const int h = herm ? 1 : 0;
  {
    ProfScope ps(cx, f64 ? "overlap_mfma_f64" : "overlap_mfma_f32");
    if (f64)
      hipLaunchKernelGGL((k_overlap_partial<double, double, false>), g, dim3(256), 0, cx.stream, (const double *)A,
                         (const double *)B, n1, n2, K, p.tiles, p.tiles_j, h, p.chunk, partial.as<double>());
    else if (wide)
      hipLaunchKernelGGL((k_overlap_partial<float, double, true>), g, dim3(256), 0, cx.stream, (const float *)A,
                         (const float *)B, n1, n2, K, p.tiles, p.tiles_j, h, p.chunk, partial.as<double>());
    else
      hipLaunchKernelGGL((k_overlap_partial<float, float, false>), g, dim3(256), 0, cx.stream, (const float *)A,
                         (const float *)B, n1, n2, K, p.tiles, p.tiles_j, h, p.chunk, partial.as<float>());
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

// ------------------------------------------------------------------------ density
// density[p][ncomp] (component ispin) += sum_i occ_i |phi_i(p)|^2, states
// state-major [nst][N]; FP64, states summed in order
template <typename T>
__global__ void __launch_bounds__(256) k_density_add(const cplx<T> *phi, const double *occ, int nst, long N,
                                                    int ncomp, int ispin, double *den) {
  for (long p = (long)blockIdx.x * blockDim.x + threadIdx.x; p < N; p += (long)gridDim.x * blockDim.x) {
    double acc = 0.0;
    for (int i = 0; i < nst; ++i) {
      const cplx<T> v = lgp(phi)[(size_t)i * N + p];
      acc += lgp(occ)[i] * ((double)v.x * v.x + (double)v.y * v.y);
    }
    lgw(den)[p * ncomp + ispin] += acc;
  }
}

void launch_density_add(Ctx &cx, int prec, const void *phi, const double *occ, int nst, long N, int ncomp,
                        int ispin, double *den) {
  const int grid = (int)std::max<long>(1, std::min<long>((N + 255) / 256, (long)cx.num_cu * 16));
  ProfScope ps(cx, "density_add");
  if (prec == INQX_FP64)
    hipLaunchKernelGGL(k_density_add<double>, dim3(grid), dim3(256), 0, cx.stream, (const cplx<double> *)phi, occ,
                       nst, N, ncomp, ispin, den);
  else
    hipLaunchKernelGGL(k_density_add<float>, dim3(grid), dim3(256), 0, cx.stream, (const cplx<float> *)phi, occ,
                       nst, N, ncomp, ispin, den);
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
  if (n <= kCholSmall) {
    const size_t lds = sizeof(double2) * (size_t)n * (n + 1) / 2;
    static DeviceOnce attr;
    if (!attr.test_and_set(cx.device))
      INQX_HIP(hipFuncSetAttribute((const void *)k_chol_small, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)(sizeof(double2) * kCholSmall * (kCholSmall + 1) / 2)));
    hipLaunchKernelGGL(k_chol_small, dim3(1), dim3(1024), lds, cx.stream, S, n, info);
    INQX_HIP(hipGetLastError());
    return;
  }
  for (int c0 = 0; c0 < n; c0 += kChB) {
    hipLaunchKernelGGL(k_chol_diag, dim3(1), dim3(256), 0, cx.stream, S, n, c0, info);
    INQX_HIP(hipGetLastError());
    const int rest = n - c0 - kChB;
    if (rest <= 0) break;
    hipLaunchKernelGGL(k_chol_panel, dim3((rest + 255) / 256), dim3(256), 0, cx.stream, S, n, c0, (const int *)info);
    INQX_HIP(hipGetLastError());
    const int m = (rest + kChB - 1) / kChB;
    hipLaunchKernelGGL(k_chol_update, dim3(m, m), dim3(256), 0, cx.stream, S, n, c0, (const int *)info);
    INQX_HIP(hipGetLastError());
  }
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

void launch_trinv(Ctx &cx, int n, const double *L, double *X) {
  ProfScope ps(cx, "trinv_f64");
  const int nb = (n + kChB - 1) / kChB;
  hipLaunchKernelGGL(k_trinv_diag, dim3(nb, nb), dim3(256), 0, cx.stream, L, n, X);
  INQX_HIP(hipGetLastError());
  for (int r = 1; r < nb; ++r) {
    hipLaunchKernelGGL(k_trinv_row, dim3(r), dim3(256), 0, cx.stream, L, n, r, X);
    INQX_HIP(hipGetLastError());
  }
}

}  // namespace inqx
