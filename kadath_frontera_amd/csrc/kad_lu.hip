// Dense LU with partial pivoting + solves + mixed-precision refinement, single MI355X.
//
// Replaces the ScaLAPACK solve of System_of_eqs::do_newton
// (reference src_par/do_newton.cpp:317-320, pdgesv_) and the single-process
// LAPACK path (src/Matrice/matrice.cpp:192-250, dgetrf_/dgetrs_).
//
// Layout: the n x n Jacobian is column-major with leading dimension lda (the
// reference packs J_in column-major before pdgemr2d/pdgesv, do_newton.cpp:178-185).
// Pivots are 0-based global row indices, LAPACK semantics: at step i row i was
// interchanged with row ipiv[i] (ipiv[i] >= i).
//
// Factorisation: right-looking, outer panel width NB; each panel is factored by
// a recursive split (LAPACK getrf2 style) whose base is a per-column kernel that
// performs exact partial pivoting (first index of max |a|, as idamax) and whose
// internal updates are MFMA GEMMs.  The trailing update A22 -= L21 U12 is the
// MFMA GEMM of kad_gemm.hip in the factor precision (f64, f32, or bf16 operands
// with f32 accumulation).  U12 = L11^{-1} A12 is a blocked substitution,
// one launch per 256 rows.  Trailing-update
// tile pairs whose L21 row tile or U12 column tile is exactly zero are skipped
// (structural zeros of a block-sparse Jacobian); the result is unchanged.
#include "kad_common.hpp"
#include "kad_ctx.hpp"
#include "kad_lanes.hpp"
#include <vector>
#include <cmath>
#include <algorithm>

namespace kad {

int gemm_launch(int prec, int op, int m, int n, int k, const void* A, int64_t lda, const void* B, int64_t ldb, void* C,
                int64_t ldc, hipStream_t s);
int gemm_launch_masked(int prec, int op, int m, int n, int k, const void* A, int64_t lda, const void* B, int64_t ldb,
                       void* C, int64_t ldc, const int* rmask, const int* cmask, hipStream_t s);
int gemm_launch_sel(int prec, int op, int m, int n, int k, const void* A, int64_t lda, const void* B, int64_t ldb,
                    void* C, int64_t ldc, const TileSel& sel, hipStream_t s);
int gemm_launch_batched(int prec, int op, int m, int n, int k, const void* A, int64_t lda, int64_t sa, const void* B,
                        int64_t ldb, int64_t sb, void* C, int64_t ldc, int64_t sc, int nbat, hipStream_t s);
constexpr int GOP_SUB = 0, GOP_SET = 1;

constexpr int PANEL_BASE = 32;  // columns factored by the per-column kernel

// An argument error of the factorisation or its solves, with its reason on stderr.
inline int arg_error(const char* why) {
  std::fprintf(stderr, "[kadath_amd] %s\n", why);
  return KAD_ERR_ARG;
}

// |a| as the pivot search compares it, as idamax does: a NaN is passed over (it takes the
// least value, and no row comes before row j), except in row j itself, where the search
// starts and no later entry exceeds it.
__device__ __forceinline__ double pivot_abs(double a, bool row_j) {
  return a == a ? fabs(a) : (row_j ? (double)INFINITY : 0.0);
}

// Block-wide (max |a|, first index) reduction.
template <typename T>
__device__ void block_argmax(double v, int idx, double* sv, int* si, double& bv, int& bi) {
  const int tid = threadIdx.x;
  sv[tid] = v;
  si[tid] = idx;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (tid < s) {
      const double ov = sv[tid + s];
      const int oi = si[tid + s];
      if (ov > sv[tid] || (ov == sv[tid] && oi < si[tid] && oi >= 0) || si[tid] < 0) {
        if (oi >= 0) {
          sv[tid] = ov;
          si[tid] = oi;
        }
      }
    }
    __syncthreads();
  }
  bv = sv[0];
  bi = si[0];
}

// Row interchanges of pivots [k1, k2) applied to columns [c0, c1): one thread per column.
template <typename T>
__global__ void laswp_kernel(T* A, int64_t lda, int c0, int c1, const int* __restrict__ ipiv, int k1, int k2,
                             int64_t sA, int sP) {
  A += (int64_t)blockIdx.y * sA;  // matrix blockIdx.y of a batch
  ipiv += (int64_t)blockIdx.y * sP;
  const int c = c0 + blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= c1) return;
  T* col = A + (int64_t)c * lda;
  for (int i = k1; i < k2; ++i) {
    const int p = ipiv[i];
    if (p != i) {
      const T t = col[i];
      col[i] = col[p];
      col[p] = t;
    }
  }
}

template <typename T>
__global__ void copy2d_kernel(const T* src, int64_t lds, T* dst, int64_t ldd, int m, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int c = blockIdx.y;
  if (i < m && c < n) dst[i + (int64_t)c * ldd] = src[i + (int64_t)c * lds];
}

template <typename T> constexpr int prec_of() { return sizeof(T) == 8 ? F64 : F32; }

// Structural-zero masks of the trailing update: per 128-row tile of the L panel
// (rows x ncols) and per 128-column tile of the U row panel (nrows x cols): 1 if the
// tile holds any entry != 0 (NaN counts as nonzero), else 0.
// 1024 threads and 8 loads in flight each: a tile's 256 columns are 4 round trips to
// memory (128 dependent ones took 36 us).
template <typename T>
__global__ __launch_bounds__(1024) void row_tile_mask_kernel(const T* __restrict__ A, int64_t lda, int nrows,
                                                             int ncols, int* __restrict__ mask, int nzrows = -1) {
  // rows at or past nzrows (when given) are known to be zero: those tiles are not read
  if (nzrows >= 0 && (int)blockIdx.x * 128 >= nzrows) {
    if (threadIdx.x == 0) mask[blockIdx.x] = 0;
    return;
  }
  const int r = blockIdx.x * 128 + (threadIdx.x & 127);
  int any = 0;
  if (r < nrows)
    for (int c0 = threadIdx.x >> 7; c0 < ncols; c0 += 64) {
      T v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = c0 + 8 * u < ncols ? A[r + (int64_t)(c0 + 8 * u) * lda] : T(0);
#pragma unroll
      for (int u = 0; u < 8; ++u) any |= v[u] != T(0);
    }
  any = __syncthreads_or(any);
  if (threadIdx.x == 0) mask[blockIdx.x] = any;
}
// Last nonzero row of each 128-column tile: out[tile] = max over the 256-row chunks
// (workgroup (tile, chunk)); -1 where there is none, with several chunks only if out starts
// there.  A chunk is read from its end, 32 rows at
// a time, until a nonzero is met, so a dense matrix costs one step of it (a full scan
// took 180 us at n = 1215, 470 at 8191).
template <typename T>
__global__ __launch_bounds__(256) void col_extent_kernel(const T* __restrict__ A, int64_t lda, int n,
                                                         int* __restrict__ out) {
  const int c0 = blockIdx.x * 128, r0 = blockIdx.y * 256;
  const int ce = min(c0 + 128, n), re = min(r0 + 256, n);
  const int tr = threadIdx.x & 31, tc = threadIdx.x >> 5;  // row within a step, one of 8 column groups
  if (gridDim.y == 1) {
    if (threadIdx.x == 0) out[blockIdx.x] = -1;
    __syncthreads();
  }
  for (int rb = r0 + (re - r0 - 1) / 32 * 32; rb >= r0; rb -= 32) {
    const int r = rb + tr;
    int any = 0;
    if (r < re) {
      T v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = c0 + tc + 8 * u < ce ? A[r + (int64_t)(c0 + tc + 8 * u) * lda] : T(0);
#pragma unroll
      for (int u = 0; u < 16; ++u) any |= v[u] != T(0);
    }
    if (any) atomicMax(&out[blockIdx.x], r);
    if (__syncthreads_or(any)) return;
  }
}

// Compacted lists of the active row / column tiles: list[0..) rows, list[stride..)
// columns, list[2 stride] and list[2 stride + 1] their counts.  One thread (a few
// hundred tiles).
__global__ void tile_lists_kernel(const int* __restrict__ rmask, int nr, const int* __restrict__ cmask, int nc,
                                  int* __restrict__ list, int stride) {
  if (blockIdx.x != 0 || threadIdx.x != 0) return;
  int a = 0, b = 0;
  for (int i = 0; i < nr; ++i)
    if (rmask[i]) list[a++] = i;
  for (int j = 0; j < nc; ++j)
    if (cmask[j]) list[stride + b++] = j;
  list[2 * stride] = a;
  list[2 * stride + 1] = b;
}

template <typename T>
__global__ __launch_bounds__(1024) void col_tile_mask_kernel(const T* __restrict__ A, int64_t lda, int nrows,
                                                             int ncols, int* __restrict__ mask) {
  const int c0 = blockIdx.x * 128 + (threadIdx.x >> 8);
  const int ce = min((int)blockIdx.x * 128 + 128, ncols);
  int any = 0;
  for (int r = threadIdx.x & 255; r < nrows; r += 256)
    for (int c = c0; c < ce; c += 32) {
      T v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = c + 4 * u < ce ? A[r + (int64_t)(c + 4 * u) * lda] : T(0);
#pragma unroll
      for (int u = 0; u < 8; ++u) any |= v[u] != T(0);
    }
  any = __syncthreads_or(any);
  if (threadIdx.x == 0) mask[blockIdx.x] = any;
}

// Where a batch's right-hand sides are known to be zero (a batch of sparse right-hand
// sides such as unit vectors); the solves skip that work, whose results would be zero.
struct ZeroRhs {
  const int* cols = nullptr;   // device, nbat entries: system z is zero past column cols[z]
  const int* start = nullptr;  // device, nbat x ng: group g (columns 64g .. 64g+63) of system z
                               // is zero above row start[z ng + g] (lower solves only)
  int ng = 0;
  int row0 = 0;  // the sub-system's first row in the full system (rows of start)
};

// Triangular solves of up to 256 rows in one launch: L X = B (unit lower) or, UP, U X = B
// (non-unit upper), in place, 16 columns of B per workgroup, held in LDS.
// The rows are taken 32 at a time (from the last for UP):
// - substitution with the 32 x 32 diagonal block, in LAPACK xTRSM's order of operations:
//   a column of B is spread over the 16 lanes of a DPP row, two rows per lane (reversed
//   for UP), and the solved entry of each step reaches the other lanes by a row
//   broadcast, so a step is one broadcast and two multiply-adds (and a division for UP);
// - the rows not yet solved subtract the block's product with the matrix cores (16 x 16
//   tiles, k = 32), whose operands were loaded before the substitution.
// Bound by latency, not by arithmetic: it replaces 8 launches of a 32-row leaf (a lane
// per column, 15-20 us each) and 7 products between them (10-13 us) per 256 rows, which
// were on the panel's critical path.  One launch takes 13 us inside the panels of n = 1215;
// with it that LU went from 9.3 to 7.7 ms, n = 8191 from 67 to 57.
constexpr int TRB = 32;          // rows per step
constexpr int TRSM_ROWS = 256;   // most rows of one launch
constexpr int TRSM_COLS = 16;    // columns per workgroup

template <typename T>
struct Mfma16;  // 16 x 16 x 4 tile: register r of lane l holds row(l, r), column l % 16
template <>
struct Mfma16<double> {
  typedef d4v V;
  static __device__ __forceinline__ V mul(double a, double b, V c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * r + (lane >> 4); }
};
template <>
struct Mfma16<float> {
  typedef f4v V;
  static __device__ __forceinline__ V mul(float a, float b, V c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};

// Steps K .. 31 of the substitution: lane g of a row holds rows 2g and 2g + 1 (y0, y1).
template <typename T, bool UP, int K>
__device__ __forceinline__ void trsm_steps(T& y0, T& y1, const T* __restrict__ Ls, const T* __restrict__ ds, int g) {
  const T l0 = Ls[K * TRB + 2 * g], l1 = Ls[K * TRB + 2 * g + 1];
  T q = (K & 1) ? y1 : y0;
  if constexpr (UP) {
    q = q / ds[K];
    if (g == K / 2) ((K & 1) ? y1 : y0) = q;
  }
  const T x = lane16<K / 2>(q);
  y0 = 2 * g > K ? y0 - l0 * x : y0;
  y1 = 2 * g + 1 > K ? y1 - l1 * x : y1;
  if constexpr (K + 1 < TRB) trsm_steps<T, UP, K + 1>(y0, y1, Ls, ds, g);
}

// r <= 256 rows (UP: a multiple of 32); system blockIdx.y of a batch.  cmask (optional):
// 128-column tiles of B that are structurally zero stay untouched; zr: as ZeroRhs.
template <typename T, bool UP>
__global__ __launch_bounds__(256) void trsm_block_kernel(const T* __restrict__ L, int64_t lda, T* __restrict__ B,
                                                         int64_t ldb, int r, int ncols, const int* __restrict__ cmask,
                                                         int64_t sL, int64_t sB, ZeroRhs zr) {
  constexpr int LD = TRSM_ROWS + 2;  // 16 columns x 4 words apart: conflict-free tile reads
  __shared__ __align__(16) T X[TRSM_COLS * LD];
  __shared__ __align__(16) T Ls[TRB * TRB];
  __shared__ T ds[TRB];
  const int c0 = blockIdx.x * TRSM_COLS;
  if (cmask && !cmask[c0 / 128]) return;
  if (zr.cols && c0 >= zr.cols[blockIdx.y]) return;
  if (zr.start && zr.start[(int)blockIdx.y * zr.ng + c0 / 64] >= zr.row0 + r) return;
  __builtin_amdgcn_s_setprio(2);  // on the critical path, beside the bulk GEMM
  L += (int64_t)blockIdx.y * sL;
  B += (int64_t)blockIdx.y * sB;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, lk = lane >> 4;
  const int nbk = (r + TRB - 1) / TRB;
  // 32 x 32 diagonal block of step `it`: column-major, rows and columns reversed for UP;
  // only the part below the diagonal is used, and the diagonal (UP)
  auto diag = [&](int it, T (&v)[4]) {
    const int o = (UP ? nbk - 1 - it : it) * TRB;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = u * 256 + tid;
      const int i = UP ? TRB - 1 - e % TRB : e % TRB, k = UP ? TRB - 1 - e / TRB : e / TRB;
      v[u] = (o + i < r && o + k < r) ? L[(o + i) + (int64_t)(o + k) * lda] : T(0);
    }
  };
  T lv[4];
  diag(0, lv);
  {
    T v[TRSM_COLS];
#pragma unroll
    for (int c = 0; c < TRSM_COLS; ++c)
      v[c] = (tid < r && c0 + c < ncols) ? B[tid + (int64_t)(c0 + c) * ldb] : T(0);
#pragma unroll
    for (int c = 0; c < TRSM_COLS; ++c) X[c * LD + tid] = v[c];
  }
  for (int it = 0; it < nbk; ++it) {
    const int kb = UP ? nbk - 1 - it : it;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = u * 256 + tid;
      Ls[e] = lv[u];
      if (e % TRB == e / TRB) ds[e % TRB] = lv[u];
    }
    // this wave's 16-row tiles of the update and their operands
    const int t0 = (UP ? 0 : 2 * (kb + 1)) + wave, t1 = UP ? 2 * kb : 2 * nbk;
    T a[4][8];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = 16 * (t0 + 4 * q) + l16;
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const int k = kb * TRB + 4 * s + lk;
        a[q][s] = (t0 + 4 * q < t1 && row < r && k < r) ? L[row + (int64_t)k * lda] : T(0);
      }
    }
    if (it + 1 < nbk) diag(it + 1, lv);
    __syncthreads();
    {
      T* const xc = X + (wave * 4 + lk) * LD + kb * TRB;
      const int i0 = UP ? TRB - 1 - 2 * l16 : 2 * l16, i1 = UP ? i0 - 1 : i0 + 1;
      T y0 = xc[i0], y1 = xc[i1];
      trsm_steps<T, UP, 0>(y0, y1, Ls, ds, l16);
      xc[i0] = y0;
      xc[i1] = y1;
    }
    __syncthreads();
    T b[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) b[s] = X[l16 * LD + kb * TRB + 4 * s + lk];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (t0 + 4 * q < t1) {
        typename Mfma16<T>::V acc = {};
#pragma unroll
        for (int s = 0; s < 8; ++s) acc = Mfma16<T>::mul(a[q][s], b[s], acc);
        T* const xr = X + l16 * LD + 16 * (t0 + 4 * q);
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) xr[Mfma16<T>::row(lane, rr)] -= acc[rr];
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < TRSM_COLS; ++c)
    if (tid < r && c0 + c < ncols) B[tid + (int64_t)(c0 + c) * ldb] = X[c * LD + tid];
}

// C_z -= A_z B_z over a batch at strides (sa, sb, sc).  zr (may be NULL): B_z is zero
// past column zr->cols[z], and (with start) the rows of B, which are rows zr->row0 ..
// zr->row0 + k - 1 of the full system, are zero in the 64-column groups that start
// below them: the tiles of C that would only subtract zeros are skipped.
static int batched_sub(int prec, int m, int n, int k, const void* A, int64_t lda, int64_t sa, const void* B,
                       int64_t ldb, int64_t sb, void* C, int64_t ldc, int64_t sc, int nbat, const ZeroRhs* zr,
                       hipStream_t s) {
  if (!zr) return gemm_launch_batched(prec, GOP_SUB, m, n, k, A, lda, sa, B, ldb, sb, C, ldc, sc, nbat, s);
  TileSel sel;
  sel.nbat = nbat;
  sel.sa = sa;
  sel.sb = sb;
  sel.sc = sc;
  sel.zcols = zr->cols;
  sel.zstart = zr->start;
  sel.zng = zr->ng;
  sel.zthr = zr->row0 + k;
  return gemm_launch_sel(prec, GOP_SUB, m, n, k, A, lda, B, ldb, C, ldc, sel, s);
}

// A12 <- L^{-1} A12 with L unit lower (r x r): X1 = L11^{-1} B1, B2 -= L21 X1,
// X2 = L22^{-1} B2, recursively, as LAPACK's dtrsm, down to blocks of one launch.
// nbat > 1: nbat systems at L + z sL, A12 + z sB (no masks).  zr (may be NULL): where the
// batch's right-hand sides are zero; the work on those parts, which stay zero, is skipped.
template <typename T>
int trsm_left_unit_lower(const T* L, int64_t lda, int r, T* A12, int64_t ld12, int ncols, LuWork& w, int gemm_prec,
                         const int* cmask = nullptr, int nbat = 1, int64_t sL = 0, int64_t sB = 0,
                         const ZeroRhs* zr = nullptr) {
  if (ncols <= 0 || r <= 0) return KAD_OK;
  if (nbat > 1 && cmask) return arg_error("trsm_left_unit_lower: masks with a batch");
  if (zr && (nbat < 2 || (zr->start && zr->ng < cdiv(ncols, 64))))
    return arg_error("trsm_left_unit_lower: zero right-hand-side parts need a batch and a group per 64 columns");
  if (r <= TRSM_ROWS) {
    trsm_block_kernel<T, false><<<dim3((unsigned)cdiv(ncols, TRSM_COLS), nbat), 256, 0, w.stream>>>(
        L, lda, A12, ld12, r, ncols, cmask, sL, sB, zr ? *zr : ZeroRhs());
    KAD_HIP_CHECK(hipGetLastError());
    return KAD_OK;
  }
  const int h = std::max(TRSM_ROWS, (r / 2) / TRSM_ROWS * TRSM_ROWS);
  int rc = trsm_left_unit_lower<T>(L, lda, h, A12, ld12, ncols, w, gemm_prec, cmask, nbat, sL, sB, zr);
  if (rc) return rc;
  const int gp = gemm_prec == BF16 ? F32 : gemm_prec;
  rc = nbat > 1
           ? batched_sub(gp, r - h, ncols, h, L + h, lda, sL, A12, ld12, sB, A12 + h, ld12, sB, nbat, zr, w.stream)
           : gemm_launch_masked(gp, GOP_SUB, r - h, ncols, h, L + h, lda, A12, ld12, A12 + h, ld12, nullptr, cmask,
                                w.stream);
  if (rc) return rc;
  ZeroRhs z2;
  if (zr) {
    z2 = *zr;
    z2.row0 += h;
  }
  return trsm_left_unit_lower<T>(L + h + (int64_t)h * lda, lda, r - h, A12 + h, ld12, ncols, w, gemm_prec, cmask, nbat,
                                 sL, sB, zr ? &z2 : nullptr);
}

// B <- U^{-1} B with U non-unit upper (r x r, r a multiple of 32): X2 = U22^{-1} B2,
// B1 -= U12 X2, X1 = U11^{-1} B1, recursively down to blocks of one launch.  nbat systems
// at U + z sU, B + z sB; zcols (device, nbat entries, may be NULL): B_z is zero past
// column zcols[z], and those columns are skipped.
template <typename T>
int trsm_left_upper(const T* U, int64_t ldu, int r, T* B, int64_t ldb, int ncols, LuWork& w, int gemm_prec, int nbat,
                    int64_t sU, int64_t sB, const int* zcols = nullptr) {
  if (ncols <= 0 || r <= 0) return KAD_OK;
  if (r % TRB != 0) return arg_error("trsm_left_upper: order not a multiple of 32");
  ZeroRhs zc;
  zc.cols = zcols;
  if (r <= TRSM_ROWS) {
    trsm_block_kernel<T, true><<<dim3((unsigned)cdiv(ncols, TRSM_COLS), nbat), 256, 0, w.stream>>>(
        U, ldu, B, ldb, r, ncols, nullptr, sU, sB, zc);
    KAD_HIP_CHECK(hipGetLastError());
    return KAD_OK;
  }
  const int h = std::max(TRSM_ROWS, (r / 2) / TRSM_ROWS * TRSM_ROWS);
  int rc =
      trsm_left_upper<T>(U + h + (int64_t)h * ldu, ldu, r - h, B + h, ldb, ncols, w, gemm_prec, nbat, sU, sB, zcols);
  if (rc) return rc;
  rc = batched_sub(gemm_prec, h, ncols, r - h, U + (int64_t)h * ldu, ldu, sU, B + h, ldb, sB, B, ldb, sB, nbat,
                   zcols ? &zc : nullptr, w.stream);
  if (rc) return rc;
  return trsm_left_upper<T>(U, ldu, h, B, ldb, ncols, w, gemm_prec, nbat, sU, sB, zcols);
}

// B <- A^{-1} B for nbat factored matrices of order n (n a multiple of 32) whose
// right-hand sides are already in pivoted row order (B_z rows permuted by perm_z):
// the unit-lower, then the upper triangular solve, in FP64.  zcols (device, nbat
// entries, may be NULL): B_z is zero past its first zcols[z] columns, which are skipped;
// zstart (device, nbat x zng, may be NULL, needs zcols): columns 64g .. 64g+63 of B_z are
// zero above row zstart[z zng + g], which the unit-lower solve skips.
int lu_solve_permuted_batched(const double* LU, int64_t lda, int n, int nbat, int64_t sA, double* B, int64_t ldb,
                              int64_t sB, int nrhs, LuWork& w, const int* zcols, const int* zstart, int zng) {
  if (n % TRB != 0 || nbat < 1) return arg_error("lu_solve_permuted_batched: order or batch");
  if (zstart && !zcols) return arg_error("lu_solve_permuted_batched: row starts without column counts");
  ZeroRhs zr;
  zr.cols = zcols;
  zr.start = zstart;
  zr.ng = zng;
  int rc = trsm_left_unit_lower<double>(LU, lda, n, B, ldb, nrhs, w, F64, nullptr, nbat, sA, sB,
                                        zcols && nbat > 1 ? &zr : nullptr);
  if (rc) return rc;
  return trsm_left_upper<double>(LU, lda, n, B, ldb, nrhs, w, F64, nbat, sA, sB, zcols);
}

// Row interchanges of pivots [k1, k2) (at most NSW) applied to COLS columns per
// workgroup.  The affected rows are k1 .. k2-1 and the pivot rows below them (2 nsw
// entries; a row that occurs twice carries the same value both times); entry e's content
// comes from the row found by undoing the interchanges in reverse order, every entry at
// once from the pivots in LDS.  Then one gather (COLS loads per entry in flight) and one
// scatter.  Bound by latency: replaying the interchanges in LDS, one thread per column,
// cost most of the kernel's 52 us (256 interchanges, n = 1215; 60 us at 8191); this one
// takes 14 (24).
template <typename T, int NSW, int COLS>
__global__ __launch_bounds__(256) void laswp_gather_kernel(T* __restrict__ A, int64_t lda, int c0, int c1,
                                                           const int* __restrict__ ipiv, int k1, int k2, int64_t sA,
                                                           int sP) {
  A += (int64_t)blockIdx.y * sA;  // matrix blockIdx.y of a batch
  ipiv += (int64_t)blockIdx.y * sP;
  constexpr int NE = 2 * NSW / 256;  // entries per thread
  __shared__ int piv[NSW];
  const int nsw = k2 - k1;           // <= NSW (checked by the launcher)
  const int t = threadIdx.x;
  const int cb = c0 + blockIdx.x * COLS;
  const int nc = min(COLS, c1 - cb);
  for (int j = t; j < nsw; j += 256) piv[j] = ipiv[k1 + j];
  __syncthreads();
  int row[NE], src[NE];
#pragma unroll
  for (int u = 0; u < NE; ++u) {
    const int e = u * 256 + t;
    row[u] = e < nsw ? k1 + e : (e < 2 * nsw && piv[e - nsw] >= k2 ? piv[e - nsw] : -1);
    src[u] = row[u];
  }
  for (int j = nsw - 1; j >= 0; --j) {
    const int r = k1 + j, p = piv[j];
#pragma unroll
    for (int u = 0; u < NE; ++u) src[u] = src[u] == r ? p : (src[u] == p ? r : src[u]);
  }
  T val[NE][COLS];
#pragma unroll
  for (int u = 0; u < NE; ++u)
#pragma unroll
    for (int c = 0; c < COLS; ++c)
      if (row[u] >= 0 && c < nc) val[u][c] = A[src[u] + (int64_t)(cb + c) * lda];
  __syncthreads();  // every read of these columns precedes every write
#pragma unroll
  for (int u = 0; u < NE; ++u)
#pragma unroll
    for (int c = 0; c < COLS; ++c)
      if (row[u] >= 0 && c < nc) A[row[u] + (int64_t)(cb + c) * lda] = val[u][c];
}

template <typename T>
int laswp(T* A, int64_t lda, int c0, int c1, const int* ipiv, int k1, int k2, LuWork& w,
          const LuBatch& bt = LuBatch()) {
  if (c1 <= c0 || k2 <= k1) return KAD_OK;
  const int nsw = k2 - k1;
  const unsigned nz = (unsigned)bt.nbat;
  if (nsw <= 256) {
    laswp_gather_kernel<T, 256, 8><<<dim3((unsigned)cdiv(c1 - c0, 8), nz), 256, 0, w.stream>>>(A, lda, c0, c1, ipiv, k1,
                                                                                           k2, bt.sA, bt.sP);
  } else if (nsw <= 512) {
    laswp_gather_kernel<T, 512, 4><<<dim3((unsigned)cdiv(c1 - c0, 4), nz), 256, 0, w.stream>>>(A, lda, c0, c1, ipiv, k1,
                                                                                           k2, bt.sA, bt.sP);
  } else {
    laswp_kernel<T><<<dim3((unsigned)cdiv(c1 - c0, 256), nz), 256, 0, w.stream>>>(A, lda, c0, c1, ipiv, k1, k2, bt.sA,
                                                                                bt.sP);
  }
  KAD_HIP_CHECK(hipGetLastError());
  return KAD_OK;
}

// ---------------------------------------------------------------------------
// Base panel without atomics or device-scope fences.  Inside the panel rows are
// never moved: a logical -> physical row map (double-buffered per step) tracks
// the interchanges, and every block re-reduces the previous step's per-block
// maxima, so all communication between blocks goes through kernel boundaries.
// The interchange sequence is LAPACK's (first index of max |a| among the
// logical rows >= j); the panel rows are permuted physically once at the end.
// ---------------------------------------------------------------------------
constexpr int FF_ROWS = 64;  // logical rows per block (x 4 column groups = 256 threads)

template <typename T>
__device__ void ff_reduce_partials(const double* __restrict__ pv, const int* __restrict__ pi, int np, double* sv,
                                   int* si, double& bv, int& bi) {
  double v = -1.0;
  int id = -1;
  for (int b = threadIdx.x; b < np; b += blockDim.x) {
    const double ov = pv[b];
    const int oi = pi[b];
    if (oi >= 0 && (id < 0 || ov > v || (ov == v && oi < id))) {
      v = ov;
      id = oi;
    }
  }
  block_argmax<T>(v, id, sv, si, bv, bi);
}

// Partial maxima of column c0 over logical rows [c0, n) (identity map).
template <typename T>
__global__ __launch_bounds__(256) void ff_first_kernel(const T* __restrict__ A, int64_t lda, int n, int c0,
                                                       int* __restrict__ map_out, double* __restrict__ pv,
                                                       int* __restrict__ pi) {
  __shared__ double sv[256];
  __shared__ int si[256];
  const int i = c0 + blockIdx.x * 256 + threadIdx.x;
  double v = -1.0;
  int id = -1;
  if (i < n) {
    map_out[i] = i;
    v = pivot_abs((double)A[i + (int64_t)c0 * lda], i == c0);
    id = i;
  }
  double bv;
  int bi;
  block_argmax<T>(v, id, sv, si, bv, bi);
  if (threadIdx.x == 0) {
    pv[blockIdx.x] = bv;
    pi[blockIdx.x] = bi;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void ff_step_kernel(T* __restrict__ A, int64_t lda, int n, int c0, int j, int c1,
                                                      const int* __restrict__ map_in, int* __restrict__ map_out,
                                                      const double* __restrict__ pv_in, const int* __restrict__ pi_in,
                                                      int np_in, double* __restrict__ pv_out, int* __restrict__ pi_out,
                                                      int* __restrict__ ipiv, int* __restrict__ info) {
  __shared__ double sv[256];
  __shared__ int si[256];
  __shared__ T urow[PANEL_BASE];
  __shared__ T lcol[FF_ROWS];
  __shared__ int pshared;
  double bv;
  int p;
  ff_reduce_partials<T>(pv_in, pi_in, np_in, sv, si, bv, p);
  if (p < 0) p = j;
  const int phys_piv = map_in[p];  // physical row that becomes logical row j
  const int phys_j = map_in[j];    // physical row that moves to logical row p
  const int w = c1 - j;
  for (int c = threadIdx.x; c < w; c += blockDim.x) urow[c] = A[phys_piv + (int64_t)(j + c) * lda];
  if (blockIdx.x == 0) {
    // logical rows [c0, j) are final: carry them into the other map buffer
    for (int k = threadIdx.x; k < j - c0; k += blockDim.x) map_out[c0 + k] = map_in[c0 + k];
    if (threadIdx.x == 0) {
      ipiv[j] = p;
      map_out[j] = phys_piv;
      if (bv == 0.0 && *info == 0) *info = j + 1;
    }
  }
  const int tx = threadIdx.x % FF_ROWS, ty = threadIdx.x / FF_ROWS;
  const int i = j + 1 + blockIdx.x * FF_ROWS + tx;  // logical row
  int phys = -1;
  if (i < n) phys = (i == p) ? phys_j : map_in[i];
  __syncthreads();
  const T piv = urow[0];
  if (ty == 0) {
    T l = T(0);
    if (i < n) {
      l = A[phys + (int64_t)j * lda];
      if (piv != T(0)) l = l / piv;
      A[phys + (int64_t)j * lda] = l;
      map_out[i] = phys;
    }
    lcol[tx] = l;
  }
  __syncthreads();
  double v = -1.0;
  int id = -1;
  if (i < n) {
    const T l = lcol[tx];
    T* ai = A + phys;
    for (int c = 1 + ty; c < w; c += 4) {
      T x = ai[(int64_t)(j + c) * lda];
      x -= l * urow[c];
      ai[(int64_t)(j + c) * lda] = x;
      if (c == 1) {
        v = pivot_abs((double)x, i == j + 1);
        id = i;
      }
    }
  }
  if (j + 1 >= c1) return;  // uniform: no partials after the last column
  int bi;
  block_argmax<T>(v, id, sv, si, bv, bi);
  if (threadIdx.x == 0) {
    pv_out[blockIdx.x] = bv;
    pi_out[blockIdx.x] = bi;
  }
  (void)pshared;
}

// Physical permutation of the panel rows: tmp[i - c0][c] = A[map[i]][c], then back.
template <typename T>
__global__ void ff_gather_kernel(const T* __restrict__ A, int64_t lda, int n, int c0, int c1,
                                 const int* __restrict__ map, T* __restrict__ tmp) {
  const int i = c0 + blockIdx.x * blockDim.x + threadIdx.x;
  const int c = c0 + blockIdx.y;
  if (i < n && c < c1) tmp[(i - c0) + (int64_t)(c - c0) * (n - c0)] = A[map[i] + (int64_t)c * lda];
}
template <typename T>
__global__ void ff_scatter_kernel(T* __restrict__ A, int64_t lda, int n, int c0, int c1, const T* __restrict__ tmp) {
  const int i = c0 + blockIdx.x * blockDim.x + threadIdx.x;
  const int c = c0 + blockIdx.y;
  if (i < n && c < c1) A[i + (int64_t)c * lda] = tmp[(i - c0) + (int64_t)(c - c0) * (n - c0)];
}

// ---------------------------------------------------------------------------
// Persistent base panel: one launch factors columns [c0, c1) (c1 - c0 <= W) of rows
// [c0, n).  Every thread keeps one row of the block in registers for the whole launch,
// with its logical position: an interchange swaps the positions of two rows, no row
// moves, and every row is written to its final position at the end.  Per column j:
//   1. every wave takes its candidate (the largest |a| of its rows, the first position
//      among ties); after one barrier every wave knows the workgroup's best, and the
//      wave that owns it stages that row in LDS;
//   2. with several workgroups, each publishes its candidate's position and the columns
//      >= j of its row, reads all candidates (four slots per thread and round trip: in
//      FP64 1 to 5 round trips for up to 64 workgroups of 256 rows), each word flagged with its column
//      (no grid barrier: a word is current when its flag is), and reduces them itself --
//      LAPACK's choice, the first index of max |a|;
//   3. positions, multipliers and the rank-1 update, with the per-column kernel's
//      operations.
// At the end the interchanges are applied to the panel's other columns [k0, c0) and
// [c1, k1) (exact: those columns are not read in between).
// Bound by latency: the chain of its columns is the factorisation's critical path.
// 3.6 us per column with several workgroups, 1.8 with one (5.1 before, when every row moved
// with its interchange, row j was published beside the candidates and every wave read the
// pivot row by LDS broadcasts).
// The grid must be resident at once: the host launches at most one workgroup per
// CU, and nothing else on the device waits on this kernel.  Every wait is bounded: a
// workgroup that reaches the spin limit raises the abort flag (sync[2]), every waiter
// leaves on it, and the host reports the failure.
// ---------------------------------------------------------------------------
constexpr int FFP_MAX_GRID = 64;

// Exchange slots.  Every 64-bit slot holds one 32-bit data word and, in its high half,
// the flag of the column that wrote it (launch sequence x 32 + column).  Slots are
// read and written as agent-scope relaxed atomics (sc1: written through to, and read
// from, the level the XCDs share), so a reader that sees the flag it expects holds
// that column's word: each slot validates itself, no slot is ordered against another,
// and no device-scope fence (a write-back and invalidate of the XCD's whole L2, the
// concurrent GEMM's working set) or arrival counter is needed.  A column's slots are
// one record per workgroup, packed: its candidate's position (and for FP64 a pad word
// that keeps the values 8-byte aligned), then the row's values from the column on, one
// word each for FP32 and two for FP64.
template <typename T, int W>
struct FfpSlots {
  static constexpr int VW = (int)(sizeof(T) / 4);  // words per value (and of a record's head)
  static constexpr int REC = VW * (1 + W);         // the first column's record, the longest
  static constexpr int COL = FFP_MAX_GRID * REC;   // one column's stride
};

__device__ __forceinline__ void slot_store(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long slot_load(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// |v| as an unsigned key that orders as the value does (high and low words; FP32: one);
// a NaN's key as pivot_abs: the least, or in row j the largest.
__device__ __forceinline__ void abs_key(double v, bool row_j, unsigned& hi, unsigned& lo) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  hi = v == v ? (unsigned)(b >> 32) & 0x7fffffffu : (row_j ? ~0u : 0u);
  lo = v == v ? (unsigned)b : 0u;
}
__device__ __forceinline__ void abs_key(float v, bool row_j, unsigned& hi, unsigned& lo) {
  hi = v == v ? __builtin_bit_cast(unsigned, v) & 0x7fffffffu : (row_j ? ~0u : 0u);
  lo = 0;
}

// Largest value over a wave (DPP row shifts, then the two row broadcasts; lane 63 holds it).
__device__ __forceinline__ unsigned wave_umax(unsigned v) {
  auto step = [&v](int o) { v = (unsigned)o > v ? (unsigned)o : v; };
  step(__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, false));
  step(__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, false));
  step(__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, false));
  step(__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, false));
  step(__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false));
  step(__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false));
  return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// The lane of the largest (hi, lo) among a wave's lanes with pos >= 0, the smallest pos
// among equal ones; -1 when there is none.  Uniform.  One 32-bit reduction decides it
// unless the high words tie (a column of zeros, the structural zeros of a Jacobian).
__device__ __forceinline__ int wave_best(unsigned hi, unsigned lo, int pos) {
  const bool in = pos >= 0;
  const unsigned m = wave_umax(in ? hi : 0u);
  unsigned long long c = __ballot(in && hi == m);
  if (__popcll(c) > 1) {
    bool tie = in && hi == m;
    const unsigned ml = wave_umax(tie ? lo : 0u);
    tie = tie && lo == ml;
    const unsigned mp = wave_umax(tie ? ~(unsigned)pos : 0u);
    c = __ballot(tie && ~(unsigned)pos == mp);
  }
  return c ? __ffsll((long long)c) - 1 : -1;
}

// TH threads, one row each.
template <typename T, int W, int TH>
__global__ __launch_bounds__(TH) void ffp_kernel(T* __restrict__ A, int64_t lda, int n, int c0, int c1, int k0, int k1,
                                                 int rpw, unsigned long long* __restrict__ xbuf, unsigned flag0,
                                                 int* __restrict__ ipiv, int* __restrict__ info,
                                                 int* __restrict__ sync, int spin_limit, int64_t sA, int sP,
                                                 int64_t sX) {
  static_assert(FFP_MAX_GRID <= 64, "one candidate per lane of a wave");
  constexpr int R4 = 4;  // columns between two rotations of the row registers
  static_assert(W % R4 == 0, "rotation");
  using S = FfpSlots<T, W>;
  constexpr int VW = S::VW, NW = TH / 64;
  // issue priority over the GEMM waves that share the SIMDs: every column waits for
  // the slowest workgroup, and the GEMM's MFMA chains leave issue slots to spare
  __builtin_amdgcn_s_setprio(3);
  __shared__ __align__(16) unsigned xim[TH == 1024 ? 4 : S::COL];  // this column's records, data words only
  __shared__ __align__(16) T stage[W];         // the workgroup's candidate row
  __shared__ unsigned wk[2][NW][4];            // the waves' candidates: key and position, by column parity
  __shared__ int s_piv[W];
  __shared__ int s_rows[2 * W];
  __shared__ int s_src[2 * W];
  // matrix blockIdx.y of a batch: its own rows, interchanges, exchange slots and info
  // word; the workgroups of one matrix (blockIdx.x) exchange only among themselves
  A += (int64_t)blockIdx.y * sA;
  ipiv += (int64_t)blockIdx.y * sP;
  xbuf += (int64_t)blockIdx.y * sX;
  info += blockIdx.y;
  const int G = TH == 1024 ? 1 : (int)gridDim.x, g = blockIdx.x, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int r0 = c0 + g * rpw;
  const int nr = max(0, min(rpw, n - r0));
  const int w = c1 - c0;
  const bool own = tid < nr;
  int pos = own ? r0 + tid : -1;  // this row's logical position; rows above the current column are done
  // the row's columns; columns past the panel's end hold zeros (rotated by R4 positions
  // every R4 columns: after jj columns, row[q] holds column (q + jj / R4 R4) mod W, so
  // every index into the array is a compile-time constant)
  T row[W];
#pragma unroll
  for (int c = 0; c < W; ++c) row[c] = own && c < w ? A[(int64_t)(r0 + tid) + (int64_t)(c0 + c) * lda] : T(0);
  bool live = true;  // uniform: false once a wait was abandoned
  int jfail = w;     // first column not factored (after an abandoned wait)
  for (int j0 = 0; j0 < w && live; j0 += R4) {
    static_for<R4>([&](auto sc) {
      constexpr int s = decltype(sc)::value;
      const int jj = j0 + s;
      if (jj >= w || !live) return;
      const int j = c0 + jj, par = s & 1;
      // 1. the wave's candidate among its rows at positions >= j, then the workgroup's
      unsigned hi, lo;
      abs_key(row[s], pos == j, hi, lo);
      const int best = wave_best(hi, lo, pos >= j ? pos : -1);
      if (lane == (best < 0 ? 0 : best)) {
        wk[par][wave][0] = hi;
        wk[par][wave][1] = lo;
        wk[par][wave][2] = best < 0 ? ~0u : (unsigned)pos;
      }
      __syncthreads();
      unsigned khi = 0, klo = 0;
      int kpos = -1;
      if (lane < NW) {
        khi = wk[par][lane][0];
        klo = wk[par][lane][1];
        kpos = (int)wk[par][lane][2];
      }
      const int bw = wave_best(khi, klo, kpos);
      int p = bw < 0 ? -1 : __builtin_amdgcn_readlane(kpos, bw);
      if (wave == bw && lane == best) {
#pragma unroll
        for (int q = s; q < W; ++q) stage[q - s] = row[q];  // values from column jj on
      }
      const T* urow = stage;
      if (G == 1) {
        __syncthreads();
      } else {
        // 2. publish (position -1: no candidate), then read every record
        const unsigned flag = flag0 + (unsigned)jj;
        const unsigned long long tag = (unsigned long long)flag << 32;
        unsigned long long* const col = xbuf + (size_t)jj * S::COL;
        const int rec = VW * (1 + W - jj);
        if (wave == (bw < 0 ? 0 : bw)) {  // the wave that staged the row
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
          for (int e = lane; e < rec; e += 64) {
            const unsigned word = e < VW ? (unsigned)p : reinterpret_cast<const unsigned*>(stage)[e - VW];
            slot_store(col + g * rec + e, tag | word);
          }
        }
        const int nused = G * rec;
        int bad = 0;
        // groups of 4 strips of TH slots, loaded together and read again until every slot
        // carries this column's flag.  Bounded: at the spin limit the workgroup raises
        // the abort flag, and every waiter leaves on it; the host reports the failure.
        for (int e0 = 0; e0 < nused && !bad; e0 += 4 * TH) {
          for (int it = 0;; ++it) {
            unsigned long long x[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) x[u] = e0 + u * TH + tid < nused ? slot_load(col + e0 + u * TH + tid) : tag;
            bool pend = false;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              if (e0 + u * TH + tid < nused) xim[e0 + u * TH + tid] = (unsigned)x[u];
              pend |= (unsigned)(x[u] >> 32) != flag;
            }
            if (!pend) break;
            if (it >= spin_limit) {
              __hip_atomic_store(&sync[2], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              bad = 1;
              break;
            }
            if ((it & 255) == 255 && __hip_atomic_load(&sync[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) {
              bad = 1;
              break;
            }
          }
        }
        if (__syncthreads_or(bad)) {  // uniform; the host sees sync[2] and reports the failure
          live = false;
          jfail = jj;
          return;
        }
        // the pivot: every wave reduces the G <= 64 candidates itself
        unsigned chi = 0, clo = 0;
        int cpos = -1;
        if (lane < G) {
          cpos = (int)xim[lane * rec];
          abs_key(reinterpret_cast<const T*>(xim + lane * rec + VW)[0], cpos == j, chi, clo);
        }
        const int bg = wave_best(chi, clo, cpos);
        p = bg < 0 ? -1 : __builtin_amdgcn_readlane(cpos, bg);
        urow = reinterpret_cast<const T*>(xim + (bg < 0 ? 0 : bg) * rec + VW);
      }
      if (p < j || p >= n) {
        // only reachable with corrupt candidates: keep every index in range and fail
        p = j;
        if (tid == 0) __hip_atomic_store(&sync[2], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      // 3. the interchange: row p moves to position j, the row there to p; the pivot row
      //    is then final
      const T piv = urow[0];
      if (tid == 0) s_piv[jj] = p;
      if (g == 0 && tid == 0) {
        ipiv[j] = p;
        if (piv == T(0) && *info == 0) *info = j + 1;
      }
      if (pos == p) pos = j;
      else if (pos == j) pos = p;
      // rows below j: the multiplier (row[s]) and the rank-1 update of the columns after
      // it (row[q]: column jj + q - s, no wrap below W - j0; columns past the panel's end
      // are never written back).  The pivot row's values sit in the lanes of each 16-lane
      // row, 16 in each of u0 and u1, and reach the multiply-adds by row broadcasts (as
      // broadcast LDS reads by every wave they filled the LDS pipe).
      const T u0 = urow[lane & 15], u1 = urow[16 + (lane & 15)];
      const bool below = pos > j;
      T l = row[s];
      if (below) {
        if (piv != T(0)) l = l / piv;
        row[s] = l;
      }
      static_for<W / R4>([&](auto bc) {
        constexpr int q0 = decltype(bc)::value * R4;
        if (q0 >= W - j0) return;  // uniform
        T ub[R4];
        static_for<R4>([&](auto qc) {
          constexpr int v = q0 + decltype(qc)::value - s;  // the value's place in the record
          if constexpr (v > 0 && v < 16) ub[decltype(qc)::value] = lane16<v>(u0);
          if constexpr (v >= 16) ub[decltype(qc)::value] = lane16<v - 16>(u1);
        });
        if (below) {
#pragma unroll
          for (int q = 0; q < R4; ++q)
            if (q0 + q > s) row[q0 + q] = row[q0 + q] - l * ub[q];
        }
      });
    });
    T t[R4];
#pragma unroll
    for (int q = 0; q < R4; ++q) t[q] = row[q];
#pragma unroll
    for (int q = 0; q < W - R4; ++q) row[q] = row[q + R4];
#pragma unroll
    for (int q = 0; q < R4; ++q) row[W - R4 + q] = t[q];
  }
  if (!live) {
    // the columns not factored get identity interchanges: later kernels index rows
    // with ipiv, which must stay within the matrix (the factors are reported invalid)
    if (g == 0)
      for (int jj = jfail + tid; jj < w; jj += TH) ipiv[c0 + jj] = c0 + jj;
    return;
  }
  // rows to their final positions: every row of the block was read before the first
  // column's exchange (one workgroup: its barrier) ended, so none is overwritten unread
  const int turn = (w + R4 - 1) / R4 * R4;  // row[q] holds column (q + turn) mod W
  if (own) {
#pragma unroll
    for (int q = 0; q < W; ++q) {
      const int c = (q + turn) & (W - 1);
      if (c < w) A[(int64_t)pos + (int64_t)(c0 + c) * lda] = row[q];
    }
  }
  __syncthreads();  // s_piv of the last column
  // the interchanges on the panel's other columns: the affected rows are rows
  // c0 .. c1-1 and the pivot rows (2 w entries, duplicates harmless: they carry the
  // same value); entry k's content comes from the row found by undoing the
  // interchanges in reverse order
  if (tid < 2 * w) {
    const int r = tid < w ? c0 + tid : s_piv[tid - w];
    int x = r;
    for (int jj = w - 1; jj >= 0; --jj) {
      const int a = c0 + jj, b = s_piv[jj];
      x = (x == a) ? b : ((x == b) ? a : x);
    }
    s_rows[tid] = r;
    s_src[tid] = x;
  }
  __syncthreads();
  // (column, affected row) pairs, columns split over the workgroups: every thread
  // gathers up to FFP_TAIL of them into registers, the workgroup synchronises, then
  // every thread scatters them -- one round trip per batch, and no row of a column is
  // written before all of that column's reads (a column stays in one workgroup)
  constexpr int FFP_TAIL = 16;
  const int nrw = 2 * w, nleft = c0 - k0, nother = (c0 - k0) + (k1 - c1);
  const int cpg = (int)cdiv(nother, G);  // columns of this workgroup: [g cpg, (g + 1) cpg)
  const int qa = min(nother, g * cpg), qe = min(nother, qa + cpg);
  const int npairs = (qe - qa) * nrw;
  const int step = ((FFP_TAIL * TH) / nrw) * nrw;  // whole columns per batch (nrw <= 2 W)
  for (int b0 = 0; b0 < npairs; b0 += step) {
    const int bend = min(npairs, b0 + step);
    T val[FFP_TAIL];
#pragma unroll
    for (int u = 0; u < FFP_TAIL; ++u) {
      const int e = b0 + u * TH + tid;
      if (e < bend) {
        const int q = qa + e / nrw, k = e - (e / nrw) * nrw;
        const int col = q < nleft ? k0 + q : c1 + (q - nleft);
        val[u] = A[(int64_t)s_src[k] + (int64_t)col * lda];
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < FFP_TAIL; ++u) {
      const int e = b0 + u * TH + tid;
      if (e < bend) {
        const int q = qa + e / nrw, k = e - (e / nrw) * nrw;
        const int col = q < nleft ? k0 + q : c1 + (q - nleft);
        A[(int64_t)s_rows[k] + (int64_t)col * lda] = val[u];
      }
    }
    __syncthreads();
  }
}

// Exchange slots of the persistent base panel for one matrix (W columns, FP64
// records), in 64-bit words, and the bytes of the whole buffer (one region per
// matrix of a batch, LU_MAX_BATCH regions).
constexpr int64_t ffp_matrix_words() { return (int64_t)PANEL_BASE * FfpSlots<double, PANEL_BASE>::COL; }
size_t ffp_bytes() { return (size_t)LU_MAX_BATCH * ffp_matrix_words() * sizeof(unsigned long long); }

// Launch shape of the persistent base panel for m rows of each of nbat matrices: threads
// (= most rows) per workgroup, grid and rows per workgroup, or false when it does not
// fit (the per-column kernels run).  Up to 1024 rows one workgroup needs no exchange.
// A batch launches the workgroups of every matrix together; all of them must be
// resident at once, so it holds at most one workgroup per CU in total.
struct FfpShape {
  int th = 0, grid = 0, rpw = 0;
};
inline bool ffp_shape(int m, int nbat, int ncu, FfpShape& s) {
  if (m < 1) return false;
  // one workgroup of 1024 rows against several of 256: n = 600 2.05 ms against 2.39, 1215
  // 4.07 against 4.74; beyond that 256 rows per workgroup (n = 5000 20.4 ms, 20.9 with
  // 512), 512 where 256 would need too many workgroups (one matrix: a batch of orders
  // above 64 x 256 is refused)
  for (int th : {1024, 256, 512}) {
    if (th == 512 && nbat > 1) break;
    s.th = th;
    s.grid = (int)cdiv(m, th);
    if (s.grid <= (th == 1024 ? 1 : FFP_MAX_GRID) && s.grid * nbat <= ncu) break;
    s.grid = 0;
  }
  if (!s.grid) return false;
  s.rpw = (int)cdiv(m, s.grid);
  s.grid = (int)cdiv(m, s.rpw);
  return true;
}

// One persistent base panel: columns [c0, c1) of rows [c0, n), interchanges applied
// across the panel's columns [k0, k1).
template <typename T>
int ffp_launch(T* A, int64_t lda, int n, int c0, int c1, int k0, int k1, int* ipiv, LuWork& w,
               const LuBatch& bt = LuBatch()) {
  FfpShape s;
  if (c1 - c0 > PANEL_BASE || c1 > n) return arg_error("ffp_launch: panel shape");
  if (bt.nbat < 1 || bt.nbat > LU_MAX_BATCH || (bt.nbat > 1 && !bt.info) || !ffp_shape(n - c0, bt.nbat, w.ncu, s))
    return arg_error("ffp_launch: batch does not fit the CUs");
  // flags: PANEL_BASE per launch, never one the slots still hold (the buffer starts
  // zeroed and the sequence at 1; before the 32-bit flags wrap it is cleared again)
  if (++w.ffp_seq >= (1u << 26)) {
    KAD_HIP_CHECK(hipMemsetAsync(w.ffp, 0, ffp_bytes(), w.stream));
    w.ffp_seq = 1;
  }
  const unsigned flag0 = w.ffp_seq * (unsigned)PANEL_BASE;
  auto run = [&](auto kernel) {
    kernel<<<dim3(s.grid, bt.nbat), s.th, 0, w.stream>>>(A, lda, n, c0, c1, k0, k1, s.rpw, (unsigned long long*)w.ffp,
                                                         flag0, ipiv, bt.info ? bt.info : w.info, w.ffp_sync,
                                                         w.ffp_spin, bt.sA, bt.sP, ffp_matrix_words());
  };
  if (s.th == 1024) run(ffp_kernel<T, PANEL_BASE, 1024>);
  else if (s.th == 256) run(ffp_kernel<T, PANEL_BASE, 256>);
  else run(ffp_kernel<T, PANEL_BASE, 512>);
  KAD_HIP_CHECK(hipGetLastError());
  return KAD_OK;
}

// Base panel without row interchanges (static pivoting): the rows were put in the
// order of an earlier factorisation's pivots beforehand, so row j is the pivot of
// column j.  Columns [c0, c1) (at most W), rows [c0, n); matrix blockIdx.y of a batch.
// - Every workgroup factors the w x w diagonal block itself, row by row (threads
//   t < w hold its rows in registers; row j, final, goes to LDS before the rows below
//   it use it).  The operations and their order are the same in every workgroup, so
//   all hold the same factored block.
// - Its rows below the block then solve l U11 = a, one row per thread in registers,
//   with the same row operations.
// - The last workgroup to arrive (a counter, returned to zero by that workgroup) writes
//   the factored diagonal block: every other one has read the block by then, so none
//   reads a block that was already overwritten.  It also writes the identity
//   interchanges and the first zero pivot.
// - growth: the largest |multiplier| of the matrix, as the bits of a non-negative
//   double (an unsigned maximum orders them; inf and NaN above every finite value).
template <typename T, int W>
__global__ __launch_bounds__(256) void nopiv_panel_kernel(T* __restrict__ A, int64_t lda, int n, int c0, int c1,
                                                          int* __restrict__ ipiv, int* __restrict__ info,
                                                          unsigned* __restrict__ cnt,
                                                          unsigned long long* __restrict__ growth, int64_t sA,
                                                          int sP) {
  A += (int64_t)blockIdx.y * sA;
  ipiv += (int64_t)blockIdx.y * sP;
  info += blockIdx.y;
  cnt += blockIdx.y;
  growth += blockIdx.y;
  __shared__ T U[W][W + 1];  // the factored diagonal block, row j once it is final
  __shared__ unsigned long long s_g[256 / 64];
  __shared__ int s_last;
  const int w = c1 - c0, tid = threadIdx.x;
  // this thread's row below the block (loaded first: its latency overlaps the block)
  const int64_t i = (int64_t)c0 + (int64_t)blockIdx.x * 256 + tid;
  const bool mine = i >= c0 + w && i < n;
  T row[W];
#pragma unroll
  for (int c = 0; c < W; ++c) row[c] = mine && c < w ? A[i + (int64_t)(c0 + c) * lda] : T(0);
  // the diagonal block, row t per thread t < w
  T drow[W];
#pragma unroll
  for (int c = 0; c < W; ++c) drow[c] = tid < w && c < w ? A[(int64_t)(c0 + tid) + (int64_t)(c0 + c) * lda] : T(0);
#pragma unroll
  for (int j = 0; j < W; ++j) {
    if (j < w) {
      if (tid == j) {
#pragma unroll
        for (int c = 0; c < W; ++c) U[j][c] = drow[c];
      }
      __syncthreads();
      if (tid > j && tid < w) {
        const T l = drow[j] / U[j][j];
        drow[j] = l;
#pragma unroll
        for (int c = j + 1; c < W; ++c) drow[c] -= l * U[j][c];
      }
    }
  }
  __syncthreads();
  // every thread has read its part of the diagonal block (its values are in LDS, behind
  // the barrier): count this workgroup in
  if (tid == 0)
    s_last = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
  unsigned long long g = 0;
  auto take = [&g](T l) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(fabs((double)l));
    g = b > g ? b : g;
  };
  if (mine) {
#pragma unroll
    for (int j = 0; j < W; ++j) {
      if (j < w) {
        const T l = row[j] / U[j][j];
        row[j] = l;
        take(l);
#pragma unroll
        for (int c = j + 1; c < W; ++c) row[c] -= l * U[j][c];
      }
    }
#pragma unroll
    for (int c = 0; c < W; ++c)
      if (c < w) A[i + (int64_t)(c0 + c) * lda] = row[c];
  }
  __syncthreads();  // s_last
  if (s_last) {
    if (tid < w) {
#pragma unroll
      for (int c = 0; c < W; ++c) {
        if (c < w) A[(int64_t)(c0 + tid) + (int64_t)(c0 + c) * lda] = U[tid][c];
        if (c < tid && c < w) take(U[tid][c]);
      }
      ipiv[c0 + tid] = c0 + tid;
    }
    if (tid == 0) {
      __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      for (int j = 0; j < w; ++j)
        if (U[j][j] == T(0)) {
          if (*info == 0) *info = c0 + j + 1;
          break;
        }
    }
  }
  // the workgroup's largest multiplier, then the matrix's
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const unsigned long long h = __shfl_xor(g, o);
    g = h > g ? h : g;
  }
  if ((tid & 63) == 0) s_g[tid >> 6] = g;
  __syncthreads();
  if (tid == 0) {
    for (int q = 1; q < 256 / 64; ++q) g = s_g[q] > g ? s_g[q] : g;
    __hip_atomic_fetch_max(growth, g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

template <typename T>
int nopiv_launch(T* A, int64_t lda, int n, int c0, int c1, int* ipiv, LuWork& w, const LuBatch& bt) {
  if (c1 - c0 > PANEL_BASE || c1 <= c0 || c1 > n) return arg_error("nopiv_launch: panel shape");
  if (bt.nbat < 1 || bt.nbat > LU_MAX_BATCH || !bt.growth || !w.bcnt) return arg_error("nopiv_launch: batch");
  const dim3 grid((unsigned)cdiv(n - c0, 256), (unsigned)bt.nbat);
  nopiv_panel_kernel<T, PANEL_BASE><<<grid, 256, 0, w.stream>>>(A, lda, n, c0, c1, ipiv, bt.info ? bt.info : w.info,
                                                                 w.bcnt, bt.growth, bt.sA, bt.sP);
  KAD_HIP_CHECK(hipGetLastError());
  return KAD_OK;
}

// Base panel: columns [c0, c1) (c1 - c0 <= PANEL_BASE), rows [c0, n).
template <typename T>
int panel_base(T* A, int64_t lda, int n, int c0, int c1, int* ipiv, LuWork& w) {
  const int nb0 = (int)cdiv(n - c0, 256);
  const int nbs = (int)cdiv(n - c0, FF_ROWS);
  if (nb0 > w.red_cap || nbs > w.red_cap) return KAD_ERR_ARG;
  int* map[2] = {w.map, w.map + n};
  double* pv[2] = {w.red_val, w.red_val + w.red_cap};
  int* pi[2] = {w.red_idx, w.red_idx + w.red_cap};
  ff_first_kernel<T><<<nb0, 256, 0, w.stream>>>(A, lda, n, c0, map[0], pv[0], pi[0]);
  int np = nb0, cur = 0;
  for (int j = c0; j < c1; ++j) {
    const int rows = n - j - 1;
    const int nbk = rows > 0 ? (int)cdiv(rows, FF_ROWS) : 1;
    ff_step_kernel<T><<<nbk, 256, 0, w.stream>>>(A, lda, n, c0, j, c1, map[cur], map[cur ^ 1], pv[cur], pi[cur], np,
                                                 pv[cur ^ 1], pi[cur ^ 1], ipiv, w.info);
    np = nbk;
    cur ^= 1;
  }
  KAD_HIP_CHECK(hipGetLastError());
  // map[cur] now holds the final logical -> physical order of rows [c0, n)
  const size_t need = (size_t)(n - c0) * (c1 - c0) * sizeof(T);
  if (need > w.tmp2_bytes) return KAD_ERR_ARG;
  dim3 g((unsigned)cdiv(n - c0, 256), c1 - c0);
  ff_gather_kernel<T><<<g, 256, 0, w.stream>>>(A, lda, n, c0, c1, map[cur], (T*)w.tmp2);
  ff_scatter_kernel<T><<<g, 256, 0, w.stream>>>(A, lda, n, c0, c1, (const T*)w.tmp2);
  KAD_HIP_CHECK(hipGetLastError());
  return KAD_OK;
}

// Recursive panel factorisation of columns [c0, c1), rows [c0, n), inside the panel
// [pk0, pk1).  fused: the base panels are the persistent kernel, which applies its
// interchanges across [pk0, pk1) itself, so the recursion swaps no rows.
// A batch (bt.nbat > 1) runs the persistent kernel only.
template <typename T>
int panel_rec(T* A, int64_t lda, int n, int c0, int c1, int* ipiv, LuWork& w, int pk0, int pk1, bool fused,
              const LuBatch& bt = LuBatch()) {
  const int wdt = c1 - c0;
  if (bt.nbat > 1 && !fused && !bt.nopiv) return arg_error("panel_rec: a batch needs the persistent panel");
  if (wdt <= PANEL_BASE) {
    if (bt.nopiv) return nopiv_launch<T>(A, lda, n, c0, c1, ipiv, w, bt);
    return fused ? ffp_launch<T>(A, lda, n, c0, c1, pk0, pk1, ipiv, w, bt) : panel_base<T>(A, lda, n, c0, c1, ipiv, w);
  }
  int h = wdt / 2;
  h = (h + PANEL_BASE - 1) / PANEL_BASE * PANEL_BASE;
  const int cm = c0 + h;
  int rc = panel_rec<T>(A, lda, n, c0, cm, ipiv, w, pk0, pk1, fused, bt);
  if (rc) return rc;
  if (!fused && (rc = laswp<T>(A, lda, cm, c1, ipiv, c0, cm, w))) return rc;
  rc = trsm_left_unit_lower<T>(A + c0 + (int64_t)c0 * lda, lda, h, A + c0 + (int64_t)cm * lda, lda, c1 - cm, w,
                               prec_of<T>(), nullptr, bt.nbat, bt.sA, bt.sA);
  if (rc) return rc;
  rc = gemm_launch_batched(prec_of<T>(), GOP_SUB, n - cm, c1 - cm, h, A + cm + (int64_t)c0 * lda, lda, bt.sA,
                           A + c0 + (int64_t)cm * lda, lda, bt.sA, A + cm + (int64_t)cm * lda, lda, bt.sA, bt.nbat,
                           w.stream);
  if (rc) return rc;
  rc = panel_rec<T>(A, lda, n, cm, c1, ipiv, w, pk0, pk1, fused, bt);
  if (rc) return rc;
  return fused ? KAD_OK : laswp<T>(A, lda, c0, cm, ipiv, cm, c1, w);
}

// dst[i + c ldt] = A[map[i] + c lda] for i < nrows, c < ncols (row gather of a column block).
template <typename T>
__global__ void gather_rows_kernel(const T* __restrict__ A, int64_t lda, const int* __restrict__ map, int nrows,
                                   T* __restrict__ dst, int64_t ldt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int c = blockIdx.y;
  if (i < nrows) dst[i + (int64_t)c * ldt] = A[map[i] + (int64_t)c * lda];
}

// The interchanges of later panels applied to the L columns of earlier panels, once,
// after the factorisation (those columns are never read again while factoring, so
// deferring them is exact).  For panel p the interchanges of steps k1_p .. n-1,
// composed on the host, are one row gather per column of rows [k1_p, n).
template <typename T>
int apply_left_swaps(T* A, int64_t lda, int n, const int* ipiv, int nb, LuWork& w) {
  const int np = (int)cdiv(n, nb);
  if (np < 2) return KAD_OK;
  std::vector<int> hp(n);
  KAD_HIP_CHECK(hipMemcpyAsync(hp.data(), ipiv, n * sizeof(int), hipMemcpyDeviceToHost, w.stream));
  KAD_HIP_CHECK(hipStreamSynchronize(w.stream));
  // the interchanges index host memory below: a factorisation that did not complete
  // (an abandoned panel barrier) leaves entries unwritten
  for (int i = 0; i < n; ++i)
    if (hp[i] < i || hp[i] >= n) return KAD_ERR_HIP;
  size_t tot = 0;
  for (int p = 0; p + 1 < np; ++p) tot += (size_t)(n - (p + 1) * nb);
  if (tot > w.swap_cap) {
    if (w.swap_map) KAD_HIP_CHECK(hipFree(w.swap_map));
    w.swap_map = nullptr;
    w.swap_cap = 0;
    KAD_HIP_CHECK(hipMalloc((void**)&w.swap_map, tot * sizeof(int)));
    w.swap_cap = tot;
  }
  std::vector<int> maps(tot);
  std::vector<size_t> moff(np, 0);
  size_t o = 0;
  for (int p = 0; p + 1 < np; ++p) {
    const int k1 = (p + 1) * nb;
    moff[p] = o;
    int* idx = maps.data() + o;
    for (int i = 0; i < n - k1; ++i) idx[i] = k1 + i;
    for (int i = k1; i < n; ++i) {
      const int q = hp[i];
      if (q != i) std::swap(idx[i - k1], idx[q - k1]);
    }
    o += (size_t)(n - k1);
  }
  KAD_HIP_CHECK(hipMemcpyAsync(w.swap_map, maps.data(), tot * sizeof(int), hipMemcpyHostToDevice, w.stream));
  for (int p = 0; p + 1 < np; ++p) {
    const int k0 = p * nb, k1 = k0 + nb;
    const int nrows = n - k1;
    const int chunk = (int)std::max<size_t>(1, std::min<size_t>(k1 - k0, w.tmp_bytes / sizeof(T) / nrows));
    for (int c = k0; c < k1; c += chunk) {
      const int nc = std::min(chunk, k1 - c);
      dim3 g((unsigned)cdiv(nrows, 256), nc);
      gather_rows_kernel<T><<<g, 256, 0, w.stream>>>(A + (int64_t)c * lda, lda, w.swap_map + moff[p], nrows,
                                                     (T*)w.tmp, nrows);
      copy2d_kernel<T><<<g, 256, 0, w.stream>>>((const T*)w.tmp, nrows, A + k1 + (int64_t)c * lda, lda, nrows, nc);
      KAD_HIP_CHECK(hipGetLastError());
    }
  }
  // the host map buffer must outlive its asynchronous upload
  KAD_HIP_CHECK(hipStreamSynchronize(w.stream));
  return KAD_OK;
}

// Full factorisation.  gemm_prec selects the trailing-update MFMA precision
// (F64 for double storage; F32 or BF16 for float storage).
//
// Look-ahead of depth one on two streams of the same priority.  For step p (panel
// [k0, k1), next panel [k1, k2), the one after [k2, k3)):
//   panel stream: interchanges, U12 and update of the next panel's columns
//     [k1, k2), then the next panel's factorisation and its L21 row-tile mask;
//   main stream, part A: interchanges, U12 and update of [k2, k3) only, then the
//     signal the panel stream waits for at step p+1;
//   main stream, part B: interchanges, U12 and update of [k3, n) -- the bulk of the
//     step, which runs beside the next panel instead of ahead of it.
// Events (ping-pong by step parity so a new record never overtakes a pending
// wait): ev_panel "panel p and its mask are done", ev_next "columns of the panel
// after next are up to date".  The two streams work on disjoint columns, and the L21
// row-tile masks rotate over three buffers: part B of step p still reads panel p's mask
// while the panel stream writes panel p+2's.
//
// A batch (bt.nbat > 1) factors bt.nbat matrices of order n together: every launch
// covers all of them, so the panel chain is that of one matrix.  The matrices are
// taken as dense (no structural-zero masks or row extents).
template <typename T>
int getrf(T* A, int64_t lda, int n, int* ipiv, int nb, int gemm_prec, LuWork& w, const LuBatch& bt) {
  // both streams' scratch must exist before anything is launched
  if (!w.stream2 || !w.tmp || !w.tmp2 ||
      !w.mask_r || !w.mask_r2 || !w.mask_r3 || !w.ext)
    return KAD_ERR_ALLOC;
  LuWork wp = w;  // panel stream: tmp, tmp2 and the panel reductions
  wp.stream = w.stream2;
  // the persistent panel's launch sequence advances in wp; it outlives this call on
  // every return path (reused flags would let stale exchange slots look current)
  struct SeqBack {
    LuWork& to;
    const LuWork& from;
    ~SeqBack() { to.ffp_seq = from.ffp_seq; }
  } seq_back{w, wp};
  int* mask_rows[3] = {w.mask_r, w.mask_r2, w.mask_r3};
  const int stride = (int)cdiv(n, 128) + 1;
  // Row extent of every 128-column tile of the input (one pass, one readback).
  // A panel's rows at or below R are zero in its columns and stay zero: the
  // interchanges and the update of an earlier panel q touch rows above R_q only,
  // so R_p = max(initial extent of p's columns, R_q for q < p) bounds them.
  // a batch, or static pivoting: no masks, no row extents, the persistent panel or the
  // static-pivot panel (no interchanges at all)
  const bool bat = bt.nbat > 1 || bt.nopiv;
  const bool piv = !bt.nopiv;
  if (bt.nbat < 1 || bt.nbat > LU_MAX_BATCH) return arg_error("getrf: batch size");
  if (bt.nopiv) {
    if (!bt.growth) return arg_error("getrf: static pivoting needs growth words");
    KAD_HIP_CHECK(hipMemsetAsync(bt.growth, 0, bt.nbat * sizeof(unsigned long long), w.stream));
  }
  const int ntc = (int)cdiv(n, 128), nrc = (int)cdiv(n, 256);
  std::vector<int> ext(ntc, bat ? n - 1 : -1);
  if (!bat) {
    if (nrc > 1) KAD_HIP_CHECK(hipMemsetAsync(w.ext, 0xff, ntc * sizeof(int), w.stream));  // -1
    col_extent_kernel<T><<<dim3(ntc, nrc), 256, 0, w.stream>>>(A, lda, n, w.ext);
    KAD_HIP_CHECK(hipGetLastError());
    KAD_HIP_CHECK(hipMemcpyAsync(ext.data(), w.ext, ntc * sizeof(int), hipMemcpyDeviceToHost, w.stream));
    KAD_HIP_CHECK(hipStreamSynchronize(w.stream));
  }
  int r_prev = 0;
  // factor panel [k0, k1) on the panel stream (rows [k0, R)), then its L21 mask
  auto panel = [&](int k0, int k1, int* mask) -> int {
    int R = std::max(k1, r_prev);
    for (int t = k0 / 128; t <= (k1 - 1) / 128; ++t) R = std::max(R, ext[t] + 1);
    R = std::min(R, n);
    r_prev = R;
    FfpShape fs;
    const bool fused = bt.nopiv || (wp.ffp && !wp.ffp_off && ffp_shape(R - k0, bt.nbat, wp.ncu, fs));
    int rc = panel_rec<T>(A, lda, R, k0, k1, ipiv, wp, k0, k1, fused, bt);
    if (rc) return rc;
    if (k1 < n && mask) {
      // the panel's rows at or below R are zero in its columns
      row_tile_mask_kernel<T><<<(unsigned)cdiv(n - k1, 128), 1024, 0, wp.stream>>>(A + k1 + (int64_t)k0 * lda, lda,
                                                                                 n - k1, k1 - k0, mask, R - k1);
      KAD_HIP_CHECK(hipGetLastError());
    }
    return KAD_OK;
  };
  // the caller's work on the main stream precedes the first panel
  KAD_HIP_CHECK(hipEventRecord(w.ev_start, w.stream));
  KAD_HIP_CHECK(hipStreamWaitEvent(wp.stream, w.ev_start, 0));
  int rc = panel(0, std::min(nb, n), bat ? nullptr : mask_rows[0]);
  if (rc) return rc;
  KAD_HIP_CHECK(hipEventRecord(w.ev_panel[0], wp.stream));
  for (int p = 0, k0 = 0; k0 < n; ++p, k0 += nb) {
    const int k1 = std::min(k0 + nb, n);
    const int k2 = std::min(k1 + nb, n);
    const int k3 = std::min(k2 + nb, n);
    const int par = p & 1;
    const int* mrows = bat ? nullptr : mask_rows[p % 3];
    const T* L21 = A + k1 + (int64_t)k0 * lda;
    const T* L11 = A + k0 + (int64_t)k0 * lda;
    // ---- main stream, part A: columns [k2, k3)
    KAD_HIP_CHECK(hipStreamWaitEvent(w.stream, w.ev_panel[par], 0));
    if (k1 >= n) break;
    if (k2 < n && bat) {
      if (piv && (rc = laswp<T>(A, lda, k2, k3, ipiv, k0, k1, w, bt))) return rc;
      rc = trsm_left_unit_lower<T>(L11, lda, k1 - k0, A + k0 + (int64_t)k2 * lda, lda, k3 - k2, w, gemm_prec,
                                   nullptr, bt.nbat, bt.sA, bt.sA);
      if (rc) return rc;
      rc = gemm_launch_batched(gemm_prec, GOP_SUB, n - k1, k3 - k2, k1 - k0, L21, lda, bt.sA,
                               A + k0 + (int64_t)k2 * lda, lda, bt.sA, A + k1 + (int64_t)k2 * lda, lda, bt.sA,
                               bt.nbat, w.stream);
      if (rc) return rc;
    } else if (k2 < n) {
      rc = laswp<T>(A, lda, k2, k3, ipiv, k0, k1, w);
      if (rc) return rc;
      // structural zeros of A12 (column tiles; U12 = L11^{-1} A12 keeps them)
      col_tile_mask_kernel<T><<<(unsigned)cdiv(k3 - k2, 128), 1024, 0, w.stream>>>(A + k0 + (int64_t)k2 * lda, lda,
                                                                                 k1 - k0, k3 - k2, w.mask_c);
      KAD_HIP_CHECK(hipGetLastError());
      rc = trsm_left_unit_lower<T>(L11, lda, k1 - k0, A + k0 + (int64_t)k2 * lda, lda, k3 - k2, w, gemm_prec,
                                   w.mask_c);
      if (rc) return rc;
      rc = gemm_launch_masked(gemm_prec, GOP_SUB, n - k1, k3 - k2, k1 - k0, L21, lda, A + k0 + (int64_t)k2 * lda, lda,
                              A + k1 + (int64_t)k2 * lda, lda, mrows, w.mask_c, w.stream);
      if (rc) return rc;
    }
    KAD_HIP_CHECK(hipEventRecord(w.ev_next[par], w.stream));
    // ---- main stream, part B: columns [k3, n), beside the next panel
    if (k3 < n && bat) {
      if (piv && (rc = laswp<T>(A, lda, k3, n, ipiv, k0, k1, w, bt))) return rc;
      rc = trsm_left_unit_lower<T>(L11, lda, k1 - k0, A + k0 + (int64_t)k3 * lda, lda, n - k3, w, gemm_prec,
                                   nullptr, bt.nbat, bt.sA, bt.sA);
      if (rc) return rc;
      rc = gemm_launch_batched(gemm_prec, GOP_SUB, n - k1, n - k3, k1 - k0, L21, lda, bt.sA,
                               A + k0 + (int64_t)k3 * lda, lda, bt.sA, A + k1 + (int64_t)k3 * lda, lda, bt.sA,
                               bt.nbat, w.stream);
      if (rc) return rc;
    } else if (k3 < n) {
      rc = laswp<T>(A, lda, k3, n, ipiv, k0, k1, w);
      if (rc) return rc;
      col_tile_mask_kernel<T><<<(unsigned)cdiv(n - k3, 128), 1024, 0, w.stream>>>(A + k0 + (int64_t)k3 * lda, lda,
                                                                                k1 - k0, n - k3, w.mask_c2);
      KAD_HIP_CHECK(hipGetLastError());
      rc = trsm_left_unit_lower<T>(L11, lda, k1 - k0, A + k0 + (int64_t)k3 * lda, lda, n - k3, w, gemm_prec,
                                   w.mask_c2);
      if (rc) return rc;
      // active tile pairs of the update, compacted on the grid (all XCDs busy)
      tile_lists_kernel<<<1, 64, 0, w.stream>>>(mrows, (int)cdiv(n - k1, 128), w.mask_c2, (int)cdiv(n - k3, 128),
                                                w.tile_list, stride);
      KAD_HIP_CHECK(hipGetLastError());
      TileSel sel;
      sel.rlist = w.tile_list;
      sel.clist = w.tile_list + stride;
      sel.cnt = w.tile_list + 2 * stride;
      rc = gemm_launch_sel(gemm_prec, GOP_SUB, n - k1, n - k3, k1 - k0, L21, lda, A + k0 + (int64_t)k3 * lda, lda,
                           A + k1 + (int64_t)k3 * lda, lda, sel, w.stream);
      if (rc) return rc;
    }
    // ---- panel stream: the next panel's columns [k1, k2), then the next panel
    if (p > 0) KAD_HIP_CHECK(hipStreamWaitEvent(wp.stream, w.ev_next[par ^ 1], 0));
    if (piv && (rc = laswp<T>(A, lda, k1, k2, ipiv, k0, k1, wp, bt))) return rc;
    rc = trsm_left_unit_lower<T>(L11, lda, k1 - k0, A + k0 + (int64_t)k1 * lda, lda, k2 - k1, wp, gemm_prec, nullptr,
                                 bt.nbat, bt.sA, bt.sA);
    if (rc) return rc;
    rc = bat ? gemm_launch_batched(gemm_prec, GOP_SUB, n - k1, k2 - k1, k1 - k0, L21, lda, bt.sA,
                                   A + k0 + (int64_t)k1 * lda, lda, bt.sA, A + k1 + (int64_t)k1 * lda, lda, bt.sA,
                                   bt.nbat, wp.stream)
             : gemm_launch_masked(gemm_prec, GOP_SUB, n - k1, k2 - k1, k1 - k0, L21, lda, A + k0 + (int64_t)k1 * lda,
                                  lda, A + k1 + (int64_t)k1 * lda, lda, mrows, nullptr, wp.stream);
    if (rc) return rc;
    rc = panel(k1, k2, bat ? nullptr : mask_rows[(p + 1) % 3]);
    if (rc) return rc;
    KAD_HIP_CHECK(hipEventRecord(w.ev_panel[par ^ 1], wp.stream));
  }
  for (int z = 0; z < bt.nbat && piv; ++z)
    if ((rc = apply_left_swaps<T>(A + z * bt.sA, lda, n, ipiv + (int64_t)z * bt.sP, nb, w))) return rc;
  return KAD_OK;
}

template int getrf<double>(double*, int64_t, int, int*, int, int, LuWork&, const LuBatch&);
template int getrf<float>(float*, int64_t, int, int*, int, int, LuWork&, const LuBatch&);

// perm from LAPACK-style ipiv (host side, O(n)).
// Returns false (perm unspecified) if some ipiv[i] is outside [i, n): interchanges read
// back from the device are checked before they index host memory.
bool ipiv_to_perm(const int* ipiv, int n, int* perm) {
  for (int i = 0; i < n; ++i) perm[i] = i;
  for (int i = 0; i < n; ++i) {
    const int p = ipiv[i];
    if (p < i || p >= n) return false;
    if (p != i) std::swap(perm[i], perm[p]);
  }
  return true;
}

// ---------------------------------------------------------------------------
// fp64 GEMV  y = b - A x  (or y = A x when b == nullptr), A column-major n x n.
// Two passes: partial sums per (row block, column chunk), then a fixed-order
// reduction, so results are bitwise reproducible.
// ---------------------------------------------------------------------------
constexpr int GEMV_CHUNK = 1024;

__global__ __launch_bounds__(256) void gemv_partial_kernel(const double* __restrict__ A, int64_t lda, int n,
                                                           const double* __restrict__ x, double* __restrict__ part,
                                                           int trans) {
  const int chunk = blockIdx.y;
  const int c0 = chunk * GEMV_CHUNK, c1 = min(n, c0 + GEMV_CHUNK);
  if (!trans) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double s = 0.0;
    const double* a = A + i;
    for (int c = c0; c < c1; ++c) s += a[(int64_t)c * lda] * x[c];
    part[(int64_t)chunk * n + i] = s;
  }
}

__global__ void gemv_reduce_kernel(const double* __restrict__ part, int nchunk, int n, const double* __restrict__ b,
                                   double* __restrict__ y) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double s = 0.0;
  for (int c = 0; c < nchunk; ++c) s += part[(int64_t)c * n + i];
  y[i] = b ? b[i] - s : s;
}

// y = A^T x  (one workgroup per column)
__global__ __launch_bounds__(256) void gemv_t_kernel(const double* __restrict__ A, int64_t lda, int n,
                                                     const double* __restrict__ x, const double* __restrict__ b,
                                                     double* __restrict__ y) {
  __shared__ double red[256];
  const int c = blockIdx.x;
  const double* a = A + (int64_t)c * lda;
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) s += a[i] * x[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if (threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) y[c] = b ? b[c] - red[0] : red[0];
}

int gemv64(const double* A, int64_t lda, int n, const double* x, const double* b, double* y, int trans, double* part,
           hipStream_t s) {
  if (!trans) {
    const int nchunk = (int)cdiv(n, GEMV_CHUNK);
    dim3 g((unsigned)cdiv(n, 256), nchunk);
    gemv_partial_kernel<<<g, 256, 0, s>>>(A, lda, n, x, part, 0);
    gemv_reduce_kernel<<<(unsigned)cdiv(n, 256), 256, 0, s>>>(part, nchunk, n, b, y);
  } else {
    gemv_t_kernel<<<n, 256, 0, s>>>(A, lda, n, x, b, y);
  }
  KAD_HIP_CHECK(hipGetLastError());
  return KAD_OK;
}

// ---------------------------------------------------------------------------
// Small vector kernels.
// ---------------------------------------------------------------------------
__global__ void axpy_kernel(int n, double a, const double* x, double* y) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] += a * x[i];
}
__global__ void cast_d2f_kernel(const double* __restrict__ a, float* __restrict__ b, int64_t nel) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nel) b[i] = (float)a[i];
}
// Column-major n x n copy with leading dimensions, fp64 -> fp32.
__global__ void cast_mat_d2f_kernel(const double* __restrict__ a, int64_t lda, float* __restrict__ b, int64_t ldb,
                                    int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int c = blockIdx.y;
  if (i < n) b[i + (int64_t)c * ldb] = (float)a[i + (int64_t)c * lda];
}
// Equilibration by powers of two (LAPACK dgeequb-style, exact in fp64):
// R_i = 2^-round(log2 max_j |a_ij|), then C_j = 2^-round(log2 max_i |R_i a_ij|).
__device__ inline double pow2_recip(double m) {
  if (!(m > 0.0) || !isfinite(m)) return 1.0;
  int e;
  frexp(m, &e);  // m = f 2^e, f in [0.5, 1)
  return ldexp(1.0, 1 - e);
}
__global__ __launch_bounds__(256) void row_absmax_kernel(const double* __restrict__ A, int64_t lda, int n,
                                                         double* __restrict__ R) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double m = 0.0;
  for (int c = 0; c < n; ++c) m = fmax(m, fabs(A[i + (int64_t)c * lda]));
  R[i] = pow2_recip(m);
}
__global__ __launch_bounds__(256) void col_scale_kernel(double* __restrict__ A, int64_t lda, int n,
                                                        const double* __restrict__ R, double* __restrict__ C) {
  __shared__ double red[256];
  const int c = blockIdx.x;
  double* a = A + (int64_t)c * lda;
  double m = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) m = fmax(m, fabs(R[i] * a[i]));
  red[threadIdx.x] = m;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  const double cj = pow2_recip(red[0]);
  if (threadIdx.x == 0) C[c] = cj;
  for (int i = threadIdx.x; i < n; i += 256) a[i] = R[i] * a[i] * cj;
}
// Column scales of diag(R) A without modifying A.
__global__ __launch_bounds__(256) void col_scale_only_kernel(const double* __restrict__ A, int64_t lda, int n,
                                                             const double* __restrict__ R, double* __restrict__ C) {
  __shared__ double red[256];
  const int c = blockIdx.x;
  const double* a = A + (int64_t)c * lda;
  double m = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) m = fmax(m, fabs(R[i] * a[i]));
  red[threadIdx.x] = m;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) C[c] = pow2_recip(red[0]);
}
// B = (float)(R_i A_ij C_j)
__global__ void cast_scaled_kernel(const double* __restrict__ a, int64_t lda, float* __restrict__ b, int64_t ldb,
                                   int n, const double* __restrict__ R, const double* __restrict__ C) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int c = blockIdx.y;
  if (i < n) b[i + (int64_t)c * ldb] = (float)(R[i] * a[i + (int64_t)c * lda] * C[c]);
}
__global__ void vec_scale_kernel(int n, const double* __restrict__ s, double* __restrict__ v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] *= s[i];
}

// Block reduction for max |x| and for dot products (fixed order, two passes).
__global__ __launch_bounds__(256) void absmax_partial_kernel(const double* x, int n, double* part) {
  __shared__ double red[256];
  double m = 0.0;
  // NaN propagates (fmax would drop it): a NaN residual must never read as converged
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const double a = fabs(x[i]);
    m = (a > m || a != a) ? a : m;
  }
  red[threadIdx.x] = m;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) {
      const double o = red[threadIdx.x + s];
      if (o > red[threadIdx.x] || o != o) red[threadIdx.x] = o;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}
// h[i] = <V_i, w> for i < k  (V: k vectors of length n, contiguous), one workgroup per i
__global__ __launch_bounds__(256) void multidot_kernel(const double* __restrict__ V, int n, int k,
                                                       const double* __restrict__ w, double* __restrict__ h) {
  __shared__ double red[256];
  const double* v = V + (int64_t)blockIdx.x * n;
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) s += v[i] * w[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if (threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) h[blockIdx.x] = red[0];
}
// w -= sum_i h[i] V_i   (or, with sub = 0, w = sum_i h[i] V_i)
__global__ void multiaxpy_kernel(const double* __restrict__ V, int n, int k, const double* __restrict__ h,
                                 double* __restrict__ w, int sub) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  double s = 0.0;
  for (int i = 0; i < k; ++i) s += h[i] * V[(int64_t)i * n + e];
  w[e] = sub ? w[e] - s : s;
}
__global__ __launch_bounds__(256) void dot_partial_kernel(const double* x, const double* y, int n, double* part) {
  __shared__ double red[256];
  double m = 0.0;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) m += x[i] * y[i];
  red[threadIdx.x] = m;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

}  // namespace kad
