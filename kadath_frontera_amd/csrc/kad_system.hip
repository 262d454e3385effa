// Device-resident Newton step of the XCTS system: executes the traced programs
// (value program -> residual F; tangent programs -> Jacobian columns, batched
// over unit seeds), factors and solves, and updates the fields in place.
//
// Replaces System_of_eqs::do_newton (src_par/do_newton.cpp:65-430):
//   sec_member / check_equations   -> value program + |F|_inf
//   do_col_J over all columns      -> tangent programs, at most B columns of each at a time
//   pdgesv_                        -> kad LU (fp64) or low-precision LU + fp64 refinement
//   xx_to_vars + old - var         -> CSR update kernel on the coefficient arrays
#include "kad_common.hpp"
#include "kad_ctx.hpp"
#include "kad_apply3d.hpp"
#include "kad_group.hpp"
#include "host/xcts.hpp"
#include "host/parsed_system.hpp"
#include "../../include/kadath_amd.h"
#include <array>
#include <map>
#include <vector>
#include <chrono>
#include <algorithm>
#include <stdexcept>
#include <cstring>
#include <functional>

namespace kad {
template <typename T>
int getrf(T* A, int64_t lda, int n, int* ipiv, int nb, int gemm_prec, LuWork& w, const LuBatch& bt = LuBatch());
bool ipiv_to_perm(const int* ipiv, int n, int* perm);
// kad_dd_solve right after a factorisation of the same, unchanged J (kad_dd.hip)
int dd_solve_after_factor(kad_dd* dd, const double* J, int64_t ldj, const double* b, double* x, double tol,
                          int max_outer, int* iters, double* resid);
}  // namespace kad

using namespace kadhost;

namespace {

using kad::DevRow;
using kad::ew_op;
static_assert(EW_ADD == kad::EWOP_ADD && EW_SUB == kad::EWOP_SUB && EW_MUL == kad::EWOP_MUL &&
                  EW_DIV == kad::EWOP_DIV && EW_SCAL == kad::EWOP_SCAL && EW_ADDS == kad::EWOP_ADDS &&
                  EW_COPY == kad::EWOP_COPY && EW_SDIV == kad::EWOP_SDIV,
              "the tracer's element-wise kinds are the kernels'");

// The same over 16-byte-aligned rows of even length: every thread takes EW_U pairs of
// elements, their loads issued together (one element per thread left each wave
// waiting out one load's latency at a time).
constexpr int EW_U = 2;
__global__ __launch_bounds__(256) void ew2_kernel(int kind, double* __restrict__ dst, int64_t dstride,
                                                  const double* __restrict__ a, int64_t astride,
                                                  const double* __restrict__ bsrc, int64_t bstride, double s,
                                                  int size2, int nbatch) {
  for (int bb = blockIdx.y; bb < nbatch; bb += gridDim.y) {
    const double2* ar = reinterpret_cast<const double2*>(a + (int64_t)bb * astride);
    const double2* br = bsrc ? reinterpret_cast<const double2*>(bsrc + (int64_t)bb * bstride) : nullptr;
    double2* dr = reinterpret_cast<double2*>(dst + (int64_t)bb * dstride);
    const int e0 = (blockIdx.x * 256 * EW_U) + threadIdx.x;
    double2 x[EW_U], y[EW_U];
#pragma unroll
    for (int u = 0; u < EW_U; ++u) {
      const int e = e0 + u * 256;
      x[u] = e < size2 ? ar[e] : double2{0.0, 0.0};
      y[u] = (br && e < size2) ? br[e] : double2{0.0, 0.0};
    }
#pragma unroll
    for (int u = 0; u < EW_U; ++u) {
      const int e = e0 + u * 256;
      if (e < size2) dr[e] = double2{ew_op(kind, x[u].x, y[u].x, s), ew_op(kind, x[u].y, y[u].y, s)};
    }
  }
}

// An element-wise instruction followed by the ones it absorbed (kad::PostOp): the
// first instruction's result goes through the chain and only the last one is stored.
__global__ __launch_bounds__(256) void ewc_kernel(int kind, const double* __restrict__ a, int64_t astride,
                                                  const double* __restrict__ bsrc, int64_t bstride, double s,
                                                  kad::PostOp post, int size, int nbatch) {
  for (int bb = blockIdx.y; bb < nbatch; bb += gridDim.y) {
    const double* ar = a + (int64_t)bb * astride;
    const double* br = bsrc ? bsrc + (int64_t)bb * bstride : nullptr;
    double* dr = post.dst + (int64_t)bb * post.ds;
    const int e0 = blockIdx.x * 256 * EW_U + threadIdx.x;
    // every load of the EW_U elements first (operands of the head and of every step)
    double x[EW_U], y[EW_U], o[EW_U][kad::kMaxChain];
#pragma unroll
    for (int u = 0; u < EW_U; ++u) {
      const int e = e0 + u * 256;
      const bool in = e < size;
      x[u] = in ? ar[e] : 0.0;
      y[u] = (in && br) ? br[e] : 0.0;
      kad::post_load(post, bb, in ? e : 0, o[u]);
    }
#pragma unroll
    for (int u = 0; u < EW_U; ++u) {
      const int e = e0 + u * 256;
      if (e < size) dr[e] = kad::post_ops(post, ew_op(kind, x[u], y[u], s), o[u]);
    }
  }
}

// dst[b][e] = op(a[b or 0][e], b[b or 0][e], s)
// Element-wise instruction over a batch: blockIdx.y walks the batch rows (a stride of
// 0 broadcasts one array to every row), blockIdx.x / threadIdx.x the elements.
__global__ void ew_kernel(int kind, double* __restrict__ dst, int64_t dstride, const double* __restrict__ a,
                          int64_t astride, const double* __restrict__ bsrc, int64_t bstride, double s, int size,
                          int nbatch) {
  for (int bb = blockIdx.y; bb < nbatch; bb += gridDim.y) {
    const double* ar = a + (int64_t)bb * astride;
    const double* br = bsrc ? bsrc + (int64_t)bb * bstride : nullptr;
    double* dr = dst + (int64_t)bb * dstride;
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < size; e += gridDim.x * blockDim.x) {
      const double x = ar[e];
      double r;
      switch (kind) {
        case EW_ADD: r = x + br[e]; break;
        case EW_SUB: r = x - br[e]; break;
        case EW_MUL: r = x * br[e]; break;
        case EW_DIV: r = x / br[e]; break;
        case EW_SCAL: r = x * s; break;
        case EW_SDIV: r = x / s; break;
        case EW_ADDS: r = x + s; break;
        default: r = x; break;
      }
      dr[e] = r;
    }
  }
}

// Inside rows: out[(row0 + r) + (col0 + b) ldo] (+)= sign (src[pos] - gw src[gpos])
template <typename T>
__global__ void export_in_kernel(const DevRow* __restrict__ rows, int nrows, const double* __restrict__ src,
                                 int64_t sstride, T* __restrict__ out, int row0, int64_t col0, int64_t ldo,
                                 double sign, int acc, int nbatch) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)nrows * nbatch) return;
  const int64_t bb = t / nrows;
  const int r = (int)(t % nrows);
  const DevRow R = rows[r];
  const double* x = src + bb * sstride;
  double v = x[R.pos];
  if (R.gpos >= 0) v -= R.gw * x[R.gpos];
  T* o = out + (row0 + r) + (col0 + bb) * ldo;
  *o = acc ? (T)((double)*o + sign * v) : (T)(sign * v);
}

// Boundary rows: X(line) = sum_i bsign^i cf(i, line)  (val_boundary, domain_shell_systems.cpp:43-74)
template <typename T>
__global__ void export_bd_kernel(const DevRow* __restrict__ rows, int nrows, const double* __restrict__ src,
                                 int64_t sstride, int nr, int bsign, T* __restrict__ out, int row0,
                                 int64_t col0, int64_t ldo, double sign, int acc, int nbatch) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)nrows * nbatch) return;
  const int64_t bb = t / nrows;
  const int r = (int)(t % nrows);
  const DevRow R = rows[r];
  const double* x = src + bb * sstride;
  double v = 0.0, g = 0.0, sg = 1.0;
  for (int i = 0; i < nr; ++i) {
    v += sg * x[i + (int64_t)nr * R.pos];
    if (R.gpos >= 0) g += sg * x[i + (int64_t)nr * R.gpos];
    sg *= bsign;
  }
  if (R.gpos >= 0) v -= R.gw * g;
  T* o = out + (row0 + r) + (col0 + bb) * ldo;
  *o = acc ? (T)((double)*o + sign * v) : (T)(sign * v);
}

// Transposed exports (the VJP of the row export): for every column b of the batch,
// out[col0 + b] += sign * sum_r w[row0 + r] row_r(b), where row_r is the inside
// (bd = 0) or boundary (bd = 1) row recipe above.  One workgroup per column, a
// fixed-order reduction, and instructions run in stream order: deterministic.
__global__ __launch_bounds__(256) void export_dot_kernel(const DevRow* __restrict__ rows, int nrows, int bd,
                                                         const double* __restrict__ src, int64_t sstride, int nr,
                                                         int bsign, const double* __restrict__ w, int row0,
                                                         double* __restrict__ out, int64_t col0, double sign) {
  __shared__ double red[256];
  const int bb = blockIdx.x;
  const double* x = src + (int64_t)bb * sstride;
  double acc = 0.0;
  for (int r = threadIdx.x; r < nrows; r += 256) {
    const DevRow R = rows[r];
    double v;
    if (!bd) {
      v = x[R.pos];
      if (R.gpos >= 0) v -= R.gw * x[R.gpos];
    } else {
      double g = 0.0, sg = 1.0;
      v = 0.0;
      for (int i = 0; i < nr; ++i) {
        v += sg * x[i + (int64_t)nr * R.pos];
        if (R.gpos >= 0) g += sg * x[i + (int64_t)nr * R.gpos];
        sg *= bsign;
      }
      if (R.gpos >= 0) v -= R.gw * g;
    }
    acc += w[row0 + r] * v;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if (threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[col0 + bb] += sign * red[0];
}

// Unit seeds of unknowns u0 .. u0 + nbatch - 1 (affecte_tau_one_coef), zero elsewhere.
__global__ void seed_kernel(double* __restrict__ dst, int64_t dstride, int size, const int* __restrict__ spos,
                            const double* __restrict__ sval, const int* __restrict__ scnt, int u0, int nu,
                            int nbatch) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)size * nbatch) return;
  const int bb = (int)(t / size);
  const int e = (int)(t % size);
  const int u = u0 + bb;
  double v = 0.0;
  if (u < nu)
    for (int q = 0; q < scnt[u]; ++q)
      if (spos[3 * u + q] == e) v = sval[3 * u + q];
  dst[(int64_t)bb * dstride + e] = v;
}

// cf[q] += scale * sum_t w[t] X[off + col[t]]   (affecte_tau as a sparse map)
__global__ void csr_update_kernel(double* __restrict__ cf, const int* __restrict__ rowptr, const int* __restrict__ col,
                                  const double* __restrict__ w, const double* __restrict__ X, int off, int ncf,
                                  double scale) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= ncf) return;
  double s = 0.0;
  for (int t = rowptr[q]; t < rowptr[q + 1]; ++t) s += w[t] * X[off + col[t]];
  cf[q] += scale * s;
}

// max |x| over one workgroup.  A NaN propagates (fmax would drop it): a residual
// holding a NaN must read as NaN, so that do_newton never reports it as converged
// (the reference's max starts from data[0] and keeps a NaN there too).
__global__ void absmax_kernel(const double* x, int n, double* out) {
  __shared__ double red[256];
  double m = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) {
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
  if (threadIdx.x == 0) *out = red[0];
}

// sum of squares (compute_f of the line search, do_newton.cpp:594-599) and signed maximum
// (Array max, array_math.cpp:308-314) of x[0..n), one workgroup; out[0] = sum, out[1] = max.
// A NaN reaches both results.
__global__ void sumsq_max_kernel(const double* x, int n, double* out) {
  __shared__ double rs[256], rm[256];
  double s = 0.0, m = n > 0 ? x[0] : 0.0;
  for (int i = threadIdx.x; i < n; i += 256) {
    const double a = x[i];
    s += a * a;
    m = (a > m || a != a) ? a : m;
  }
  rs[threadIdx.x] = s;
  rm[threadIdx.x] = m;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (threadIdx.x < k) {
      rs[threadIdx.x] += rs[threadIdx.x + k];
      const double o = rm[threadIdx.x + k];
      if (o > rm[threadIdx.x] || o != o) rm[threadIdx.x] = o;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = rs[0];
    out[1] = rm[0];
  }
}

// B = A^T for an n x n column-major matrix: 64 x 64 tiles through LDS (padded row), both
// sides coalesced.  Grid (cdiv(n, 64), cdiv(n, 64)), 256 threads.
__global__ __launch_bounds__(256) void transpose_kernel(const double* __restrict__ A, int64_t lda,
                                                        double* __restrict__ B, int64_t ldb, int n) {
  __shared__ double t[64][65];
  const int r0 = blockIdx.x * 64, c0 = blockIdx.y * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int c = ty; c < 64; c += 4) {
    const int gr = r0 + tx, gc = c0 + c;
    t[c][tx] = (gr < n && gc < n) ? A[gr + (int64_t)gc * lda] : 0.0;
  }
  __syncthreads();
  // B(c0 + tx, r0 + r) = A(r0 + r, c0 + tx)
  for (int r = ty; r < 64; r += 4) {
    const int gr = c0 + tx, gc = r0 + r;
    if (gr < n && gc < n) B[gr + (int64_t)gc * ldb] = t[tx][r];
  }
}

// Surface integral of one quantity (Domain_compact::integ, domain_compact.cpp:89-121):
// cf holds the coefficients of r r sin(theta) so; value on the boundary x = bsign of
// phi coefficient 0, theta weights pi (COS_EVEN, j = 0) or 2/(2j+1) (SIN_ODD), times
// 2 pi and fac.  One workgroup.
__global__ void surface_integral_kernel(const double* __restrict__ cf, int nr, int nt, int bt0, int bsign,
                                        double fac, double* __restrict__ out) {
  __shared__ double red[64];
  const int j = threadIdx.x;
  double v = 0.0;
  if (j < nt && (bt0 == COS_EVEN || bt0 == SIN_ODD)) {
    double b = 0.0, sg = 1.0;
    for (int i = 0; i < nr; ++i) {
      b += sg * cf[i + (int64_t)nr * j];
      sg *= bsign;
    }
    if (bt0 == COS_EVEN) v = (j == 0) ? M_PI * b : 0.0;
    else v = 2.0 / (2.0 * j + 1.0) * b;
  }
  red[threadIdx.x] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int q = 0; q < 64; ++q) t += red[q];
    *out = t * 2.0 * M_PI * fac;
  }
}

// Per column b: fac * 2 pi * sum_j w_j sum_i cf_b(i, j, k = 0) (the integ weights of
// surface_integral_kernel at the outer boundary) into out[b + q ldo].
__global__ void export_int_kernel(const double* __restrict__ src, int64_t sstride, int nr, int nt, int bt0,
                                  double fac, double* __restrict__ out, int q, int64_t col0, int64_t ldo,
                                  int nbatch) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nbatch) return;
  const double* x = src + (int64_t)b * sstride;
  double tot = 0.0;
  if (bt0 == COS_EVEN || bt0 == SIN_ODD) {
    for (int j = 0; j < nt; ++j) {
      const double w = bt0 == COS_EVEN ? (j == 0 ? M_PI : 0.0) : 2.0 / (2.0 * j + 1.0);
      if (w == 0.0) continue;
      double v = 0.0;
      for (int i = 0; i < nr; ++i) v += x[i + (int64_t)nr * j];
      tot += w * v;
    }
  }
  out[col0 + b + (int64_t)q * ldo] = tot * 2.0 * M_PI * fac;
}

// Integral-equation row (Domain::integ at x = bsign of the coefficients of r r sin(theta)
// so, theta weights of phi coefficient 0 (pi for COS_EVEN j = 0, 2/(2j+1) for SIN_ODD),
// times 2 pi and fac): value programs write out[row] = v + c0 (or add v); tangent
// programs write J(row, col0 + b) (column-major, ld ldo, always added: J is cleared);
// with w, the transposed export adds w[row] v to out[col0 + b].  src == nullptr: the
// constant alone.
template <typename T>
__global__ void export_gl_kernel(const double* __restrict__ src, int64_t sstride, int nr, int nt, int bt0,
                                 int bsign, double fac, double c0, int acc, int pt, T* __restrict__ out, int row,
                                 int64_t col0, int64_t ldo, const double* __restrict__ w, int nbatch) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nbatch) return;
  double tot = 0.0;
  if (src && pt) {
    // point value of a constant field (a parameter): entry 0 of its array, times fac
    const double val = src[(int64_t)b * sstride] * fac;
    if (w) {
      ((double*)out)[col0 + b] += w[row] * val;
      return;
    }
    T* o = out + row + (col0 + b) * ldo;
    *o = acc ? (T)((double)*o + val + c0) : (T)(val + c0);
    return;
  }
  if (src && (bt0 == COS_EVEN || bt0 == SIN_ODD)) {
    const double* x = src + (int64_t)b * sstride;
    for (int j = 0; j < nt; ++j) {
      const double wj = bt0 == COS_EVEN ? (j == 0 ? M_PI : 0.0) : 2.0 / (2.0 * j + 1.0);
      if (wj == 0.0) continue;
      double v = 0.0, sg = 1.0;
      for (int i = 0; i < nr; ++i) {
        v += sg * x[i + (int64_t)nr * j];
        sg *= bsign;
      }
      tot += wj * v;
    }
  }
  const double val = tot * 2.0 * M_PI * fac;
  if (w) {
    ((double*)out)[col0 + b] += w[row] * val;
    return;
  }
  T* o = out + row + (col0 + b) * ldo;
  *o = acc ? (T)((double)*o + val + c0) : (T)(val + c0);
}

// Double unknowns' fields (constant fields of the value arena): v[e] += scale * X[k].
__global__ void double_update_kernel(double* __restrict__ v, int size, const double* __restrict__ X, int k,
                                     double scale) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < size) v[e] += scale * X[k];
}


struct DevProgram {
  std::vector<Instr> code;       // slots of tangent operands remapped to physical slots
  int nphys = 0;
  int seed_tab = -1;
  int field = 0, dom = 0, off = 0, cnt = 0;
};

// A program's instructions by dependency level (kad_group.hip): ops [op0 + lev[l],
// op0 + lev[l + 1]) of the device table run together.
struct GroupProg {
  bool ok = false;             // false: the program runs instruction by instruction
  int op0 = 0, nphys = 0;      // nphys: tangent slots of one column
  std::vector<int> lev;
  std::vector<int> ncl;        // per level: clusters among them (the last ones)
  std::vector<int> clsize;     // per level: elements of the largest cluster
  std::vector<size_t> lds;     // per level: the most LDS of an instruction
  std::vector<double> bytes;   // per level: algorithmic HBM bytes of one column (passes and element-wise)
};
// Columns [u0, u0 + nb) of a program, results in column col0 + (0 .. nb).
struct GroupItem {
  const GroupProg* p;
  int u0, nb;
  int64_t col0;
};

double now_s() {
  return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

}  // namespace

struct kad_system_impl {
  kad::Ctx* ctx = nullptr;
  SystemBase* sys = nullptr;
  XctsSystem* xsys = nullptr;  // the same object when the system is the hand-traced XCTS one
  int B = 256;
  int64_t stride = 0;          // doubles per slot per batch element
  double* val_arena = nullptr;  // nval_slots * stride
  double* tan_arena = nullptr;  // nphys_max * B * stride (grow_arena may give it more)
  size_t tan_cap = 0;           // doubles
  double* F = nullptr;          // n_rows
  double* scratch = nullptr;    // small
  std::vector<kad::LinePlan> plans;  // by the tracer's plan ids; npass 0: no instruction uses it
  std::vector<DevRow*> row_tabs;
  std::vector<int*> seed_pos;
  std::vector<double*> seed_val;
  std::vector<int*> seed_cnt;
  std::vector<int*> csr_rowptr, csr_col;
  std::vector<double*> csr_w;
  std::vector<DevProgram> tprogs;
  std::vector<DevProgram> obs_tprogs;  // d(observables)/d(unknowns)
  std::vector<DevProgram> par_progs;   // dF/dp of each parameter
  std::vector<DevProgram> glob_tprogs;      // dQ/du of the global quantities, per layout entry
  std::vector<DevProgram> glob_par_progs;   // dQ/dp at fixed fields, per parameter
  double* dQ = nullptr;                // 3 x n, row q contiguous
  double* dFdp = nullptr;              // n per parameter
  int nphys_max = 0;
  // dense linear algebra buffers (lazily allocated)
  double* J = nullptr;
  float* Jlo = nullptr;
  int* ipiv = nullptr;
  int* perm = nullptr;
  double* X = nullptr;
  double* Fsave = nullptr;
  double* Jt = nullptr;   // Gauss-Newton: J^T and J^T J
  double* JtJ = nullptr;
  double* held = nullptr;   // line search: the unknowns' storage at the start of the search
  size_t held_cap = 0;
  double* Rs = nullptr;  // equilibration scales
  double* Cs = nullptr;
  std::vector<void*> allocs;
  double last_times[4] = {0, 0, 0, 0};
  int last_iters[2] = {0, 0};
  double last_resid = 0;
  int last_fallback = 0;  // the last low-precision step fell back to an fp64 factorisation
  int last_factored = 0;  // the last step factored J (0: it reused earlier low-precision factors)
  // low-precision solve options (kad_system_set_option)
  double forcing = 0.0;   // refinement target max(1e-13, forcing * min(1, ||F||_inf)); 0: 1e-13
  int reuse_inner = 0;    // reuse the low-precision factors while the previous refinement took
                          // at most this many inner steps (0: factor every step)
  bool lo_valid = false;  // Jlo / perm / Rs / Cs hold usable low-precision factors
  int lo_prec = -1;
  int prev_inner = 0;     // inner steps of the previous refinement
  double* Jfac = nullptr;  // solver 5: fp64 factors of an earlier Jacobian (J and Jfac alternate)
  bool fac_valid = false;  // Jfac / perm hold usable fp64 factors
  kad_dd* dd = nullptr;    // solvers 6-7: the domain-decomposed factors (their own copy of the blocks)
  bool dd_valid = false;
  // solvers 6-7: factor with the pivot orders of the solve's last factorisation with
  // partial pivoting (static pivoting, kad_dd_factor_static) once there is one
  bool dd_static = true;
  bool dd_orders = false;  // this solve has such a factorisation (option 2 forgets it)
  // Jacobian fill on several streams (kad_system_set_option 3): the tangent programs are
  // dealt to the streams by estimated cost, each stream with its own tangent arena;
  // every program writes only its own columns of J, so the streams never touch the
  // same memory.  Stream 0 is the context's stream with tan_arena.
  bool fuse_ew = true;  // apply marked element-wise instructions in the preceding pass (option 5)
  static constexpr int kFillMax = 4;
  int nfill = 3;  // 17x13x12 x 5 domains, batch 4096: 0.241 s on one stream, 0.207 / 0.201 / 0.210 on 2 / 3 / 4
  hipStream_t fstream[kFillMax] = {};
  double* ftan[kFillMax] = {};
  hipEvent_t fev[kFillMax] = {};

  ~kad_system_impl() {
    if (dd) kad_dd_destroy(dd);
    for (int i = 0; i < kFillMax; ++i) {
      if (fstream[i]) (void)hipStreamDestroy(fstream[i]);
      if (fev[i]) (void)hipEventDestroy(fev[i]);
    }
    for (void* p : allocs) (void)hipFree(p);
    if (tan_arena) (void)hipFree(tan_arena);
    delete sys;
  }
  int dmalloc(void** p, size_t bytes) {
    KAD_HIP_CHECK(hipMalloc(p, bytes < 16 ? 16 : bytes));
    allocs.push_back(*p);
    return KAD_OK;
  }
  template <typename T>
  int upload(const std::vector<T>& h, T** d) {
    int rc = dmalloc((void**)d, h.size() * sizeof(T));
    if (rc) return rc;
    if (!h.empty()) KAD_HIP_CHECK(hipMemcpy(*d, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
    return KAD_OK;
  }
  double* slot_ptr(const Opnd& o, double* tan) const {
    return o.space == SP_VAL ? val_arena + (int64_t)o.slot * stride : tan + (int64_t)o.slot * B * stride;
  }
  int64_t slot_stride(const Opnd& o) const { return o.space == SP_VAL ? 0 : stride; }
  int setup();
  int upload_plans();
  // out: fp64 (dtype 0) or fp32 (dtype 1) column-major rows x columns with leading
  // dimension ldo, columns from col0; with w != nullptr the exports are transposed
  // instead (out: fp64 per column, += w . row).  st / tan: the stream and tangent arena
  // (default: the context's stream and tan_arena).
  int run(const std::vector<Instr>& code, int nb, int u0, int seed_tab, void* out, int64_t col0, int64_t ldo,
          int dtype = 0, const double* w = nullptr, hipStream_t st = nullptr, double* tan = nullptr);
  // every tangent program's columns of J (fp64, ld ldj), after the value pass and the
  // double unknowns' columns, on nfill streams; the context's stream waits for all
  int fill_columns(double* Jd, int64_t ldj);
  // the side streams (and, with arenas, their tangent arenas) and events for ns streams
  int ensure_streams(int ns, bool arenas);
  // the value program split by domain over ns streams (value_pass); false: not splittable
  bool split_values(int ns);
  int vsplit_ns = 0;
  bool vsplit_ok = false;
  std::vector<std::vector<Instr>> vparts;
  std::vector<Instr> vexports;
  // grouped execution: the instruction table, the value program, the tangent programs
  // (one per layout entry) and the parameters' programs by dependency level
  kad::GroupOp* gops = nullptr;
  kad::ClusterStep* gsteps = nullptr;
  GroupProg gval;
  std::vector<GroupProg> gtan, gpar;
  bool gtan_ok = false;         // every tangent program can be grouped
  bool tan_sized = false;       // the arena has its size for the levels
  bool levels_ready();
  void grow_arena();
  int group_build(std::vector<Instr> code, int nvirt, bool value, int seed_tab, GroupProg& gp,
                  std::vector<kad::GroupOp>& ops, std::vector<kad::ClusterStep>& steps);
  int group_round(const std::vector<GroupItem>& items, void* out, int64_t ldo, int dtype, const double* w);
  int group_columns(std::vector<GroupItem> items, void* out, int64_t ldo, int dtype, const double* w);
  // columns [c0, c1) of J (or, with w, entries of J^T w) into out, whose column 0 is
  // column col_base of J: the double unknowns' programs, then the tangent programs'
  int columns(int c0, int c1, int64_t col_base, void* out, int64_t ldo, int dtype = 0, const double* w = nullptr);
  bool vals_current = false;  // the value arena holds the value pass of the current fields
  int ensure_values() { return vals_current ? KAD_OK : value_pass(); }
  int value_pass();
  int jacobian(double* Jd, int64_t ldj);
  int update(const double* Xd, double scale);
  // columns [c0, c1) of the double unknowns (their parameter programs) into J, whose
  // column c0 sits at Jout + (c0 - col_base) ld
  int double_columns(void* Jout, int64_t ld, int c0, int c1, int col_base, int dtype = 0) {
    for (int k = c0; k < c1 && k < sys->ndouble; ++k) {
      const DevProgram& pp = par_progs[sys->dvar_par[k]];
      int rc = run(pp.code, 1, 0, pp.seed_tab, Jout, (int64_t)k - col_base, ld, dtype);
      if (rc) return rc;
    }
    return KAD_OK;
  }
};

// Chains of element-wise instructions that run inside the instruction before them: an
// instruction (a spectral pass or an element-wise one) whose result feeds only the
// element-wise instruction right after it absorbs that instruction, which then applies
// to the value as it is stored, and so on up to kad::kMaxChain of them.  The
// intermediate arrays never go to HBM (one launch and two array transfers fewer per
// absorbed instruction).  Conditions, on the virtual slots (before allocate_slots):
// tangent destinations (the slots are the program's own), the result is the next
// instruction's a or b but not both, it is read nowhere else, and the next
// instruction covers the whole array.  code[t].fuse = the number absorbed.
// A pass read by a single element-wise instruction a few places later moves down to just
// before it (the slots are written once, so the instructions in between read neither
// its result nor anything it overwrites), unless the instruction before that reader
// already feeds it.
static void pull_passes_to_readers(std::vector<Instr>& code, int nvirt) {
  constexpr int kReach = 3;
  auto reader_of = [&](int slot, size_t from) -> long {
    long at = -1;
    for (size_t u = from; u < code.size(); ++u) {
      const Instr& in = code[u];
      const bool ra = in.a.space == SP_TAN && in.a.slot == slot, rb = in.b.slot >= 0 && in.b.space == SP_TAN && in.b.slot == slot;
      if (ra || rb) {
        if (at >= 0) return -1;  // read twice
        at = (long)u;
      }
    }
    return at;
  };
  (void)nvirt;
  for (size_t t = 0; t + 2 < code.size(); ++t) {
    const Instr& l = code[t];
    if (l.kind != I_LIN || l.dst.space != SP_TAN || l.dst.slot < 0) continue;
    const long u = reader_of(l.dst.slot, t + 1);
    if (u < (long)t + 2 || u > (long)t + 1 + kReach || code[u].kind != I_EW) continue;
    const Instr& e = code[u];
    const Instr& pv = code[u - 1];
    const bool fed_by_prev = pv.dst.space == SP_TAN && pv.dst.slot >= 0 &&
                             ((e.a.space == SP_TAN && e.a.slot == pv.dst.slot) ||
                              (e.b.slot >= 0 && e.b.space == SP_TAN && e.b.slot == pv.dst.slot));
    if (fed_by_prev) continue;
    std::rotate(code.begin() + t, code.begin() + t + 1, code.begin() + u);  // the pass now at u - 1
    --t;  // look again at what moved into position t
  }
}

static void mark_fusions(std::vector<Instr>& code, int nvirt, const std::vector<kad::LinePlan>& plans) {
  pull_passes_to_readers(code, nvirt);
  std::vector<int> reads(nvirt, 0);
  for (Instr& in : code) {
    in.fuse = 0;
    if (in.a.slot >= 0 && in.a.space == SP_TAN) reads[in.a.slot]++;
    if (in.b.slot >= 0 && in.b.space == SP_TAN) reads[in.b.slot]++;
  }
  for (size_t t = 0; t < code.size(); ++t) {
    Instr& h = code[t];
    if ((h.kind != I_LIN && h.kind != I_EW) || h.dst.space != SP_TAN || h.dst.slot < 0) continue;
    int size = h.size;
    if (h.kind == I_LIN) {
      if (h.plan < 0 || h.plan >= (int)plans.size()) continue;
      size = plans[h.plan].size_out;
    }
    int m = 0;
    while (m < kad::kMaxChain && t + m + 1 < code.size()) {
      const Instr& prev = code[t + m];
      const Instr& e = code[t + m + 1];
      if (e.kind != I_EW || e.dst.space != SP_TAN || e.size != size || e.ew < 0 || e.ew > EW_SDIV) break;
      const bool in_a = e.a.space == SP_TAN && e.a.slot == prev.dst.slot;
      const bool in_b = e.b.slot >= 0 && e.b.space == SP_TAN && e.b.slot == prev.dst.slot;
      if (in_a == in_b || reads[prev.dst.slot] != 1) break;
      ++m;
    }
    h.fuse = m;
    t += m;  // the absorbed instructions run inside this one
  }
}

// The absorbed instructions code[t+1 .. t+fuse] as steps on the value of code[t].
static kad::PostOp chain_of(const std::vector<Instr>& code, size_t t, const std::function<double*(const Opnd&)>& ptr,
                            const std::function<int64_t(const Opnd&)>& stride) {
  kad::PostOp post;
  const int m = code[t].fuse;
  for (int k = 0; k < m; ++k) {
    const Instr& prev = code[t + k];
    const Instr& e = code[t + k + 1];
    // the chain value is prev's result; the other operand is the instruction's other one
    const int side = (e.a.space == SP_TAN && e.a.slot == prev.dst.slot) ? 0 : 1;
    const Opnd& other = side == 0 ? e.b : e.a;
    kad::EwStep& st = post.op[k];
    st.kind = e.ew;
    st.side = side;
    st.o = other.slot >= 0 ? ptr(other) : nullptr;
    st.os = other.slot >= 0 ? stride(other) : 0;
    st.s = e.s;
  }
  post.n = m;
  post.dst = ptr(code[t + m].dst);
  post.ds = stride(code[t + m].dst);
  return post;
}

// Liveness-based reuse of tangent slots within one program.
static int allocate_slots(std::vector<Instr>& code, int nvirt, const std::vector<kad::LinePlan>& plans) {
  mark_fusions(code, nvirt, plans);
  std::vector<int> last(nvirt, -1);
  auto use = [&](const Opnd& o, int t) {
    if (o.slot >= 0 && o.space == SP_TAN) last[o.slot] = std::max(last[o.slot], t);
  };
  for (int t = 0; t < (int)code.size(); ++t) {
    const Instr& in = code[t];
    use(in.a, t);
    use(in.b, t);
    use(in.dst, t);
  }
  std::vector<int> phys(nvirt, -1), freelist;
  int nphys = 0;
  for (int t = 0; t < (int)code.size(); ++t) {
    Instr& in = code[t];
    auto map_read = [&](Opnd& o) {
      if (o.slot >= 0 && o.space == SP_TAN) o.slot = phys[o.slot];
    };
    const int dv = (in.dst.space == SP_TAN) ? in.dst.slot : -1;
    const int av = (in.a.space == SP_TAN) ? in.a.slot : -1;
    const int bv = (in.b.space == SP_TAN) ? in.b.slot : -1;
    map_read(in.a);
    map_read(in.b);
    if (dv >= 0) {
      if (phys[dv] < 0) {
        if (!freelist.empty()) {
          phys[dv] = freelist.back();
          freelist.pop_back();
        } else {
          phys[dv] = nphys++;
        }
      }
      in.dst.slot = phys[dv];
    }
    // release operands whose last use is this instruction (after the destination is taken,
    // so an instruction never writes the slot it reads)
    for (int v : {av, bv}) {
      if (v >= 0 && last[v] == t && v != dv) {
        freelist.push_back(phys[v]);
        last[v] = -2;
      }
    }
    if (dv >= 0 && last[dv] == t) {
      freelist.push_back(phys[dv]);
      last[dv] = -2;
    }
  }
  return nphys;
}

// The line tables and matrices of every plan, for the array its instructions run it on
// (a plan belongs to one domain and one layout of it).
int kad_system_impl::upload_plans() {
  Tracer& tr = sys->tr;
  std::vector<std::array<int, 3>> din(tr.plans.size(), {0, 0, 0});
  bool one = true;
  auto scan = [&](const std::vector<Instr>& code) {
    for (const Instr& in : code) {
      if (in.kind != I_LIN) continue;
      if (in.plan < 0 || in.plan >= (int)tr.plans.size()) {
        one = false;
        continue;
      }
      const std::array<int, 3> d = {in.din[0], in.din[1], in.din[2]};
      if (din[in.plan][0] == 0) din[in.plan] = d;
      one = one && din[in.plan] == d;
    }
  };
  scan(tr.val.code);
  scan(sys->obs_prog.code);
  scan(sys->glob_prog.code);
  for (auto* v : {&sys->tprog, &sys->obs_tprog, &sys->par_prog, &sys->glob_tprog, &sys->glob_par_prog})
    for (auto& p : *v) scan(p.code);
  if (!one) return KAD_ERR_ARG;
  std::vector<double> pools;
  std::vector<kad::LineEnt> tabs;
  std::vector<std::array<size_t, kad::MAX_PASSES + 1>> where(tr.plans.size());
  plans.assign(tr.plans.size(), kad::LinePlan());
  for (size_t q = 0; q < tr.plans.size(); ++q) {
    if (din[q][0] == 0) continue;
    const HostPlan& hp = tr.plans[q];
    std::vector<kad::PassDesc> pd;
    for (auto& ps : hp.passes) pd.push_back({ps.axis, ps.nout, ps.line_mat.data()});
    size_t lines = 0, used = 0, size = (size_t)din[q][0] * din[q][1] * din[q][2];
    int nin[3] = {din[q][0], din[q][1], din[q][2]};
    size_t toff[kad::MAX_PASSES];
    for (const kad::PassDesc& ps : pd) {
      lines += size / nin[ps.axis];
      size = size / nin[ps.axis] * ps.nout;
      nin[ps.axis] = ps.nout;
    }
    std::vector<kad::LineEnt> tab(std::max<size_t>(1, lines));
    if (!kad::lines_build(din[q][0], din[q][1], din[q][2], pd.data(), (int)pd.size(), (int)hp.pool.size(), plans[q],
                          tab.data(), tab.size(), &used, toff))
      return KAD_ERR_ARG;
    for (int p = 0; p < plans[q].npass; ++p) where[q][p] = tabs.size() + toff[p];
    where[q][kad::MAX_PASSES] = pools.size();
    tabs.insert(tabs.end(), tab.begin(), tab.begin() + used);
    pools.insert(pools.end(), hp.pool.begin(), hp.pool.end());
  }
  double* dp;
  kad::LineEnt* dt;
  int rc;
  if ((rc = upload(pools, &dp)) || (rc = upload(tabs, &dt))) return rc;
  for (size_t q = 0; q < plans.size(); ++q) {
    plans[q].pool = dp + where[q][kad::MAX_PASSES];
    for (int p = 0; p < plans[q].npass; ++p) plans[q].p[p].tab = dt + where[q][p];
  }
  return KAD_OK;
}

int kad_system_impl::setup() {
  Tracer& tr = sys->tr;
  // slot stride: the largest domain array (coef layout), rounded to 8 doubles
  int maxsz = 0;
  for (int d = sys->dmin; d <= sys->dmax; ++d) maxsz = std::max(maxsz, sys->doms[d].coef_size());
  stride = (maxsz + 7) / 8 * 8;
  int rc = dmalloc((void**)&val_arena, (size_t)std::max(1, tr.nval_slots) * stride * sizeof(double));
  if (rc) return rc;
  KAD_HIP_CHECK(hipMemset(val_arena, 0, (size_t)std::max(1, tr.nval_slots) * stride * sizeof(double)));
  for (auto& cs : tr.const_slots)
    KAD_HIP_CHECK(hipMemcpy(val_arena + (int64_t)cs.first * stride, cs.second.data(),
                            cs.second.size() * sizeof(double), hipMemcpyHostToDevice));
  if ((rc = upload_plans())) return rc;
  for (auto& rt : tr.row_tabs) {
    std::vector<DevRow> h(rt.size());
    for (size_t i = 0; i < rt.size(); ++i) h[i] = {rt[i].pos, rt[i].gpos, rt[i].gw};
    DevRow* d;
    if ((rc = upload(h, &d))) return rc;
    row_tabs.push_back(d);
  }
  for (auto& st : sys->seeds) {
    int* p;
    double* v;
    int* c;
    if ((rc = upload(st.pos, &p)) || (rc = upload(st.val, &v)) || (rc = upload(st.cnt, &c))) return rc;
    seed_pos.push_back(p);
    seed_val.push_back(v);
    seed_cnt.push_back(c);
  }
  for (auto& m : sys->tau_maps) {
    int *rp, *cl;
    double* w;
    if ((rc = upload(m.rowptr, &rp)) || (rc = upload(m.col, &cl)) || (rc = upload(m.w, &w))) return rc;
    csr_rowptr.push_back(rp);
    csr_col.push_back(cl);
    csr_w.push_back(w);
  }
  // tangent programs: physical slots
  for (size_t p = 0; p < sys->tprog.size(); ++p) {
    DevProgram dp;
    dp.code = sys->tprog[p].code;
    dp.nphys = allocate_slots(dp.code, sys->tprog[p].nslots, plans);
    dp.field = sys->layout[p][0];
    dp.dom = sys->layout[p][1];
    dp.off = sys->layout[p][2];
    dp.cnt = sys->layout[p][3];
    for (auto& in : dp.code)
      if (in.kind == I_SEED) dp.seed_tab = in.seed_tab;
    nphys_max = std::max(nphys_max, dp.nphys);
    tprogs.push_back(std::move(dp));
  }
  for (size_t p = 0; p < sys->obs_tprog.size(); ++p) {
    DevProgram dp;
    dp.code = sys->obs_tprog[p].code;
    dp.nphys = allocate_slots(dp.code, sys->obs_tprog[p].nslots, plans);
    dp.field = sys->obs_tprog_lay[p][0];
    dp.dom = sys->obs_tprog_lay[p][1];
    dp.off = sys->obs_tprog_lay[p][2];
    dp.cnt = sys->obs_tprog_lay[p][3];
    dp.seed_tab = sys->obs_tprog_tab[p];
    nphys_max = std::max(nphys_max, dp.nphys);
    obs_tprogs.push_back(std::move(dp));
  }
  for (size_t p = 0; p < sys->par_prog.size(); ++p) {
    DevProgram dp;
    dp.code = sys->par_prog[p].code;
    dp.nphys = allocate_slots(dp.code, sys->par_prog[p].nslots, plans);
    dp.seed_tab = sys->par_tab[p];
    dp.cnt = 1;
    nphys_max = std::max(nphys_max, dp.nphys);
    par_progs.push_back(std::move(dp));
  }
  for (size_t p = 0; p < sys->glob_tprog.size(); ++p) {
    DevProgram dp;
    dp.code = sys->glob_tprog[p].code;
    dp.nphys = allocate_slots(dp.code, sys->glob_tprog[p].nslots, plans);
    dp.field = sys->layout[p][0];
    dp.dom = sys->layout[p][1];
    dp.off = sys->layout[p][2];
    dp.cnt = sys->layout[p][3];
    dp.seed_tab = tprogs[p].seed_tab;
    nphys_max = std::max(nphys_max, dp.nphys);
    glob_tprogs.push_back(std::move(dp));
  }
  for (size_t p = 0; p < sys->glob_par_prog.size(); ++p) {
    DevProgram dp;
    dp.code = sys->glob_par_prog[p].code;
    dp.nphys = allocate_slots(dp.code, sys->glob_par_prog[p].nslots, plans);
    dp.seed_tab = sys->par_tab[p];
    dp.cnt = 1;
    nphys_max = std::max(nphys_max, dp.nphys);
    glob_par_progs.push_back(std::move(dp));
  }
  tan_cap = (size_t)std::max(1, nphys_max) * B * stride;
  KAD_HIP_CHECK(hipMalloc((void**)&tan_arena, tan_cap * sizeof(double)));
  // the same programs by dependency level (adds 0.6 ms to a set-up of 26.3 ms at 9x7x4, 0.7 to
  // 44.5 at 13x9x8, 1.3 to 88 at 17x13x12, systems given by strings)
  std::vector<kad::GroupOp> ops;
  std::vector<kad::ClusterStep> steps;
  size_t most = tr.val.code.size();  // (an entry is some 500 bytes: no copies as the table grows)
  for (auto& p : sys->tprog) most += p.code.size();
  for (auto& p : sys->par_prog) most += p.code.size();
  ops.reserve(most);
  if ((rc = group_build(tr.val.code, 0, true, -1, gval, ops, steps))) return rc;
  gtan.resize(sys->tprog.size());
  gtan_ok = !gtan.empty();
  for (size_t p = 0; p < sys->tprog.size(); ++p) {
    if ((rc = group_build(sys->tprog[p].code, sys->tprog[p].nslots, false, tprogs[p].seed_tab, gtan[p], ops, steps)))
      return rc;
    gtan_ok = gtan_ok && gtan[p].ok;
  }
  gpar.resize(sys->par_prog.size());
  for (int k = 0; k < sys->ndouble; ++k) {
    const int p = sys->dvar_par[k];
    if ((rc = group_build(sys->par_prog[p].code, sys->par_prog[p].nslots, false, sys->par_tab[p], gpar[p], ops, steps)))
      return rc;
    gtan_ok = gtan_ok && gpar[p].ok;
  }
  if ((rc = upload(ops, &gops)) || (rc = upload(steps, &gsteps))) return rc;
  if ((rc = dmalloc((void**)&F, (size_t)sys->n_rows * sizeof(double)))) return rc;
  if ((rc = dmalloc((void**)&scratch, 64 * sizeof(double)))) return rc;
  return KAD_OK;
}

int kad_system_impl::run(const std::vector<Instr>& code, int nb, int u0, int seed_tab, void* out, int64_t col0,
                         int64_t ldo, int dtype, const double* w, hipStream_t st, double* tan) {
  hipStream_t s = st ? st : ctx->stream;
  if (!tan) tan = tan_arena;
  auto slot_ptr = [&](const Opnd& o) { return this->slot_ptr(o, tan); };
  for (size_t t = 0; t < code.size(); ++t) {
    const Instr& in = code[t];
    const Domain& dm = sys->doms[in.dom];
    switch (in.kind) {
      case I_LIN: {
        const int batch = (in.dst.space == SP_VAL) ? 1 : nb;
        kad::PostOp post;
        if (in.fuse > 0 && fuse_ew) {
          // the following element-wise instructions, applied in this pass's store phase
          post = chain_of(code, t, slot_ptr, [&](const Opnd& o) { return slot_stride(o); });
          t += in.fuse;
        }
        int rc = kad::apply3d_launch(slot_ptr(in.a), stride, slot_ptr(in.dst), stride, batch, plans[in.plan], s, &post);
        if (rc) return rc;
        break;
      }
      case I_EW: {
        const int batch = (in.dst.space == SP_VAL) ? 1 : nb;
        double* dp = slot_ptr(in.dst);
        const double* ap = slot_ptr(in.a);
        const double* bp = in.b.slot >= 0 ? slot_ptr(in.b) : nullptr;
        const int64_t ds = slot_stride(in.dst), as = slot_stride(in.a), bs = in.b.slot >= 0 ? slot_stride(in.b) : 0;
        if (in.fuse > 0 && fuse_ew) {
          // this instruction and the ones it absorbed, in one pass over the arrays
          const kad::PostOp post = chain_of(code, t, slot_ptr, [&](const Opnd& o) { return slot_stride(o); });
          t += in.fuse;
          const dim3 grid((unsigned)kad::cdiv(in.size, 256 * EW_U), (unsigned)std::min(batch, 65535));
          ewc_kernel<<<grid, 256, 0, s>>>(in.ew, ap, as, bp, bs, in.s, post, in.size, batch);
          break;
        }
        auto a16 = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
        if (in.size % 2 == 0 && ds % 2 == 0 && as % 2 == 0 && bs % 2 == 0 && a16(dp) && a16(ap) &&
            (!bp || a16(bp))) {
          const int size2 = in.size / 2;
          const dim3 grid((unsigned)kad::cdiv(size2, 256 * EW_U), (unsigned)std::min(batch, 65535));
          ew2_kernel<<<grid, 256, 0, s>>>(in.ew, dp, ds, ap, as, bp, bs, in.s, size2, batch);
        } else {
          const dim3 grid((unsigned)kad::cdiv(in.size, 256), (unsigned)std::min(batch, 65535));
          ew_kernel<<<grid, 256, 0, s>>>(in.ew, dp, ds, ap, as, bp, bs, in.s, in.size, batch);
        }
        break;
      }
      case I_EXPORT_IN:
      case I_EXPORT_BD: {
        const int batch = (in.a.space == SP_VAL) ? 1 : nb;
        const int64_t tot = (int64_t)in.nrows * batch;
        const unsigned g = (unsigned)kad::cdiv(tot, 256);
        if (w) {
          export_dot_kernel<<<(unsigned)batch, 256, 0, s>>>(row_tabs[in.rows], in.nrows, in.kind == I_EXPORT_BD,
                                                            slot_ptr(in.a), slot_stride(in.a), dm.nr, in.bsign, w,
                                                            in.row0, (double*)out, col0, in.sign);
        } else if (in.kind == I_EXPORT_IN) {
          if (dtype == 0)
            export_in_kernel<double><<<g, 256, 0, s>>>(row_tabs[in.rows], in.nrows, slot_ptr(in.a), slot_stride(in.a),
                                                       (double*)out, in.row0, col0, ldo, in.sign, in.accumulate,
                                                       batch);
          else
            export_in_kernel<float><<<g, 256, 0, s>>>(row_tabs[in.rows], in.nrows, slot_ptr(in.a), slot_stride(in.a),
                                                      (float*)out, in.row0, col0, ldo, in.sign, in.accumulate, batch);
        } else {
          if (dtype == 0)
            export_bd_kernel<double><<<g, 256, 0, s>>>(row_tabs[in.rows], in.nrows, slot_ptr(in.a), slot_stride(in.a),
                                                       dm.nr, in.bsign, (double*)out, in.row0, col0, ldo, in.sign,
                                                       in.accumulate, batch);
          else
            export_bd_kernel<float><<<g, 256, 0, s>>>(row_tabs[in.rows], in.nrows, slot_ptr(in.a), slot_stride(in.a),
                                                      dm.nr, in.bsign, (float*)out, in.row0, col0, ldo, in.sign,
                                                      in.accumulate, batch);
        }
        break;
      }
      case I_EXPORT_INT: {
        if (w || dtype != 0) return KAD_ERR_ARG;
        const int batch = (in.a.space == SP_VAL) ? 1 : nb;
        export_int_kernel<<<(unsigned)kad::cdiv(batch, 64), 64, 0, s>>>(slot_ptr(in.a), slot_stride(in.a), dm.nr,
                                                                         dm.nt, in.aux, in.s, (double*)out, in.row0,
                                                                         col0, ldo, batch);
        break;
      }
      case I_EXPORT_GL: {
        const bool val = in.a.slot < 0 || in.a.space == SP_VAL;
        const int batch = val ? 1 : nb;
        const double* src = in.a.slot >= 0 ? slot_ptr(in.a) : nullptr;
        const int64_t ss = in.a.slot >= 0 ? slot_stride(in.a) : 0;
        const unsigned g = (unsigned)kad::cdiv(batch, 64);
        if (w || dtype == 0)
          export_gl_kernel<double><<<g, 64, 0, s>>>(src, ss, dm.nr, dm.nt, in.aux, in.bsign, in.s, in.c0,
                                                    in.accumulate, in.pt, (double*)out, in.row0, col0, ldo, w,
                                                    batch);
        else
          export_gl_kernel<float><<<g, 64, 0, s>>>(src, ss, dm.nr, dm.nt, in.aux, in.bsign, in.s, in.c0,
                                                   in.accumulate, in.pt, (float*)out, in.row0, col0, ldo, nullptr,
                                                   batch);
        break;
      }
      case I_SEED: {
        const int64_t tot = (int64_t)in.size * nb;
        const int nu = (int)sys->seeds[seed_tab].cnt.size();
        seed_kernel<<<(unsigned)kad::cdiv(tot, 256), 256, 0, s>>>(slot_ptr(in.dst), stride, in.size,
                                                                    seed_pos[seed_tab], seed_val[seed_tab],
                                                                    seed_cnt[seed_tab], u0, nu, nb);
        break;
      }
      default:
        return KAD_ERR_ARG;
    }
  }
  KAD_HIP_CHECK(hipGetLastError());
  return KAD_OK;
}

int kad_system_impl::ensure_streams(int ns, bool arenas) {
  for (int i = 1; i < ns; ++i) {
    if (!fstream[i]) KAD_HIP_CHECK(hipStreamCreateWithFlags(&fstream[i], hipStreamNonBlocking));
    if (arenas && !ftan[i]) {
      const int rc = dmalloc((void**)&ftan[i], (size_t)std::max(1, nphys_max) * B * stride * sizeof(double));
      if (rc) return rc;
    }
  }
  for (int i = 0; i < ns && ns > 1; ++i)
    if (!fev[i]) KAD_HIP_CHECK(hipEventCreateWithFlags(&fev[i], hipEventDisableTiming));
  return KAD_OK;
}

// The value program split over ns streams: every instruction but the row exports goes to
// the stream of its domain, in program order; the exports follow on the context's
// stream once all have finished.  Valid when no instruction reads a value slot that
// an instruction of another stream writes (the domains' arrays are their own) and the
// exports feed nothing but their rows.
bool kad_system_impl::split_values(int ns) {
  if (vsplit_ns == ns) return vsplit_ok;
  vsplit_ns = ns;
  vsplit_ok = false;
  vparts.assign(ns, {});
  vexports.clear();
  std::vector<int> writer(std::max(1, sys->tr.nval_slots), -1);
  auto is_export = [](const Instr& in) {
    return in.kind == I_EXPORT_IN || in.kind == I_EXPORT_BD || in.kind == I_EXPORT_INT || in.kind == I_EXPORT_GL;
  };
  for (const Instr& in : sys->tr.val.code) {
    if (is_export(in)) {
      vexports.push_back(in);
      continue;
    }
    const int k = ((in.dom - sys->dmin) % ns + ns) % ns;
    for (const Opnd* o : {&in.a, &in.b})
      if (o->slot >= 0 && o->space == SP_VAL && o->slot < (int)writer.size() && writer[o->slot] >= 0 &&
          writer[o->slot] != k)
        return false;
    if (in.dst.slot >= 0) {
      if (in.dst.space != SP_VAL || in.dst.slot >= (int)writer.size()) return false;
      writer[in.dst.slot] = k;
    }
    vparts[k].push_back(in);
  }
  int used = 0;
  for (auto& v : vparts) used += !v.empty();
  vsplit_ok = used > 1;
  return vsplit_ok;
}

// Instructions that run as one unit of the grouped execution: a pass with the
// element-wise chain it absorbed (code[t[1..]]), a cluster of element-wise instructions, or
// one other instruction.
struct GroupUnit {
  std::vector<int> t;
  bool cluster = false;
  int level = 0;
};

// The next readers in a list of instructions: next[3 i] and next[3 i + 1] are the places in
// the list of the next instruction after ts[i] that reads its operand a or b, next[3 i + 2]
// that of its result (kNever: none).  seen: every slot of the two spaces at kNever, as on
// return.
constexpr int kNever = 1 << 30;
static void next_readers(const std::vector<Instr>& code, const std::vector<int>& ts, std::vector<int> (&seen)[2],
                         std::vector<int>& next) {
  next.assign(3 * ts.size(), kNever);
  for (int i = (int)ts.size() - 1; i >= 0; --i) {
    const Instr& in = code[ts[i]];
    next[3 * i + 2] = seen[in.dst.space][in.dst.slot];
    if (in.a.slot >= 0) next[3 * i] = seen[in.a.space][in.a.slot];
    if (in.b.slot >= 0) next[3 * i + 1] = seen[in.b.space][in.b.slot];
    for (const Opnd* o : {&in.a, &in.b})
      if (o->slot >= 0) seen[o->space][o->slot] = i;
  }
  for (int t : ts)
    for (const Opnd* o : {&code[t].a, &code[t].b})
      if (o->slot >= 0) seen[o->space][o->slot] = kNever;
}

// How many of the element-wise instructions code[ts[i]], i from begin to end (program order),
// fit the temporaries of one cluster, and if steps is given, its steps.  An operand from
// outside that is used again is kept in a temporary while one is free (else it is read
// again); a value made inside must be kept until its last use inside.  next: next_readers of
// ts.  stored(slot): the value is read outside the cluster.
static int cluster_steps(const std::vector<Instr>& code, const std::vector<int>& ts, const std::vector<int>& next,
                         int begin, int end, const std::function<bool(int)>& stored,
                         const std::function<kad::GroupOpnd(const Opnd&)>& opnd,
                         std::vector<kad::ClusterStep>* steps) {
  struct Temp {
    int space = -1, slot = -1;  // -1: free
    int next = kNever;          // the place of its next reader
    bool input = false;
  };
  Temp tmp[kad::kClusterTemps];
  auto find = [&](int space, int slot) {
    for (int q = 0; q < kad::kClusterTemps; ++q)
      if (tmp[q].space == space && tmp[q].slot == slot) return q;
    return -1;
  };
  for (int i = begin; i < end; ++i) {
    const Instr& in = code[ts[i]];
    kad::ClusterStep st;
    st.kind = in.ew;
    st.s = in.s;
    auto operand = [&](const Opnd& o, int nx, int& where, int& cache, kad::GroupOpnd& g) {
      if (o.slot < 0) return;
      const int q = find(o.space, o.slot);
      if (q >= 0) {
        where = q;
        tmp[q].next = nx;
        return;
      }
      where = -2;
      if (steps) g = opnd(o);
      if (nx >= end) return;
      const int f = find(-1, -1);
      if (f >= 0) {
        tmp[f] = {o.space, o.slot, nx, true};
        cache = f;
      }
    };
    operand(in.a, next[3 * i], st.a, st.ca, st.ga);
    if (in.b.slot >= 0 && in.b.space == in.a.space && in.b.slot == in.a.slot) {
      st.b = st.a;  // both operands are the same value
      st.gb = st.ga;
    } else {
      operand(in.b, next[3 * i + 1], st.b, st.cb, st.gb);
    }
    for (Temp& q : tmp)  // free those whose value is not read after this instruction
      if (q.next >= end) q = Temp();
    if (next[3 * i + 2] < end) {
      int f = find(-1, -1);
      if (f < 0) {  // give up the outside operand that is used last
        int far = -1;
        for (int q = 0; q < kad::kClusterTemps; ++q)
          if (tmp[q].input && tmp[q].next > far) {
            far = tmp[q].next;
            f = q;
          }
        if (f < 0) return i - begin;
        // (this very step may have put it there: then it is read from its array again)
        if (f == st.ca) st.ca = -1;
        if (f == st.cb) st.cb = -1;
      }
      tmp[f] = {in.dst.space, in.dst.slot, next[3 * i + 2], false};
      st.d = f;
    }
    if (steps) {
      if (stored(in.dst.slot)) st.gd = opnd(in.dst);
      steps->push_back(st);
    }
  }
  return end - begin;
}

// The instructions of a program by dependency level: an instruction's level is one past
// the last of its operands' (ASAP), so the instructions of a level are independent.
// Exports add to rows that earlier exports may have written: in the value program an
// export follows every earlier one that shares a row, in a tangent program every
// earlier one (the transposed export adds all of them to one entry).
// Tangent programs: the value program's results are all kept, a tangent's are not, so
// - multiplications and divisions by one drop out (they change no bit);
// - element-wise instructions between two rounds of passes (the same number of passes on
//   the longest way to them) run as clusters, split where they are not connected;
// - a pass whose result only feeds an element-wise instruction that no cluster reads
//   takes that one (and the chain after it) into its store phase;
// - slots are reused between levels: free again after the last level that reads them.
// A program with other instructions, or a slot written twice, stays on the
// per-instruction path (ok false).
int kad_system_impl::group_build(std::vector<Instr> code, int nvirt, bool value, int seed_tab, GroupProg& gp,
                                 std::vector<kad::GroupOp>& ops, std::vector<kad::ClusterStep>& steps) {
  gp = GroupProg();
  const int space = value ? SP_VAL : SP_TAN;
  const int nslots = std::max(1, value ? sys->tr.nval_slots : nvirt);
  const int N = (int)code.size();
  auto is_export = [](const Instr& in) {
    return in.kind == I_EXPORT_IN || in.kind == I_EXPORT_BD || in.kind == I_EXPORT_GL;
  };
  // the form that can be grouped
  std::vector<int> writer(nslots, -1);
  for (int t = 0; t < N; ++t) {
    const Instr& in = code[t];
    if (!is_export(in) && in.kind != I_LIN && in.kind != I_EW && !(in.kind == I_SEED && !value)) return KAD_OK;
    if (in.kind != I_SEED)
      for (const Opnd* o : {&in.a, &in.b}) {
        if (o->slot < 0) continue;
        if (o->space != space && (value || is_export(in))) return KAD_OK;
        if (o->space == space && (o->slot >= nslots || (!value && writer[o->slot] < 0))) return KAD_OK;
      }
    if (!is_export(in)) {
      const Opnd& d = in.dst;
      if (d.space != space || d.slot < 0 || d.slot >= nslots || writer[d.slot] >= 0) return KAD_OK;
      if (in.kind == I_EW && (in.ew < 0 || in.ew > EW_SDIV || in.a.slot < 0)) return KAD_OK;
      if (in.kind == I_LIN && (in.plan < 0 || in.plan >= (int)plans.size() ||
                               kad::lines_lds(plans[in.plan]) > kad::kMaxLds))
        return KAD_OK;
      writer[d.slot] = t;
    }
  }
  // x * 1 and x / 1: later reads take x
  std::vector<char> skip(N, 0);
  if (!value) {
    std::vector<int> alias(nslots);
    for (int s = 0; s < nslots; ++s) alias[s] = s;
    for (int t = 0; t < N; ++t) {
      Instr& in = code[t];
      if (in.kind != I_SEED)
        for (Opnd* o : {&in.a, &in.b})
          if (o->slot >= 0 && o->space == SP_TAN) o->slot = alias[o->slot];
      if (in.kind == I_EW && (in.ew == EW_SCAL || in.ew == EW_SDIV) && in.s == 1.0 && in.a.space == SP_TAN) {
        alias[in.dst.slot] = in.a.slot;
        skip[t] = 1;
      }
    }
  }
  // readers of every slot of this space, in program order
  std::vector<std::vector<int>> readers(nslots);
  auto for_reads = [&](int t, const std::function<void(int)>& f) {
    const Instr& in = code[t];
    if (in.kind == I_SEED) return;
    int first = -1;
    for (const Opnd* o : {&in.a, &in.b})
      if (o->slot >= 0 && o->space == space && o->slot != first) {
        f(o->slot);
        first = o->slot;
      }
  };
  for (int t = 0; t < N; ++t)
    if (!skip[t]) for_reads(t, [&](int s) { readers[s].push_back(t); });
  // units
  std::vector<GroupUnit> units;
  std::vector<int> unit_of(N, -1);
  std::vector<int> seen[2], next;  // next_readers
  seen[SP_VAL].assign(std::max(1, sys->tr.nval_slots), kNever);
  seen[SP_TAN].assign(nslots, kNever);
  if (value) {
    for (int t = 0; t < N; ++t) {
      unit_of[t] = (int)units.size();
      units.push_back({{t}, false, 0});
    }
  } else {
    std::vector<int> depth(N, 0);  // passes on the longest way to the instruction's result
    for (int t = 0; t < N; ++t) {
      if (skip[t]) continue;
      for_reads(t, [&](int s) { depth[t] = std::max(depth[t], depth[writer[s]]); });
      if (code[t].kind == I_LIN) ++depth[t];
    }
    auto out_size = [&](const Instr& l) { return plans[l.plan].size_out; };
    // chains absorbed by a pass: each value has one reader, an element-wise instruction
    // that reads it once, and no element-wise instruction reads the chain's end
    for (int t = 0; t < N; ++t) {
      if (skip[t] || code[t].kind != I_LIN) continue;
      std::vector<int> chain{t};
      while ((int)chain.size() <= kad::kMaxChain) {
        const int v = code[chain.back()].dst.slot;
        if (readers[v].size() != 1) break;
        const int r = readers[v][0];
        const Instr& e = code[r];
        if (e.kind != I_EW || e.size != out_size(code[t])) break;
        if (e.a.space == SP_TAN && e.a.slot == v && e.b.slot >= 0 && e.b.space == SP_TAN && e.b.slot == v) break;
        // another tangent operand must be ready before this pass's round
        const Opnd& o = (e.a.space == SP_TAN && e.a.slot == v) ? e.b : e.a;
        if (o.slot >= 0 && o.space == SP_TAN && depth[writer[o.slot]] >= depth[t]) break;
        chain.push_back(r);
      }
      while (chain.size() > 1) {  // back to an end that no element-wise instruction reads
        bool ew = false;
        for (int r : readers[code[chain.back()].dst.slot]) ew = ew || code[r].kind == I_EW;
        if (!ew) break;
        chain.pop_back();
      }
      for (int q : chain) unit_of[q] = (int)units.size();
      units.push_back({chain, false, 0});
    }
    // clusters: connected through tangent values, of one depth and array size
    std::vector<int> root(N);
    for (int t = 0; t < N; ++t) root[t] = t;
    std::function<int(int)> top = [&](int x) { return root[x] == x ? x : root[x] = top(root[x]); };
    auto member = [&](int t) { return !skip[t] && code[t].kind == I_EW && unit_of[t] < 0; };
    for (int s = 0; s < nslots; ++s) {
      std::vector<int> m;
      if (writer[s] >= 0 && member(writer[s])) m.push_back(writer[s]);
      for (int r : readers[s])
        if (member(r)) m.push_back(r);
      for (size_t x = 0; x < m.size(); ++x)
        for (size_t y = x + 1; y < m.size(); ++y)
          if (depth[m[x]] == depth[m[y]] && code[m[x]].size == code[m[y]].size) {
            root[top(m[x])] = top(m[y]);  // the later ones follow from m[y]
            break;
          }
    }
    std::map<int, std::vector<int>> clusters;
    for (int t = 0; t < N; ++t)
      if (member(t)) clusters[top(t)].push_back(t);
    for (auto& c : clusters) {
      const std::vector<int>& all = c.second;
      next_readers(code, all, seen, next);
      for (int done = 0; done < (int)all.size();) {
        // (the first 64 instructions decide: the temporaries end a region long before)
        const int k = cluster_steps(code, all, next, done, std::min((int)all.size(), done + 64),
                                    [](int) { return false; }, nullptr, nullptr);
        if (k == 0) return KAD_OK;  // (one instruction always fits)
        const std::vector<int> part(all.begin() + done, all.begin() + done + k);
        for (int t : part) unit_of[t] = (int)units.size();
        units.push_back({part, true, 0});
        done += k;
      }
    }
    for (int t = 0; t < N; ++t)
      if (!skip[t] && unit_of[t] < 0) {
        unit_of[t] = (int)units.size();
        units.push_back({{t}, false, 0});
      }
  }
  // levels: longest way over the units' dependencies (an acyclic graph: a cluster's
  // instructions have the same number of passes before them)
  std::vector<std::vector<int>> after(units.size());
  std::vector<int> waits(units.size(), 0);
  auto edge = [&](int from, int to) {
    if (from == to) return;
    after[from].push_back(to);
    ++waits[to];
  };
  std::vector<int> exported;
  for (int t = 0; t < N; ++t) {
    if (skip[t]) continue;
    for_reads(t, [&](int s) {
      if (writer[s] >= 0) edge(unit_of[writer[s]], unit_of[t]);
    });
    if (is_export(code[t])) {
      const int n = code[t].kind == I_EXPORT_GL ? 1 : code[t].nrows;
      for (int q : exported) {
        const int nq = code[q].kind == I_EXPORT_GL ? 1 : code[q].nrows;
        if (!value || (code[t].row0 < code[q].row0 + nq && code[q].row0 < code[t].row0 + n))
          edge(unit_of[q], unit_of[t]);
      }
      exported.push_back(t);
    }
  }
  std::vector<int> ready;
  for (size_t u = 0; u < units.size(); ++u)
    if (waits[u] == 0) ready.push_back((int)u);
  size_t done = 0;
  int depth = 0;
  while (!ready.empty()) {
    const int u = ready.back();
    ready.pop_back();
    ++done;
    depth = std::max(depth, units[u].level + 1);
    for (int v : after[u]) {
      units[v].level = std::max(units[v].level, units[u].level + 1);
      if (--waits[v] == 0) ready.push_back(v);
    }
  }
  if (done != units.size()) return KAD_OK;
  // slots: a unit stores what other units read; reused once no level reads them any more
  std::vector<int> rlev(nslots, -1);
  std::vector<char> live(nslots, 0);
  for (int t = 0; t < N; ++t) {
    if (skip[t]) continue;
    for_reads(t, [&](int s) {
      if (writer[s] < 0 || unit_of[writer[s]] == unit_of[t]) return;
      live[s] = 1;
      rlev[s] = std::max(rlev[s], units[unit_of[t]].level);
    });
  }
  std::vector<std::vector<int>> by_level(depth);
  for (size_t u = 0; u < units.size(); ++u) by_level[units[u].level].push_back((int)u);
  std::vector<int> phys(nslots, -1), freelist;
  if (!value) {
    std::vector<std::vector<int>> dies(depth);
    for (int l = 0; l < depth; ++l) {
      for (int u : by_level[l])
        for (int t : units[u].t) {
          if (is_export(code[t]) || !(live[code[t].dst.slot] || (!units[u].cluster && t == units[u].t.back()))) continue;
          const int s = code[t].dst.slot;
          if (freelist.empty()) {
            phys[s] = gp.nphys++;
          } else {
            phys[s] = freelist.back();
            freelist.pop_back();
          }
          dies[std::max(l, rlev[s])].push_back(s);
        }
      for (int s : dies[l]) freelist.push_back(phys[s]);
    }
  }
  auto opnd = [&](const Opnd& o) {
    kad::GroupOpnd g;
    g.slot = o.slot;
    g.tan = (o.slot >= 0 && o.space == SP_TAN) ? 1 : 0;
    if (g.tan) g.slot = phys[o.slot];
    return g;
  };
  gp.op0 = (int)ops.size();
  gp.lev.assign(1, 0);
  for (int l = 0; l < depth; ++l) {
    size_t lds = 0;
    double bytes = 0.0;
    std::vector<kad::GroupOp> lv;
    std::vector<std::pair<double, int>> order;  // cost, instruction: the longest start first
    lv.reserve(by_level[l].size());
    for (int u : by_level[l]) {
      const std::vector<int>& ts = units[u].t;
      const Instr& in = code[ts[0]];
      const Domain& dm = sys->doms[in.dom];
      kad::GroupOp op;
      double cost = 0.0;
      if (units[u].cluster) {
        op.kind = kad::GK_CLUSTER;
        op.size = in.size;
        op.step0 = (int)steps.size();
        next_readers(code, ts, seen, next);
        if (cluster_steps(code, ts, next, 0, (int)ts.size(), [&](int s) { return live[s] != 0; }, opnd, &steps) !=
            (int)ts.size())
          return KAD_ERR_ARG;
        op.nsteps = (int)steps.size() - op.step0;
        for (int q = op.step0; q < (int)steps.size(); ++q) {
          kad::ClusterStep& s = steps[q];
          for (int* w : {&s.ca, &s.cb, &s.d})
            if (*w < 0) *w = kad::kClusterTemps;
          bytes += 8.0 * in.size * ((s.a == -2 && s.ga.tan) + (s.b == -2 && s.gb.tan) + (s.gd.slot >= 0));
        }
        order.push_back({100.0 * op.nsteps * (double)kad::cdiv(in.size, 256), (int)lv.size()});
        lv.push_back(op);
        continue;
      }
      op.a = opnd(in.a);
      const int m = (int)ts.size() - 1;
      op.nstep = m;
      for (int k = 0; k < m; ++k) {
        const Instr& e = code[ts[k + 1]];
        const int v = code[ts[k]].dst.slot;
        const int side = (e.a.space == SP_TAN && e.a.slot == v) ? 0 : 1;
        op.st[k].kind = e.ew;
        op.st[k].side = side;
        op.st[k].o = opnd(side == 0 ? e.b : e.a);
        op.st[k].s = e.s;
      }
      if (!is_export(in)) op.dst = opnd(code[ts.back()].dst);
      int nout = in.size;
      switch (in.kind) {
        case I_LIN: {
          op.kind = kad::GK_LIN;
          op.P = plans[in.plan];
          lds = std::max(lds, kad::lines_lds(op.P));
          nout = op.P.size_out;
          bytes += 8.0 * ((double)op.P.size_in + nout);
          cost = 2000.0 * op.P.npass + nout;
          break;
        }
        case I_EW:
          op.kind = kad::GK_EW;
          op.ew = in.ew;
          op.size = in.size;
          op.s = in.s;
          op.b = opnd(in.b);
          bytes += 8.0 * in.size * (2.0 + (in.b.slot >= 0 ? 1.0 : 0.0));
          cost = 0.1 * in.size;
          break;
        case I_SEED: {
          op.kind = kad::GK_SEED;
          op.size = in.size;
          op.spos = seed_pos[seed_tab];
          op.sval = seed_val[seed_tab];
          op.scnt = seed_cnt[seed_tab];
          op.nu = (int)sys->seeds[seed_tab].cnt.size();
          cost = 0.1 * in.size;
          break;
        }
        case I_EXPORT_GL:
          op.kind = kad::GK_EXPORT_GL;
          op.row0 = in.row0;
          op.nr = dm.nr;
          op.nt = dm.nt;
          op.aux = in.aux;
          op.bsign = in.bsign;
          op.s = in.s;
          op.c0 = in.c0;
          op.accumulate = in.accumulate;
          op.pt = in.pt;
          cost = 1e6;
          break;
        default:
          op.kind = in.kind == I_EXPORT_BD ? kad::GK_EXPORT_BD : kad::GK_EXPORT_IN;
          op.rows = row_tabs[in.rows];
          op.nrows = in.nrows;
          op.row0 = in.row0;
          op.accumulate = in.accumulate;
          op.bsign = in.bsign;
          op.sign = in.sign;
          op.nr = dm.nr;
          lds = std::max(lds, (size_t)256 * sizeof(double));  // the transposed export's reduction
          cost = in.nrows;
          break;
      }
      for (int k = 0; k < m; ++k) bytes += op.st[k].o.tan ? 8.0 * nout : 0.0;
      order.push_back({cost, (int)lv.size()});
      lv.push_back(op);
    }
    std::stable_sort(order.begin(), order.end(), [&](const auto& x, const auto& y) {
      const bool cx = lv[x.second].kind == kad::GK_CLUSTER, cy = lv[y.second].kind == kad::GK_CLUSTER;
      return cx != cy ? cy : x.first > y.first;  // the clusters last
    });
    int ncl = 0, clsize = 0;
    for (auto& x : order) {
      const kad::GroupOp& op = lv[x.second];
      ops.push_back(op);
      if (op.kind != kad::GK_CLUSTER) continue;
      ++ncl;
      clsize = std::max(clsize, op.size);
    }
    gp.ncl.push_back(ncl);
    gp.clsize.push_back(clsize);
    gp.lev.push_back((int)ops.size() - gp.op0);
    gp.lds.push_back(lds);
    gp.bytes.push_back(bytes);
  }
  gp.ok = true;
  return KAD_OK;
}

// One round: every level of the items' programs, all items of a level in one launch (at
// most kGroupEntries items).
int kad_system_impl::group_round(const std::vector<GroupItem>& items, void* out, int64_t ldo, int dtype,
                                 const double* w) {
  kad::GroupArgs g;
  g.ops = gops;
  g.steps = gsteps;
  g.val = val_arena;
  g.tan = tan_arena;
  g.stride = stride;
  g.out = out;
  g.ldo = ldo;
  g.dtype = dtype;
  g.w = w;
  size_t depth = 0;
  for (const GroupItem& it : items) depth = std::max(depth, it.p->lds.size());
  for (size_t l = 0; l < depth; ++l) {
    double bytes = 0.0;
    for (const GroupItem& it : items) bytes += l < it.p->lds.size() ? it.p->bytes[l] * it.nb : 0.0;
    kad::GemmTimer* tm = kad::g_apply_timer;
    const int trc = tm && bytes > 0.0 ? tm->begin(ctx->stream, bytes) : 1;
    if (trc < 0) return trc;
    for (const bool clusters : {false, true}) {
      int blocks = 0, n = 0;
      size_t lds = 0;
      int64_t base = 0;
      for (const GroupItem& it : items) {
        const GroupProg& p = *it.p;
        const int64_t b0 = base;
        base += (int64_t)p.nphys * it.nb * stride;
        if (l >= p.lds.size()) continue;
        const int first = clusters ? p.lev[l + 1] - p.ncl[l] : p.lev[l];
        const int nops = (clusters ? p.lev[l + 1] : p.lev[l + 1] - p.ncl[l]) - first;
        if (nops == 0) continue;
        // a column's workgroups keep their residue modulo 8, so the round-robin dispatch
        // puts it on the same XCD (and its L2) at every level
        const int nbp = it.nb == 1 ? 1 : (int)kad::cdiv(it.nb, 8) * 8;
        if (nbp > 1) blocks = (int)kad::cdiv(blocks, 8) * 8;
        g.blk0[n] = blocks;
        const int nch = clusters ? (int)kad::cdiv(p.clsize[l], kad::kClusterChunk) : 1;
        g.e[n++] = {nops, p.op0 + first, it.nb, nbp, it.u0, nch, b0, it.col0};
        blocks += nops * nch * nbp;
        lds = std::max(lds, p.lds[l]);
      }
      g.nent = n;
      const int rc = kad::group_launch(g, blocks, clusters, lds, ctx->stream);
      if (rc) return rc;
    }
    if (trc == 0 && tm->end(ctx->stream)) return KAD_ERR_HIP;
  }
  return KAD_OK;
}

// The tangent arena with room for what the levels take, once: at most B columns of a program
// run at a time, and those of every program together have room (a region's arrays stay for a
// whole level, so a column takes about three times the slots it takes instruction by
// instruction).  At most 6 GiB (with the regions' temporaries in LDS, 5001 columns at
// 17x13x12 took 29.7, 25.7, 25.4 ms with 3, 6, 12 GiB, J^T w at 13x9x8 32.7, 32.2, 32.4), and
// at most half of the card's free memory, which leaves the other half to the caller.  Where
// that is less than the arena of the set-up, that one serves, in more rounds.
void kad_system_impl::grow_arena() {
  if (tan_sized) return;
  tan_sized = true;
  size_t want = 0, free = 0, total = 0;
  for (size_t p = 0; p < gtan.size(); ++p) want += (size_t)gtan[p].nphys * std::min(tprogs[p].cnt, B) * stride;
  for (auto& p : gpar) want += (size_t)p.nphys * stride;
  want = std::min(want, (size_t)6 << 27);
  if (want <= tan_cap) return;
  // (work on the present arena ends on the context's stream)
  bool ok = hipStreamSynchronize(ctx->stream) == hipSuccess && hipMemGetInfo(&free, &total) == hipSuccess;
  want = std::min(want, free / 2 / sizeof(double));
  double* more = nullptr;
  if (ok && want > tan_cap) ok = hipMalloc((void**)&more, want * sizeof(double)) == hipSuccess;
  if (!ok) (void)hipGetLastError();  // no room: the present arena serves
  if (ok && more) {
    (void)hipFree(tan_arena);
    tan_arena = more;
    tan_cap = want;
  }
}

// Whether the tangent programs run by levels: the arena holds one column of any of them
// (otherwise they run instruction by instruction).
bool kad_system_impl::levels_ready() {
  if (!gtan_ok || !fuse_ew) return false;
  size_t one = 0;
  for (auto* v : {&gtan, &gpar})
    for (auto& p : *v) one = std::max(one, (size_t)p.nphys * stride);
  if (one > tan_cap) grow_arena();
  return tan_cap >= one;
}

// The items in rounds that fit the arena.
int kad_system_impl::group_columns(std::vector<GroupItem> items, void* out, int64_t ldo, int dtype, const double* w) {
  size_t need = 0;
  for (const GroupItem& it : items) need += (size_t)it.p->nphys * it.nb * stride;
  if (need > tan_cap) grow_arena();
  std::vector<GroupItem> round;
  size_t used = 0;
  auto flush = [&]() -> int {
    if (round.empty()) return KAD_OK;
    const int rc = group_round(round, out, ldo, dtype, w);
    round.clear();
    used = 0;
    return rc;
  };
  for (GroupItem it : items) {
    const size_t per = std::max<size_t>(1, (size_t)it.p->nphys * stride);
    while (it.nb > 0) {
      const int64_t room = (int64_t)((tan_cap - used) / per);
      if ((int)round.size() >= kad::kGroupEntries || (room < std::min({it.nb, B, 64}) && !round.empty())) {
        const int rc = flush();
        if (rc) return rc;
        continue;
      }
      GroupItem q = it;
      q.nb = (int)std::min<int64_t>(std::min(it.nb, B), room);
      if (q.nb < 1) return KAD_ERR_ALLOC;  // (levels_ready: one column fits)
      round.push_back(q);
      used += per * q.nb;
      it.u0 += q.nb;
      it.col0 += q.nb;
      it.nb -= q.nb;
    }
  }
  return flush();
}

int kad_system_impl::columns(int c0, int c1, int64_t col_base, void* out, int64_t ldo, int dtype, const double* w) {
  std::vector<GroupItem> items;
  for (int k = c0; k < c1 && k < sys->ndouble; ++k) items.push_back({&gpar[sys->dvar_par[k]], 0, 1, k - col_base});
  for (size_t p = 0; p < tprogs.size(); ++p) {
    const int lo = std::max(c0, tprogs[p].off), hi = std::min(c1, tprogs[p].off + tprogs[p].cnt);
    if (lo < hi) items.push_back({&gtan[p], lo - tprogs[p].off, hi - lo, lo - col_base});
  }
  return group_columns(std::move(items), out, ldo, dtype, w);
}

int kad_system_impl::value_pass() {
  int rc;
  if (gval.ok && fuse_ew) {
    rc = group_round({{&gval, 0, 1, 0}}, F, 0, 0, nullptr);
    vals_current = (rc == KAD_OK);
    return rc;
  }
  const int ns = std::max(1, std::min(nfill, kFillMax));
  if (ns > 1 && split_values(ns)) {
    hipStream_t s0 = ctx->stream;
    if ((rc = ensure_streams(ns, false))) return rc;
    KAD_HIP_CHECK(hipEventRecord(fev[0], s0));
    for (int i = 1; i < ns; ++i) KAD_HIP_CHECK(hipStreamWaitEvent(fstream[i], fev[0], 0));
    for (int i = 0; i < ns && rc == KAD_OK; ++i)
      rc = run(vparts[i], 1, 0, -1, F, 0, 0, 0, nullptr, i ? fstream[i] : s0, tan_arena);
    for (int i = 1; i < ns; ++i) {
      KAD_HIP_CHECK(hipEventRecord(fev[i], fstream[i]));
      KAD_HIP_CHECK(hipStreamWaitEvent(s0, fev[i], 0));
    }
    if (rc == KAD_OK) rc = run(vexports, 1, 0, -1, F, 0, 0);
  } else {
    rc = run(sys->tr.val.code, 1, 0, -1, F, 0, 0);
  }
  vals_current = (rc == KAD_OK);
  return rc;
}

int kad_system_impl::jacobian(double* Jd, int64_t ldj) {
  int rc = value_pass();
  if (rc) return rc;
  KAD_HIP_CHECK(hipMemsetAsync(Jd, 0, (size_t)ldj * sys->n_unknowns * sizeof(double), ctx->stream));
  return fill_columns(Jd, ldj);
}

int kad_system_impl::fill_columns(double* Jd, int64_t ldj) {
  // Programs of 2048 columns and more fill the chip with each instruction (8 workgroups
  // per CU); their launches on nfill streams overlap and keep an instruction's arrays
  // closer together than a whole level's.  ms by levels and on streams, columns per program:
  // 675 13.5, 14.6; 798 18.2, 18.4; 1006 26.4, 25.7 (2 domains 13.0, 13.7); 1214 36.0, 34.3;
  // 1719 47.1, 45.5; 2079 64.2, 62.2; 2356 79.2, 79.7 (5 domains 137.7, 135.5).  From 1000
  // the streams lead by up to 5% where a whole program runs at once; with a smaller batch
  // they trail (798, batch 512, 18.3, 24.8; 1214, batch 1024, 36.0, 39.9).
  const bool wide = (int64_t)sys->n_unknowns >= (int64_t)2048 * (int64_t)tprogs.size();
  if (!wide && levels_ready()) return columns(0, sys->n_unknowns, 0, Jd, ldj);
  {
    const int rc = double_columns(Jd, ldj, 0, sys->ndouble, 0);
    if (rc) return rc;
  }
  hipStream_t s0 = ctx->stream;
  const int ns = std::max(1, std::min(nfill, (int)tprogs.size()));
  {
    const int rc = ensure_streams(ns, true);
    if (rc) return rc;
  }
  if (ns > 1) {
    KAD_HIP_CHECK(hipEventRecord(fev[0], s0));  // J cleared, value pass done
    for (int i = 1; i < ns; ++i) KAD_HIP_CHECK(hipStreamWaitEvent(fstream[i], fev[0], 0));
  }
  // longest programs first, each to the stream with the least work so far
  std::vector<int> order(tprogs.size());
  for (size_t q = 0; q < order.size(); ++q) order[q] = (int)q;
  auto cost = [&](int q) { return (double)tprogs[q].cnt * (double)tprogs[q].code.size(); };
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return cost(a) > cost(b); });
  double load[kFillMax] = {0, 0, 0, 0};
  for (int q : order) {
    int i = 0;
    for (int k = 1; k < ns; ++k)
      if (load[k] < load[i]) i = k;
    load[i] += cost(q);
    const DevProgram& p = tprogs[q];
    for (int u0 = 0; u0 < p.cnt; u0 += B) {
      const int nb = std::min(B, p.cnt - u0);
      // exports write columns off+u0 .. off+u0+nb-1
      const int rc = run(p.code, nb, u0, p.seed_tab, Jd, (int64_t)p.off + u0, ldj, 0, nullptr, i ? fstream[i] : s0,
                         i ? ftan[i] : tan_arena);
      if (rc) return rc;
    }
  }
  for (int i = 1; i < ns; ++i) {
    KAD_HIP_CHECK(hipEventRecord(fev[i], fstream[i]));
    KAD_HIP_CHECK(hipStreamWaitEvent(s0, fev[i], 0));
  }
  return KAD_OK;
}

int kad_system_impl::update(const double* Xd, double scale) {
  vals_current = false;
  for (int k = 0; k < sys->ndouble; ++k) {
    const std::string& name = sys->par_names[sys->dvar_par[k]];
    for (int d = sys->dmin; d <= sys->dmax; ++d) {
      const int slot = sys->param_slot(name, d);
      if (slot < 0) continue;
      const int size = sys->doms[d].conf_size();
      double_update_kernel<<<(unsigned)kad::cdiv(size, 256), 256, 0, ctx->stream>>>(val_arena + (int64_t)slot * stride,
                                                                                   size, Xd, k, scale);
    }
  }
  for (size_t q = 0; q < sys->layout.size(); ++q) {
    const int f = sys->layout[q][0], d = sys->layout[q][1], off = sys->layout[q][2];
    const int ncf = sys->doms[d].coef_size();
    double* cf = val_arena + (int64_t)sys->field_slot[f][d] * stride;
    csr_update_kernel<<<(unsigned)kad::cdiv(ncf, 256), 256, 0, ctx->stream>>>(cf, csr_rowptr[q], csr_col[q], csr_w[q],
                                                                              Xd, off, ncf, scale);
  }
  KAD_HIP_CHECK(hipGetLastError());
  return KAD_OK;
}

extern "C" {

int kad_xcts_create(kad_ctx* ctx, int nr, int nt, int np, const double* bounds, int nbounds, int dmin, int dmax,
                    double n0, double a, double ome, int order, int batch, kad_system** out) {
  if (!ctx || !bounds || nbounds < 2 || !out || batch <= 0 || order < 0 || order > 1) return KAD_ERR_ARG;
  auto* S = new kad_system_impl();
  S->ctx = reinterpret_cast<kad::Ctx*>(ctx);
  S->B = batch;
  XctsParams p;
  p.nr = nr;
  p.nt = nt;
  p.np = np;
  p.bounds.assign(bounds, bounds + nbounds);
  p.dmin = dmin;
  p.dmax = dmax;
  p.n0 = n0;
  p.a = a;
  p.ome = ome;
  p.order = order;
  try {
    S->xsys = new XctsSystem(p);
    S->sys = S->xsys;
    S->sys->build();
  } catch (const std::exception& e) {
    fprintf(stderr, "[kadath_amd] kad_xcts_create: %s\n", e.what());
    delete S;
    return KAD_ERR_ARG;
  }
  int rc = S->setup();
  if (rc) {
    delete S;
    return rc;
  }
  *out = reinterpret_cast<kad_system*>(S);
  return KAD_OK;
}

int kad_xcts_destroy(kad_system* s) {
  if (!s) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  (void)hipStreamSynchronize(S->ctx->stream);
  delete S;
  return KAD_OK;
}

int kad_xcts_sizes(kad_system* s, int* n_unknowns, int* n_rows, int* stats) {
  if (!s) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  if (n_unknowns) *n_unknowns = S->sys->n_unknowns;
  if (n_rows) *n_rows = S->sys->n_rows;
  if (stats) {
    size_t tcode = 0;
    for (auto& p : S->tprogs) tcode += p.code.size();
    stats[0] = (int)S->sys->tr.val.code.size();
    stats[1] = (int)tcode;
    stats[2] = S->sys->tr.nval_slots;
    stats[3] = S->nphys_max;
  }
  return KAD_OK;
}

// layout: 4 ints per (field, domain): field (0 P, 1 N, 2-4 bet x,y,z), domain, offset, count
int kad_xcts_layout(kad_system* s, int* out, int cap) {
  if (!s || !out) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  const int n = (int)S->sys->layout.size();
  if (cap < 4 * n) return KAD_ERR_ARG;
  for (int q = 0; q < n; ++q)
    for (int c = 0; c < 4; ++c) out[4 * q + c] = S->sys->layout[q][c];
  return n;
}

// 5 ints per (equation, component), in row order: kind (0 inside, 1 matching
// d|d+1, 2 outer bc, 3 inner bc), domain, component, first row, row count.
// Returns the number of entries.
int kad_xcts_row_layout(kad_system* s, int* out, int cap) {
  if (!s || !out) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  int q = 0;
  for (const auto& e : S->sys->eqs) {
    int row = e.row0;
    for (int c = 0; c < e.ncomp; ++c) {
      if (5 * (q + 1) > cap) return KAD_ERR_ARG;
      const int v[5] = {e.kind, e.d, c, row, e.nrows[c]};
      for (int t = 0; t < 5; ++t) out[5 * q + t] = v[t];
      row += e.nrows[c];
      ++q;
    }
  }
  return q;
}

// Coefficients of configuration values on the host, with the device's tables
// (Base_spectral::coef, coef.cpp:96-104: phi, then theta, then r).
static std::vector<double> host_coef(const Domain& dm, const Base& b, const std::vector<double>& conf) {
  Mat Mp = coef_matrix(b.bp, dm.np);
  std::vector<double> t1((size_t)dm.nr * dm.nt * dm.npc, 0.0), t2(t1.size(), 0.0), t3(t1.size(), 0.0);
  for (int kk = 0; kk < dm.npc; ++kk)
    for (int k = 0; k < dm.np; ++k)
      for (int j = 0; j < dm.nt; ++j)
        for (int i = 0; i < dm.nr; ++i)
          t1[i + dm.nr * (j + (size_t)dm.nt * kk)] += Mp(kk, k) * conf[i + dm.nr * (j + (size_t)dm.nt * k)];
  for (int k = 0; k < dm.npc; ++k) {
    Mat Mt = coef_matrix(b.bt[k], dm.nt);
    for (int jj = 0; jj < dm.nt; ++jj)
      for (int j = 0; j < dm.nt; ++j)
        for (int i = 0; i < dm.nr; ++i)
          t2[i + dm.nr * (jj + (size_t)dm.nt * k)] += Mt(jj, j) * t1[i + dm.nr * (j + (size_t)dm.nt * k)];
  }
  Mat Mr = coef_matrix(CHEB, dm.nr);
  for (int k = 0; k < dm.npc; ++k)
    for (int j = 0; j < dm.nt; ++j)
      for (int ii = 0; ii < dm.nr; ++ii)
        for (int i = 0; i < dm.nr; ++i)
          t3[ii + dm.nr * (j + (size_t)dm.nt * k)] += Mr(ii, i) * t2[i + dm.nr * (j + (size_t)dm.nt * k)];
  return t3;
}

// fields += affecte_tau(X0), X0 HOST (n_unknowns)
static int add_unknowns_host(kad_system_impl* S, const double* X0) {
  hipStream_t st = S->ctx->stream;
  double* dX;
  KAD_HIP_CHECK(hipMalloc(&dX, (size_t)S->sys->n_unknowns * sizeof(double)));
  KAD_HIP_CHECK(hipMemcpyAsync(dX, X0, (size_t)S->sys->n_unknowns * sizeof(double), hipMemcpyHostToDevice, st));
  int rc = S->update(dX, 1.0);
  KAD_HIP_CHECK(hipStreamSynchronize(st));
  (void)hipFree(dX);
  return rc;
}

// Fields := flat guess (P = 1 + a/r, N = 1, bet = 0; codes/Par_version/Kerr/kerr.cpp:36-52)
// + affecte_tau(X0).  X0: HOST, n_unknowns doubles (may be NULL for the flat guess).
int kad_xcts_set_guess(kad_system* s, const double* X0) {
  if (!s) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  if (!S->xsys) return KAD_ERR_ARG;
  XctsSystem& sy = *S->xsys;
  hipStream_t st = S->ctx->stream;
  for (int d = sy.dmin; d <= sy.dmax; ++d) {
    const Domain& dm = sy.doms[d];
    for (int f = 0; f < XctsSystem::NF; ++f) {
      std::vector<double> conf(dm.conf_size(), 0.0);
      for (size_t q = 0; q < conf.size(); ++q) {
        if (f == 0) {
          const double v = 1.0 + sy.prm.a / dm.R[q];
          conf[q] = std::isfinite(v) ? v : 1.0;
        } else if (f == 1) {
          conf[q] = 1.0;
        }
      }
      const std::vector<double> cf = host_coef(dm, sy.field_base(f, d), conf);
      S->vals_current = false;
      KAD_HIP_CHECK(hipMemcpyAsync(S->val_arena + (int64_t)sy.field_slot[f][d] * S->stride, cf.data(),
                                   cf.size() * sizeof(double), hipMemcpyHostToDevice, st));
    }
  }
  KAD_HIP_CHECK(hipStreamSynchronize(st));
  if (X0) return add_unknowns_host(S, X0);
  return KAD_OK;
}

// sec_member: F (device, n_rows) for the current fields.
int kad_xcts_residual(kad_system* s, double* Fout) {
  if (!s || !Fout) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  int rc = S->value_pass();
  if (rc) return rc;
  KAD_HIP_CHECK(hipMemcpyAsync(Fout, S->F, (size_t)S->sys->n_rows * sizeof(double), hipMemcpyDeviceToDevice,
                               S->ctx->stream));
  KAD_HIP_CHECK(hipStreamSynchronize(S->ctx->stream));
  return KAD_OK;
}

// Full Jacobian (device, column-major, ld ldj >= n_rows), all do_col_J columns.
int kad_xcts_jacobian(kad_system* s, double* Jd, int64_t ldj) {
  if (!s || !Jd) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  if (ldj < S->sys->n_rows) return KAD_ERR_ARG;
  int rc = S->jacobian(Jd, ldj);
  if (rc) return rc;
  KAD_HIP_CHECK(hipStreamSynchronize(S->ctx->stream));
  return KAD_OK;
}

// fields -= affecte_tau(X)  (X device, n_unknowns)
int kad_xcts_update(kad_system* s, const double* Xd) {
  if (!s || !Xd) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  int rc = S->update(Xd, -1.0);
  if (rc) return rc;
  KAD_HIP_CHECK(hipStreamSynchronize(S->ctx->stream));
  return KAD_OK;
}

// Coefficients of field f (0 P, 1 N, 2-4 bet) in domain d: HOST out, nr*nt*(np+2) doubles.
int kad_xcts_get_coef(kad_system* s, int f, int d, double* out) {
  if (!s || !out) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  SystemBase& sy = *S->sys;
  if (f < 0 || f >= sy.nfields || d < sy.dmin || d > sy.dmax) return KAD_ERR_ARG;
  KAD_HIP_CHECK(hipMemcpyAsync(out, S->val_arena + (int64_t)sy.field_slot[f][d] * S->stride,
                               (size_t)sy.doms[d].coef_size() * sizeof(double), hipMemcpyDeviceToHost,
                               S->ctx->stream));
  KAD_HIP_CHECK(hipStreamSynchronize(S->ctx->stream));
  return KAD_OK;
}

// Overwrite the coefficients of field f in domain d (HOST in, nr*nt*(np+2)): the
// counterpart of kad_xcts_get_coef, for fields prepared elsewhere (Scalar::set_domain).
int kad_xcts_set_coef(kad_system* s, int f, int d, const double* in) {
  if (!s || !in) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  SystemBase& sy = *S->sys;
  if (f < 0 || f >= sy.nfields || d < sy.dmin || d > sy.dmax) return KAD_ERR_ARG;
  S->vals_current = false;
  KAD_HIP_CHECK(hipMemcpyAsync(S->val_arena + (int64_t)sy.field_slot[f][d] * S->stride, in,
                               (size_t)sy.doms[d].coef_size() * sizeof(double), hipMemcpyHostToDevice,
                               S->ctx->stream));
  KAD_HIP_CHECK(hipStreamSynchronize(S->ctx->stream));
  return KAD_OK;
}

// Global quantities of the current fields at the outer boundary of the compactified
// domain (codes/Par_version/Kerr/reader.cpp:114-125): out[0] ADM mass, out[1] Komar
// mass, out[2] ADM angular momentum about z.  HOST out.
int kad_xcts_observables(kad_system* s, double* out) {
  if (!s || !out) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  SystemBase& sy = *S->sys;
  if (sy.obs.empty() || sy.obs.size() > 32) return KAD_ERR_ARG;
  hipStream_t st = S->ctx->stream;
  int rc = S->value_pass();
  if (rc) return rc;
  if ((rc = S->run(sy.obs_prog.code, 1, 0, -1, S->F, 0, 0))) return rc;
  const Domain& dm = sy.doms[sy.dmax];
  const int nq = (int)sy.obs.size();
  for (int q = 0; q < nq; ++q) {
    const auto& r = sy.obs[q];
    if (r.slot < 0) {
      KAD_HIP_CHECK(hipMemsetAsync(S->scratch + q, 0, sizeof(double), st));
      continue;
    }
    surface_integral_kernel<<<1, 64, 0, st>>>(S->val_arena + (int64_t)r.slot * S->stride, dm.nr, dm.nt, r.bt0, 1,
                                              r.fac, S->scratch + q);
    KAD_HIP_CHECK(hipGetLastError());
  }
  KAD_HIP_CHECK(hipMemcpyAsync(out, S->scratch, nq * sizeof(double), hipMemcpyDeviceToHost, st));
  KAD_HIP_CHECK(hipStreamSynchronize(st));
  return KAD_OK;
}

// The solvers need as many equations as unknowns (System_of_eqs::check_size_VS_unknowns,
// do_newton.cpp:113-118 and :600-609, which abort).
static int check_square(const SystemBase& sy) {
  if (sy.n_rows == sy.n_unknowns) return KAD_OK;
  fprintf(stderr, "Number of unknowns is different from the number of equations\nnbr equations = %d\n"
                  "nbr unknowns  = %d\n", sy.n_rows, sy.n_unknowns);
  return KAD_ERR_ARG;
}

// An interface condition that matches normal derivatives ("dn..." of the hand-traced
// system, or a string holding dn( or dr( ) rather than values.
static bool matches_derivative(const std::string& which) {
  return which.rfind("dn", 0) == 0 || which.find("dn(") != std::string::npos ||
         which.find("dr(") != std::string::npos;
}

// Blocks of the domain-decomposed solve: one per domain, with the domain's unknowns
// and the rows of the equations that live there.  An interface's matching condition
// lives in the inner domain when it matches values and in the outer one when it
// matches normal derivatives, which makes every block square (the domain's operator
// with a Dirichlet-type outer and a Neumann-type inner interface condition).  Integral
// equations and double unknowns couple every domain: such systems have no blocks.
static int dd_blocks(const SystemBase& sy, std::vector<int>& size, std::vector<int>& rows, std::vector<int>& cols) {
  if (sy.ndouble > 0 || sy.n_rows != sy.n_unknowns) return KAD_ERR_ARG;
  const int nb = sy.dmax - sy.dmin + 1;
  std::vector<std::vector<int>> R(nb), C(nb);
  for (auto& e : sy.eqs) {
    if (e.kind == 4) return KAD_ERR_ARG;
    const int d = (e.kind == 1 && matches_derivative(e.which)) ? e.d + 1 : e.d;
    if (d < sy.dmin || d > sy.dmax) return KAD_ERR_ARG;
    int len = 0;
    for (int c : e.nrows) len += c;
    for (int q = 0; q < len; ++q) R[d - sy.dmin].push_back(e.row0 + q);
  }
  for (auto& L : sy.layout)
    for (int q = 0; q < L[3]; ++q) C[L[1] - sy.dmin].push_back(L[2] + q);
  size.clear();
  rows.clear();
  cols.clear();
  for (int b = 0; b < nb; ++b) {
    if (R[b].size() != C[b].size() || R[b].empty()) return KAD_ERR_ARG;
    std::sort(R[b].begin(), R[b].end());
    size.push_back((int)R[b].size());
    rows.insert(rows.end(), R[b].begin(), R[b].end());
    cols.insert(cols.end(), C[b].begin(), C[b].end());
  }
  return KAD_OK;
}

// Set a parameter of the system: which indexes its parameters (XCTS: 0 = Ome, the
// horizon rotation of kerr.cpp:91-95).  The constant field is rewritten in every
// domain that holds it.
static int set_param_impl(kad_system_impl* S, int which, double value) {
  SystemBase& sy = *S->sys;
  if (which < 0 || which >= (int)sy.par_names.size()) return KAD_ERR_ARG;
  for (int d = sy.dmin; d <= sy.dmax; ++d) {
    const int slot = sy.param_slot(sy.par_names[which], d);
    if (slot < 0) continue;
    std::vector<double> h(sy.doms[d].conf_size(), value);
    S->vals_current = false;
    KAD_HIP_CHECK(hipMemcpyAsync(S->val_arena + (int64_t)slot * S->stride, h.data(), h.size() * sizeof(double),
                                 hipMemcpyHostToDevice, S->ctx->stream));
    KAD_HIP_CHECK(hipStreamSynchronize(S->ctx->stream));
  }
  if (S->xsys && sy.par_names[which] == "ome") S->xsys->prm.ome = value;
  return KAD_OK;
}

int kad_xcts_set_param(kad_system* s, int which, double value) {
  if (!s || which != 0) return KAD_ERR_ARG;
  return set_param_impl(reinterpret_cast<kad_system_impl*>(s), which, value);
}

// Sensitivities of the global quantities Q_q at a solution F(u, p) = 0 with respect
// to the parameter p = par, by the adjoint method:
//   J^T lambda_q = dQ_q/du   (the transposed solve reuses the LU factors of J),
//   dQ_q/dp = dQ_q/dp|_u - lambda_q . dF/dp   (the first term is 0: the quantities
//   read no parameter).
// dQ/du comes from tangent programs of the quantities, dF/dp from the tangent
// program of the parameter; J is refilled and factored at the current fields.
// out: HOST, one per quantity; dQdu (HOST, nq x n, may be NULL) receives dQ/du.
static int sensitivity_impl(kad_system_impl* S, int par, double* out, double* dQdu) {
  SystemBase& sy = *S->sys;
  hipStream_t st = S->ctx->stream;
  const int n = sy.n_unknowns;
  if (check_square(sy)) return KAD_ERR_ARG;
  const int nq = (int)sy.obs.size();
  if (nq == 0 || par < 0 || par >= (int)S->par_progs.size()) return KAD_ERR_ARG;
  int rc;
  if (!S->J) {
    if ((rc = S->dmalloc((void**)&S->J, (size_t)n * n * sizeof(double)))) return rc;
    if ((rc = S->dmalloc((void**)&S->ipiv, (size_t)n * sizeof(int)))) return rc;
    if ((rc = S->dmalloc((void**)&S->perm, (size_t)n * sizeof(int)))) return rc;
    if ((rc = S->dmalloc((void**)&S->X, (size_t)n * sizeof(double)))) return rc;
  }
  if (!S->dQ) {
    if ((rc = S->dmalloc((void**)&S->dQ, (size_t)nq * n * sizeof(double)))) return rc;
    if ((rc = S->dmalloc((void**)&S->dFdp, (size_t)n * sizeof(double)))) return rc;
  }
  if ((rc = S->jacobian(S->J, n))) return rc;  // includes the value pass at the current fields
  if ((rc = S->run(sy.obs_prog.code, 1, 0, -1, S->F, 0, 0))) return rc;
  KAD_HIP_CHECK(hipMemsetAsync(S->dQ, 0, (size_t)nq * n * sizeof(double), st));
  KAD_HIP_CHECK(hipMemsetAsync(S->dFdp, 0, (size_t)n * sizeof(double), st));
  for (auto& p : S->obs_tprogs)
    for (int u0 = 0; u0 < p.cnt; u0 += S->B) {
      const int nb = std::min(S->B, p.cnt - u0);
      if ((rc = S->run(p.code, nb, u0, p.seed_tab, S->dQ, (int64_t)p.off + u0, n))) return rc;
    }
  const DevProgram& pp = S->par_progs[par];
  if ((rc = S->run(pp.code, 1, 0, pp.seed_tab, S->dFdp, 0, n))) return rc;
  if (dQdu) {
    KAD_HIP_CHECK(hipMemcpyAsync(dQdu, S->dQ, (size_t)nq * n * sizeof(double), hipMemcpyDeviceToHost, st));
  }
  rc = kad_lu_factor(reinterpret_cast<kad_ctx*>(S->ctx), KAD_PREC_F64, n, S->J, n, S->ipiv, S->perm, 0);
  if (rc < 0) return rc;
  if (rc > 0) return KAD_ERR_SINGULAR;
  for (int q = 0; q < nq; ++q) {
    KAD_HIP_CHECK(hipMemcpyAsync(S->X, S->dQ + (size_t)q * n, (size_t)n * sizeof(double), hipMemcpyDeviceToDevice,
                                 st));
    if ((rc = kad_lu_solve(reinterpret_cast<kad_ctx*>(S->ctx), KAD_PREC_F64, n, S->J, n, S->perm, S->X, 1)))
      return rc;
    out[q] = -S->ctx->dot(S->X, S->dFdp, n);
  }
  KAD_HIP_CHECK(hipStreamSynchronize(st));
  return KAD_OK;
}

// dst[q n + k] = src[q] for every quantity q (a double unknown's column of dQ/du)
__global__ void scatter_q_kernel(const double* __restrict__ src, int nq, double* __restrict__ dst, int64_t n, int k) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < nq) dst[(int64_t)q * n + k] = src[q];
}

// Global quantities of a parsed system at the current fields: out[q] (HOST).
static int globals_impl(kad_system_impl* S, double* out) {
  SystemBase& sy = *S->sys;
  const int nq = (int)sy.glob_names.size();
  if (nq == 0 || nq > 32) return KAD_ERR_ARG;
  int rc = S->ensure_values();
  if (rc) return rc;
  if ((rc = S->run(sy.glob_prog.code, 1, 0, -1, S->scratch, 0, 0))) return rc;
  KAD_HIP_CHECK(hipMemcpyAsync(out, S->scratch, nq * sizeof(double), hipMemcpyDeviceToHost, S->ctx->stream));
  KAD_HIP_CHECK(hipStreamSynchronize(S->ctx->stream));
  return KAD_OK;
}

// Adjoint sensitivities of the parsed system's global quantities:
// dQ_q/dp = dQ_q/dp|_u - lambda_q . dF/dp with J^T lambda_q = dQ_q/du, J refilled and
// factored at the current fields.  out[q] HOST; dQdu (HOST nq x n, may be NULL).
static int glob_sensitivity_impl(kad_system_impl* S, int par, double* out, double* dQdu) {
  SystemBase& sy = *S->sys;
  hipStream_t st = S->ctx->stream;
  const int n = sy.n_unknowns;
  if (check_square(sy)) return KAD_ERR_ARG;
  const int nq = (int)sy.glob_names.size();
  if (nq == 0 || nq > 16 || par < 0 || par >= (int)S->par_progs.size()) return KAD_ERR_ARG;
  int rc;
  if (!S->J) {
    if ((rc = S->dmalloc((void**)&S->J, (size_t)n * n * sizeof(double)))) return rc;
    if ((rc = S->dmalloc((void**)&S->ipiv, (size_t)n * sizeof(int)))) return rc;
    if ((rc = S->dmalloc((void**)&S->perm, (size_t)n * sizeof(int)))) return rc;
    if ((rc = S->dmalloc((void**)&S->X, (size_t)n * sizeof(double)))) return rc;
  }
  if (!S->dQ) {
    if ((rc = S->dmalloc((void**)&S->dQ, (size_t)std::max(3, nq) * n * sizeof(double)))) return rc;
    if ((rc = S->dmalloc((void**)&S->dFdp, (size_t)n * sizeof(double)))) return rc;
  }
  if ((rc = S->jacobian(S->J, n))) return rc;  // value pass + every column, doubles included
  double* tmp = S->scratch + 32;   // nq: a double unknown's dQ column, then dQ/dp at fixed fields
  KAD_HIP_CHECK(hipMemsetAsync(S->dQ, 0, (size_t)nq * n * sizeof(double), st));
  KAD_HIP_CHECK(hipMemsetAsync(S->dFdp, 0, (size_t)n * sizeof(double), st));
  for (int k = 0; k < sy.ndouble; ++k) {
    const DevProgram& gp = S->glob_par_progs[sy.dvar_par[k]];
    KAD_HIP_CHECK(hipMemsetAsync(tmp, 0, nq * sizeof(double), st));
    if ((rc = S->run(gp.code, 1, 0, gp.seed_tab, tmp, 0, 1))) return rc;
    scatter_q_kernel<<<1, 64, 0, st>>>(tmp, nq, S->dQ, n, k);
  }
  for (auto& p : S->glob_tprogs)
    for (int u0 = 0; u0 < p.cnt; u0 += S->B) {
      const int nb = std::min(S->B, p.cnt - u0);
      if ((rc = S->run(p.code, nb, u0, p.seed_tab, S->dQ, (int64_t)p.off + u0, 1))) return rc;
    }
  const DevProgram& pp = S->par_progs[par];
  if ((rc = S->run(pp.code, 1, 0, pp.seed_tab, S->dFdp, 0, n))) return rc;
  KAD_HIP_CHECK(hipMemsetAsync(tmp, 0, nq * sizeof(double), st));
  if ((rc = S->run(S->glob_par_progs[par].code, 1, 0, S->glob_par_progs[par].seed_tab, tmp, 0, 1))) return rc;
  double direct[16];
  KAD_HIP_CHECK(hipMemcpyAsync(direct, tmp, nq * sizeof(double), hipMemcpyDeviceToHost, st));
  if (dQdu) KAD_HIP_CHECK(hipMemcpyAsync(dQdu, S->dQ, (size_t)nq * n * sizeof(double), hipMemcpyDeviceToHost, st));
  rc = kad_lu_factor(reinterpret_cast<kad_ctx*>(S->ctx), KAD_PREC_F64, n, S->J, n, S->ipiv, S->perm, 0);
  if (rc < 0) return rc;
  if (rc > 0) return KAD_ERR_SINGULAR;
  KAD_HIP_CHECK(hipStreamSynchronize(st));
  for (int q = 0; q < nq; ++q) {
    KAD_HIP_CHECK(hipMemcpyAsync(S->X, S->dQ + (size_t)q * n, (size_t)n * sizeof(double), hipMemcpyDeviceToDevice,
                                 st));
    if ((rc = kad_lu_solve(reinterpret_cast<kad_ctx*>(S->ctx), KAD_PREC_F64, n, S->J, n, S->perm, S->X, 1)))
      return rc;
    out[q] = direct[q] - S->ctx->dot(S->X, S->dFdp, n);
  }
  KAD_HIP_CHECK(hipStreamSynchronize(st));
  return KAD_OK;
}

// XCTS: out[3] = d(M_ADM, M_Komar, J_ADM)/dOme.
int kad_xcts_sensitivity(kad_system* s, double* out, double* dQdu) {
  if (!s || !out) return KAD_ERR_ARG;
  return sensitivity_impl(reinterpret_cast<kad_system_impl*>(s), 0, out, dQdu);
}

// ||F||_inf at the current fields (the value pass leaves F on the device).
static int newton_residual(kad_system_impl* S, double* err) {
  hipStream_t st = S->ctx->stream;
  int rc;
  if ((rc = S->value_pass())) return rc;
  absmax_kernel<<<1, 256, 0, st>>>(S->F, S->sys->n_rows, S->scratch);
  KAD_HIP_CHECK(hipMemcpyAsync(err, S->scratch, sizeof(double), hipMemcpyDeviceToHost, st));
  KAD_HIP_CHECK(hipStreamSynchronize(st));
  return KAD_OK;
}

// The Newton direction X (S->X) with J X = F: Jacobian fill, then the solver's
// factorisation and solve.  err = ||F||_inf (the forcing term of the low-precision
// refinement).  Gauss-Newton (solver 4) solves J^T J X = J^T F instead, as
// do_newton.cpp:264-311 (pdgemv_ 'T', pdgemm_ 'T','N', pdgesv_).  times as for
// kad_xcts_do_newton from index 1; t1 = wall clock at entry.
static int newton_direction(kad_system_impl* S, int solver, double err, double* times, double t1) {
  SystemBase& sy = *S->sys;
  hipStream_t st = S->ctx->stream;
  kad_ctx* cx = reinterpret_cast<kad_ctx*>(S->ctx);
  const int n = sy.n_unknowns;
  int rc;
  if ((rc = check_square(sy))) return rc;
  if (!S->J) {
    if ((rc = S->dmalloc((void**)&S->J, (size_t)n * n * sizeof(double)))) return rc;
    if ((rc = S->dmalloc((void**)&S->ipiv, (size_t)n * sizeof(int)))) return rc;
    if ((rc = S->dmalloc((void**)&S->perm, (size_t)n * sizeof(int)))) return rc;
    if ((rc = S->dmalloc((void**)&S->X, (size_t)n * sizeof(double)))) return rc;
  }
  if ((solver == 1 || solver == 2 || solver == 3) && !S->Jlo)
    if ((rc = S->dmalloc((void**)&S->Jlo, (size_t)n * n * sizeof(float)))) return rc;
  if (solver == 5 && !S->Jfac)
    if ((rc = S->dmalloc((void**)&S->Jfac, (size_t)n * n * sizeof(double)))) return rc;
  if (solver == 4 && !S->Jt) {
    if ((rc = S->dmalloc((void**)&S->Jt, (size_t)n * n * sizeof(double)))) return rc;
    if ((rc = S->dmalloc((void**)&S->JtJ, (size_t)n * n * sizeof(double)))) return rc;
  }
  // Jacobian (the value pass of the residual already holds the intermediates)
  if (!S->vals_current)
    if ((rc = S->value_pass())) return rc;
  KAD_HIP_CHECK(hipMemsetAsync(S->J, 0, (size_t)n * n * sizeof(double), st));
  if ((rc = S->fill_columns(S->J, n))) return rc;
  KAD_HIP_CHECK(hipStreamSynchronize(st));
  double t2 = now_s();
  if (times) times[1] = t2 - t1;
  int info = 0;
  double tf0 = 0, tf1 = 0;
  // The refinement target of the iterative solvers.  The default runs it to its
  // attainable accuracy (the tau system's near-null modes, high radial orders in the
  // compactified domain, are barely seen by a residual test).  With a forcing factor c
  // the target follows ||F||: c min(1, ||F||) relative, which keeps Newton quadratic
  // while early iterations need only a few inner steps.
  const double eta = S->forcing > 0.0 ? std::max(1e-13, S->forcing * std::min(1.0, err)) : 1e-13;
  // A refinement result is a usable Newton direction below this relative residual.
  constexpr double kAcceptResid = 1e-6;
  // Static pivoting (solvers 6-7): the kept orders are rejected above this multiplier
  // (partial pivoting keeps every one at most 1), and their factors are replaced when
  // the refinement needs more inner steps than this (2 with the exact Woodbury solve).
  // The refinement on the fp64 J is the real check: on the 17x13x12 spinning hole the
  // orders of one Newton step give the next step's blocks multipliers up to 4e5 (in
  // columns of rounding-level entries) and the preconditioned refinement still reaches
  // 2e-15 in two inner steps, as with partial pivoting; the bound only turns away
  // factors past any use (and the infinities of an exactly zero pivot).
  constexpr double kDdMaxGrowth = 1e8;
  constexpr int kDdStaticInner = 6;
  // Orders kept over several steps drift from the Jacobian (the same hole: multipliers
  // 4e5, 6e9, 4e14 one, two, three steps on, and then 700 inner steps), so a step whose
  // static factors show multipliers above this takes them, and the next step factors
  // with partial pivoting again for fresh orders.
  constexpr double kDdRefresh = 1e3;
  if (solver == 6 || solver == 7) {
    // domain-decomposed factors (the blocks factored together, then the Woodbury
    // coupling) precondition flexible GMRES on the current J; solver 7 keeps them for
    // later Jacobians while the refinement takes at most `limit` inner steps
    S->lo_valid = false;
    S->fac_valid = false;
    if (!S->dd) {
      std::vector<int> bs, rows, cols;
      if (dd_blocks(sy, bs, rows, cols)) {
        fprintf(stderr, "domain-decomposed solve: the system's domain blocks are not square\n");
        return KAD_ERR_ARG;
      }
      if ((rc = kad_dd_create(cx, n, (int)bs.size(), bs.data(), rows.data(), cols.data(), &S->dd))) return rc;
    }
    const int limit = S->reuse_inner > 0 ? S->reuse_inner : 30;
    bool solved = false;
    if (solver == 7 && S->dd_valid && S->prev_inner <= limit) {
      rc = kad_dd_solve(S->dd, S->J, n, S->F, S->X, eta, 8, S->last_iters, &S->last_resid);
      if (rc < 0 && rc != KAD_ERR_NOCONV) return rc;
      S->prev_inner = S->last_iters[1];
      solved = rc == KAD_OK || S->last_resid <= std::max(eta, kAcceptResid);
      S->last_factored = 0;
    }
    if (!solved) {
      KAD_HIP_CHECK(hipStreamSynchronize(st));
      const double tg0 = now_s();
      // static pivoting first when the solve has pivot orders; partial pivoting when
      // they do not apply (a multiplier above kDdMaxGrowth, other coupling rows)
      int dd_info = 1;
      bool stat = false;
      if (S->dd_static && S->dd_orders) {
        if ((rc = kad_dd_factor_static(S->dd, S->J, n, kDdMaxGrowth)) < 0) return rc;
        dd_info = rc;
        stat = rc == 0;
        double growth = 0.0;
        if (stat && kad_dd_pivoting(S->dd, nullptr, &growth) == KAD_OK && growth > kDdRefresh)
          S->dd_orders = false;  // used once; the next step refreshes them
      }
      // keep: with static pivoting on, the capacitance matrix keeps its order through
      // the blocks' partial pivoting while its multipliers stay within kDdMaxGrowth
      auto factor_pivoting = [&](bool keep) -> int {
        const int frc = keep ? kad_dd_factor_keep(S->dd, S->J, n, kDdMaxGrowth) : kad_dd_factor(S->dd, S->J, n);
        S->dd_orders = frc == 0;
        return frc;
      };
      bool kept_cap = false;
      if (!stat) {
        if ((dd_info = factor_pivoting(S->dd_static)) < 0) return dd_info;
        double cg = 0.0;
        kept_cap = dd_info == 0 && S->dd_static && kad_dd_pivoting(S->dd, nullptr, &cg) == KAD_OK && cg > 0.0;
      }
      tf1 += now_s() - tg0;
      // dd_info > 0: a singular domain block or capacitance matrix
      S->dd_valid = (dd_info == 0);
      S->last_factored = 1;
      bool fallback = dd_info != 0;
      if (dd_info == 0) {
        rc = kad::dd_solve_after_factor(S->dd, S->J, n, S->F, S->X, eta, 8, S->last_iters, &S->last_resid);
        if (rc < 0 && rc != KAD_ERR_NOCONV) return rc;
        bool poor = rc == KAD_ERR_NOCONV && !(S->last_resid <= std::max(eta, kAcceptResid));
        if ((stat || kept_cap) && (poor || S->last_iters[1] > kDdStaticInner)) {
          // the kept orders made a poor preconditioner: partial pivoting throughout,
          // solved again
          KAD_HIP_CHECK(hipStreamSynchronize(st));
          const double tg2 = now_s();
          if ((dd_info = factor_pivoting(false)) < 0) return dd_info;
          tf1 += now_s() - tg2;
          S->dd_valid = (dd_info == 0);
          poor = dd_info != 0;
          if (dd_info == 0) {
            rc = kad::dd_solve_after_factor(S->dd, S->J, n, S->F, S->X, eta, 8, S->last_iters, &S->last_resid);
            if (rc < 0 && rc != KAD_ERR_NOCONV) return rc;
            poor = rc == KAD_ERR_NOCONV && !(S->last_resid <= std::max(eta, kAcceptResid));
          }
        }
        S->prev_inner = S->last_iters[1];
        fallback = poor;
      }
      if (fallback) {
        // a singular block (J itself need not be singular) or not a usable Newton
        // direction: the fp64 LU of the same, untouched J decides
        S->last_fallback = 1;
        const double tg1 = now_s();
        if ((rc = kad_lu_factor(cx, KAD_PREC_F64, n, S->J, n, S->ipiv, S->perm, 0)) < 0) return rc;
        tf1 += now_s() - tg1;
        info = rc;
        S->dd_valid = false;
        if (info == 0) {
          KAD_HIP_CHECK(hipMemcpyAsync(S->X, S->F, (size_t)n * sizeof(double), hipMemcpyDeviceToDevice, st));
          if ((rc = kad_lu_solve(cx, KAD_PREC_F64, n, S->J, n, S->perm, S->X, 0))) return rc;
        }
      }
    }
  } else if (solver == 5) {
    // fp64 factors of an earlier J precondition flexible GMRES on the current J while
    // the previous refinement took at most `limit` inner steps; otherwise the current J
    // is factored in place and solved directly, and its factors are kept (the next fill
    // goes to the other buffer)
    S->lo_valid = false;
    const int limit = S->reuse_inner > 0 ? S->reuse_inner : 30;
    bool solved = false;
    if (S->fac_valid && S->prev_inner <= limit) {
      rc = kad_ir_solve_scaled(cx, n, S->J, n, KAD_PREC_F64, S->Jfac, n, S->perm, nullptr, nullptr, S->F, S->X,
                               eta, 8, 1, 0, S->last_iters, &S->last_resid);
      if (rc < 0 && rc != KAD_ERR_NOCONV) return rc;
      S->prev_inner = S->last_iters[1];
      solved = rc == KAD_OK || S->last_resid <= std::max(eta, kAcceptResid);
      S->last_factored = 0;
    }
    if (!solved) {
      KAD_HIP_CHECK(hipStreamSynchronize(st));
      const double tg0 = now_s();
      if ((rc = kad_lu_factor(cx, KAD_PREC_F64, n, S->J, n, S->ipiv, S->perm, 0)) < 0) return rc;
      tf1 += now_s() - tg0;
      info = rc;
      if (info == 0) {
        KAD_HIP_CHECK(hipMemcpyAsync(S->X, S->F, (size_t)n * sizeof(double), hipMemcpyDeviceToDevice, st));
        if ((rc = kad_lu_solve(cx, KAD_PREC_F64, n, S->J, n, S->perm, S->X, 0))) return rc;
      }
      std::swap(S->J, S->Jfac);
      S->fac_valid = (info == 0);
      S->prev_inner = 0;
      S->last_factored = 1;
    }
  } else if (solver == 0 || solver == 4) {
    S->lo_valid = false;  // the fp64 factorisation takes over ipiv / perm
    S->fac_valid = false;
    S->dd_valid = false;
    S->last_factored = 1;
    double* M = S->J;
    if (solver == 4) {
      // J^T F, then J^T J = (J^T) J with an explicit transpose and the MFMA GEMM; J
      // itself stays unfactored
      if ((rc = kad_gemv64(cx, n, S->J, n, S->F, nullptr, S->X, 1))) return rc;
      dim3 g((unsigned)kad::cdiv(n, 64), (unsigned)kad::cdiv(n, 64));
      transpose_kernel<<<g, 256, 0, st>>>(S->J, n, S->Jt, n, n);
      KAD_HIP_CHECK(hipGetLastError());
      if ((rc = kad_gemm(cx, KAD_PREC_F64, 1, n, n, n, S->Jt, n, S->J, n, S->JtJ, n))) return rc;
      M = S->JtJ;
    }
    KAD_HIP_CHECK(hipStreamSynchronize(st));
    tf0 = now_s();
    if ((rc = kad_lu_factor(cx, KAD_PREC_F64, n, M, n, S->ipiv, S->perm, 0)) < 0) return rc;
    tf1 = now_s();
    info = rc;
    if (info == 0) {
      if (solver == 0)
        KAD_HIP_CHECK(hipMemcpyAsync(S->X, S->F, (size_t)n * sizeof(double), hipMemcpyDeviceToDevice, st));
      if ((rc = kad_lu_solve(cx, KAD_PREC_F64, n, M, n, S->perm, S->X, 0))) return rc;
    }
  } else {
    S->fac_valid = false;  // the low-precision factorisation takes over ipiv / perm
    // low-precision factors of the equilibrated R J C (exact powers of two); the
    // refinement keeps the unscaled fp64 J, so its stopping test is on ||F - J X||.
    if (!S->Rs) {
      if ((rc = S->dmalloc((void**)&S->Rs, (size_t)n * sizeof(double)))) return rc;
      if ((rc = S->dmalloc((void**)&S->Cs, (size_t)n * sizeof(double)))) return rc;
    }
    const int prec = (solver == 3) ? KAD_PREC_BF16 : KAD_PREC_F32;
    // The factors of an earlier J precondition the refinement on the current one as
    // long as it keeps converging quickly; J itself (the residuals) is always current.
    bool reuse = S->reuse_inner > 0 && S->lo_valid && S->lo_prec == prec && S->prev_inner <= S->reuse_inner;
    for (int attempt = 0; attempt < 2; ++attempt) {
      if (!reuse) {
        if ((rc = kad_cast_equilibrated(cx, n, S->J, n, S->Jlo, n, S->Rs, S->Cs))) return rc;
        KAD_HIP_CHECK(hipStreamSynchronize(st));
        const double tg0 = now_s();
        if ((rc = kad_lu_factor(cx, prec, n, S->Jlo, n, S->ipiv, S->perm, 0)) < 0) return rc;
        tf1 += now_s() - tg0;
        info = rc;
        S->lo_valid = (info == 0);
        S->lo_prec = prec;
        S->last_factored = 1;
        if (info != 0) break;
      }
      rc = kad_ir_solve_scaled(cx, n, S->J, n, prec, S->Jlo, n, S->perm, S->Rs, S->Cs, S->F, S->X, eta,
                               solver == 1 ? 30 : 8, solver == 1 ? 0 : 1, 0, S->last_iters, &S->last_resid);
      if (rc < 0 && rc != KAD_ERR_NOCONV) return rc;
      S->prev_inner = S->last_iters[1];
      // reused factors that no longer precondition well: factor the current J and retry
      if (reuse && rc == KAD_ERR_NOCONV && !(S->last_resid <= std::max(eta, 1e-6))) {
        reuse = false;
        continue;
      }
      break;
    }
    if (info == 0) {
      // The refinement stops at its attainable accuracy.  A step whose relative linear
      // residual is above kAcceptResid is not a usable Newton direction (a refinement
      // that made no progress leaves X = 0): the step is then solved with an fp64
      // factorisation of the same (unscaled, untouched) J, as the reference's pdgesv_
      // would, and the fallback is reported through kad_xcts_last_solve.
      if (rc == KAD_ERR_NOCONV && !(S->last_resid <= std::max(eta, kAcceptResid))) {
        S->last_fallback = 1;
        S->lo_valid = false;  // the fp64 factorisation below takes over ipiv / perm
        const double tg0 = now_s();
        rc = kad_lu_factor(cx, KAD_PREC_F64, n, S->J, n, S->ipiv, S->perm, 0);
        if (rc < 0) return rc;
        tf1 += now_s() - tg0;  // both factorisations count as factor time
        info = rc;
        if (info == 0) {
          KAD_HIP_CHECK(hipMemcpyAsync(S->X, S->F, (size_t)n * sizeof(double), hipMemcpyDeviceToDevice, st));
          if ((rc = kad_lu_solve(cx, KAD_PREC_F64, n, S->J, n, S->perm, S->X, 0))) return rc;
        }
      }
    }
  }
  if (times) times[4] = (solver == 0 || solver == 4) ? tf1 - tf0 : tf1;  // the others accumulate in tf1
  if (info != 0) {
    fprintf(stderr, "Jacobian is singular! Stopping.\n");
    return KAD_ERR_SINGULAR;
  }
  KAD_HIP_CHECK(hipStreamSynchronize(st));
  if (times) times[2] = now_s() - t2;
  return KAD_OK;
}

static void reset_solve_record(kad_system_impl* S) {
  S->last_iters[0] = S->last_iters[1] = 0;
  S->last_resid = 0.0;
  S->last_fallback = 0;
  S->last_factored = 0;
}

// One Newton-Raphson iteration (System_of_eqs::do_newton, src_par/do_newton.cpp:65-430).
// solver: 0 fp64 LU; 1 fp32 LU + fp64 IR; 2 fp32 LU + fp64 GMRES-IR; 3 bf16-update LU +
// fp64 GMRES-IR; 4 Gauss-Newton (fp64 J^T J X = J^T F, the reference's GAUSS_NEWTON);
// 5 fp64 LU of an earlier J (refactored when it stops preconditioning well) + fp64
// flexible GMRES on the current J; 6 domain-decomposed fp64 factors (kad_dd_factor) +
// fp64 flexible GMRES; 7 the same, the factors of an earlier J kept while they
// precondition well.
// Returns 1 when ||F||_inf < precision at entry (converged; no step taken), 0 after a step,
// < 0 on error, KAD_ERR_SINGULAR (-5) when the factorisation meets an exact zero pivot.
// times[5] (may be NULL): residual, Jacobian fill, factor+solve, update, factor alone (seconds).
int kad_xcts_do_newton(kad_system* s, double precision, double* error, int solver, double* times) {
  if (!s || !error || solver < 0 || solver > 7) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  hipStream_t st = S->ctx->stream;
  int rc;
  double t0 = now_s();
  double err = 0;
  if ((rc = newton_residual(S, &err))) return rc;
  *error = err;
  double t1 = now_s();
  if (times) times[0] = t1 - t0;
  reset_solve_record(S);
  if (err < precision) return 1;  // false for a NaN error: a NaN residual is never converged
  if ((rc = newton_direction(S, solver, err, times, t1))) return rc;
  double t3 = now_s();
  if ((rc = S->update(S->X, -1.0))) return rc;
  KAD_HIP_CHECK(hipStreamSynchronize(st));
  if (times) times[3] = now_s() - t3;
  return 0;
}

// Newton iteration with a backtracking line search
// (System_of_eqs::do_newton_with_linesearch, src_par/do_newton.cpp:454-517, after
// Numerical Recipes 2007 section 9.7.1).  f = sum F^2 (compute_f, :594-599), slope =
// -2 f_old; the Newton step p (J p = F, by `solver`) is scaled by stepmax / max(p) when
// its (signed) maximum exceeds stepmax; u(lambda) = u_old - lambda p.  lambda starts at
// 1 and is taken from the quadratic model, then the cubic one, kept in [0.1, 0.5] of the
// previous lambda, until f <= 5e-13, f <= f_old + 1e-4 lambda slope, lambda <= 1e-10, or
// ntrymax tries (the last computed lambda is then applied).
// Returns 1 when ||F||_inf < precision at entry, 0 after a step; KAD_ERR_NOCONV where the
// reference aborts on roundoff ("roundoff error in do_newton_with_linesearch": a
// non-negative slope or a negative cubic discriminant).  lambda_out, ntry_out (may be
// NULL): the lambda applied and the number of residual evaluations of the search.
int kad_system_do_newton_linesearch(kad_system* s, double precision, double* error, int ntrymax, double stepmax,
                                    int solver, double* lambda_out, int* ntry_out) {
  if (!s || !error || ntrymax < 1 || !(stepmax > 0.0) || solver < 0 || solver > 7) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  SystemBase& sy = *S->sys;
  hipStream_t st = S->ctx->stream;
  int rc;
  double err = 0;
  if ((rc = newton_residual(S, &err))) return rc;
  *error = err;
  reset_solve_record(S);
  if (lambda_out) *lambda_out = 0.0;
  if (ntry_out) *ntry_out = 0;
  if (err < precision) return 1;
  auto sumsq_max = [&](const double* x, int n, double out[2]) -> int {
    sumsq_max_kernel<<<1, 256, 0, st>>>(x, n, S->scratch + 8);
    KAD_HIP_CHECK(hipMemcpyAsync(out, S->scratch + 8, 2 * sizeof(double), hipMemcpyDeviceToHost, st));
    KAD_HIP_CHECK(hipStreamSynchronize(st));
    return KAD_OK;
  };
  double r[2];
  if ((rc = sumsq_max(S->F, sy.n_rows, r))) return rc;
  const double fold = r[0], slope = -2.0 * fold;
  if (!(slope < 0.0)) {
    fprintf(stderr, "roundoff error in do_newton_with_linesearch\n");
    return KAD_ERR_NOCONV;
  }
  if ((rc = newton_direction(S, solver, err, nullptr, now_s()))) return rc;
  if ((rc = sumsq_max(S->X, sy.n_unknowns, r))) return rc;
  const double pmax = r[1];
  const double pscale = (pmax > stepmax) ? stepmax / pmax : 1.0;
  // snapshot of the unknowns' storage: field coefficients and double-unknown constants
  std::vector<std::pair<double*, int>> held;
  for (auto& L : sy.layout)
    held.push_back({S->val_arena + (int64_t)sy.field_slot[L[0]][L[1]] * S->stride, sy.doms[L[1]].coef_size()});
  for (int k = 0; k < sy.ndouble; ++k)
    for (int d = sy.dmin; d <= sy.dmax; ++d) {
      const int slot = sy.param_slot(sy.par_names[sy.dvar_par[k]], d);
      if (slot >= 0) held.push_back({S->val_arena + (int64_t)slot * S->stride, sy.doms[d].conf_size()});
    }
  size_t total = 0;
  for (auto& h : held) total += (size_t)h.second;
  if (S->held_cap < total) {
    if ((rc = S->dmalloc((void**)&S->held, total * sizeof(double)))) return rc;
    S->held_cap = total;
  }
  auto copy_held = [&](bool save) -> int {
    size_t o = 0;
    for (auto& h : held) {
      double* a = S->held + o;
      KAD_HIP_CHECK(hipMemcpyAsync(save ? a : h.first, save ? h.first : a, (size_t)h.second * sizeof(double),
                                   hipMemcpyDeviceToDevice, st));
      o += (size_t)h.second;
    }
    return KAD_OK;
  };
  auto apply = [&](double lam) -> int {
    int q = copy_held(false);
    if (q) return q;
    return S->update(S->X, -lam * pscale);
  };
  if ((rc = copy_held(true))) return rc;
  const double alpha = 1.0e-4, lambdamin = 1.0e-10;
  double lambda = 1.0, lambda2 = 0.0, f2 = 0.0;
  int tries = 0;
  for (int itry = 1; itry <= ntrymax; ++itry) {
    if ((rc = apply(lambda))) return rc;
    if ((rc = S->value_pass())) return rc;
    if ((rc = sumsq_max(S->F, sy.n_rows, r))) return rc;
    const double f = r[0];
    tries = itry;
    if (f <= 5.0e-13) break;
    if (f <= fold + alpha * lambda * slope || lambda <= lambdamin) break;
    double lt;
    if (lambda == 1.0) {
      lt = -0.5 * slope / (f - fold - slope);
    } else {
      const double rhs1 = f - fold - lambda * slope, rhs2 = f2 - fold - lambda2 * slope;
      const double a = (rhs1 / (lambda * lambda) - rhs2 / (lambda2 * lambda2)) / (lambda - lambda2);
      const double b = (-lambda2 * rhs1 / (lambda * lambda) + lambda * rhs2 / (lambda2 * lambda2)) / (lambda - lambda2);
      if (a == 0.0) {
        lt = -0.5 * slope / b;
      } else {
        const double delta = b * b - 3.0 * a * slope;
        if (delta < 0.0) {
          fprintf(stderr, "roundoff error in do_newton_with_linesearch\n");
          return KAD_ERR_NOCONV;
        }
        lt = (-b + std::sqrt(delta)) / (3.0 * a);
      }
      if (lt > 0.5 * lambda) lt = 0.5 * lambda;
    }
    lambda2 = lambda;
    f2 = f;
    lambda = std::max(lt, 0.1 * lambda);
    if (itry == ntrymax)
      if ((rc = apply(lambda))) return rc;
  }
  S->vals_current = false;
  KAD_HIP_CHECK(hipStreamSynchronize(st));
  if (lambda_out) *lambda_out = lambda;
  if (ntry_out) *ntry_out = tries;
  return 0;
}

// Seeded initial perturbation amp * 2^-(i+j+k) * U(-1,1) on every admissible
// coefficient, in unknown order (HOST out, n_unknowns).  U from splitmix64.
int kad_xcts_perturbation(kad_system* s, uint64_t seed, double amp, double* out) {
  if (!s || !out) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  SystemBase& sy = *S->sys;
  uint64_t x = seed;
  auto next = [&]() {
    uint64_t z = (x += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= (z >> 31);
    return (double)(z >> 11) * (1.0 / 9007199254740992.0);
  };
  // draws in the reference unknown order (variables, then domains, then components),
  // stored at this system's layout offsets, so both orderings start from the same guess;
  // the double unknowns are not perturbed
  for (int k = 0; k < sy.ndouble; ++k) out[k] = 0.0;
  for (auto& var : sy.var_fields)
    for (int d = sy.dmin; d <= sy.dmax; ++d)
      for (int f : var) {
        int u = -1;
        for (auto& L : sy.layout)
          if (L[0] == f && L[1] == d) u = L[2];
        if (u < 0) return KAD_ERR_ARG;
        const Domain& dm = sy.doms[d];
        for (auto& kj : dm.unknown_slots(sy.field_base(f, d).bt))
          for (int i = 0; i < dm.nr; ++i)
            out[u++] = amp * std::ldexp(1.0, -(i + kj.second + kj.first)) * (2 * next() - 1);
      }
  return KAD_OK;
}

int kad_xcts_last_solve(kad_system* s, int* iters, double* resid) {
  if (!s) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  if (iters) {
    iters[0] = S->last_iters[0];
    iters[1] = S->last_iters[1];
    iters[2] = S->last_fallback;
    iters[3] = S->last_factored;
  }
  if (resid) *resid = S->last_resid;
  return KAD_OK;
}

}  // extern "C"

extern "C" {
// Host-only tracing (no device work): sizes of the system and of its programs.
// info[0] n_unknowns, [1] n_rows, [2] value instructions, [3] tangent instructions,
// [4] value slots, [5] tangent programs.  layout: 4 ints per (field, domain) entry.
// kad_system_dd_blocks of the hand-traced system, traced on the host only.
int kad_xcts_host_dd_blocks(int nr, int nt, int np, const double* bounds, int nbounds, int dmin, int dmax, int order,
                            int* sizes, int cap, int* rows, int* cols) {
  if (!bounds || !sizes || order < 0 || order > 1) return KAD_ERR_ARG;
  XctsParams p;
  p.nr = nr;
  p.nt = nt;
  p.np = np;
  p.bounds.assign(bounds, bounds + nbounds);
  p.dmin = dmin;
  p.dmax = dmax;
  p.order = order;
  try {
    XctsSystem sy(p);
    sy.build();
    std::vector<int> bs, rr, cc;
    const int rc = dd_blocks(sy, bs, rr, cc);
    if (rc) return rc;
    for (int b = 0; b < (int)bs.size() && b < cap; ++b) sizes[b] = bs[b];
    if (rows) std::copy(rr.begin(), rr.end(), rows);
    if (cols) std::copy(cc.begin(), cc.end(), cols);
    return (int)bs.size();
  } catch (const std::exception& e) {
    fprintf(stderr, "kad_xcts_host_dd_blocks: %s\n", e.what());
    return KAD_ERR_ARG;
  }
}

int kad_xcts_host_info(int nr, int nt, int np, const double* bounds, int nbounds, int dmin, int dmax, double n0,
                       double a, double ome, int order, int* info, int* layout, int cap) {
  if (!bounds || !info || order < 0 || order > 1) return KAD_ERR_ARG;
  XctsParams p;
  p.nr = nr;
  p.nt = nt;
  p.np = np;
  p.bounds.assign(bounds, bounds + nbounds);
  p.dmin = dmin;
  p.dmax = dmax;
  p.n0 = n0;
  p.a = a;
  p.ome = ome;
  p.order = order;
  try {
    XctsSystem sy(p);
    sy.build();
    size_t tcode = 0;
    for (auto& pr : sy.tprog) tcode += pr.code.size();
    info[0] = sy.n_unknowns;
    info[1] = sy.n_rows;
    info[2] = (int)sy.tr.val.code.size();
    info[3] = (int)tcode;
    info[4] = sy.tr.nval_slots;
    info[5] = (int)sy.tprog.size();
    if (layout) {
      if (cap < 4 * (int)sy.layout.size()) return KAD_ERR_ARG;
      for (size_t q = 0; q < sy.layout.size(); ++q)
        for (int c = 0; c < 4; ++c) layout[4 * q + c] = sy.layout[q][c];
    }
    return (int)sy.layout.size();
  } catch (const std::exception& e) {
    fprintf(stderr, "[kadath_amd] kad_xcts_host_info: %s\n", e.what());
    return KAD_ERR_ARG;
  }
}
}

// ---------------------------------------------------------------------------
// Systems given as equation strings, and the entry points common to every system
// ---------------------------------------------------------------------------
struct kad_sysdef_impl {
  ParsedSystem* ps = nullptr;
  std::string err;
  ~kad_sysdef_impl() { delete ps; }
};

template <typename F>
static int guarded(kad_sysdef* def, F f) {
  if (!def) return KAD_ERR_ARG;
  auto* D = reinterpret_cast<kad_sysdef_impl*>(def);
  if (!D->ps) return KAD_ERR_ARG;
  try {
    f(*D->ps);
  } catch (const std::exception& e) {
    D->err = e.what();
    fprintf(stderr, "[kadath_amd] %s\n", e.what());
    return KAD_ERR_ARG;
  }
  return KAD_OK;
}

extern "C" {

int kad_sysdef_create(int nr, int nt, int np, const double* bounds, int nbounds, int dmin, int dmax,
                      kad_sysdef** out) {
  if (!bounds || nbounds < 1 || !out) return KAD_ERR_ARG;
  auto* D = new kad_sysdef_impl();
  try {
    D->ps = new ParsedSystem(nr, nt, np, std::vector<double>(bounds, bounds + nbounds), dmin, dmax, 0);
  } catch (const std::exception& e) {
    fprintf(stderr, "[kadath_amd] kad_sysdef_create: %s\n", e.what());
    delete D;
    return KAD_ERR_ARG;
  }
  *out = reinterpret_cast<kad_sysdef*>(D);
  return KAD_OK;
}

int kad_sysdef_destroy(kad_sysdef* def) {
  if (!def) return KAD_ERR_ARG;
  delete reinterpret_cast<kad_sysdef_impl*>(def);
  return KAD_OK;
}

int kad_sysdef_add_var(kad_sysdef* def, const char* name, int valence) {
  if (!name) return KAD_ERR_ARG;
  return guarded(def, [&](ParsedSystem& p) { p.add_var(name, valence); });
}
int kad_sysdef_add_cst(kad_sysdef* def, const char* name, double value) {
  if (!name) return KAD_ERR_ARG;
  return guarded(def, [&](ParsedSystem& p) { p.add_cst(name, value); });
}
int kad_sysdef_add_var_double(kad_sysdef* def, const char* name, double value) {
  if (!name) return KAD_ERR_ARG;
  int idx = -1;
  int rc = guarded(def, [&](ParsedSystem& p) { idx = p.add_var_double(name, value); });
  return rc ? rc : idx;
}
int kad_sysdef_add_global(kad_sysdef* def, const char* name, int dom, int bound, const char* expr) {
  if (!name || !expr) return KAD_ERR_ARG;
  int idx = -1;
  int rc = guarded(def, [&](ParsedSystem& p) { idx = p.add_global(name, dom, bound, expr); });
  return rc ? rc : idx;
}
int kad_sysdef_add_eq_int(kad_sysdef* def, int dom, int bound, const char* eq) {
  if (!eq) return KAD_ERR_ARG;
  return guarded(def, [&](ParsedSystem& p) { p.add_eq_int(dom, bound, eq); });
}
int kad_sysdef_add_param(kad_sysdef* def, const char* name, double value) {
  if (!name) return KAD_ERR_ARG;
  int idx = -1;
  int rc = guarded(def, [&](ParsedSystem& p) { idx = p.add_param(name, value); });
  return rc ? rc : idx;
}
int kad_sysdef_add_cst_field(kad_sysdef* def, const char* name, int valence, const double* conf, int64_t count) {
  if (!name || !conf || count <= 0) return KAD_ERR_ARG;
  return guarded(def, [&](ParsedSystem& p) { p.add_cst_field(name, valence, std::vector<double>(conf, conf + count)); });
}
int kad_sysdef_set_flat_metric(kad_sysdef* def, const char* name) {
  if (!name) return KAD_ERR_ARG;
  return guarded(def, [&](ParsedSystem& p) { p.set_flat_metric(name); });
}
int kad_sysdef_add_def(kad_sysdef* def, const char* text) {
  if (!text) return KAD_ERR_ARG;
  return guarded(def, [&](ParsedSystem& p) { p.add_def(text); });
}
int kad_sysdef_add_eq_inside(kad_sysdef* def, int dom, const char* eq, int order) {
  if (!eq) return KAD_ERR_ARG;
  return guarded(def, [&](ParsedSystem& p) { p.add_eq_inside(dom, eq, order); });
}
int kad_sysdef_add_eq_bc(kad_sysdef* def, int dom, int bound, const char* eq) {
  if (!eq) return KAD_ERR_ARG;
  return guarded(def, [&](ParsedSystem& p) { p.add_eq_bc(dom, bound, eq); });
}
int kad_sysdef_add_eq_matching(kad_sysdef* def, int dom, int bound, const char* expr) {
  if (!expr) return KAD_ERR_ARG;
  return guarded(def, [&](ParsedSystem& p) { p.add_eq_matching(dom, bound, expr); });
}
int kad_sysdef_space_add_eq(kad_sysdef* def, const char* eq, const char* m1, const char* m2) {
  if (!eq || !m1 || !m2) return KAD_ERR_ARG;
  return guarded(def, [&](ParsedSystem& p) { p.space_add_eq(eq, m1, m2); });
}
int kad_sysdef_space_add_bc(kad_sysdef* def, int bound, const char* eq) {
  if (!eq) return KAD_ERR_ARG;
  return guarded(def, [&](ParsedSystem& p) {
    if (bound == INNER_BC) p.space_add_inner_bc(eq);
    else p.space_add_outer_bc(eq);
  });
}

// Collocation points of the conf grid of domain d (r fastest, then theta, then phi):
// r (compactified domain: infinity at x = 1 is reported as +inf), theta, phi.  HOST out.
// Mark domain d as a shell of an adapted space with round boundaries (the homothetic
// shells of Space_adapted_bh): its surface integrals weight in configuration space
// (Domain_shell_inner_adapted::integ, domain_shell_inner_adapted.cpp:1134-1208).
int kad_sysdef_set_adapted(kad_sysdef* def, int d) {
  return guarded(def, [&](ParsedSystem& p) {
    if (d < p.dmin || d > p.dmax) throw std::runtime_error("kad_sysdef_set_adapted: domain out of range");
    if (p.doms[d].compact) throw std::runtime_error("kad_sysdef_set_adapted: the compactified domain is not adapted");
    p.doms[d].adapted = true;
  });
}

int kad_sysdef_coloc(kad_sysdef* def, int d, double* r, double* theta, double* phi) {
  return guarded(def, [&](ParsedSystem& p) {
    if (d < p.dmin || d > p.dmax) throw std::runtime_error("kad_sysdef_coloc: domain out of range");
    const Domain& dm = p.doms[d];
    for (int k = 0; k < dm.np; ++k)
      for (int j = 0; j < dm.nt; ++j)
        for (int i = 0; i < dm.nr; ++i) {
          const size_t q = (size_t)i + dm.nr * (j + (size_t)dm.nt * k);
          if (r) r[q] = std::isfinite(dm.R[q]) ? dm.R[q] : HUGE_VAL;
          if (theta) theta[q] = dm.th[j];
          if (phi) phi[q] = dm.ph[k];
        }
  });
}

// Host-only trace (no device): sizes and row layout of the declared system.
int kad_sysdef_host_trace(kad_sysdef* def, int order, int* info, int* row_layout, int cap) {
  if (!info || (order != 0 && order != 1)) return KAD_ERR_ARG;
  int q = 0;
  int rc = guarded(def, [&](ParsedSystem& p) {
    p.order_mode = order;
    p.build();
    size_t tcode = 0;
    for (auto& pr : p.tprog) tcode += pr.code.size();
    info[0] = p.n_unknowns;
    info[1] = p.n_rows;
    info[2] = (int)p.tr.val.code.size();
    info[3] = (int)tcode;
    info[4] = p.tr.nval_slots;
    info[5] = (int)p.tprog.size();
    for (const auto& e : p.eqs) {
      int row = e.row0;
      for (int c = 0; c < e.ncomp; ++c) {
        if (row_layout) {
          if (5 * (q + 1) > cap) throw std::runtime_error("kad_sysdef_host_trace: row layout capacity");
          const int v[5] = {e.kind, e.d, c, row, e.nrows[c]};
          for (int t = 0; t < 5; ++t) row_layout[5 * q + t] = v[t];
        }
        row += e.nrows[c];
        ++q;
      }
    }
  });
  if (rc) return rc;
  // a traced declaration is not built again
  auto* D = reinterpret_cast<kad_sysdef_impl*>(def);
  delete D->ps;
  D->ps = nullptr;
  return q;
}

// Trace the declared system into device programs and upload them.  The declaration
// is consumed (def is freed, also on failure).
int kad_system_build(kad_ctx* ctx, kad_sysdef* def, int order, int batch, kad_system** out) {
  if (!def) return KAD_ERR_ARG;
  auto* D = reinterpret_cast<kad_sysdef_impl*>(def);
  if (!ctx || !out || batch <= 0 || (order != 0 && order != 1) || !D->ps) {
    delete D;
    return KAD_ERR_ARG;
  }
  auto* S = new kad_system_impl();
  S->ctx = reinterpret_cast<kad::Ctx*>(ctx);
  S->B = batch;
  S->sys = D->ps;
  D->ps = nullptr;
  delete D;
  try {
    static_cast<ParsedSystem*>(S->sys)->order_mode = order;
    S->sys->build();
  } catch (const std::exception& e) {
    fprintf(stderr, "[kadath_amd] kad_system_build: %s\n", e.what());
    delete S;
    return KAD_ERR_ARG;
  }
  int rc = S->setup();
  if (rc) {
    delete S;
    return rc;
  }
  *out = reinterpret_cast<kad_system*>(S);
  return KAD_OK;
}

int kad_system_destroy(kad_system* s) { return kad_xcts_destroy(s); }

// n_unknowns, n_rows, scalar field components
int kad_system_sizes(kad_system* s, int* n_unknowns, int* n_rows, int* nfields) {
  if (!s) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  if (n_unknowns) *n_unknowns = S->sys->n_unknowns;
  if (n_rows) *n_rows = S->sys->n_rows;
  if (nfields) *nfields = S->sys->nfields;
  return KAD_OK;
}

int kad_system_layout(kad_system* s, int* out, int cap) { return kad_xcts_layout(s, out, cap); }
int kad_system_row_layout(kad_system* s, int* out, int cap) { return kad_xcts_row_layout(s, out, cap); }

// Values of field component f in domain d at the collocation points (HOST in, conf
// order): the field's coefficients become their transform (Scalar::set_domain then
// std_base / coef, tensor.cpp:609-650).
int kad_system_set_field(kad_system* s, int f, int d, const double* conf) {
  if (!s || !conf) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  SystemBase& sy = *S->sys;
  if (f < 0 || f >= sy.nfields || d < sy.dmin || d > sy.dmax) return KAD_ERR_ARG;
  const Domain& dm = sy.doms[d];
  std::vector<double> c(conf, conf + dm.conf_size());
  for (double& x : c)
    if (!std::isfinite(x)) return KAD_ERR_ARG;
  const std::vector<double> cf = host_coef(dm, sy.field_base(f, d), c);
  S->vals_current = false;
  KAD_HIP_CHECK(hipMemcpyAsync(S->val_arena + (int64_t)sy.field_slot[f][d] * S->stride, cf.data(),
                               cf.size() * sizeof(double), hipMemcpyHostToDevice, S->ctx->stream));
  KAD_HIP_CHECK(hipStreamSynchronize(S->ctx->stream));
  return KAD_OK;
}

// Values of field component f in domain d at the collocation points (HOST out):
// the synthesis of its coefficients (Val_domain::coef_i).
int kad_system_get_field(kad_system* s, int f, int d, double* conf) {
  if (!s || !conf) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  SystemBase& sy = *S->sys;
  if (f < 0 || f >= sy.nfields || d < sy.dmin || d > sy.dmax) return KAD_ERR_ARG;
  const Domain& dm = sy.doms[d];
  std::vector<double> cf(dm.coef_size());
  int rc = kad_xcts_get_coef(s, f, d, cf.data());
  if (rc) return rc;
  const Base b = sy.field_base(f, d);
  // coef_i: r, then theta, then phi (coef_i.cpp:96-104)
  Mat Mr = coef_i_matrix(CHEB, dm.nr);
  std::vector<double> t1(cf.size(), 0.0), t2(cf.size(), 0.0);
  for (int k = 0; k < dm.npc; ++k)
    for (int j = 0; j < dm.nt; ++j)
      for (int i = 0; i < dm.nr; ++i)
        for (int ii = 0; ii < dm.nr; ++ii)
          t1[i + dm.nr * (j + (size_t)dm.nt * k)] += Mr(i, ii) * cf[ii + dm.nr * (j + (size_t)dm.nt * k)];
  for (int k = 0; k < dm.npc; ++k) {
    Mat Mt = coef_i_matrix(b.bt[k], dm.nt);
    for (int j = 0; j < dm.nt; ++j)
      for (int jj = 0; jj < dm.nt; ++jj)
        for (int i = 0; i < dm.nr; ++i)
          t2[i + dm.nr * (j + (size_t)dm.nt * k)] += Mt(j, jj) * t1[i + dm.nr * (jj + (size_t)dm.nt * k)];
  }
  Mat Mp = coef_i_matrix(b.bp, dm.np);
  for (int k = 0; k < dm.np; ++k)
    for (int j = 0; j < dm.nt; ++j)
      for (int i = 0; i < dm.nr; ++i) {
        double v = 0.0;
        for (int kk = 0; kk < dm.npc; ++kk) v += Mp(k, kk) * t2[i + dm.nr * (j + (size_t)dm.nt * kk)];
        conf[i + dm.nr * (j + (size_t)dm.nt * k)] = v;
      }
  return KAD_OK;
}

int kad_system_get_coef(kad_system* s, int f, int d, double* out) { return kad_xcts_get_coef(s, f, d, out); }
int kad_system_set_coef(kad_system* s, int f, int d, const double* in) { return kad_xcts_set_coef(s, f, d, in); }
int kad_system_update(kad_system* s, const double* X) { return kad_xcts_update(s, X); }
int kad_system_perturbation(kad_system* s, uint64_t seed, double amp, double* out) {
  return kad_xcts_perturbation(s, seed, amp, out);
}
int kad_system_add_unknowns(kad_system* s, const double* X0) {
  if (!s || !X0) return KAD_ERR_ARG;
  return add_unknowns_host(reinterpret_cast<kad_system_impl*>(s), X0);
}
// Number of double unknowns (unknowns 0 .. count-1).
int kad_system_ndouble(kad_system* s) {
  if (!s) return KAD_ERR_ARG;
  return reinterpret_cast<kad_system_impl*>(s)->sys->ndouble;
}
// Current value of double unknown k (HOST out).
int kad_system_get_double(kad_system* s, int k, double* value) {
  if (!s || !value) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  SystemBase& sy = *S->sys;
  if (k < 0 || k >= sy.ndouble) return KAD_ERR_ARG;
  const std::string& name = sy.par_names[sy.dvar_par[k]];
  for (int d = sy.dmin; d <= sy.dmax; ++d) {
    const int slot = sy.param_slot(name, d);
    if (slot < 0) continue;
    KAD_HIP_CHECK(hipMemcpyAsync(value, S->val_arena + (int64_t)slot * S->stride, sizeof(double),
                                 hipMemcpyDeviceToHost, S->ctx->stream));
    KAD_HIP_CHECK(hipStreamSynchronize(S->ctx->stream));
    return KAD_OK;
  }
  return KAD_ERR_ARG;  // the unknown appears in no equation
}
// Global quantities (kad_sysdef_add_global) at the current fields, HOST out.
int kad_system_globals(kad_system* s, double* out) {
  if (!s || !out) return KAD_ERR_ARG;
  return globals_impl(reinterpret_cast<kad_system_impl*>(s), out);
}
// dQ_q/dp of the global quantities with respect to parameter `which`, by the adjoint
// method at the current (converged) fields; HOST out[nq], dQdu (HOST nq x n) may be NULL.
int kad_system_sensitivity(kad_system* s, int which, double* out, double* dQdu) {
  if (!s || !out) return KAD_ERR_ARG;
  return glob_sensitivity_impl(reinterpret_cast<kad_system_impl*>(s), which, out, dQdu);
}
int kad_system_set_param(kad_system* s, int which, double value) {
  if (!s) return KAD_ERR_ARG;
  return set_param_impl(reinterpret_cast<kad_system_impl*>(s), which, value);
}
int kad_system_do_newton(kad_system* s, double precision, double* error, int solver, double* times) {
  return kad_xcts_do_newton(s, precision, error, solver, times);
}
int kad_system_last_solve(kad_system* s, int* iters, double* resid) { return kad_xcts_last_solve(s, iters, resid); }

// The domain blocks of solvers 6-7 (HOST out): sizes (cap entries), rows and cols (n
// each, may be NULL).  Returns the number of blocks, KAD_ERR_ARG when they are not
// square (integral equations, double unknowns, unpaired interface conditions).
int kad_system_dd_blocks(kad_system* s, int* sizes, int cap, int* rows, int* cols) {
  if (!s || !sizes) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  std::vector<int> bs, rr, cc;
  int rc = dd_blocks(*S->sys, bs, rr, cc);
  if (rc) return rc;
  for (int b = 0; b < (int)bs.size() && b < cap; ++b) sizes[b] = bs[b];
  if (rows) std::copy(rr.begin(), rr.end(), rows);
  if (cols) std::copy(cc.begin(), cc.end(), cols);
  return (int)bs.size();
}

// Sizes and set-up times of the last domain-decomposed factorisation (kad_dd_info).
int kad_system_dd_info(kad_system* s, int* sizes, double* times) {
  if (!s) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  if (!S->dd) return KAD_ERR_ARG;
  return kad_dd_info(S->dd, sizes, times);
}

// Pivoting of the last domain-decomposed factorisation (kad_dd_pivoting).
int kad_system_dd_pivoting(kad_system* s, int* static_orders, double* growth) {
  if (!s) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  if (!S->dd) return KAD_ERR_ARG;
  return kad_dd_pivoting(S->dd, static_orders, growth);
}

// F(u) (device, n_rows): System_of_eqs::sec_member.
int kad_residual(kad_system* s, double* F) { return kad_xcts_residual(s, F); }

// Per (equation, component) max |F| over its rows (HOST out, cap entries), in row-layout
// order: System_of_eqs::check_equations (solver.cpp:24-47).  Returns the entry count.
int kad_check_equations(kad_system* s, double* errors, int cap) {
  if (!s || !errors) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  int rc = S->value_pass();
  if (rc) return rc;
  std::vector<double> h(S->sys->n_rows);
  KAD_HIP_CHECK(hipMemcpyAsync(h.data(), S->F, h.size() * sizeof(double), hipMemcpyDeviceToHost, S->ctx->stream));
  KAD_HIP_CHECK(hipStreamSynchronize(S->ctx->stream));
  int q = 0;
  for (const auto& e : S->sys->eqs) {
    int row = e.row0;
    for (int c = 0; c < e.ncomp; ++c) {
      if (q >= cap) return KAD_ERR_ARG;
      double m = 0.0;
      for (int r = row; r < row + e.nrows[c]; ++r) {
        const double a = std::fabs(h[r]);
        if (a > m || a != a) m = a;
      }
      errors[q++] = m;
      row += e.nrows[c];
    }
  }
  return q;
}

// Columns [col_begin, col_begin + col_count) of J (every do_col_J of that range,
// solver.cpp:120-214) into the device tile J_tile (column-major, ld >= n_rows), fp64
// (dtype 0) or fp32 (dtype 1).  The tile's columns are cleared first; the values are
// those of the current fields (the value pass runs when they changed).
int kad_jvp_fill(kad_system* s, int col_begin, int col_count, void* J_tile, int64_t ld, int dtype) {
  if (!s || !J_tile || col_begin < 0 || col_count <= 0 || (dtype != 0 && dtype != 1)) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  const int n = S->sys->n_unknowns, m = S->sys->n_rows;
  if (ld < m || col_begin + (int64_t)col_count > n) return KAD_ERR_ARG;
  hipStream_t st = S->ctx->stream;
  int rc = S->ensure_values();
  if (rc) return rc;
  const size_t es = dtype == 0 ? sizeof(double) : sizeof(float);
  KAD_HIP_CHECK(hipMemset2DAsync(J_tile, (size_t)ld * es, 0, (size_t)m * es, (size_t)col_count, st));
  const int c1 = col_begin + col_count;
  if (S->levels_ready()) {
    if ((rc = S->columns(col_begin, c1, col_begin, J_tile, ld, dtype))) return rc;
    KAD_HIP_CHECK(hipStreamSynchronize(st));
    return KAD_OK;
  }
  if ((rc = S->double_columns(J_tile, ld, col_begin, c1, col_begin, dtype))) return rc;
  for (auto& p : S->tprogs) {
    const int lo = std::max(col_begin, p.off), hi = std::min(c1, p.off + p.cnt);
    for (int u = lo; u < hi; u += S->B) {
      const int nb = std::min(S->B, hi - u);
      if ((rc = S->run(p.code, nb, u - p.off, p.seed_tab, J_tile, (int64_t)u - col_begin, ld, dtype))) return rc;
    }
  }
  KAD_HIP_CHECK(hipStreamSynchronize(st));
  return KAD_OK;
}

// out = J^T w (device, n_unknowns; w device, n_rows), matrix-free: every tangent
// program runs as for the fill, and its row exports are replaced by their transposes
// (per column, the dot product of w with the exported rows), so J is never formed.
int kad_vjp(kad_system* s, const double* w, double* out) {
  if (!s || !w || !out) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  hipStream_t st = S->ctx->stream;
  int rc = S->ensure_values();
  if (rc) return rc;
  KAD_HIP_CHECK(hipMemsetAsync(out, 0, (size_t)S->sys->n_unknowns * sizeof(double), st));
  if (S->levels_ready()) {
    if ((rc = S->columns(0, S->sys->n_unknowns, 0, out, 0, 0, w))) return rc;
    KAD_HIP_CHECK(hipStreamSynchronize(st));
    return KAD_OK;
  }
  for (int k = 0; k < S->sys->ndouble; ++k) {
    const DevProgram& pp = S->par_progs[S->sys->dvar_par[k]];
    if ((rc = S->run(pp.code, 1, 0, pp.seed_tab, out, k, 0, 0, w))) return rc;
  }
  for (auto& p : S->tprogs)
    for (int u0 = 0; u0 < p.cnt; u0 += S->B) {
      const int nb = std::min(S->B, p.cnt - u0);
      if ((rc = S->run(p.code, nb, u0, p.seed_tab, out, (int64_t)p.off + u0, 0, 0, w))) return rc;
    }
  KAD_HIP_CHECK(hipStreamSynchronize(st));
  return KAD_OK;
}

// dF/dp of parameter `which` at the current fields (device out, n_rows).
int kad_param_tangent(kad_system* s, int which, double* out) {
  if (!s || !out) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  if (which < 0 || which >= (int)S->par_progs.size()) return KAD_ERR_ARG;
  int rc = S->ensure_values();
  if (rc) return rc;
  KAD_HIP_CHECK(hipMemsetAsync(out, 0, (size_t)S->sys->n_rows * sizeof(double), S->ctx->stream));
  const DevProgram& pp = S->par_progs[which];
  if ((rc = S->run(pp.code, 1, 0, pp.seed_tab, out, 0, S->sys->n_rows))) return rc;
  KAD_HIP_CHECK(hipStreamSynchronize(S->ctx->stream));
  return KAD_OK;
}

}  // extern "C"

extern "C" {
// Options of the low-precision solvers: which 0 = forcing factor c (refinement target
// max(1e-13, c min(1, ||F||_inf)); 0, the default, runs it to its attainable
// accuracy), which 1 = reuse the low-precision factors while the previous refinement
// took at most `value` inner steps (0, the default: factor every step).
int kad_system_set_option(kad_system* s, int which, double value) {
  if (!s || !(value >= 0.0)) return KAD_ERR_ARG;
  auto* S = reinterpret_cast<kad_system_impl*>(s);
  if (which == 0) {
    S->forcing = value;
  } else if (which == 1) {
    S->reuse_inner = (int)value;
  } else if (which == 2) {
    // forget every factorisation kept for reuse, and the kept pivot orders: the next
    // step factors its own J with partial pivoting
    S->lo_valid = S->fac_valid = S->dd_valid = S->dd_orders = false;
    S->prev_inner = 0;
  } else if (which == 5) {
    // element-wise instructions applied in the spectral pass that feeds them (1, the
    // default) or launched on their own (0)
    if (value != 0.0 && value != 1.0) return KAD_ERR_ARG;
    S->fuse_ew = value != 0.0;
  } else if (which == 4) {
    // static pivoting in solvers 6-7 (1, the default) or partial pivoting at every
    // factorisation (0)
    if (value != 0.0 && value != 1.0) return KAD_ERR_ARG;
    S->dd_static = value != 0.0;
  } else if (which == 3) {
    // streams of the Jacobian fill
    if (value < 1.0 || value > (double)kad_system_impl::kFillMax || value != (double)(int)value) return KAD_ERR_ARG;
    S->nfill = (int)value;
  } else {
    return KAD_ERR_ARG;
  }
  return KAD_OK;
}
}  // extern "C"
