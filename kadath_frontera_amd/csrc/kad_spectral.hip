// Batched spectral transforms and 1-D coefficient-space operators.
//
// Replaces Base_spectral::coef / coef_i (src/Coef/coef.cpp:28-104,
// src/Coef/coef_i.cpp:28-104) and Base_spectral::ope_1d
// (include/implementation/ope_1d.cpp:25-82), which gather each 1-D line of a
// Val_domain, call FFTW (or a coefficient recurrence) on it and scatter back.
//
// Here every 1-D operation on a line of length <= 64 is a small dense matrix
// (chosen per line by the line's basis), and a whole 3-D domain array
// (<= ~33x33x34 doubles) is staged in LDS: one coalesced HBM read, any number of
// 1-D passes along r, theta, phi in LDS, one coalesced HBM write.
//
// Array layout: index 0 (r) fastest, then theta, then phi -- the reference's
// Array/Index order (include/implementation/index.cpp:84-96).
#include "kad_common.hpp"
#include "kad_apply3d.hpp"
#include "kad_ctx.hpp"
#include <algorithm>

namespace kad {

// One workgroup per batch element.
__global__ __launch_bounds__(256) void apply3d_kernel(const double* __restrict__ in, int64_t in_stride,
                                                      double* __restrict__ out, int64_t out_stride, LinePlan P,
                                                      PostOp post) {
  extern __shared__ double lds[];
  const int64_t b = blockIdx.x;
  apply3d_body(in + b * in_stride, out + b * out_stride, P, post, b, lds);
}

// Contiguous 1-D lines: in [L][nin] -> out [L][nout], one matrix for all lines.
// A workgroup stages LINES_PER_WG lines in LDS (coalesced) together with M.
constexpr int LINES_PER_WG = 64;
__global__ __launch_bounds__(256) void apply_lines_kernel(const double* __restrict__ in, double* __restrict__ out,
                                                          int64_t L, int nin, int nout, const double* __restrict__ M) {
  extern __shared__ double lds[];
  double* Ms = lds;                    // nout*nin
  double* xs = lds + nout * nin;       // LINES_PER_WG*nin
  const int64_t l0 = (int64_t)blockIdx.x * LINES_PER_WG;
  const int nl = (int)min<int64_t>(LINES_PER_WG, L - l0);
  for (int e = threadIdx.x; e < nout * nin; e += blockDim.x) Ms[e] = M[e];
  const double* src = in + l0 * nin;
  for (int e = threadIdx.x; e < nl * nin; e += blockDim.x) xs[e] = src[e];
  __syncthreads();
  double* dst = out + l0 * nout;
  for (int e = threadIdx.x; e < nl * nout; e += blockDim.x) {
    const int l = e / nout, o = e % nout;
    const double* m = Ms + o * nin;
    const double* x = xs + l * nin;
    double s = 0.0;
    for (int q = 0; q < nin; ++q) s += m[q] * x[q];
    dst[e] = s;
  }
}

bool lines_build(int d0, int d1, int d2, const PassDesc* passes, int npass, int pool_size, LinePlan& P,
                 LineEnt* tab, size_t cap, size_t* used, size_t* toff) {
  if (npass < 1 || npass > MAX_PASSES) return false;
  int dm[3] = {d0, d1, d2};
  P = LinePlan();
  P.npass = npass;
  P.pool_size = pool_size;
  P.size_in = P.maxsize = d0 * d1 * d2;
  P.single = P.small = 1;
  size_t n = 0;
  for (int p = 0; p < npass; ++p) {
    const int ax = passes[p].axis;
    LinePlan::Pass& q = P.p[p];
    int od[3] = {dm[0], dm[1], dm[2]};
    od[ax] = passes[p].nout;
    q.nin = dm[ax];
    q.nout = passes[p].nout;
    q.sin = ax == 0 ? 1 : (ax == 1 ? dm[0] : dm[0] * dm[1]);
    q.sout = ax == 0 ? 1 : (ax == 1 ? od[0] : od[0] * od[1]);
    toff[p] = n;
    const int na = ax == 0 ? dm[1] : dm[0], nb = ax == 2 ? dm[1] : dm[2];
    q.nlines = na * nb;
    if (n + q.nlines > cap) return false;
    for (int b = 0; b < nb; ++b)
      for (int a = 0; a < na; ++a) {
        LineEnt e{0, 0, 0, 0};
        if (ax == 0) {  // line (j, k) = (a, b)
          e = {dm[0] * (a + dm[1] * b), od[0] * (a + od[1] * b), passes[p].line_mat[a + dm[1] * b], 0};
        } else if (ax == 1) {  // (i, k)
          e = {a + dm[0] * dm[1] * b, a + od[0] * od[1] * b, passes[p].line_mat[b], 0};
        } else {  // (i, j)
          e = {a + dm[0] * b, a + od[0] * b, passes[p].line_mat[0], 0};
        }
        tab[n++] = e;
      }
    // lines with one matrix together: few waves hold lines of two
    std::stable_sort(tab + toff[p], tab + n, [](const LineEnt& x, const LineEnt& y) { return x.off < y.off; });
    if (q.nlines * q.nout > kSmallArray) P.small = 0;
    if ((q.nlines > 256 && q.nin != q.nout) || q.nin > kLineTemplates) P.single = 0;
    dm[0] = od[0];
    dm[1] = od[1];
    dm[2] = od[2];
    P.maxsize = std::max(P.maxsize, dm[0] * dm[1] * dm[2]);
  }
  if (P.small) P.single = 0;  // outputs by other threads than read the line: two buffers
  P.size_out = dm[0] * dm[1] * dm[2];
  *used = n;
  return true;
}

int apply3d_launch(const double* in, int64_t in_stride, double* out, int64_t out_stride, int nbatch, const LinePlan& P,
                   hipStream_t s, const PostOp* post) {
  if (nbatch <= 0) return KAD_OK;
  if (post && post->n > 0 && (post->n > kMaxChain || !post->dst)) return KAD_ERR_ARG;
  const PostOp pop = post ? *post : PostOp();
  const size_t lds = lines_lds(P);
  if (lds > kMaxLds || P.npass < 1) return KAD_ERR_ARG;
  GemmTimer* tm = g_apply_timer;
  bool timed = false;
  if (tm) {
    // algorithmic HBM bytes: the input arrays read once, the output arrays written once;
    // the matrices are cache-resident (each fused instruction's other operand adds its
    // array per batch element)
    double extra = 0.0;
    for (int k = 0; k < pop.n; ++k)
      if (pop.op[k].o && pop.op[k].os != 0) extra += P.size_out;
    const int rc = tm->begin(s, 8.0 * nbatch * ((double)P.size_in + P.size_out + extra));
    if (rc < 0) return rc;
    timed = rc == 0;
  }
  apply3d_kernel<<<nbatch, 256, lds, s>>>(in, in_stride, out, out_stride, P, pop);
  KAD_HIP_CHECK(hipGetLastError());
  if (timed && tm->end(s)) return KAD_ERR_HIP;
  return KAD_OK;
}

int apply_lines_launch(const double* in, double* out, int64_t L, int nin, int nout, const double* M, hipStream_t s) {
  if (L <= 0) return KAD_OK;
  const size_t lds = ((size_t)nout * nin + (size_t)LINES_PER_WG * nin) * sizeof(double);
  if (lds > 160 * 1024) return KAD_ERR_ARG;
  apply_lines_kernel<<<(unsigned)cdiv(L, LINES_PER_WG), 256, lds, s>>>(in, out, L, nin, nout, M);
  KAD_HIP_CHECK(hipGetLastError());
  return KAD_OK;
}

}  // namespace kad
