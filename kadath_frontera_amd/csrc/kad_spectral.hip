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

namespace kad {

// One workgroup per batch element.
__global__ __launch_bounds__(256) void apply3d_kernel(const double* __restrict__ in, int64_t in_stride,
                                                      double* __restrict__ out, int64_t out_stride, int d0, int d1,
                                                      int d2, Passes P, const double* __restrict__ pool,
                                                      int accumulate, double scale, int stage_pool, int inplace,
                                                      PostOp post) {
  extern __shared__ double lds[];
  const int64_t b = blockIdx.x;
  apply3d_body(in + b * in_stride, out + b * out_stride, d0, d1, d2, P, pool, accumulate, scale, stage_pool, inplace,
               post, b, lds);
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

int apply3d_launch(const double* in, int64_t in_stride, double* out, int64_t out_stride, int nbatch, int d0, int d1,
                   int d2, const Passes& P, const double* pool, int accumulate, double scale, hipStream_t s,
                   const PostOp* post) {
  if (nbatch <= 0) return KAD_OK;
  if (post && post->n > 0 && (post->n > kMaxChain || accumulate || scale != 1.0 || !post->dst)) return KAD_ERR_ARG;
  const PostOp pop = post ? *post : PostOp();
  const Apply3dShape sh = apply3d_shape(d0, d1, d2, P);
  if (sh.lds > 160 * 1024) return KAD_ERR_ARG;
  GemmTimer* tm = g_apply_timer;
  bool timed = false;
  if (tm) {
    // algorithmic HBM bytes: the input arrays read once, the output arrays written
    // once (accumulate also reads them); the per-line matrices are cache-resident
    int od[3] = {d0, d1, d2};
    for (int p = 0; p < P.npass; ++p) od[P.axis[p]] = P.nout[p];
    const double nin = (double)d0 * d1 * d2, nout = (double)od[0] * od[1] * od[2];
    // (each fused instruction's other operand adds its array per batch element)
    double extra = 0.0;
    for (int k = 0; k < pop.n; ++k)
      if (pop.op[k].o && pop.op[k].os != 0) extra += nout;
    const int rc = tm->begin(s, 8.0 * nbatch * (nin + nout * (accumulate ? 2 : 1) + extra));
    if (rc < 0) return rc;
    timed = rc == 0;
  }
  apply3d_kernel<<<nbatch, 256, sh.lds, s>>>(in, in_stride, out, out_stride, d0, d1, d2, P, pool, accumulate, scale,
                                          sh.stage_pool, sh.inplace, pop);
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
