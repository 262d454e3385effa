// Grouped execution of the device programs (value program, tangent programs).
//
// A traced program is a few hundred to a few thousand instructions on small arrays, but
// its dependency depth is about 32: run one launch per instruction, a residual at 9x7x4
// is 2004 dependent launches of a single workgroup each.  Here one launch executes every
// instruction of a dependency level, over all columns of every program in the group
// (element-wise regions by a second one), one workgroup per (instruction, column); the instruction is read from a device table
// with scalar loads (the workgroup's index is uniform), so all its branches are uniform.
// Instructions of one level never touch the same memory, and the launch boundary orders
// the levels.  The operations are those of the per-instruction kernels, in the same
// order per element, so results are the same bit for bit.
#include "kad_group.hpp"
#include "kad_apply3d.hpp"
#include "kad_ctx.hpp"
#include "host/spectral.hpp"

namespace kad {

namespace {
typedef const __attribute__((address_space(4))) GroupOp COp;
typedef const __attribute__((address_space(4))) ClusterStep CStep;

struct Where {
  double* val;
  double* tan;
  int64_t stride;
  int nb, b;
  // (32-bit factors: the arrays of an arena are fewer than 2^31, an array has fewer elements)
  template <typename O>
  __device__ __forceinline__ double* at(const O& o) const {
    const unsigned n = o.tan ? (unsigned)o.slot * (unsigned)nb + (unsigned)b : (unsigned)o.slot;
    return (o.tan ? tan : val) + (uint64_t)n * (unsigned)stride;
  }
};

// Value of one exported row (inside: a coefficient minus its Galerkin partner; boundary:
// the line's value at x = bsign).
__device__ __forceinline__ double row_value(const DevRow R, const double* x, bool bd, int nr, int bsign) {
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
  return v;
}

// An element-wise region of the program, U elements per lane from element e0: every array
// it needs from outside is read once (or kept in a temporary), its intermediate values live
// in registers (temporary d of element u is entry d of t[u], addressed through the register
// index), only what other instructions read is stored.  The array operands of the next Q
// steps are loaded while Q steps run.  Bound by instruction issue (about 150 instructions per
// step and wave, 2/3 of them decoding and register indexing) and, 44% of a wave's time, by
// the loads; hence four elements per lane, one decoding for them, and no partly filled
// sweeps.  With one element per lane and the temporaries in LDS J^T w at 13x9x8 took 31.8 ms
// and 5001 fp32 columns at 17x13x12 25.4, now 26.2 and 20.9 (15 temporaries and two waves
// per SIMD were 2% slower than 7 and three).
template <int U>
__device__ __forceinline__ void cluster_body(const GroupArgs& g, const Where& at, const COp& op, int e0) {
  typedef double Temps __attribute__((ext_vector_type(kClusterTemps + 1)));
  const int size = op.size, n = op.nsteps;
  const CStep* const st = (const CStep*)g.steps + op.step0;
  constexpr int Q = 2;
  Temps t[U];
#pragma unroll
  for (int u = 0; u < U; ++u) t[u] = Temps(0.0);
  unsigned at_e[U];
#pragma unroll
  for (int u = 0; u < U; ++u) at_e[u] = min(e0 + u * 64, size - 1);
  double ga[Q][U], gb[Q][U];
  auto load = [&](int i0) {
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      if (i0 + i < n) {
        if (st[i0 + i].a == -2) {
          const double* const p = at.at(st[i0 + i].ga);
#pragma unroll
          for (int u = 0; u < U; ++u) ga[i][u] = p[at_e[u]];
        }
        if (st[i0 + i].b == -2) {
          const double* const p = at.at(st[i0 + i].gb);
#pragma unroll
          for (int u = 0; u < U; ++u) gb[i][u] = p[at_e[u]];
        }
      }
    }
  };
  load(0);
  for (int i0 = 0; i0 < n; i0 += Q) {
    double xa[Q][U], xb[Q][U];
#pragma unroll
    for (int i = 0; i < Q; ++i)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        xa[i][u] = ga[i][u];
        xb[i][u] = gb[i][u];
      }
    load(i0 + Q);  // the next steps' operands, while these run
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      if (i0 + i >= n) break;
      const CStep& s = st[i0 + i];
      const int a = s.a, b = s.b;
      // unconditional register accesses (temporary kClusterTemps takes what nothing reads):
      // with a branch around each, the compiler selected between copies of all temporaries
      const int ca = s.ca, cb = s.cb, d = s.d;
      double x[U], y[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        t[u][ca] = xa[i][u];
        t[u][cb] = xb[i][u];
        x[u] = a < 0 ? xa[i][u] : t[u][a < 0 ? 0 : a];
        y[u] = b < 0 ? xb[i][u] : t[u][b < 0 ? 0 : b];
      }
      ew_ops<U>(s.kind, x, y, s.s);
#pragma unroll
      for (int u = 0; u < U; ++u) t[u][d] = x[u];
      if (s.gd.slot >= 0) {
        double* const out = at.at(s.gd);
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (e0 + u * 64 < size) out[at_e[u]] = x[u];
      }
    }
  }
}

template <typename T>
__device__ __forceinline__ void put_row(void* out, int64_t at, int acc, double v, double c0 = 0.0) {
  T* o = (T*)out + at;
  *o = acc ? (T)((double)*o + v + c0) : (T)(v + c0);
}
}  // namespace

// The entry of this workgroup and its place in it.
__device__ __forceinline__ void group_entry(const GroupArgs& g, int& q, int& oi, int& b) {
  int blk = 0;
  q = 0;
#pragma unroll
  for (int i = 1; i < kGroupEntries; ++i)
    if (i < g.nent && (int)blockIdx.x >= g.blk0[i]) {
      q = i;
      blk = g.blk0[i];
    }
  const int loc = blockIdx.x - blk, nbp = g.e[q].nbp;
  oi = loc / nbp;
  b = loc - oi * nbp;
}

// The element-wise regions of a level, in a launch of their own, a wave per
// kClusterChunk elements of (region, column): their temporaries leave three waves per SIMD,
// the passes have five.
__global__ __launch_bounds__(64, 3) void cluster_kernel(GroupArgs g) {
  int q, oi, b;
  group_entry(g, q, oi, b);
  const int nch = g.e[q].nch, op_i = oi / nch, e0 = (oi - op_i * nch) * kClusterChunk;
  if (op_i >= g.e[q].nops || b >= g.e[q].nb) return;  // padding
  const COp& op = *((COp*)g.ops + g.e[q].op0 + op_i);
  if (e0 >= op.size) return;
  const Where at{g.val, g.tan + g.e[q].base, g.stride, g.e[q].nb, b};
  cluster_body<kClusterChunk / 64>(g, at, op, e0 + threadIdx.x);
}

__global__ __launch_bounds__(256) void group_kernel(GroupArgs g) {
  extern __shared__ double lds[];
  const int tid = threadIdx.x;
  int q, oi, b;
  group_entry(g, q, oi, b);
  if (oi >= g.e[q].nops || b >= g.e[q].nb) return;  // padding
  const COp& op = *((COp*)g.ops + g.e[q].op0 + oi);
  const Where at{g.val, g.tan + g.e[q].base, g.stride, g.e[q].nb, b};
  const int64_t col = g.e[q].col0 + b;
  const int kind = op.kind;
  if (kind == GK_LIN || kind == GK_EW) {
    PostOp post;
    post.n = op.nstep;
    post.dst = at.at(op.dst);
#pragma unroll
    for (int k = 0; k < kMaxChain; ++k)
      if (k < post.n) {
        post.op[k].kind = op.st[k].kind;
        post.op[k].side = op.st[k].side;
        post.op[k].o = op.st[k].o.slot >= 0 ? at.at(op.st[k].o) : nullptr;
        post.op[k].s = op.st[k].s;
      }
    const double* a = at.at(op.a);
    if (kind == GK_LIN) {
      apply3d_body(a, post.dst, op.P, post, 0, lds);
      return;
    }
    const double* y = op.b.slot >= 0 ? at.at(op.b) : nullptr;
    const int size = op.size, ew = op.ew;
    const double s = op.s;
    // every load of U elements first (operands of the head and of every step)
    constexpr int U = 4;
    for (int e0 = 0; e0 < size; e0 += 256 * U) {
      double xv[U], yv[U], o[U][kMaxChain];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = e0 + u * 256 + tid;
        const bool in = e < size;
        xv[u] = in ? a[e] : 0.0;
        yv[u] = (in && y) ? y[e] : 0.0;
        post_load(post, 0, in ? e : 0, o[u]);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = e0 + u * 256 + tid;
        if (e < size) post.dst[e] = post_ops(post, ew_op(ew, xv[u], yv[u], s), o[u]);
      }
    }
    return;
  }
  if (kind == GK_SEED) {
    // unit seed of unknown u (affecte_tau_one_coef), zero elsewhere
    double* d = at.at(op.dst);
    const int u = g.e[q].u0 + b, size = op.size;
    const int n = u < op.nu ? op.scnt[u] : 0;
    for (int e = tid; e < size; e += 256) {
      double v = 0.0;
      for (int t = 0; t < n; ++t)
        if (op.spos[3 * u + t] == e) v = op.sval[3 * u + t];
      d[e] = v;
    }
    return;
  }
  const double* x = op.a.slot >= 0 ? at.at(op.a) : nullptr;
  if (kind == GK_EXPORT_GL) {
    // one row: fac * surface integral of x at a boundary (or its point value) + c0
    if (tid != 0) return;
    double val = 0.0;
    if (x && op.pt) {
      val = x[0] * op.s;
    } else {
      double tot = 0.0;
      if (x && (op.aux == kadhost::COS_EVEN || op.aux == kadhost::SIN_ODD)) {
        for (int j = 0; j < op.nt; ++j) {
          const double wj = op.aux == kadhost::COS_EVEN ? (j == 0 ? M_PI : 0.0) : 2.0 / (2.0 * j + 1.0);
          if (wj == 0.0) continue;
          double v = 0.0, sg = 1.0;
          for (int i = 0; i < op.nr; ++i) {
            v += sg * x[i + (int64_t)op.nr * j];
            sg *= op.bsign;
          }
          tot += wj * v;
        }
      }
      val = tot * 2.0 * M_PI * op.s;
    }
    if (g.w) {
      ((double*)g.out)[col] += g.w[op.row0] * val;
      return;
    }
    const int64_t o = op.row0 + col * g.ldo;
    if (g.dtype == 0) put_row<double>(g.out, o, op.accumulate, val, op.c0);
    else put_row<float>(g.out, o, op.accumulate, val, op.c0);
    return;
  }
  const bool bd = kind == GK_EXPORT_BD;
  const int nrows = op.nrows, row0 = op.row0, nr = op.nr, bsign = op.bsign;
  const DevRow* rows = op.rows;
  if (g.w) {
    // transposed export: a fixed-order reduction over the rows; a program's exports are
    // on different levels, in program order, so the column's sum is deterministic
    double acc = 0.0;
    for (int r = tid; r < nrows; r += 256) acc += g.w[row0 + r] * row_value(rows[r], x, bd, nr, bsign);
    lds[tid] = acc;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
      if (tid < st) lds[tid] += lds[tid + st];
      __syncthreads();
    }
    if (tid == 0) ((double*)g.out)[col] += op.sign * lds[0];
    return;
  }
  for (int r = tid; r < nrows; r += 256) {
    const double v = row_value(rows[r], x, bd, nr, bsign);
    const int64_t o = (row0 + r) + col * g.ldo;
    if (g.dtype == 0) put_row<double>(g.out, o, op.accumulate, op.sign * v);
    else put_row<float>(g.out, o, op.accumulate, op.sign * v);
  }
}

int group_launch(const GroupArgs& g, int blocks, bool clusters, size_t lds, hipStream_t s) {
  if (blocks <= 0) return KAD_OK;
  if (g.nent < 1 || g.nent > kGroupEntries || lds > kMaxLds) return KAD_ERR_ARG;
  if (clusters) cluster_kernel<<<blocks, 64, 0, s>>>(g);
  else group_kernel<<<blocks, 256, lds, s>>>(g);
  KAD_HIP_CHECK(hipGetLastError());
  return KAD_OK;
}

}  // namespace kad
