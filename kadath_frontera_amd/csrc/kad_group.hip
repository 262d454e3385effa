// Grouped execution of the device programs (value program, tangent programs).
//
// A traced program is a few hundred to a few thousand instructions on small arrays, but
// its dependency depth is about 32: run one launch per instruction, a residual at 9x7x4
// is 2004 dependent launches of a single workgroup each.  Here one launch executes every
// instruction of a dependency level, over all columns of every program in the group,
// one workgroup per (instruction, column); the instruction is read from a device table
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
  template <typename O>
  __device__ __forceinline__ double* at(const O& o) const {
    return o.tan ? tan + ((int64_t)o.slot * nb + b) * stride : val + (int64_t)o.slot * stride;
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

// An element-wise region of the program: every array it needs from outside is read once
// (or kept in a temporary), its intermediate values live in LDS temporaries
// (lds[temporary][element of the thread][thread]), only what other instructions read is
// stored.  U elements per thread and 8 / U steps have their array operands loaded
// together: one at a time, a step waited out a memory latency and the decoding of the
// next one (1900 cycles per step of 256 elements).  Bound by that latency and by the few
// workgroups that the temporaries' LDS leaves per CU: J^T w at 13x9x8 moves 66 GB at 2.05
// TB/s.  One instruction at a time it moved more arrays through memory: 34.2 ms, 31.8 now;
// 5001 fp32 columns at 17x13x12 36.4 and 25.3.
template <int U>
__device__ __forceinline__ void cluster_body(const GroupArgs& g, const Where& at, const COp& op, double* lds, int tid) {
  const int size = op.size, n = op.nsteps;
  const CStep* const st = (const CStep*)g.steps + op.step0;
  constexpr int Q = 8 / U > 4 ? 4 : 8 / U;
  for (int e0 = 0; e0 < size; e0 += 256 * U) {
    double ga[Q][U], gb[Q][U];
    auto load = [&](int i0) {
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        if (i0 + i < n) {
          if (st[i0 + i].a == -2) {
            const double* const p = at.at(st[i0 + i].ga);
#pragma unroll
            for (int u = 0; u < U; ++u) ga[i][u] = p[min(e0 + u * 256 + tid, size - 1)];
          }
          if (st[i0 + i].b == -2) {
            const double* const p = at.at(st[i0 + i].gb);
#pragma unroll
            for (int u = 0; u < U; ++u) gb[i][u] = p[min(e0 + u * 256 + tid, size - 1)];
          }
        }
      }
    };
    load(0);
    for (int i0 = 0; i0 < n; i0 += Q) {
      double ca_[Q][U], cb_[Q][U];
#pragma unroll
      for (int i = 0; i < Q; ++i)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          ca_[i][u] = ga[i][u];
          cb_[i][u] = gb[i][u];
        }
      load(i0 + Q);  // the next steps' operands, while these run
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        if (i0 + i >= n) break;
        const CStep& s = st[i0 + i];
        const int a = s.a, b = s.b, ca = s.ca, cb = s.cb, d = s.d, kind = s.kind;
        double* const out = s.gd.slot >= 0 ? at.at(s.gd) : nullptr;
        const double sc = s.s;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          double* const l = lds + u * 256 + tid;
          if (ca >= 0) l[ca * 256 * U] = ca_[i][u];
          if (cb >= 0) l[cb * 256 * U] = cb_[i][u];
          const double x = a >= 0 ? l[a * 256 * U] : ca_[i][u];
          const double y = b >= 0 ? l[b * 256 * U] : cb_[i][u];
          const double r = ew_op(kind, x, y, sc);
          if (d >= 0) l[d * 256 * U] = r;
          if (out && e0 + u * 256 + tid < size) out[e0 + u * 256 + tid] = r;
        }
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

__global__ __launch_bounds__(256) void group_kernel(GroupArgs g) {
  extern __shared__ double lds[];
  const int bid = blockIdx.x, tid = threadIdx.x;
  int q = 0, blk = 0;
#pragma unroll
  for (int i = 1; i < kGroupEntries; ++i)
    if (i < g.nent && bid >= g.blk0[i]) {
      q = i;
      blk = g.blk0[i];
    }
  const int loc = bid - blk, nbp = g.e[q].nbp;
  const int oi = loc / nbp, b = loc - oi * nbp;
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
  if (kind == GK_CLUSTER) {
    // few temporaries leave LDS for more elements per thread
    if (op.per == 4) cluster_body<4>(g, at, op, lds, tid);
    else if (op.per == 2) cluster_body<2>(g, at, op, lds, tid);
    else cluster_body<1>(g, at, op, lds, tid);
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

int group_launch(const GroupArgs& g, int blocks, size_t lds, hipStream_t s) {
  if (blocks <= 0) return KAD_OK;
  if (g.nent < 1 || g.nent > kGroupEntries || lds > 160 * 1024) return KAD_ERR_ARG;
  group_kernel<<<blocks, 256, lds, s>>>(g);
  KAD_HIP_CHECK(hipGetLastError());
  return KAD_OK;
}

}  // namespace kad
