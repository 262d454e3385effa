// Device body of a chain of 1-D passes over one 3-D domain array staged in LDS: used by
// the batched transform kernel (kad_spectral.hip) and by the grouped execution of the
// device programs (kad_group.hip), so both give the same bits.
//
// One thread per line and part of its outputs: the line goes to registers once, the
// outputs are a small dense matrix times the line.  Bound by the vector unit once warm
// (about 8 cycles per matrix entry and wave).  The matrix row of an output sits in the
// lanes of each 16-lane row of the wave (one LDS read per output) and its entries reach the
// multiply-adds by DPP row broadcasts; entries past 16 are broadcast LDS reads.  With the
// entries read by scalar loads every output waited for the scalar cache: 4096 transforms
// there and back took 247 us at 17x13x12 and 390 at 18x13x12, now 217 and 226.  Chains of
// small arrays take a thread per output.
#pragma once
#include "kad_lanes.hpp"
#include "kad_spectral.hpp"

namespace kad {

// The outputs [o0, o1) of one line per lane (ni <= NIN points from x + q sin to y + o sout;
// the entries past ni count as zeros).  Waves whose lines use different matrices are served
// one matrix at a time.  one (the output may lie over the input): every thread passes the
// barrier between its reads and its writes.
template <int NIN>
__device__ __forceinline__ void pass_lines(const double* x, double* y, const double* mats, const LineEnt en, bool act,
                                           int ni, int sin, int sout, int o0, int o1, bool one) {
  double xv[NIN];
#pragma unroll
  for (int q = 0; q < NIN; ++q) xv[q] = q < ni ? x[en.xb + q * sin] : 0.0;  // (lanes without a line read line 0)
  if (one) __syncthreads();
  const int l16 = threadIdx.x & 15;
  bool todo = act;
  while (true) {
    const unsigned long long pend = __ballot(todo);
    if (pend == 0) break;
    const int off = __builtin_amdgcn_readlane(en.off, __ffsll((long long)pend) - 1);
    const bool mine = todo && en.off == off;
    todo = todo && !mine;
    double* yl = y + en.yb + o0 * sout;
    if (off < 0) {  // a line without a matrix is zero
      if (mine)
        for (int o = o0; o < o1; ++o, yl += sout) *yl = 0.0;
      continue;
    }
    const double* M = mats + off + o0 * ni;
    double m = l16 < ni ? M[l16] : 0.0;
#pragma unroll 1
    for (int o = o0; o < o1; ++o, yl += sout) {
      const double mc = m;
      double tail[NIN > 16 ? NIN - 16 : 1];
#pragma unroll
      for (int q = 16; q < NIN; ++q) tail[q - 16] = q < ni ? M[q] : 0.0;
      M += ni;
      if (o + 1 < o1) m = l16 < ni ? M[l16] : 0.0;  // the next output's row, ahead of its use
      double s0 = 0.0, s1 = 0.0;
      static_for<NIN>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        double c;
        if constexpr (q < 16) c = lane16<q>(mc);
        else c = tail[q - 16];
        if constexpr (q % 2 == 0) s0 += c * xv[q];
        else s1 += c * xv[q];
        if constexpr (q % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // four broadcasts in registers, not all
      });
      double r = s0 + s1;
      asm volatile("" : "+v"(r));  // computed by every lane: kept out of the store's branch, with its broadcasts
      if (mine) *yl = r;
    }
  }
}

// One output: a matrix row times a line, both in LDS.
__device__ __forceinline__ double line_dot(const double* M, const double* x, int ni, int sin) {
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  int q = 0;
  for (; q + 4 <= ni; q += 4) {
    s0 += M[q] * x[q * sin];
    s1 += M[q + 1] * x[(q + 1) * sin];
    s2 += M[q + 2] * x[(q + 2) * sin];
    s3 += M[q + 3] * x[(q + 3) * sin];
  }
  for (; q < ni; ++q) s0 += M[q] * x[q * sin];
  return (s0 + s1) + (s2 + s3);
}

// One workgroup (256 threads) takes the array src (batch element b of the chain post) to
// dst.  lds: one buffer (two when a pass has more lines than threads), then the matrix
// pool.  PP: LinePlan, as a kernel argument or in the constant address space (read with
// scalar loads either way).
template <typename PP>
__device__ __forceinline__ void apply3d_body(const double* __restrict__ src, double* __restrict__ dst, const PP& P,
                                             const PostOp& post, int64_t b, double* lds) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nin = P.size_in, npass = P.npass, npool = P.pool_size, maxsize = P.maxsize;
  const bool single = P.single != 0;
  const double* const pool = P.pool;
  double* const buf0 = lds;
  double* const buf1 = single ? lds : lds + maxsize;
  double* const mats = lds + (single ? 1 : 2) * maxsize;
  // A wave takes 64 lines and a part of their outputs at a time (a unit).  One or two groups
  // of 64 lines share the four waves evenly; other remainders do so by halves or quarters
  // where lines may be read twice, with two buffers (17x13x16, 5 groups: 216 us for 3072
  // transforms there and back, 276 in whole lines).
  auto split = [&](int nlines, int& groups, int& sh) {  // 1 << sh parts
    groups = (nlines + 63) >> 6;
    sh = groups == 1 ? 2 : (groups == 2 ? 1 : (single || (groups & 3) == 0 ? 0 : (groups == 3 ? 2 : 1)));
  };
  auto entry = [&](int p, int slot) -> LineEnt {
    LineEnt e{0, 0, -1, 0};
    if (slot < P.p[p].nlines) e = P.p[p].tab[slot];
    return e;
  };
  int groups, sh;
  split(P.p[0].nlines, groups, sh);
  LineEnt en = entry(0, (wave >> sh) * 64 + lane);
  // the array and the matrices, 8 loads in flight per thread (one load per iteration
  // would wait out the memory latency ~10 times per array)
  constexpr int UL = 8;
  for (int e0 = 0; e0 < nin; e0 += UL * 256) {
    double v[UL];
#pragma unroll
    for (int u = 0; u < UL; ++u) {
      const int e = e0 + u * 256 + tid;
      v[u] = e < nin ? src[e] : 0.0;
    }
    double mv[2] = {0.0, 0.0};
    if (e0 == 0) {
#pragma unroll
      for (int u = 0; u < 2; ++u) mv[u] = u * 256 + tid < npool ? pool[u * 256 + tid] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < UL; ++u) {
      const int e = e0 + u * 256 + tid;
      if (e < nin) buf0[e] = v[u];
    }
    if (e0 == 0) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if (u * 256 + tid < npool) mats[u * 256 + tid] = mv[u];
    }
  }
  for (int e = 512 + tid; e < npool; e += 256) mats[e] = pool[e];
  __syncthreads();
  int cur = 0;
  if (P.small) {
    // up to 768 outputs per pass: three per thread, straight from LDS (a Jacobian at 9x7x4
    // takes 2.45 ms, 2.96 with a thread per line); the next pass's places are loaded ahead
    constexpr int US = kSmallArray / 256;
    LineEnt a[US];
    int oo[US];
    auto places = [&](int p) {
      const int no = P.p[p].nout, n = P.p[p].nlines * no;
#pragma unroll
      for (int u = 0; u < US; ++u) {
        const int e = u * 256 + tid;
        a[u].xb = -1;
        oo[u] = 0;
        if (e < n) {
          const int l = e / no;
          a[u] = P.p[p].tab[l];
          oo[u] = e - l * no;
        }
      }
    };
    places(0);
    for (int p = 0; p < npass; ++p) {
      const int ni = P.p[p].nin, sin = P.p[p].sin, sout = P.p[p].sout;
      const double* const x = cur ? buf1 : buf0;
      double* const y = cur ? buf0 : buf1;
      LineEnt c[US];
      int o[US];
#pragma unroll
      for (int u = 0; u < US; ++u) {
        c[u] = a[u];
        o[u] = oo[u];
      }
      if (p + 1 < npass) places(p + 1);
#pragma unroll
      for (int u = 0; u < US; ++u) {
        if (c[u].xb < 0) continue;
        y[c[u].yb + o[u] * sout] = c[u].off < 0 ? 0.0 : line_dot(mats + c[u].off + o[u] * ni, x + c[u].xb, ni, sin);
      }
      __syncthreads();
      cur ^= 1;
    }
  } else
  for (int p = 0; p < npass; ++p) {
    const int nlines = P.p[p].nlines, no = P.p[p].nout, sin = P.p[p].sin, sout = P.p[p].sout;
    const int ni = __builtin_amdgcn_readfirstlane(P.p[p].nin);
    const double* const x = cur ? buf1 : buf0;
    double* const y = single ? buf0 : (cur ? buf0 : buf1);
    const int per = (no + (1 << sh) - 1) >> sh;
    // the thread's line is all that is overwritten by it, or every line is read first
    const bool barrier = single && groups <= 4;
    LineEnt next{0, 0, -1, 0};
    int ngroups = 0, nsh = 0;
    if (p + 1 < npass) {
      split(P.p[p + 1].nlines, ngroups, nsh);
      next = entry(p + 1, (wave >> nsh) * 64 + lane);  // ahead of its use
    }
    if (ni <= kLineTemplates) {
      const int units = barrier ? 4 : groups << sh;
      for (int u = wave; u < units; u += 4) {
        const int slot = (u >> sh) * 64 + lane, o0 = min(no, (u & ((1 << sh) - 1)) * per), o1 = min(no, o0 + per);
        if (u >= 4) en = entry(p, slot);
        const bool act = slot < nlines;
        // five lengths: one per length would be 17 pieces of code, each met cold.  Without the
        // one of 16, 2349 transforms to coefficients at 17x17x16 took 293 us, now 273, and 4096
        // there and back at 15x13x12 206, now 201; it is laid out of the others' way (553 us per
        // residual at 17x13x12, which does not meet it, with it among them, 543 so, 549
        // without it).
        if (ni <= 10) {
          if (ni <= 6) pass_lines<6>(x, y, mats, en, act, ni, sin, sout, o0, o1, barrier);
          else pass_lines<10>(x, y, mats, en, act, ni, sin, sout, o0, o1, barrier);
        } else {
          if (ni <= 14) pass_lines<14>(x, y, mats, en, act, ni, sin, sout, o0, o1, barrier);
          else if (__builtin_expect(ni == 15 || ni == 16, 0))
            pass_lines<16>(x, y, mats, en, act, ni, sin, sout, o0, o1, barrier);
          else pass_lines<18>(x, y, mats, en, act, ni, sin, sout, o0, o1, barrier);
        }
      }
    } else {
      // longer lines: an output per thread, straight from LDS; the next one's place is
      // loaded ahead (without, 3315 transforms there and back at 21x13x12 took 403 us, now 392)
      const int n = nlines * no;
      auto place = [&](int e, LineEnt& l, int& o) {
        const int q = e / no;
        o = e - q * no;
        if (e < n) l = P.p[p].tab[q];
      };
      LineEnt l{0, 0, -1, 0};
      int o = 0;
      place(tid, l, o);
      for (int e = tid; e < n; e += 256) {
        LineEnt ln{0, 0, -1, 0};
        int on = 0;
        place(e + 256, ln, on);
        y[l.yb + o * sout] = l.off < 0 ? 0.0 : line_dot(mats + l.off + o * ni, x + l.xb, ni, sin);
        l = ln;
        o = on;
      }
    }
    __syncthreads();
    cur ^= 1;
    en = next;
    groups = ngroups;
    sh = nsh;
  }
  const int nfin = P.size_out;
  const double* const fin = cur ? buf1 : buf0;
  if (post.n > 0) {
    // the element-wise instructions fed by this pass; the other operands of UP elements
    // per thread are loaded together, as the inputs were
    constexpr int UP = 4;
    double* drow = post.dst + b * post.ds;
    for (int e0 = 0; e0 < nfin; e0 += UP * 256) {
      double o[UP][kMaxChain];
#pragma unroll
      for (int u = 0; u < UP; ++u) {
        const int e = e0 + u * 256 + tid;
        post_load(post, b, e < nfin ? e : 0, o[u]);
      }
#pragma unroll
      for (int u = 0; u < UP; ++u) {
        const int e = e0 + u * 256 + tid;
        if (e < nfin) drow[e] = post_ops(post, fin[e], o[u]);
      }
    }
  } else {
    for (int e = tid; e < nfin; e += 256) dst[e] = fin[e];
  }
}

}  // namespace kad
