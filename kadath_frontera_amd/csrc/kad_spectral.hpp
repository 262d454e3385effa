// Launch interface of the batched 1-D / 3-D spectral kernels.
#pragma once
#include "kad_common.hpp"
#include "kad_ew.hpp"

namespace kad {

constexpr int MAX_PASSES = 6;
constexpr int kSmallArray = 768;   // a thread per output up to here, per line above
constexpr int kLineTemplates = 18;  // longest line kept in registers

// A chain of 1-D passes over a 3-D array.  Pass p acts along axis[p] and maps
// that axis to nout[p] entries; line_mat[p] (HOST) gives, per line, the offset
// of a row-major nout x nin matrix in the pool (or -1: the line is zero).  Lines
// are numbered like the reference's per-dimension basis tables
// (src/Base_spectral/base_spectral.cpp:92-104): axis 0 by (j + d1*k), axis 1 by k,
// axis 2 by 0.
struct PassDesc {
  int axis = 0, nout = 0;
  const int* line_mat = nullptr;
};

// One line of a pass: where it starts in the pass's input and output arrays, its matrix.
struct LineEnt {
  int xb, yb, off, pad;
};

// The chain laid out for the kernels (lines_build): every pass's lines, those with one
// matrix together, with their places computed once.
struct LinePlan {
  struct Pass {
    int nlines = 0, nin = 0, nout = 0, sin = 0, sout = 0;  // lines, points in / out, strides of a line
    int pad = 0;
    const LineEnt* tab = nullptr;  // device
  };
  int npass = 0;
  int size_in = 0, size_out = 0;
  int maxsize = 0;    // largest intermediate array (doubles)
  int pool_size = 0;  // doubles of the matrix pool (staged in LDS)
  int single = 0;     // 1: one LDS buffer serves (every pass has at most 256 lines or keeps their length)
  int small = 0;      // 1: every pass has at most kSmallArray outputs: a thread per output
  const double* pool = nullptr;  // device
  Pass p[MAX_PASSES];
};

constexpr size_t kMaxLds = 160 * 1024;  // of a workgroup

// LDS bytes of a chain (kad_apply3d.hpp).
inline size_t lines_lds(const LinePlan& P) {
  return ((P.single ? 1 : 2) * (size_t)P.maxsize + (size_t)P.pool_size) * sizeof(double);
}

// The line tables of a chain over a d0 x d1 x d2 array, one after another in tab (HOST); the
// caller uploads them and sets every pass's tab to its part (toff) and the pool.  False:
// no pass or more than MAX_PASSES, or more than cap lines.  (A chain that needs more LDS than
// a workgroup has is laid out; its launches are refused.)
bool lines_build(int d0, int d1, int d2, const PassDesc* passes, int npass, int pool_size, LinePlan& P,
                 LineEnt* tab, size_t cap, size_t* used, size_t* toff);

// post (may be NULL): element-wise instructions applied in the store phase; out is then
// not written
int apply3d_launch(const double* in, int64_t in_stride, double* out, int64_t out_stride, int nbatch, const LinePlan& P,
                   hipStream_t s, const PostOp* post = nullptr);
int apply_lines_launch(const double* in, double* out, int64_t L, int nin, int nout, const double* M, hipStream_t s);

}  // namespace kad
