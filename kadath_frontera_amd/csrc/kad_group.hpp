// Grouped execution of the device programs: every instruction of one dependency level,
// of one or several programs, in one launch (kad_group.hip).
#pragma once
#include "kad_spectral.hpp"

namespace kad {

struct DevRow {
  int pos, gpos;
  double gw;
};

enum : int { GK_LIN = 0, GK_EW = 1, GK_EXPORT_IN = 2, GK_EXPORT_BD = 3, GK_EXPORT_GL = 4, GK_SEED = 5 };

// An operand: a slot of the value arena (tan = 0) or of the program's region of the
// tangent arena (tan = 1); slot < 0: none.
struct GroupOpnd {
  int slot = -1, tan = 0;
};
struct GroupStep {
  int kind = 0, side = 0;
  GroupOpnd o;
  double s = 0.0;
};

// One instruction (with the element-wise instructions it absorbed, as PostOp): the
// workgroup of (instruction, column) does all of it.
struct GroupOp {
  int kind = 0, nstep = 0;
  int d0 = 0, d1 = 0, d2 = 0;           // LIN: input dimensions
  int stage_pool = 0, inplace = 0;      // LIN: Apply3dShape
  int ew = 0, size = 0;                 // EW: kind, elements; SEED: elements
  GroupOpnd dst, a, b;
  double s = 0.0;                       // EW scalar; EXPORT_GL: factor
  GroupStep st[kMaxChain];
  Passes P;                             // LIN
  const double* pool = nullptr;
  // exports
  const DevRow* rows = nullptr;
  int nrows = 0, row0 = 0, accumulate = 0, bsign = 1;
  int nr = 0, nt = 0, aux = 0, pt = 0;
  double sign = 1.0, c0 = 0.0;
  // seeds
  const int* spos = nullptr;
  const double* sval = nullptr;
  const int* scnt = nullptr;
  int nu = 0;
};

// The columns [u0, u0 + nb) of one program in a launch: its instructions ops[op0 ..
// op0 + nops) of the level, workgroups blk0 .. blk0 + nops nbp - 1 (instruction-major,
// nbp >= nb columns each), tangent slot s of column b at base + (s nb + b) stride,
// results in column col0 + b.
struct GroupEntry {
  int blk0, nops, op0, nb, nbp, u0;
  int64_t base, col0;
};
constexpr int kGroupEntries = 32;
struct GroupArgs {
  const GroupOp* ops = nullptr;
  double* val = nullptr;
  double* tan = nullptr;
  int64_t stride = 0;
  void* out = nullptr;      // rows x columns (ldo), fp64 (dtype 0) or fp32 (dtype 1)
  int64_t ldo = 0;
  const double* w = nullptr;  // transposed exports: out[column] += w . exported rows
  int dtype = 0;
  int nent = 0;
  GroupEntry e[kGroupEntries];
};

int group_launch(const GroupArgs& g, int blocks, size_t lds, hipStream_t s);

}  // namespace kad
