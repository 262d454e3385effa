// Grouped execution of the device programs: every instruction of one dependency level,
// of one or several programs, in one launch (kad_group.hip).
#pragma once
#include "kad_spectral.hpp"

namespace kad {

struct DevRow {
  int pos, gpos;
  double gw;
};

enum : int { GK_LIN = 0, GK_EW = 1, GK_EXPORT_IN = 2, GK_EXPORT_BD = 3, GK_EXPORT_GL = 4, GK_SEED = 5, GK_CLUSTER = 6 };

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

// One element-wise instruction of a cluster, in execution order.  Operand a / b: a
// temporary (>= 0), none (-1), or an array (-2: ga / gb), kept in temporary ca / cb when
// that is >= 0.  The result goes to temporary d (>= 0) and to array gd (slot >= 0).
// In the device table ca, cb and d are kClusterTemps where there is none.
constexpr int kClusterTemps = 7;
constexpr int kClusterChunk = 256;  // elements of a wave
struct ClusterStep {
  int kind = 0, a = -1, b = -1, ca = -1, cb = -1, d = -1;
  GroupOpnd ga, gb, gd;
  double s = 0.0;
};

// One instruction (with the element-wise instructions it absorbed, as PostOp): the
// workgroup of (instruction, column) does all of it.
struct GroupOp {
  int kind = 0, nstep = 0;
  int ew = 0, size = 0;                 // EW: kind, elements; SEED: elements
  GroupOpnd dst, a, b;
  double s = 0.0;                       // EW scalar; EXPORT_GL: factor
  GroupStep st[kMaxChain];
  int step0 = 0, nsteps = 0;            // CLUSTER: its steps in the step table
  LinePlan P;                           // LIN
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
  int nops, op0, nb, nbp, u0, nch;
  int64_t base, col0;
};
constexpr int kGroupEntries = 32;
struct GroupArgs {
  const GroupOp* ops = nullptr;
  const ClusterStep* steps = nullptr;
  double* val = nullptr;
  double* tan = nullptr;
  int64_t stride = 0;
  void* out = nullptr;      // rows x columns (ldo), fp64 (dtype 0) or fp32 (dtype 1)
  int64_t ldo = 0;
  const double* w = nullptr;  // transposed exports: out[column] += w . exported rows
  int dtype = 0;
  int nent = 0;
  int blk0[kGroupEntries];  // first workgroup of each entry
  GroupEntry e[kGroupEntries];
};

// clusters: every instruction of the launch is a CLUSTER, otherwise none is
int group_launch(const GroupArgs& g, int blocks, bool clusters, size_t lds, hipStream_t s);

}  // namespace kad
