// mgpcg.h -- multigrid-preconditioned CG for the pressure system (mgpcg.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "aqflip_internal.h"

namespace aqf {

constexpr int kMgMaxLevels = 12;  // 1,024 cells along an axis take 9

// One grid level: cells in hash order (x-major, z fastest). code[n] = 0 on cells that are
// no unknowns; else kMgFluid and one wall bit per axis end the cell touches (+x, -x, +y,
// -y, +z, -z). f: right-hand side, u: correction, t: ping-pong / residual, all FP32; u
// and t hold 0 on every non-FLUID cell throughout a solve. Every array has a guard of
// mg_guard(level) elements on both sides, so a neighbour's offset is always in range.
constexpr uint8_t kMgFluid = 0x40;
struct MgLevel {
  int X, Y, Z, n;
  FastDiv divZ, divYZ;
  uint8_t* code;
  float *f, *u, *t;
};
inline int mg_guard(const MgLevel& L) { return (L.Y * L.Z + 4 + 7) / 8 * 8; }

struct MgLevels {
  int count;  // levels; the last is solved by kMgCoarseSweeps sweeps
  int tail;   // first level of the one-workgroup kernel
  MgLevel L[kMgMaxLevels];
};

// Scalars of a solve, on the device.
struct MgScalars {
  double rz, bb, alpha, beta, res, tol;
  int it, max_iters, check_every;
  int stop;  // the residual is at or below tol, or not finite, at a checked iteration
};
// What the host polls (pinned memory), written at every checked iteration: seq last.
struct MgReport {
  double res;
  int stop, seq;
};

// FP64 vectors of the solve (guarded like level 0's arrays) and its scratch.
struct MgVectors {
  double *x, *r, *q, *d[2];
  double* part;  // per-block partial sums
  MgScalars* S;
  MgReport* report;  // device address of the pinned report
};

// Level `l` of a hierarchy over a grid of extents X, Y, Z (arrays not set).
MgLevel mg_level(int X, int Y, int Z);
// First level the one-workgroup kernel takes.
int mg_tail_level(const MgLevels& H);
// Doubles of MgVectors::part.
size_t mg_part_size(const MgLevels& H);

// Starts a solve: levels' codes, x and r = b - A x from the FLIP grid (p: the start, or
// null for zero), scalars from tol / max_iters / check_every, then the first V-cycle.
void mg_start(const Geom& G, const MgLevels& H, const MgVectors& V, const uint8_t* content, const float* rhs,
              const float* p, double tol, int max_iters, int check_every, hipStream_t s);
// One CG iteration; `odd`: the parity of its number (0 first).
void mg_iterate(const MgLevels& H, const MgVectors& V, int odd, hipStream_t s);
// p = FP32(x), 0 on non-FLUID cells.
void mg_finish(const Geom& G, const MgLevels& H, const MgVectors& V, float* p, hipStream_t s);

}  // namespace aqf
