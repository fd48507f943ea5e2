// mgpcg.hip -- multigrid-preconditioned conjugate gradients for the pressure system.
//
// The accuracy reference and second fallback beside Jacobi. It solves the same
// system as jacobiImpl's fixed point (Fluid/Fluid_3D_kernels.cu:460-505) -- the
// operator of the FP64 residual, (A p)_i = (6 - walls_i) p_i - sum of FLUID
// neighbours, AIR cells Dirichlet 0 -- which is the matrix the reference's legacy
// sparse path assembles (Fluid/Legacy/PressureEquation.cuh:216-328) and solves with
// AMGX-preconditioned CG (Fluid/Legacy/SPD_Solver.h:102-160). Here it is matrix-free:
// CG in FP64 on dense vectors in hash order, preconditioned by one geometric V-cycle
// in FP32 (levels halve every axis; a coarse cell is FLUID when any child is; damped
// Jacobi, omega 2/3, two sweeps before and after; cell-centred trilinear prolongation
// and its exact transpose as restriction, scaled by 1/2 for the coarser operator; a
// fixed number of sweeps on the coarsest level). Every piece is a fixed linear map
// and pre/post smoothing match, so the preconditioner is symmetric positive definite
// as CG requires.
//
// One CG iteration is 16 launches at 128^3, most of them a few microseconds:
//   * a cell's byte code holds "FLUID" and its wall bits, and every vector that is read
//     at a neighbour holds 0 on non-FLUID cells, so a stencil is the cell's code and
//     seven values at fixed linear offsets: no coordinates, no neighbour flags. In the CG
//     passes a thread owns four consecutive cells on large levels (16-byte loads) and
//     returns after reading their codes when none is FLUID.
//   * vector updates ride on passes that read the vectors anyway: d = z + beta d inside
//     the operator's pass (recomputed at the neighbours, d ping-ponged), x, r, the FP32
//     copy of r and the first smoothing sweep (from zero) in one pass, r.z in the last
//     smoothing sweep.
//   * a level below kVecCells takes one launch down (sweep, residual, restriction, the
//     coarse level's first sweep) and one up (prolongation, two sweeps), on LDS tiles with
//     recomputed margins.
//   * all levels of at most kTailCells cells run in one workgroup, in LDS (launches on 64
//     to 4,096 cells were 60 of the cycle's 75).
//   * scalars stay on the device. r.r, and with it whether to stop, is known before an
//     iteration's V-cycle starts and is written to pinned memory there, so the host
//     queues the next iteration while the V-cycle runs.
// 128^3 system of 0.59 M unknowns to 1e-5, 12 iterations, with the read-back of the
// pressure (0.8 ms): 7.9 -> 2.5 ms. Before, every operator, sweep, transfer and update was a
// launch of its own (some 75 per cycle) with a thread per cell, a host synchronisation per
// iteration and single-thread folds of 26 us.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "aqflip_internal.h"
#include "mgpcg.h"

#pragma clang fp contract(off)

namespace aqf {

constexpr int kMgBlock = 256;
constexpr int kMgCoarseSweeps = 40;  // sweeps on the coarsest level
constexpr int kTailCells = 4096;     // largest level of the one-workgroup kernel
constexpr int kTailLds = 6144;        // cells of all its levels together
constexpr int kTailThreads = 1024;
constexpr int kVecCells = 1 << 19;   // levels this large take four cells per thread

typedef float f32x4a __attribute__((ext_vector_type(4), aligned(4)));
typedef double f64x4a __attribute__((ext_vector_type(4), aligned(8)));

__device__ __forceinline__ int mg_block() {  // neighbouring cells in one XCD's L2
  const int nb = gridDim.x, bid = blockIdx.x;
  const int per = nb / 8, rem = nb % 8, xcd = bid % 8;
  return xcd * per + min(xcd, rem) + bid / 8;
}

// V consecutive values.
template <int V, typename T>
struct Vals {
  T v[V];
};
template <int V>
__device__ __forceinline__ Vals<V, float> ld(const float* p) {
  Vals<V, float> o;
  if constexpr (V == 4) {
    const f32x4a t = *(const f32x4a*)p;
#pragma unroll
    for (int i = 0; i < 4; ++i) o.v[i] = t[i];
  } else {
    o.v[0] = *p;
  }
  return o;
}
template <int V>
__device__ __forceinline__ Vals<V, double> ld(const double* p) {
  Vals<V, double> o;
  if constexpr (V == 4) {
    const f64x4a t = *(const f64x4a*)p;
#pragma unroll
    for (int i = 0; i < 4; ++i) o.v[i] = t[i];
  } else {
    o.v[0] = *p;
  }
  return o;
}
template <int V>
__device__ __forceinline__ void st(float* p, const Vals<V, float>& v) {
  if constexpr (V == 4)
    *(f32x4a*)p = f32x4a{v.v[0], v.v[1], v.v[2], v.v[3]};
  else
    *p = v.v[0];
}
template <int V>
__device__ __forceinline__ void st(double* p, const Vals<V, double>& v) {
  if constexpr (V == 4)
    *(f64x4a*)p = f64x4a{v.v[0], v.v[1], v.v[2], v.v[3]};
  else
    *p = v.v[0];
}
// The codes of V consecutive cells from n (n a multiple of V), cell i in byte i.
template <int V>
__device__ __forceinline__ uint32_t ld_codes(const uint8_t* code, int n) {
  if constexpr (V == 4)
    return *(const uint32_t*)(code + n);
  else
    return code[n];
}
__device__ __forceinline__ uint32_t code_of(uint32_t codes, int i) { return (codes >> (8 * i)) & 0xff; }
template <int V>
__device__ __forceinline__ bool any_fluid(uint32_t codes) {
  return (codes & (V == 4 ? 0x40404040u : 0x40u)) != 0;
}

// Values at the six neighbours and the centre of V consecutive cells.
template <int V, typename T>
struct Star {
  Vals<V, T> c, xp, xm, yp, ym;
  T zm, zp;
  __device__ __forceinline__ T zprev(int i) const { return i == 0 ? zm : c.v[i > 0 ? i - 1 : 0]; }
  __device__ __forceinline__ T znext(int i) const { return i == V - 1 ? zp : c.v[i < V - 1 ? i + 1 : i]; }
};
template <int V, typename T>
__device__ __forceinline__ Star<V, T> ld_star(const T* u, int n, int sy, int sx) {
  Star<V, T> s;
  s.c = ld<V>(u + n);
  s.xp = ld<V>(u + n + sx);
  s.xm = ld<V>(u + n - sx);
  s.yp = ld<V>(u + n + sy);
  s.ym = ld<V>(u + n - sy);
  s.zm = u[n - 1];
  s.zp = u[n + V];
  return s;
}
// (A u) at a cell (unit spacing): walls are clamp-to-edge (Neumann), non-FLUID neighbours
// are Dirichlet 0.
template <typename T>
__device__ __forceinline__ T stencil(uint32_t code, T uc, T xp, T xm, T yp, T ym, T zp, T zm) {
  T a = (T)6 * uc;
  a -= code & 1 ? uc : xp;
  a -= code & 2 ? uc : xm;
  a -= code & 4 ? uc : yp;
  a -= code & 8 ? uc : ym;
  a -= code & 16 ? uc : zp;
  a -= code & 32 ? uc : zm;
  return a;
}
template <int V, typename T>
__device__ __forceinline__ T apply_at(uint32_t code, const Star<V, T>& s, int i) {
  return stencil<T>(code, s.c.v[i], s.xp.v[i], s.xm.v[i], s.yp.v[i], s.ym.v[i], s.znext(i), s.zprev(i));
}
__device__ __forceinline__ float diag_of(uint32_t code) { return (float)(6 - __popc(code & 63u)); }
constexpr float kOmega = 2.f / 3.f;
// The first damped Jacobi sweep (from zero) at a cell, 0 on non-FLUID cells.
__device__ __forceinline__ float smooth0(uint32_t code, float f) {
  return code & kMgFluid ? kOmega * f / diag_of(code) : 0.f;
}

__device__ __forceinline__ void cell_xyz(const MgLevel& L, int n, int& x, int& y, int& z) {
  x = (int)fast_div((uint32_t)n, L.divYZ);
  const int r = n - x * (L.Y * L.Z);
  y = (int)fast_div((uint32_t)r, L.divZ);
  z = r - y * L.Z;
}
__device__ __forceinline__ uint8_t make_code(const MgLevel& L, int x, int y, int z) {
  return (uint8_t)(kMgFluid | (x + 1 >= L.X ? 1 : 0) | (x <= 0 ? 2 : 0) | (y + 1 >= L.Y ? 4 : 0) | (y <= 0 ? 8 : 0) |
                   (z + 1 >= L.Z ? 16 : 0) | (z <= 0 ? 32 : 0));
}

// Sum over the block, in a fixed order; the result is returned to thread 0.
template <int N>
__device__ __forceinline__ double block_sum(double v) {
  __shared__ double w[N / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0;
#pragma unroll
  for (int i = 0; i < N / 64; ++i) s += w[i];
  return s;
}

// ---- start of a solve
// Level 0 from the FLIP grid: code, x (the start p, or 0) and r = b; u, t and both search
// directions cleared; partial sums of b.b. The FP64 vectors are also cleared in the guard
// cells that the last thread of a pass updates with its own (0 times a scalar, but a solve
// that overflowed multiplied by an infinity there).
__global__ void k_mg_gather(Geom G, const uint8_t* __restrict__ content, const float* __restrict__ rhs,
                            const float* __restrict__ p, MgLevel L, MgVectors V) {
  const int n = mg_block() * kMgBlock + (int)threadIdx.x;
  double bb = 0;
  if (n < L.n) {
    int i, j, k;
    cell_xyz(L, n, i, j, k);
    const long long g = G.g(i, j, k);
    const bool fl = content[g] == FLUID;
    const double b = fl ? (double)rhs[g] : 0.0;
    L.code[n] = fl ? make_code(L, i, j, k) : 0;
    V.x[n] = fl && p ? (double)p[g] : 0.0;
    V.r[n] = b;
    V.d[0][n] = 0.0;
    V.d[1][n] = 0.0;
    L.u[n] = 0.f;
    L.t[n] = 0.f;
    bb = b * b;
  } else if (n < (L.n + 3) / 4 * 4) {
    V.x[n] = 0.0;
    V.r[n] = 0.0;
    V.d[0][n] = 0.0;
    V.d[1][n] = 0.0;
  }
  bb = block_sum<kMgBlock>(bb);
  if (threadIdx.x == 0) V.part[blockIdx.x] = bb;
}
// A coarse cell is FLUID when any child is; u and t cleared.
__global__ void k_mg_coarsen(MgLevel F, MgLevel C) {
  const int n = mg_block() * kMgBlock + (int)threadIdx.x;
  if (n >= C.n) return;
  int x, y, z;
  cell_xyz(C, n, x, y, z);
  uint32_t any = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int fx = min(2 * x + (k >> 2), F.X - 1), fy = min(2 * y + ((k >> 1) & 1), F.Y - 1),
              fz = min(2 * z + (k & 1), F.Z - 1);  // a missing child repeats its sibling
    any |= F.code[(fx * F.Y + fy) * F.Z + fz];
  }
  C.code[n] = any & kMgFluid ? make_code(C, x, y, z) : 0;
  C.u[n] = 0.f;
  C.t[n] = 0.f;
}

// r (given b - 0, or computed as b - A x), its FP32 copy f, the first smoothing sweep
// t = omega f / diag, and partial sums of r.r.
template <int V>
__global__ void k_mg_residual0(MgLevel L, MgVectors W, int use_x) {
  const int n = (mg_block() * kMgBlock + (int)threadIdx.x) * V;
  double rr = 0;
  if (n < L.n) {
    const uint32_t codes = ld_codes<V>(L.code, n);
    if (any_fluid<V>(codes)) {
      Vals<V, double> r = ld<V>(W.r + n);
      if (use_x) {
        const Star<V, double> s = ld_star<V>(W.x, n, L.Z, L.Y * L.Z);
#pragma unroll
        for (int i = 0; i < V; ++i)
          if (code_of(codes, i) & kMgFluid) r.v[i] = r.v[i] - apply_at(code_of(codes, i), s, i);
      }
      Vals<V, float> f, t;
#pragma unroll
      for (int i = 0; i < V; ++i) {  // r is 0 on non-FLUID cells
        f.v[i] = (float)r.v[i];
        t.v[i] = smooth0(code_of(codes, i), f.v[i]);
        rr += r.v[i] * r.v[i];
      }
      if (use_x) st<V>(W.r + n, r);
      st<V>(L.f + n, f);
      st<V>(L.t + n, t);
    }
  }
  rr = block_sum<kMgBlock>(rr);
  if (threadIdx.x == 0) W.part[blockIdx.x] = rr;
}

// ---- scalars: partial sums folded in a fixed order by one block
__device__ double fold(const double* __restrict__ part, int n) {
  double v = 0;
  for (int i = threadIdx.x; i < n; i += kTailThreads) v += part[i];
  return block_sum<kTailThreads>(v);
}
__device__ void mg_report(MgScalars* S, MgReport* report, double rr) {
  S->res = S->bb > 0 ? sqrt(rr / S->bb) : sqrt(rr);
  S->stop = !(S->res > S->tol) || isinf(S->res);  // at tol, or not finite
  report->res = S->res;
  report->stop = S->stop;
  __hip_atomic_store(&report->seq, S->it + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
__global__ __launch_bounds__(kTailThreads) void k_mg_fold_start(const double* part, int n, MgScalars* S, double tol,
                                                               int max_iters, int check_every) {
  const double bb = fold(part, n);
  if (threadIdx.x == 0) *S = MgScalars{0, bb, 0, 0, 0, tol, 0, max_iters, check_every, 0};
}
// r.r: the residual, and at a checked iteration whether to stop, for the host and for the
// V-cycle that follows (level 0 does nothing once stopped). first: before any iteration.
__global__ __launch_bounds__(kTailThreads) void k_mg_fold_rr(const double* part, int n, MgScalars* S, MgReport* report,
                                                            int first) {
  const double rr = fold(part, n);
  if (threadIdx.x != 0) return;
  if (!first) S->it += 1;
  if (first || S->it % S->check_every == 0 || S->it == S->max_iters) mg_report(S, report, rr);
}
// d.q: alpha = r.z / d.q
__global__ __launch_bounds__(kTailThreads) void k_mg_fold_dq(const double* part, int n, MgScalars* S) {
  const double dq = fold(part, n);
  if (threadIdx.x == 0) S->alpha = dq != 0.0 ? S->rz / dq : 0.0;
}
// r.z: beta = new r.z / old r.z (0 before the first iteration)
__global__ __launch_bounds__(kTailThreads) void k_mg_fold_rz(const double* part, int n, MgScalars* S) {
  const double rz = fold(part, n);
  if (threadIdx.x != 0) return;
  S->beta = S->rz != 0.0 ? rz / S->rz : 0.0;
  S->rz = rz;
}

// ---- CG passes (FP64)
// d' = z + beta d (z: the V-cycle's correction), q = A d', partial sums of d'.q.
template <int V>
__global__ void k_cg_apply(MgLevel L, MgVectors W, const float* __restrict__ zc, int odd) {
  const int n = (mg_block() * kMgBlock + (int)threadIdx.x) * V;
  double dq = 0;
  if (n < L.n) {
    const uint32_t codes = ld_codes<V>(L.code, n);
    if (any_fluid<V>(codes)) {
      const double beta = W.S->beta;
      const Star<V, double> d = ld_star<V>((const double*)W.d[odd], n, L.Z, L.Y * L.Z);
      const Star<V, float> z = ld_star<V>(zc, n, L.Z, L.Y * L.Z);
      Star<V, double> e;
#pragma unroll
      for (int i = 0; i < V; ++i) {
        e.c.v[i] = (double)z.c.v[i] + beta * d.c.v[i];
        e.xp.v[i] = (double)z.xp.v[i] + beta * d.xp.v[i];
        e.xm.v[i] = (double)z.xm.v[i] + beta * d.xm.v[i];
        e.yp.v[i] = (double)z.yp.v[i] + beta * d.yp.v[i];
        e.ym.v[i] = (double)z.ym.v[i] + beta * d.ym.v[i];
      }
      e.zm = (double)z.zm + beta * d.zm;
      e.zp = (double)z.zp + beta * d.zp;
      Vals<V, double> q;
#pragma unroll
      for (int i = 0; i < V; ++i) {  // d is 0 on non-FLUID cells
        const uint32_t c = code_of(codes, i);
        q.v[i] = c & kMgFluid ? apply_at(c, e, i) : 0.0;
        dq += e.c.v[i] * q.v[i];
      }
      st<V>(W.d[odd ^ 1] + n, e.c);
      st<V>(W.q + n, q);
    }
  }
  dq = block_sum<kMgBlock>(dq);
  if (threadIdx.x == 0) W.part[blockIdx.x] = dq;
}
// x += alpha d, r -= alpha q, f = FP32(r), t = omega f / diag, partial sums of r.r.
template <int V>
__global__ void k_cg_update(MgLevel L, MgVectors W, int odd) {
  const int n = (mg_block() * kMgBlock + (int)threadIdx.x) * V;
  double rr = 0;
  if (n < L.n) {
    const uint32_t codes = ld_codes<V>(L.code, n);
    if (any_fluid<V>(codes)) {
      const double alpha = W.S->alpha;
      Vals<V, double> x = ld<V>(W.x + n), r = ld<V>(W.r + n);
      const Vals<V, double> q = ld<V>(W.q + n), d = ld<V>(W.d[odd ^ 1] + n);
      Vals<V, float> f, t;
#pragma unroll
      for (int i = 0; i < V; ++i) {  // every vector is 0 on non-FLUID cells
        x.v[i] = x.v[i] + alpha * d.v[i];
        r.v[i] = r.v[i] - alpha * q.v[i];
        f.v[i] = (float)r.v[i];
        t.v[i] = smooth0(code_of(codes, i), f.v[i]);
        rr += r.v[i] * r.v[i];
      }
      st<V>(W.x + n, x);
      st<V>(W.r + n, r);
      st<V>(L.f + n, f);
      st<V>(L.t + n, t);
    }
  }
  rr = block_sum<kMgBlock>(rr);
  if (threadIdx.x == 0) W.part[blockIdx.x] = rr;
}
__global__ void k_mg_finish(Geom G, MgLevel L, const double* __restrict__ x, float* __restrict__ p) {
  const int n = mg_block() * kMgBlock + (int)threadIdx.x;
  if (n >= L.n) return;
  int i, j, k;
  cell_xyz(L, n, i, j, k);
  p[G.g(i, j, k)] = L.code[n] ? (float)x[n] : 0.f;
}

// ---- V-cycle passes (FP32)
// Cell-centred trilinear prolongation, per axis: fine x takes 3/4 of parent p = x/2
// and 1/4 of q = p + (x odd ? 1 : -1) clamped to the coarse range.
__device__ __forceinline__ void prolong_refs(int x, int nc, int& p, int& q) {
  p = min(x >> 1, nc - 1);
  q = min(max(p + ((x & 1) ? 1 : -1), 0), nc - 1);
}
__device__ __forceinline__ float axis_weight(int x, int a, int nc) {
  int p, q;
  prolong_refs(x, nc, p, q);
  return (p == a ? 0.75f : 0.f) + (q == a ? 0.25f : 0.f);
}
// The prolongation of e (0 on non-FLUID coarse cells) at a fine cell.
__device__ __forceinline__ float prolong_at(const float* e, int X, int Y, int Z, int x, int y, int z) {
  int px, qx, py, qy, pz, qz;
  prolong_refs(x, X, px, qx);
  prolong_refs(y, Y, py, qy);
  prolong_refs(z, Z, pz, qz);
  const int ix[2] = {px, qx}, iy[2] = {py, qy}, iz[2] = {pz, qz};
  const float w[2] = {0.75f, 0.25f};
  float v[8], s = 0.f;
#pragma unroll
  for (int k = 0; k < 8; ++k) v[k] = e[(ix[k >> 2] * Y + iy[(k >> 1) & 1]) * Z + iz[k & 1]];
#pragma unroll
  for (int k = 0; k < 8; ++k) s += w[k >> 2] * w[(k >> 1) & 1] * w[k & 1] * v[k];
  return s;
}
// The transpose of the prolongation at a coarse cell, gathered: coarse a collects the fine
// cells 2a-1 .. 2a+2 per axis of res (0 on non-FLUID fine cells).
__device__ __forceinline__ float restrict_at(const float* res, int X, int Y, int Z, int CX, int CY, int CZ, int x,
                                             int y, int z) {
  float wx[4], wy[4], wz[4];
  int gx[4], gy[4], gz[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int fx = 2 * x - 1 + k, fy = 2 * y - 1 + k, fz = 2 * z - 1 + k;
    wx[k] = fx >= 0 && fx < X ? axis_weight(fx, x, CX) : 0.f;
    wy[k] = fy >= 0 && fy < Y ? axis_weight(fy, y, CY) : 0.f;
    wz[k] = fz >= 0 && fz < Z ? axis_weight(fz, z, CZ) : 0.f;
    gx[k] = min(max(fx, 0), X - 1) * Y;
    gy[k] = min(max(fy, 0), Y - 1);
    gz[k] = min(max(fz, 0), Z - 1);
  }
  float s = 0.f;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    float v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = res[(gx[a] + gy[k >> 2]) * Z + gz[k & 3]];
#pragma unroll
    for (int k = 0; k < 16; ++k) s += wx[a] * wy[k >> 2] * wz[k & 3] * v[k];
  }
  return s;
}
// Large levels take one linear pass per step, four cells per thread. S (level 0 only):
// nothing is done once the solve has stopped.
// Damped Jacobi sweep out = in + omega (f - A in) / diag; RZ: also partial sums of r.out.
template <bool RZ>
__global__ void k_mg_smooth(MgLevel L, const float* __restrict__ in, float* __restrict__ out,
                            const double* __restrict__ r, double* __restrict__ part, const MgScalars* __restrict__ S) {
  if (S && S->stop) return;
  const int n = (mg_block() * kMgBlock + (int)threadIdx.x) * 4;
  double rz = 0;
  if (n < L.n) {
    const uint32_t codes = ld_codes<4>(L.code, n);
    if (any_fluid<4>(codes)) {
      const Star<4, float> s = ld_star<4>(in, n, L.Z, L.Y * L.Z);
      const Vals<4, float> f = ld<4>(L.f + n);
      Vals<4, double> rv;
      if (RZ) rv = ld<4>(r + n);
      Vals<4, float> o;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t c = code_of(codes, i);
        o.v[i] = c & kMgFluid ? s.c.v[i] + kOmega * (f.v[i] - apply_at(c, s, i)) / diag_of(c) : 0.f;
        if (RZ) rz += rv.v[i] * (double)o.v[i];
      }
      st<4>(out + n, o);
    }
  }
  if (RZ) {
    rz = block_sum<kMgBlock>(rz);
    if (threadIdx.x == 0) part[blockIdx.x] = rz;
  }
}
// t = f - A u
__global__ void k_mg_residual(MgLevel L, const MgScalars* __restrict__ S) {
  if (S && S->stop) return;
  const int n = (mg_block() * kMgBlock + (int)threadIdx.x) * 4;
  if (n >= L.n) return;
  const uint32_t codes = ld_codes<4>(L.code, n);
  if (!any_fluid<4>(codes)) return;
  const Star<4, float> s = ld_star<4>((const float*)L.u, n, L.Z, L.Y * L.Z);
  const Vals<4, float> f = ld<4>(L.f + n);
  Vals<4, float> o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t c = code_of(codes, i);
    o.v[i] = c & kMgFluid ? f.v[i] - apply_at(c, s, i) : 0.f;
  }
  st<4>(L.t + n, o);
}
// Coarse f = 1/2 P^T (fine residual t) and the coarse level's first smoothing sweep. The
// four fine cells along z come in one load, from the row's ends inwards where the coarse
// cell touches them (the others' weights are 0).
__global__ void k_mg_restrict(MgLevel F, MgLevel C, const MgScalars* __restrict__ S) {
  if (S && S->stop) return;
  const int n = mg_block() * kMgBlock + (int)threadIdx.x;
  if (n >= C.n) return;
  const uint32_t c = C.code[n];
  if (!c) return;
  int x, y, z;
  cell_xyz(C, n, x, y, z);
  float wx[4], wy[4], wz[4];
  int gx[4], gy[4];
  const int z0 = max(0, min(2 * z - 1, F.Z - 4));
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int fx = 2 * x - 1 + k, fy = 2 * y - 1 + k;
    wx[k] = fx >= 0 && fx < F.X ? axis_weight(fx, x, C.X) : 0.f;
    wy[k] = fy >= 0 && fy < F.Y ? axis_weight(fy, y, C.Y) : 0.f;
    wz[k] = z0 + k < F.Z ? axis_weight(z0 + k, z, C.Z) : 0.f;
    gx[k] = min(max(fx, 0), F.X - 1) * F.Y;
    gy[k] = min(max(fy, 0), F.Y - 1);
  }
  float s = 0.f;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    Vals<4, float> v[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) v[b] = ld<4>(F.t + (gx[a] + gy[b]) * F.Z + z0);
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int k = 0; k < 4; ++k) s += wx[a] * wy[b] * wz[k] * v[b].v[k];
  }
  s = 0.5f * s;
  C.f[n] = s;
  C.t[n] = smooth0(c, s);
}
// u += P cu on FLUID fine cells (cu: the coarse level's result)
__global__ void k_mg_prolong(MgLevel F, MgLevel C, const float* __restrict__ cu, const MgScalars* __restrict__ S) {
  if (S && S->stop) return;
  const int n = mg_block() * kMgBlock + (int)threadIdx.x;
  if (n >= F.n || !F.code[n]) return;
  int x, y, z;
  cell_xyz(F, n, x, y, z);
  F.u[n] += prolong_at(cu, C.X, C.Y, C.Z, x, y, z);
}

// A smaller level's way down in one launch: the second sweep u = t + omega (f - A t) / diag, the residual, its
// restriction and the coarse level's first sweep. A block owns 8 x 8 x 16 fine cells (4 x
// 4 x 8 coarse ones); the restriction reaches one cell out, the residual one more, the
// sweep one more, so t is staged in LDS with a margin of 3 and u and the residual are
// recomputed in the margins (8.6 us at 64^3 and 32^3, where the three linear passes took 14;
// at 128^3 the margins cost more than the launches: 33 against 22 us).
// Tiles without FLUID leave after reading their codes.
constexpr int kTx = 8, kTy = 8, kTz = 16;
constexpr int kTileThreads = 1024;  // about three cells of the widest margin per thread
// Box of the tile's cells with margin M.
template <int M>
struct Box {
  static constexpr int X = kTx + 2 * M, Y = kTy + 2 * M, Z = kTz + 2 * M, N = X * Y * Z;
  static constexpr int sy = Z, sx = Y * Z;
  __device__ static __forceinline__ int at(int x, int y, int z) { return ((x + M) * Y + y + M) * Z + z + M; }
  // entry e's cell relative to the tile
  __device__ static __forceinline__ void cell(int e, int& x, int& y, int& z) {
    x = e / sx;
    y = (e - x * sx) / Z;
    z = e - x * sx - y * Z - M;
    x -= M;
    y -= M;
  }
};
struct Tile {
  int x, y, z;  // first cell
};
__device__ __forceinline__ Tile tile_of(const MgLevel& L) {
  const int nz = (L.Z + kTz - 1) / kTz, ny = (L.Y + kTy - 1) / kTy;
  int b = mg_block();
  Tile t;
  t.z = (b % nz) * kTz;
  b /= nz;
  t.y = (b % ny) * kTy;
  t.x = b / ny * kTx;
  return t;
}
__device__ __forceinline__ bool inside(const MgLevel& L, int x, int y, int z) {
  return (unsigned)x < (unsigned)L.X && (unsigned)y < (unsigned)L.Y && (unsigned)z < (unsigned)L.Z;
}
__device__ __forceinline__ int cell_n(const MgLevel& L, int x, int y, int z) { return (x * L.Y + y) * L.Z + z; }
// A box's entries per thread, and the i-th one. The last entry is everyone's beyond it (the
// same value written again), so that the unrolled loads and sums need no branches.
template <int M>
constexpr int kPer = (Box<M>::N + kTileThreads - 1) / kTileThreads;
template <int M>
__device__ __forceinline__ int entry(int i) {
  return min(i * kTileThreads + (int)threadIdx.x, Box<M>::N - 1);
}
// Codes of the tile with margin 2 into LDS; whether the tile itself holds FLUID.
__device__ __forceinline__ bool stage_codes(const MgLevel& L, const Tile& t, uint8_t* code) {
  bool any = false;
#pragma unroll
  for (int i = 0; i < kPer<2>; ++i) {
    const int e = entry<2>(i);
    int x, y, z;
    Box<2>::cell(e, x, y, z);
    const bool in = inside(L, t.x + x, t.y + y, t.z + z);
    const uint8_t v = L.code[in ? cell_n(L, t.x + x, t.y + y, t.z + z) : 0], c = in ? v : 0;
    code[e] = c;
    any |= c && (unsigned)x < kTx && (unsigned)y < kTy && (unsigned)z < kTz;
  }
  return __syncthreads_or(any);
}
template <typename B>
__device__ __forceinline__ float box_apply(const float* u, int e, uint32_t c) {
  return stencil<float>(c, u[e], u[e + B::sx], u[e - B::sx], u[e + B::sy], u[e - B::sy], u[e + 1], u[e - 1]);
}
__global__ __launch_bounds__(kTileThreads) void k_mg_down(MgLevel L, MgLevel C, const MgScalars* __restrict__ S) {
  __shared__ uint8_t code[Box<2>::N];
  __shared__ float t[Box<3>::N], u[Box<2>::N];
  if (S && S->stop) return;
  const Tile o = tile_of(L);
  if (!stage_codes(L, o, code)) return;
  float tv[kPer<3>], f[kPer<2>];
  uint32_t c2[kPer<2>];
#pragma unroll
  for (int i = 0; i < kPer<3>; ++i) {
    int x, y, z;
    Box<3>::cell(entry<3>(i), x, y, z);
    const bool in = inside(L, o.x + x, o.y + y, o.z + z);
    tv[i] = L.t[in ? cell_n(L, o.x + x, o.y + y, o.z + z) : 0];
    if (!in) tv[i] = 0.f;
  }
#pragma unroll
  for (int i = 0; i < kPer<2>; ++i) {
    const int e = entry<2>(i);
    int x, y, z;
    Box<2>::cell(e, x, y, z);
    c2[i] = code[e];
    f[i] = L.f[c2[i] ? cell_n(L, o.x + x, o.y + y, o.z + z) : 0];
  }
#pragma unroll
  for (int i = 0; i < kPer<3>; ++i) t[entry<3>(i)] = tv[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPer<2>; ++i) {
    const int e = entry<2>(i);
    int x, y, z;
    Box<2>::cell(e, x, y, z);
    const int te = Box<3>::at(x, y, z);
    const float v = t[te] + kOmega * (f[i] - box_apply<Box<3>>(t, te, c2[i])) / diag_of(c2[i]);
    u[e] = c2[i] ? v : 0.f;
    if (c2[i] && (unsigned)x < kTx && (unsigned)y < kTy && (unsigned)z < kTz)
      L.u[cell_n(L, o.x + x, o.y + y, o.z + z)] = v;
  }
  __syncthreads();
  // the residual on the tile with margin 1, in t's place
  float* res = t;
#pragma unroll
  for (int i = 0; i < kPer<2>; ++i) {
    const int e = entry<2>(i);
    int x, y, z;
    Box<2>::cell(e, x, y, z);
    if ((unsigned)(x + 1) >= kTx + 2 || (unsigned)(y + 1) >= kTy + 2 || (unsigned)(z + 1) >= kTz + 2) continue;
    res[Box<1>::at(x, y, z)] = c2[i] ? f[i] - box_apply<Box<2>>(u, e, c2[i]) : 0.f;
  }
  __syncthreads();
  if (threadIdx.x >= kTx * kTy * kTz / 8) return;
  const int k = threadIdx.x;
  const int lx = k / (kTy * kTz / 4), ly = k / (kTz / 2) % (kTy / 2), lz = k % (kTz / 2);
  const int x = o.x / 2 + lx, y = o.y / 2 + ly, z = o.z / 2 + lz;
  if (x >= C.X || y >= C.Y || z >= C.Z) return;
  const int n = cell_n(C, x, y, z);
  const uint32_t c = C.code[n];
  if (!c) return;
  float wx[4], wy[4], wz[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {  // a missing fine cell's residual is 0
    wx[j] = axis_weight(2 * x - 1 + j, x, C.X);
    wy[j] = axis_weight(2 * y - 1 + j, y, C.Y);
    wz[j] = axis_weight(2 * z - 1 + j, z, C.Z);
  }
  float s = 0.f;
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        s += wx[a] * wy[b] * wz[j] * res[Box<1>::at(2 * lx - 1 + a, 2 * ly - 1 + b, 2 * lz - 1 + j)];
  s = 0.5f * s;
  C.f[n] = s;
  C.t[n] = smooth0(c, s);
}

// One level's way up: u += P e, then two sweeps. The sweeps reach one cell out each, so the
// corrected u is formed on the tile with margin 2 and the first sweep on margin 1. The
// result goes to t (other tiles still read u). cu: the coarse level's result. RZ: also
// partial sums of r.t (level 0).
template <bool RZ>
__global__ __launch_bounds__(kTileThreads) void k_mg_up(MgLevel L, MgLevel C, const float* __restrict__ cu,
                                                    const double* __restrict__ r,
                                                    double* __restrict__ part, const MgScalars* __restrict__ S) {
  constexpr int CX = kTx / 2 + 4, CY = kTy / 2 + 4, CZ = kTz / 2 + 4;  // parents of margin 2, and theirs
  __shared__ uint8_t code[Box<2>::N];
  __shared__ float u[Box<2>::N], t[Box<1>::N], ce[CX * CY * CZ];
  if (S && S->stop) return;
  const Tile o = tile_of(L);
  if (!stage_codes(L, o, code)) {
    if (RZ && threadIdx.x == 0) part[blockIdx.x] = 0.0;
    return;
  }
  const int cx0 = o.x / 2 - 2, cy0 = o.y / 2 - 2, cz0 = o.z / 2 - 2;
  static_assert(CX * CY * CZ <= kTileThreads, "one parent per thread");
  {
    const int e = min((int)threadIdx.x, CX * CY * CZ - 1);
    const int x = cx0 + e / (CY * CZ), y = cy0 + e / CZ % CY, z = cz0 + e % CZ;
    const bool in = inside(C, x, y, z);
    const float w = cu[in ? cell_n(C, x, y, z) : 0];
    ce[e] = in ? w : 0.f;
  }
  float v[kPer<2>], f[kPer<2>];
  uint32_t c2[kPer<2>];
#pragma unroll
  for (int i = 0; i < kPer<2>; ++i) {
    const int e = entry<2>(i);
    int x, y, z;
    Box<2>::cell(e, x, y, z);
    c2[i] = code[e];
    const int n = c2[i] ? cell_n(L, o.x + x, o.y + y, o.z + z) : 0;
    v[i] = L.u[n];
    f[i] = L.f[n];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPer<2>; ++i) {
    const int e = entry<2>(i);
    {
      int x, y, z, px, qx, py, qy, pz, qz;
      Box<2>::cell(e, x, y, z);
      prolong_refs(o.x + x, C.X, px, qx);
      prolong_refs(o.y + y, C.Y, py, qy);
      prolong_refs(o.z + z, C.Z, pz, qz);
      if (!c2[i]) px = qx = cx0, py = qy = cy0, pz = qz = cz0;  // may lie outside the grid
      const int ix[2] = {(px - cx0) * CY, (qx - cx0) * CY}, iy[2] = {py - cy0, qy - cy0}, iz[2] = {pz - cz0, qz - cz0};
      const float w[2] = {0.75f, 0.25f};
      float s = 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k)
        s += w[k >> 2] * w[(k >> 1) & 1] * w[k & 1] * ce[(ix[k >> 2] + iy[(k >> 1) & 1]) * CZ + iz[k & 1]];
      v[i] = c2[i] ? v[i] + s : 0.f;
    }
    u[e] = v[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPer<2>; ++i) {
    const int e = entry<2>(i);
    int x, y, z;
    Box<2>::cell(e, x, y, z);
    if ((unsigned)(x + 1) >= kTx + 2 || (unsigned)(y + 1) >= kTy + 2 || (unsigned)(z + 1) >= kTz + 2) continue;
    const uint32_t c = c2[i];
    t[Box<1>::at(x, y, z)] = c ? v[i] + kOmega * (f[i] - box_apply<Box<2>>(u, e, c)) / diag_of(c) : 0.f;
  }
  __syncthreads();
  double rz = 0;
#pragma unroll
  for (int i = 0; i < kPer<2>; ++i) {
    if (i * kTileThreads + (int)threadIdx.x >= Box<2>::N) break;
    int x, y, z;
    Box<2>::cell(entry<2>(i), x, y, z);
    const uint32_t c = c2[i];
    if (!c || (unsigned)x >= kTx || (unsigned)y >= kTy || (unsigned)z >= kTz) continue;
    const int te = Box<1>::at(x, y, z), n = cell_n(L, o.x + x, o.y + y, o.z + z);
    const float w = t[te] + kOmega * (f[i] - box_apply<Box<1>>(t, te, c)) / diag_of(c);
    L.t[n] = w;
    if (RZ) rz += r[n] * (double)w;
  }
  if (RZ) {
    rz = block_sum<kTileThreads>(rz);
    if (threadIdx.x == 0) part[blockIdx.x] = rz;
  }
}

// ---- the levels of at most kTailCells cells, in one workgroup
// Same passes on LDS arrays. A neighbour outside the level's array is read as the cell
// itself (its wall bit replaces it). The coarsest level has at most 64 cells: one wave,
// its value in a register, neighbours by lane permutation. (Its sweeps as a precomputed 64
// x 64 matrix: 1.4 us less per V-cycle, but rounded differently, which moved results of
// small systems by up to 3e-6.)
struct TailLds {
  float f[kTailLds], u[kTailLds], t[kTailLds];
  double inv[8];  // reciprocals of the diagonals by wall count
  uint8_t code[kTailLds];
};
__device__ __forceinline__ float tail_apply(const float* u, uint32_t code, int n, int sy, int sx) {
  return stencil<float>(code, u[n], u[code & 1 ? n : n + sx], u[code & 2 ? n : n - sx], u[code & 4 ? n : n + sy],
                        u[code & 8 ? n : n - sy], u[code & 16 ? n : n + 1], u[code & 32 ? n : n - 1]);
}
// The levels share one copy of the code (unrolled per level, the kernel waited for its
// instructions), and a cell's sweep divides through the reciprocal of its diagonal.
struct MgTail {
  struct Level {
    int X, Y, Z, n;
    FastDiv divZ, divYZ;
    const uint8_t* code;
  };
  int count;
  const float* f;
  float* u;
  Level L[kMgMaxLevels];
};
__device__ __forceinline__ void cell_xyz(const MgTail::Level& L, int n, int& x, int& y, int& z) {
  x = (int)fast_div((uint32_t)n, L.divYZ);
  const int r = n - x * (L.Y * L.Z);
  y = (int)fast_div((uint32_t)r, L.divZ);
  z = r - y * L.Z;
}
// x * inv, inv = the double reciprocal of d, rounds to the float quotient x / d.
__device__ __forceinline__ float over(float x, double inv) { return (float)((double)x * inv); }
// A level's cells of one thread; the last cell is everyone's beyond it.
template <int NP>
struct TailCell {
  int n[NP];
  uint32_t c[NP];
  float f[NP], v[NP];
  double inv[NP];
  int sy, sx;
  __device__ __forceinline__ TailCell(const MgTail::Level& L, const TailLds& m, int at) {
    sy = L.Z, sx = L.Y * L.Z;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      n[i] = min((int)threadIdx.x + i * kTailThreads, L.n - 1);
      c[i] = m.code[at + n[i]];
      f[i] = m.f[at + n[i]];
      inv[i] = m.inv[__popc(c[i] & 63u)];
    }
  }
  __device__ __forceinline__ void put(float* out) {
#pragma unroll
    for (int i = 0; i < NP; ++i) out[n[i]] = v[i];
    __syncthreads();
  }
  __device__ __forceinline__ void sweep(const float* in, float* out) {
#pragma unroll
    for (int i = 0; i < NP; ++i)
      v[i] = c[i] ? in[n[i]] + over(kOmega * (f[i] - tail_apply(in, c[i], n[i], sy, sx)), inv[i]) : 0.f;
    put(out);
  }
};
template <int NP>
__device__ __forceinline__ void tail_down(const MgTail::Level& L, const MgTail::Level& C, TailLds& m, int at) {
  float *u = m.u + at, *t = m.t + at;
  TailCell<NP> k(L, m, at);
#pragma unroll
  for (int i = 0; i < NP; ++i) k.v[i] = k.c[i] ? over(kOmega * k.f[i], k.inv[i]) : 0.f;
  k.put(t);
  k.sweep(t, u);
#pragma unroll
  for (int i = 0; i < NP; ++i) k.v[i] = k.c[i] ? k.f[i] - tail_apply(u, k.c[i], k.n[i], k.sy, k.sx) : 0.f;
  k.put(t);
  for (int j = threadIdx.x; j < C.n; j += kTailThreads) {
    int x, y, z;
    cell_xyz(C, j, x, y, z);
    const float s = restrict_at(t, L.X, L.Y, L.Z, C.X, C.Y, C.Z, x, y, z);
    m.f[at + L.n + j] = m.code[at + L.n + j] ? 0.5f * s : 0.f;
  }
  __syncthreads();
}
template <int NP>
__device__ __forceinline__ void tail_up(const MgTail::Level& L, const MgTail::Level& C, TailLds& m, int at) {
  float *u = m.u + at, *t = m.t + at;
  TailCell<NP> k(L, m, at);
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    int x, y, z;
    cell_xyz(L, k.n[i], x, y, z);
    const float e = prolong_at(u + L.n, C.X, C.Y, C.Z, x, y, z);
    k.v[i] = k.c[i] ? u[k.n[i]] + e : 0.f;
  }
  __syncthreads();  // the duplicates of the last cell have read it
  k.put(u);
  k.sweep(u, t);
  k.sweep(t, u);
}
__global__ __launch_bounds__(kTailThreads) void k_mg_tail(MgTail T) {
  __shared__ TailLds m;
  const int tid = threadIdx.x;
  if (tid < 8) m.inv[tid] = 1.0 / (6.0 - tid);
  int at = 0;
  for (int l = 0; l < T.count; ++l) {
    constexpr int NP = kTailCells / kTailThreads;
    if (l == 0) {
      float f[NP];
      uint8_t c[NP];
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int n = min(tid + i * kTailThreads, T.L[0].n - 1);
        f[i] = T.f[n];
        c[i] = T.L[0].code[n];
      }
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int n = min(tid + i * kTailThreads, T.L[0].n - 1);
        m.f[n] = f[i];
        m.code[n] = c[i];
      }
    } else {
      for (int n = tid; n < T.L[l].n; n += kTailThreads) m.code[at + n] = T.L[l].code[n];
    }
    at += T.L[l].n;
  }
  __syncthreads();
  at = 0;
  for (int l = 0; l + 1 < T.count; ++l) {
    if (T.L[l].n > kTailThreads)
      tail_down<kTailCells / kTailThreads>(T.L[l], T.L[l + 1], m, at);
    else
      tail_down<1>(T.L[l], T.L[l + 1], m, at);
    at += T.L[l].n;
  }
  if (tid < 64) {  // the coarsest level: one wave, the value in a register
    const MgTail::Level& L = T.L[T.count - 1];
    const int sy = L.Z, sx = L.Y * L.Z;
    const uint32_t c = tid < L.n ? m.code[at + tid] : 0;
    const float f = tid < L.n ? m.f[at + tid] : 0.f;
    const double inv = m.inv[__popc(c & 63u)];
    float v = c ? over(kOmega * f, inv) : 0.f;
    for (int k = 1; k < kMgCoarseSweeps; ++k) {
      const float a = stencil<float>(c, v, __shfl(v, tid + sx, 64), __shfl(v, tid - sx, 64), __shfl(v, tid + sy, 64),
                                     __shfl(v, tid - sy, 64), __shfl(v, tid + 1, 64), __shfl(v, tid - 1, 64));
      if (c) v = v + over(kOmega * (f - a), inv);
    }
    if (tid < L.n) m.u[at + tid] = v;
  }
  __syncthreads();
  for (int l = T.count - 2; l >= 0; --l) {
    at -= T.L[l].n;
    if (T.L[l].n > kTailThreads)
      tail_up<kTailCells / kTailThreads>(T.L[l], T.L[l + 1], m, at);
    else
      tail_up<1>(T.L[l], T.L[l + 1], m, at);
  }
  for (int n = tid; n < T.L[0].n; n += kTailThreads)
    if (m.code[n]) T.u[n] = m.u[n];
}
// r.z where level 0 itself ran in the workgroup above.
__global__ void k_mg_rz(MgLevel L, const double* __restrict__ r, double* __restrict__ part) {
  const int n = mg_block() * kMgBlock + (int)threadIdx.x;
  double v = n < L.n && L.code[n] ? r[n] * (double)L.u[n] : 0.0;
  v = block_sum<kMgBlock>(v);
  if (threadIdx.x == 0) part[blockIdx.x] = v;
}

// ---- launchers
MgLevel mg_level(int X, int Y, int Z) {
  MgLevel L{};
  L.X = X, L.Y = Y, L.Z = Z;
  L.n = X * Y * Z;
  L.divZ = make_fastdiv((uint32_t)Z);
  L.divYZ = make_fastdiv((uint32_t)(Y * Z));
  return L;
}
int mg_tail_level(const MgLevels& H) {
  int l = H.count - 1, cells = H.L[l].n;
  while (l > 0 && H.L[l - 1].n <= kTailCells && cells + H.L[l - 1].n <= kTailLds)
    cells += H.L[--l].n;
  return l;
}
static int blocks1(const MgLevel& L) { return (L.n + kMgBlock - 1) / kMgBlock; }
static int vec_of(const MgLevel& L) { return L.n >= kVecCells ? 4 : 1; }
static int blocksv(const MgLevel& L) { return (L.n + kMgBlock * vec_of(L) - 1) / (kMgBlock * vec_of(L)); }
static int tiles(const MgLevel& L) {
  return ((L.X + kTx - 1) / kTx) * ((L.Y + kTy - 1) / kTy) * ((L.Z + kTz - 1) / kTz);
}
size_t mg_part_size(const MgLevels& H) { return (size_t)std::max(blocks1(H.L[0]), tiles(H.L[0])); }

#define MG_LAUNCH_VEC(kernel, L, s, ...)                                                                   \
  do {                                                                                                     \
    if (vec_of(L) == 4)                                                                                    \
      hipLaunchKernelGGL((kernel<4>), dim3(blocksv(L)), dim3(kMgBlock), 0, s, __VA_ARGS__);                \
    else                                                                                                   \
      hipLaunchKernelGGL((kernel<1>), dim3(blocksv(L)), dim3(kMgBlock), 0, s, __VA_ARGS__);                \
  } while (0)

// Where the V-cycle leaves level l's correction: tiled levels in t, the others in u.
static bool tiled(const MgLevels& H, int l) { return l < H.tail && vec_of(H.L[l]) == 1; }
static float* correction(const MgLevels& H, int l) { return tiled(H, l) ? H.L[l].t : H.L[l].u; }
// The V-cycle of f[0] given t[0], level 0's first sweep; then r.z and beta.
static void vcycle(const MgLevels& H, const MgVectors& V, hipStream_t s) {
  const MgLevel& L0 = H.L[0];
  for (int l = 0; l < H.tail; ++l) {
    const MgLevel &L = H.L[l], &C = H.L[l + 1];
    const MgScalars* S = l == 0 ? V.S : nullptr;
    if (tiled(H, l)) {
      hipLaunchKernelGGL(k_mg_down, dim3(tiles(L)), dim3(kTileThreads), 0, s, L, C, S);
      continue;
    }
    hipLaunchKernelGGL(k_mg_smooth<false>, dim3(blocksv(L)), dim3(kMgBlock), 0, s, L, L.t, L.u, nullptr, nullptr, S);
    hipLaunchKernelGGL(k_mg_residual, dim3(blocksv(L)), dim3(kMgBlock), 0, s, L, S);
    hipLaunchKernelGGL(k_mg_restrict, dim3(blocks1(C)), dim3(kMgBlock), 0, s, L, C, S);
  }
  MgTail T{};
  T.count = H.count - H.tail;
  T.f = H.L[H.tail].f, T.u = H.L[H.tail].u;
  for (int l = 0; l < T.count; ++l) {
    const MgLevel& L = H.L[H.tail + l];
    T.L[l] = MgTail::Level{L.X, L.Y, L.Z, L.n, L.divZ, L.divYZ, L.code};
  }
  hipLaunchKernelGGL(k_mg_tail, dim3(1), dim3(kTailThreads), 0, s, T);
  int parts = blocks1(L0);
  for (int l = H.tail - 1; l >= 0; --l) {
    const MgLevel &L = H.L[l], &C = H.L[l + 1];
    const MgScalars* S = l == 0 ? V.S : nullptr;
    const float* cu = correction(H, l + 1);
    parts = tiled(H, l) ? tiles(L) : blocksv(L);
    if (tiled(H, l)) {
      if (l == 0)
        hipLaunchKernelGGL(k_mg_up<true>, dim3(parts), dim3(kTileThreads), 0, s, L, C, cu, V.r, V.part, S);
      else
        hipLaunchKernelGGL(k_mg_up<false>, dim3(parts), dim3(kTileThreads), 0, s, L, C, cu, nullptr, nullptr, S);
      continue;
    }
    hipLaunchKernelGGL(k_mg_prolong, dim3(blocks1(L)), dim3(kMgBlock), 0, s, L, C, cu, S);
    hipLaunchKernelGGL(k_mg_smooth<false>, dim3(parts), dim3(kMgBlock), 0, s, L, L.u, L.t, nullptr, nullptr, S);
    if (l == 0)
      hipLaunchKernelGGL(k_mg_smooth<true>, dim3(parts), dim3(kMgBlock), 0, s, L, L.t, L.u, V.r, V.part, S);
    else
      hipLaunchKernelGGL(k_mg_smooth<false>, dim3(parts), dim3(kMgBlock), 0, s, L, L.t, L.u, nullptr, nullptr, S);
  }
  if (H.tail == 0) hipLaunchKernelGGL(k_mg_rz, dim3(parts), dim3(kMgBlock), 0, s, L0, V.r, V.part);
  hipLaunchKernelGGL(k_mg_fold_rz, dim3(1), dim3(kTailThreads), 0, s, V.part, parts, V.S);
}

void mg_start(const Geom& G, const MgLevels& H, const MgVectors& V, const uint8_t* content, const float* rhs,
              const float* p, double tol, int max_iters, int check_every, hipStream_t s) {
  const MgLevel& L = H.L[0];
  hipLaunchKernelGGL(k_mg_gather, dim3(blocks1(L)), dim3(kMgBlock), 0, s, G, content, rhs, p, L, V);
  hipLaunchKernelGGL(k_mg_fold_start, dim3(1), dim3(kTailThreads), 0, s, V.part, blocks1(L), V.S, tol, max_iters,
                     check_every);
  for (int l = 1; l < H.count; ++l)
    hipLaunchKernelGGL(k_mg_coarsen, dim3(blocks1(H.L[l])), dim3(kMgBlock), 0, s, H.L[l - 1], H.L[l]);
  MG_LAUNCH_VEC(k_mg_residual0, L, s, L, V, p ? 1 : 0);
  hipLaunchKernelGGL(k_mg_fold_rr, dim3(1), dim3(kTailThreads), 0, s, V.part, blocksv(L), V.S, V.report, 1);
  vcycle(H, V, s);
}
void mg_iterate(const MgLevels& H, const MgVectors& V, int odd, hipStream_t s) {
  const MgLevel& L = H.L[0];
  MG_LAUNCH_VEC(k_cg_apply, L, s, L, V, correction(H, 0), odd);
  hipLaunchKernelGGL(k_mg_fold_dq, dim3(1), dim3(kTailThreads), 0, s, V.part, blocksv(L), V.S);
  MG_LAUNCH_VEC(k_cg_update, L, s, L, V, odd);
  hipLaunchKernelGGL(k_mg_fold_rr, dim3(1), dim3(kTailThreads), 0, s, V.part, blocksv(L), V.S, V.report, 0);
  vcycle(H, V, s);
}
void mg_finish(const Geom& G, const MgLevels& H, const MgVectors& V, float* p, hipStream_t s) {
  hipLaunchKernelGGL(k_mg_finish, dim3(blocks1(H.L[0])), dim3(kMgBlock), 0, s, G, H.L[0], V.x, p);
}

}  // namespace aqf
