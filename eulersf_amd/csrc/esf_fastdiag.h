// esf_fastdiag.h -- the pieces of the fast-diagonalisation preconditioned
// pressure solve shared by esf_fastdiag.hip (the preconditioner and the
// vector update) and esf_pressure.hip (the SpMV and the solve).
#pragma once
#include "esf_internal.h"

namespace esf {

// cells per axis, padded to multiples of 16, and the 32-wide tiles of x and y
struct FdGeom {
  int nx, ny, nz, PX, PY, PZ, tx, ty;
};

// the test of the recursive residual that an iteration's first kernel makes
struct PcgTest {
  int nb;               // |r|^2 partials of the update before
  const double* parts;
  double tol2;          // (relative tolerance)^2
  int iter;             // updates made so far
  CrScalars* sc;        // the solve's block
  const CrScalars* outer;  // holds |b|
};

// what the SpMV needs to form p = z + beta p: the r . z partials, and r . z of
// this and the last iteration at rz[iter & 1], rz[1 - (iter & 1)]
struct PcgDir {
  int iter;
  int nb;
  const double* parts;
  double* rz;
};

// the sums of K sets of nb partials ([k nb + i]), in every thread of the block
// (NT threads) and bitwise the same in every block; lds: K doubles per wave
template <int K, int NT = 256>
__device__ inline void blockTotals(int nb, const double* __restrict__ parts, double* lds,
                                   double (&t)[K]) {
  double a[K];
#pragma unroll
  for (int k = 0; k < K; k++) a[k] = 0;
  constexpr int nt = NT, nw = NT / 64;
  for (int i = threadIdx.x; i < nb; i += 4 * nt) {
    double v[K][4];
#pragma unroll
    for (int k = 0; k < K; k++)
#pragma unroll
      for (int u = 0; u < 4; u++)
        v[k][u] = i + nt * u < nb ? parts[(long)k * nb + i + nt * u] : 0.0;
#pragma unroll
    for (int k = 0; k < K; k++) a[k] += (v[k][0] + v[k][1]) + (v[k][2] + v[k][3]);
  }
  double w[K];
#pragma unroll
  for (int k = 0; k < K; k++) w[k] = waveSum(a[k]);
  __syncthreads();
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int k = 0; k < K; k++) lds[nw * k + (threadIdx.x >> 6)] = w[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < K; k++) {
    double r = 0;
#pragma unroll
    for (int v = 0; v < nw; v++) r += lds[nw * k + v];
    t[k] = r;
  }
  __syncthreads();
}
template <int NT = 256>
__device__ inline double blockTotal(int nb, const double* __restrict__ parts, double* lds) {
  double t[1];
  blockTotals<1, NT>(nb, parts, lds, t);
  return t[0];
}

// a solve's done flag for a launch in which a block sets it: the read of the
// block's first thread, in all its threads.  Each wave reading for itself, a
// block that starts while the flag is being set would have some waves leave
// and the others add up LDS slots that nobody wrote.  (Blocks may differ: a
// launch that sets the flag leaves the solve's vectors alone in every block.)
__device__ inline bool blockDone(int done, int* lds) {
  if (threadIdx.x == 0) *lds = done;
  __syncthreads();
  return *lds != 0;
}

FdGeom fdGeom(const Dims& d);
// whether the preconditioner takes this grid
bool fdFits(const Dims& d);
// its tables and buffers (mixed contexts, at creation)
esf_status fdCreate(esf_ctx* ctx);
// one iteration: z = S0^-1 r, p = z + beta p, q = S p, x += alpha p,
// r -= alpha q; on scalar block 1, |b| in block 0
esf_status fdIteration(esf_ctx* ctx, int it, double eps);
// the test of the residual after `it` iterations; scalar block 1 to hostOut
void fdTest(esf_ctx* ctx, int it, double eps, CrScalars* hostOut);

// esf_pressure.hip
int spmvBlocks(const esf_ctx* ctx);
int spmvPcgBlocks(const esf_ctx* ctx);
esf_status spmvPcg(esf_ctx* ctx, const double* pOld, const float* z, double* pNew, double* q,
                   CrScalars* sc, const PcgDir& dir, double* parts);

}  // namespace esf
