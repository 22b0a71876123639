// esf_pressure.hip -- the Schur pressure system S = J M^-1 J^T on the
// collocated Q1-P0 grid of the reference, and its Krylov solvers.
//
// S x (COUPLED_INTEGRATOR_3D.cpp:638-660) is never assembled.  One kernel
// streams x through LDS in 32x8-cell tiles marching along z, the next layer
// prefetched into registers: for each node layer it forms w = minv * (J^T x)
// (8 cells, signs from the corner bits, COUPLED_INTEGRATOR_3D.cpp:239-249),
// for each cell layer it forms y = J w (8 corners x 3 components).  Sums run
// in the reference's sparse row/column order, so the FP64 result is bitwise
// the reference's CSR product.  Bytes per apply: x once, y once, minv once
// (8 B each in FP64).
//
// The Krylov loop is CONJUGATE_RESIDUAL::solvePCR (CONJUGATE_RESIDUAL.inl:
// 109-192), one SpMV launch per iteration with the direction update of the
// previous iteration folded in:
//   Ap = beta Ap + s, p = beta p + r (:157-160), x += alpha p,
//   r -= alpha D^-1 Ap (recomputed on the halo), s = S r; partial sums r.s,
//   s.D^-1 s, Ap.D^-1 s, Ap.D^-1 Ap
// and one finisher: delta and beta from r.s, alpha = delta / (Ap.D^-1 Ap)
// for the next direction Ap = s + beta Ap with the square expanded, so a
// single reduction per iteration provides both (only alpha's rounding
// differs from the reference's evaluation).  s and Ap alternate between two
// buffers (halo cells read the previous values while owners write the new
// ones), as r does.  A true-residual check every 5 iterations, as the
// reference does.  Block partials are summed by a one-block finisher (fixed
// order, deterministic).
#include <limits>

#include "esf_fastdiag.h"
#include "esf_internal.h"
#include "esf_krylov.h"

namespace esf {

enum SpmvMode {
  M_APPLY = 0,
  M_SETUP_R = 1,
  M_SETUP_S = 2,
  M_UPDATE = 3,
  M_CHECK = 4,
  M_IR_RESID = 5,
  M_PCG = 6,        // p = z + beta p, q = S p, p . q (esf_fastdiag.hip)
  M_PCG_RESID = 7,  // r = b - S x, also in FP32 in the preconditioner's layout
  M_UPDATE_CHECK = 8,  // kSpmvFlat: M_UPDATE and, in blocks of its own, M_CHECK
};

template <typename T>
struct SpmvArgs {
  const T* in;       // input vector (x, r, or r_old / x_old)
  const T* minv;     // per node
  T* out;            // M_APPLY output
  const T* b;        // right-hand side
  const T* D;        // Jacobi diagonal
  const T* Dinv;     // its reciprocals (M_UPDATE)
  T* x;              // solution (M_UPDATE, M_IR_RESID)
  T* r;              // residual
  T* p;              // direction
  T* s;              // S r (M_UPDATE: the previous s, read)
  T* Ap;             // A p (M_UPDATE: the previous Ap, read)
  T* sOut;           // M_UPDATE: the new s
  T* ApOut;          // M_UPDATE: the new Ap
  const float* e32;  // M_IR_RESID: correction added to x (may be null)
  float* r32;        // M_IR_RESID: residual handed to the FP32 solve
  CrScalars* sc;
  double* partials;
  int iter;
  int first;         // M_IR_RESID: also compute |b|
  int recursive;     // M_UPDATE: the finisher tests the recursive residual
  CrScalars* hostOut;  // M_CHECK (M_UPDATE when recursive): pinned slot for the scalar block
  PcgDir dir;        // M_PCG
  // kSpmvFlat M_UPDATE: r . s of the last two iterations; the x it writes (x
  // stays as it was for a check beside it); the iterate whose check rode
  // with the update before (its verdict is this update's to find), or -1
  double* delta;
  T* xOut;
  int verdict;
  int px, pxy;       // M_PCG_RESID: the padded layout's strides
};

constexpr int TX = 32, TY = 8;
constexpr int HALO = (TX + 2) * (TY + 2);  // cells of one layer incl. halo
constexpr int NODES = (TX + 1) * (TY + 1); // nodes of one layer
constexpr int NRING = HALO - TX * TY;      // halo cells around the tile's own
constexpr int HPT = 2;                     // halo cells per thread: its own, one of the ring
constexpr int NEDGE = NODES - TX * TY;     // nodes on the tile's low x and low y edges
static_assert(TX * TY == 256 && NRING <= 256, "one 256-thread block per tile");

// One block owns a TX x TY tile of cells and `layers` cell layers of it,
// marching up in z.  Iteration k of the march forms node layer k and cell
// layer k - 2, so one barrier per layer separates producers from
// consumers:
//   - node layer k: w = minv * (J^T x) from cell layers k - 1 and k.  Each
//     thread owns the node at the upper corner of its cell and carries that
//     node's sums over its four cells of the lower layer from the previous
//     iteration, so it reads only the four of the upper layer; the NEDGE
//     nodes on the tile's low x and low y edges are formed by the first
//     threads from LDS alone (three x buffers: layers k - 1, k, k + 1);
//   - cell layer k - 2: y = J w, its sum over the corner nodes of layer
//     k - 2 carried from the previous iteration, those of layer k - 1 read
//     from LDS (two w buffers);
//   - x of layer k + 1 goes to LDS; layer k + 2 and the pointwise operands
//     of the next output layer are fetched, minv of layer k + 1 at the top
//     of the iteration.
// The additions keep the reference's sparse row/column order exactly.  A
// corner node off the interior carries w = 0 and is added like the others:
// the running sum starts at +0 and adding a zero never changes it.
// Out-of-grid halo cells are read at a clamped address and replaced by 0,
// so the loop has no per-cell branches.
template <typename T, int MODE, int DEPTH, class GridT>
__device__ __forceinline__ void kSpmv(const GridT& wg, Dims d, SpmvArgs<T> a, int tilesX, int tilesY,
                                      int tilesZ, int layers) {
  if (MODE != M_APPLY && a.sc && a.sc->done) return;
  __shared__ T xs[3 * HALO];
  __shared__ T ws[2 * NODES * 3];
  __shared__ double red[5 * 4];

  // XCD-aware tile order: each XCD gets a contiguous run of tiles, so
  // neighbouring tiles' shared halos stay in one L2
  const int tile = wg.block();
  const int tx = tile % tilesX, ty = (tile / tilesX) % tilesY,
            tz = tile / (tilesX * tilesY);
  const int x0 = tx * TX, y0 = ty * TY, z0 = tz * layers;
  const int zEnd = min(z0 + layers, d.CZ);

  T alpha = 0, beta = 0;
  if (MODE == M_UPDATE) {
    alpha = (T)a.sc->alpha;
    beta = (T)a.sc->beta;
  }
  if (MODE == M_PCG) {
    const double rz = blockTotal(a.dir.nb, a.dir.parts, red);
    const int now = a.dir.iter & 1;
    if (a.dir.iter > 0) beta = (T)(rz / a.dir.rz[1 - now]);
    if (wg.block() == 0 && threadIdx.x == 0) a.dir.rz[now] = rz;
  }
  double part0 = 0, part1 = 0, part2 = 0, part3 = 0, part4 = 0;

  const int lx = threadIdx.x % TX, ly = threadIdx.x / TX;
  const int cx = x0 + lx, cy = y0 + ly;
  const bool cellXY = cx < d.CX && cy < d.CY;
  // in-layer offset of this thread's cell (clamped into the grid)
  const int cOff = min(cx, d.CX - 1) + min(cy, d.CY - 1) * d.CX;

  // halo slots of this thread: slot 0 is its own cell, slot 1 (threads
  // below NRING) a cell of the ring around the tile -- the low row, the
  // high row, then the low and the high column between them.  Per slot:
  // in-layer offset (clamped), validity and LDS position.  Owning its cell's
  // halo values lets the CR update keep them in registers until the cell's
  // output layer instead of reading them again.
  int hOff[HPT], hIdx[HPT];
  bool hVal[HPT];
  {
    const int r = threadIdx.x < NRING ? threadIdx.x : 0;
    const int q = r - 2 * (TX + 2);
    const int rx = r < TX + 2 ? r : (r < 2 * (TX + 2) ? r - (TX + 2) : (q < TY ? 0 : TX + 1));
    const int ry = r < TX + 2 ? 0 : (r < 2 * (TX + 2) ? TY + 1 : 1 + q % TY);
    const int hx[HPT] = {lx + 1, rx}, hy[HPT] = {ly + 1, ry};
#pragma unroll
    for (int h = 0; h < HPT; h++) {
      const int gx = x0 - 1 + hx[h], gy = y0 - 1 + hy[h];
      hIdx[h] = hy[h] * (TX + 2) + hx[h];
      hVal[h] = gx >= 0 && gx < d.CX && gy >= 0 && gy < d.CY;
      hOff[h] = min(max(gx, 0), d.CX - 1) + min(max(gy, 0), d.CY - 1) * d.CX;
    }
    // a thread without a ring cell re-reads its own (no extra lines)
    if (threadIdx.x >= NRING) hOff[1] = hOff[0];
  }
  // this thread's node: tile node (lx + 1, ly + 1), the upper corner of its
  // cell; its edge node (threads below NEDGE): (0, t) for t <= TY, else
  // (t - TY, 0).  In-layer offsets clamped to the interior.
  const bool hasEdge = threadIdx.x < NEDGE;
  const int enx = threadIdx.x <= TY ? 0 : threadIdx.x - TY;
  const int eny = threadIdx.x <= TY ? threadIdx.x : 0;
  const int mI = x0 + lx + 1, mJ = y0 + ly + 1, eI = x0 + enx, eJ = y0 + eny;
  const bool mainIJ = mI >= 1 && mI <= d.X - 2 && mJ >= 1 && mJ <= d.Y - 2;
  const bool edgeIJ = hasEdge && eI >= 1 && eI <= d.X - 2 && eJ >= 1 && eJ <= d.Y - 2;
  const int mOff = min(max(mI, 1), d.X - 2) + min(max(mJ, 1), d.Y - 2) * d.X;
  // a thread without an edge node re-reads its main node's minv
  const int eOff = hasEdge ? min(max(eI, 1), d.X - 2) + min(max(eJ, 1), d.Y - 2) * d.X : mOff;
  // LDS positions
  const int mHalo = (ly + 1) * (TX + 2) + lx + 1;  // lowest of the main node's cells
  const int eHalo = eny * (TX + 2) + enx;          // lowest of the edge node's cells
  const int mW = 3 * ((ly + 1) * (TX + 1) + lx + 1);
  const int eW = 3 * (eny * (TX + 1) + enx);
  const int cW = 3 * (ly * (TX + 1) + lx);         // this cell's lowest corner node

  // Every global load of the loop is issued unconditionally at the end of
  // an iteration for the iteration DEPTH later (addresses clamped into the
  // grid and to the block's own last layers, so the loads issued past the
  // end of the march re-read lines just fetched; their values are not
  // used), in the order that iteration
  // consumes them -- minv (node stage), the output cell's operands (cell
  // stage), x (LDS store) -- so each consumer waits only for its own
  // loads.  With DEPTH 2 two such sets are in flight.
  struct Pre {
    T mvMain, mvEdge;                 // minv of the main and the edge node
    T in[HPT], ap[HPT], s[HPT], dd[HPT];  // raw values of the halo cells
    float e[HPT];
    T eB, eD, eX, eP;                 // operands of the output cell
  };
  auto fetchX = [&](Pre& P, int cz) {
    const long zb = (long)min(max(cz, 0), min(zEnd, d.CZ - 1)) * d.cslab;
#pragma unroll
    for (int h = 0; h < HPT; h++) {
      const long c = zb + hOff[h];
      P.in[h] = a.in[c];
      if (MODE == M_UPDATE) {
        P.ap[h] = a.Ap[c];
        P.s[h] = a.s[c];
        P.dd[h] = a.Dinv[c];
      } else if (MODE == M_IR_RESID) {
        P.e[h] = a.e32 ? a.e32[c] : 0.0f;
      } else if (MODE == M_PCG) {
        P.e[h] = a.e32[c];
      }
    }
  };
  // x of layer cz into LDS: the halo values (out-of-grid cells 0)
  auto store = [&](const Pre& P, T* L, int cz) {
    const bool zok = cz >= 0 && cz < d.CZ;
#pragma unroll
    for (int h = 0; h < HPT; h++) {
      if (h == 0 || threadIdx.x < NRING) {
        T v = P.in[h];
        if (MODE == M_UPDATE) {
          // r_new from r_old, Ap_old and s_old, on the halo as well (the
          // owner writes it with the cell's other updates)
          const T apn = P.ap[h] * beta + P.s[h];
          const T qq = apn * P.dd[h];
          v = P.in[h] - alpha * qq;
        } else if (MODE == M_IR_RESID) {
          // x_old (+ e); the owner writes x_new to the other buffer
          if (a.e32) v = v + (T)P.e[h];
        } else if (MODE == M_PCG) {
          // p = z + beta p (the first iteration's previous p is not read as
          // a number: its buffer may hold anything)
          v = a.dir.iter > 0 ? (T)P.e[h] + beta * P.in[h] : (T)P.e[h];
        }
        L[hIdx[h]] = zok && hVal[h] ? v : (T)0;
      }
    }
  };
  // M_UPDATE: the own cell's Ap_new = beta Ap + s, 1/D and r_old, taken from
  // its halo slot as each layer enters LDS and kept for three layers, until
  // the cell stage of that layer (the slot after every store, so the third
  // set is always the output layer's)
  T oAp0 = 0, oAp1 = 0, oAp2 = 0, oD0 = 0, oD1 = 0, oD2 = 0, oR0 = 0, oR1 = 0, oR2 = 0;
  auto keepOwn = [&](const Pre& P) {
    if (MODE != M_UPDATE) return;
    oAp2 = oAp1;
    oAp1 = oAp0;
    oAp0 = P.ap[0] * beta + P.s[0];
    oD2 = oD1;
    oD1 = oD0;
    oD0 = P.dd[0];
    oR2 = oR1;
    oR1 = oR0;
    oR0 = P.in[0];
  };
  auto fetchMinv = [&](Pre& P, int k) {
    const long kb = (long)max(min(max(k, 1), min(zEnd, d.Z - 2)), 0) * d.slab;
    P.mvMain = a.minv[kb + mOff];
    P.mvEdge = a.minv[kb + eOff];
  };
  auto fetchOut = [&](Pre& P, int cz) {
    const long c = (long)min(max(cz, 0), zEnd - 1) * d.cslab + cOff;
    if (MODE == M_SETUP_R || MODE == M_CHECK || MODE == M_IR_RESID || MODE == M_PCG_RESID)
      P.eB = a.b[c];
    if (MODE == M_SETUP_R || MODE == M_SETUP_S) P.eD = a.D[c];
    if (MODE == M_UPDATE) {
      P.eX = a.x[c];
      P.eP = a.p[c];
    }
  };
  // what iteration k consumes: minv of node layer k, the operands of output
  // cell layer k - 2, x of layer k + 1
  auto issue = [&](Pre& P, int k) {
    fetchMinv(P, k);
    if (MODE != M_APPLY) fetchOut(P, k - 2);
    fetchX(P, k + 1);
  };

  // a node's additions over its adjacent cells, in ascending cell index
  // (dz, dy, dx): lowerSums adds the four of the lower layer to zero,
  // nodeW the four of the upper layer, then scales by minv
  auto lowerSums = [&](const T (&lo)[4], T& m0, T& m1, T& m2) {
    m0 = 0;
    m1 = 0;
    m2 = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const T v = lo[q];
      m0 += (q & 1) == 0 ? v : -v;
      m1 += (q >> 1) == 0 ? v : -v;
      m2 += v;
    }
  };
  auto nodeW = [&](T m0, T m1, T m2, const T (&hi)[4], T mi, bool interior, T* W) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const T v = hi[q];
      m0 += (q & 1) == 0 ? v : -v;
      m1 += (q >> 1) == 0 ? v : -v;
      m2 += -v;
    }
    W[0] = interior ? m0 * mi : (T)0;
    W[1] = interior ? m1 * mi : (T)0;
    W[2] = interior ? m2 * mi : (T)0;
  };
  // a cell's additions over four corner nodes of one layer (oz), in
  // ascending node index (oy, ox)
  auto cornerSums = [&](T acc, const T (&wc)[12], int oz) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const T* W = &wc[3 * q];
      acc += (q & 1) ? W[0] : -W[0];
      acc += (q >> 1) ? W[1] : -W[1];
      acc += oz ? W[2] : -W[2];
    }
    return acc;
  };

  T ml0, ml1, ml2;   // main node: sums over its lower-layer cells
  T accLo = 0;       // output cell: sum over its lower-layer corners
  T own0 = 0, own1 = 0, own2 = 0;  // own input of cell layers k, k - 1, k - 2
  // LDS buffer offsets: x of layers k - 1, k, k + 1; w of layers k, k - 1
  int bLo = 0, bHi = HALO, bNx = 2 * HALO;
  int wCur = 0, wPrev = 3 * NODES;

  // one iteration of the march (k: node layer), consuming the loads in P
  // and refilling it for iteration k + DEPTH
  auto step = [&](int k, Pre& P) {
    T up0 = 0;
    if (k <= zEnd) {
      const bool kin = k >= 1 && k <= d.Z - 2;
      const T* Lhi = xs + bHi;
      T hi[4];
      hi[0] = Lhi[mHalo];
      hi[1] = Lhi[mHalo + 1];
      hi[2] = Lhi[mHalo + TX + 2];
      hi[3] = Lhi[mHalo + TX + 3];
      nodeW(ml0, ml1, ml2, hi, P.mvMain, mainIJ && kin, ws + wCur + mW);
      lowerSums(hi, ml0, ml1, ml2);
      up0 = hi[0];
      if (hasEdge) {
        const T* Llo = xs + bLo;
        T elo[4], ehi[4];
        elo[0] = Llo[eHalo];
        elo[1] = Llo[eHalo + 1];
        elo[2] = Llo[eHalo + TX + 2];
        elo[3] = Llo[eHalo + TX + 3];
        ehi[0] = Lhi[eHalo];
        ehi[1] = Lhi[eHalo + 1];
        ehi[2] = Lhi[eHalo + TX + 2];
        ehi[3] = Lhi[eHalo + TX + 3];
        T e0, e1, e2;
        lowerSums(elo, e0, e1, e2);
        nodeW(e0, e1, e2, ehi, P.mvEdge, edgeIJ && kin, ws + wCur + eW);
      }
    }
    own2 = own1;
    own1 = own0;
    own0 = up0;
    if (k >= z0 + 1) {
      // node layer k - 1: the upper corners of cell layer k - 2, the lower
      // corners of cell layer k - 1
      const T* W = ws + wPrev + cW;
      T wu[12];
#pragma unroll
      for (int c = 0; c < 3; c++) {
        wu[c] = W[c];
        wu[3 + c] = W[3 + c];
        wu[6 + c] = W[3 * (TX + 1) + c];
        wu[9 + c] = W[3 * (TX + 1) + 3 + c];
      }
      const int cz = k - 2;
      if (cz >= z0 && cz < zEnd) {
        const T acc = cornerSums(accLo, wu, 1);
        // the cell's own input; the CR update forms r_new again from the kept
        // operands, by the expression that stored it in LDS
        const T ownIn = MODE == M_UPDATE ? oR2 - alpha * (oAp2 * oD2) : own2;
        const long c = (long)cz * d.cslab + cOff;
        if (cellXY) {
          if (MODE == M_APPLY) {
            a.out[c] = acc;
          } else if (MODE == M_SETUP_R) {
            const T rv = (P.eB - acc) / P.eD;
            a.r[c] = rv;
            a.p[c] = rv;
            part0 += (double)P.eB * (double)P.eB;
          } else if (MODE == M_SETUP_S) {
            a.s[c] = acc;
            a.Ap[c] = acc;
            part0 += (double)ownIn * (double)acc;
            const T q = acc / P.eD;
            part1 += (double)acc * (double)q;
          } else if (MODE == M_UPDATE) {
            // the cell's deferred direction update (Ap, p, x) and its
            // r_new, written to the other buffers, and s = S r_new
            // (Ap_new, 1/D and r_old kept from the halo slot)
            const T apn = oAp2;
            const T pn = P.eP * beta + oR2;
            a.r[c] = ownIn;
            a.ApOut[c] = apn;
            a.p[c] = pn;
            a.x[c] = P.eX + alpha * pn;
            a.sOut[c] = acc;
            const T sq = acc * oD2;
            part0 += (double)ownIn * (double)acc;
            part1 += (double)acc * (double)sq;
            part2 += (double)apn * (double)sq;
            part3 += (double)apn * (double)(apn * oD2);
            // |b - S x| as the recursion carries it (r is D^-1 (b - S x));
            // only the FP32 inner solve tests it
            if (a.recursive) {
              const double rb = (double)ownIn / (double)oD2;
              part4 += rb * rb;
            }
          } else if (MODE == M_CHECK) {
            const T t = acc - P.eB;
            part0 += (double)t * (double)t;
          } else if (MODE == M_IR_RESID) {
            if (a.e32) a.x[c] = ownIn;
            const T rr = P.eB - acc;
            a.r32[c] = (float)rr;
            part0 += (double)rr * (double)rr;
            part1 += (double)P.eB * (double)P.eB;
          } else if (MODE == M_PCG) {
            a.p[c] = ownIn;
            a.out[c] = acc;
            part0 += (double)ownIn * (double)acc;
          } else if (MODE == M_PCG_RESID) {
            const T rr = P.eB - acc;
            a.r[c] = rr;
            a.r32[(long)cz * a.pxy + cy * a.px + cx] = (float)rr;
            part0 += (double)rr * (double)rr;
            part1 += (double)P.eB * (double)P.eB;
          }
        }
      }
      accLo = cornerSums((T)0, wu, 0);
    }
    if (k + 1 <= zEnd) store(P, xs + bNx, k + 1);
    keepOwn(P);
    issue(P, k + DEPTH);
    // rotate the LDS buffers
    const int b = bLo;
    bLo = bHi;
    bHi = bNx;
    bNx = b;
    const int w = wCur;
    wCur = wPrev;
    wPrev = w;
    __syncthreads();
  };

  Pre P[DEPTH];
  fetchX(P[0], z0 - 1);
  store(P[0], xs + bLo, z0 - 1);
  keepOwn(P[0]);
  fetchX(P[0], z0);
  store(P[0], xs + bHi, z0);
  keepOwn(P[0]);
#pragma unroll
  for (int j = 0; j < DEPTH; j++) issue(P[j], z0 + j);
  __syncthreads();
  {
    T lo[4];
    lo[0] = xs[bLo + mHalo];
    lo[1] = xs[bLo + mHalo + 1];
    lo[2] = xs[bLo + mHalo + TX + 2];
    lo[3] = xs[bLo + mHalo + TX + 3];
    lowerSums(lo, ml0, ml1, ml2);
  }
  // layers z0 - 1 .. zEnd pass through: node layers z0 .. zEnd, cell
  // layers z0 .. zEnd - 1 (two iterations behind).  The march runs in
  // groups of DEPTH iterations, one load set each (trailing iterations past
  // zEnd + 1 do nothing but load).
  if (DEPTH == 1) {
    for (int k = z0; k <= zEnd + 1; k++) step(k, P[0]);
  } else {
    for (int k = z0; k <= zEnd + 1; k += DEPTH) {
#pragma unroll
      for (int j = 0; j < DEPTH; j++) step(k + j, P[j]);
    }
  }
  if (MODE == M_APPLY) return;
  if (MODE == M_UPDATE) {
    double mine[5] = {part0, part1, part2, part3, part4};
    blockPartialsAt<5>(mine, a.partials, red, wg.blocks(), wg.block());
  } else if (MODE == M_PCG) {
    double mine[1] = {part0};
    blockPartialsAt<1>(mine, a.partials, red, wg.blocks(), wg.block());
  } else {
    double mine[2] = {part0, part1};
    blockPartialsAt<2>(mine, a.partials, red, wg.blocks(), wg.block());
  }
}
ESF_BOUNDS(kSpmv, 256);

// The same products and updates for grids of few tiles, where the march above
// is a chain of load latencies (33^3: 10 layers of it, 11.5 us, for 36 000
// cells): a block owns FX x FY x FZ cells, issues every load it needs at once,
// and runs the stages through LDS with one barrier each.  The halo makes it
// load each operand 2.1 times, so past kFlatBlocks tiles the march is ahead.
// The sums over cells and nodes keep the march's order.
// The CR update also takes over its finisher: the first thing it needs is the
// totals of the iteration before, which every block adds up itself from the
// (double-buffered) partials, in one order, instead of a one-block kernel
// between the updates (3.7 us).
constexpr int FX = 16, FY = 8, FZ = 4;
constexpr int FHX = FX + 2, FHY = FY + 2, FHZ = FZ + 2, FHALO = FHX * FHY * FHZ;
constexpr int FNX = FX + 1, FNY = FY + 1, FNZ = FZ + 1, FNODES = FNX * FNY * FNZ;
constexpr int FCELLS = FX * FY * FZ;

// The true-residual check of an iterate may ride beside the next update, in
// blocks of its own (M_UPDATE_CHECK), and a later update finds the verdict: no
// launch of the check's and of its finisher's (8.5 us at 33^3, every fifth
// iteration) stands in the chain.
template <int MODE, int FT, class GridT>
__device__ __forceinline__ void spmvFlat(const GridT& wg, const Dims& d, const SpmvArgs<double>& a,
                                         int tilesX, int tilesY, double* xs, double (*ws)[FNODES],
                                         double (*os)[FCELLS], double* red, int* flag) {
  constexpr int FHPT = (FHALO + FT - 1) / FT, FNPT = (FNODES + FT - 1) / FT, FCPT = FCELLS / FT;
  bool done = a.sc && a.sc->done;  // looked at once the loads are out
  const int tile = wg.block();
  const int x0 = FX * (tile % tilesX), y0 = FY * ((tile / tilesX) % tilesY),
            z0 = FZ * (tile / (tilesX * tilesY));
  const double* in = MODE == M_CHECK ? a.x : a.in;

  // every load of the block, addresses clamped into the grid
  double hin[FHPT], hap[FHPT], hs[FHPT], hd[FHPT];
  float he[FHPT];
#pragma unroll
  for (int u = 0; u < FHPT; u++) {
    const int h = threadIdx.x + FT * u;
    const int hx = h % FHX, hy = (h / FHX) % FHY, hz = h / (FHX * FHY);
    const int gx = min(max(x0 + hx - 1, 0), d.CX - 1), gy = min(max(y0 + hy - 1, 0), d.CY - 1),
              gz = min(max(z0 + hz - 1, 0), d.CZ - 1);
    const long c = gx + (long)gy * d.CX + gz * d.cslab;
    hin[u] = in[c];
    if (MODE == M_UPDATE) {
      hap[u] = a.Ap[c];
      hs[u] = a.s[c];
      hd[u] = a.Dinv[c];
    }
    if (MODE == M_PCG) he[u] = a.e32[c];
  }
  double mi[FNPT];
#pragma unroll
  for (int u = 0; u < FNPT; u++) {
    const int n = threadIdx.x + FT * u;
    const int i = x0 + n % FNX, j = y0 + (n / FNX) % FNY, k = z0 + n / (FNX * FNY);
    mi[u] = a.minv[min(max(i, 1), d.X - 2) + (long)min(max(j, 1), d.Y - 2) * d.X +
                   min(max(k, 1), d.Z - 2) * d.slab];
  }
  long oc[FCPT];
  bool own[FCPT];
  double oB[FCPT], oX[FCPT], oP[FCPT];
#pragma unroll
  for (int u = 0; u < FCPT; u++) {
    const int t = threadIdx.x + FT * u;
    const int cx = x0 + t % FX, cy = y0 + (t / FX) % FY, cz = z0 + t / (FX * FY);
    own[u] = cx < d.CX && cy < d.CY && cz < d.CZ;
    oc[u] = min(cx, d.CX - 1) + (long)min(cy, d.CY - 1) * d.CX + min(cz, d.CZ - 1) * d.cslab;
    if (MODE == M_CHECK || MODE == M_PCG_RESID) oB[u] = a.b[oc[u]];
    if (MODE == M_UPDATE) {
      oX[u] = a.x[oc[u]];
      oP[u] = a.p[oc[u]];
    }
  }

  const double deltaOld = MODE == M_UPDATE ? a.delta[(a.iter + 1) & 1] : 0.0;
  asm volatile("" ::: "memory");
  // (a launch that finds a verdict may set the flag while its blocks read it)
  if (MODE == M_UPDATE && a.verdict >= 0) done = blockDone(done, flag);
  if (done) return;

  double alpha = 0, beta = 0;
  if (MODE == M_UPDATE) {
    // r.s, s.D^-1 s, Ap.D^-1 s, Ap.D^-1 Ap of the iteration before: kFinish's
    // F_CR; the setup's finisher left the first iteration's in the block
    double dNew = a.sc->delta;
    if (a.verdict >= 0) {
      // kFinish's F_CHECK, by every block
      const double rn = sqrt(blockTotal<FT>(wg.blocks(), a.partials, red));
      const bool conv = rn < a.sc->eps * a.sc->bnorm;
      if (wg.block() == 0 && threadIdx.x == 0) {
        a.sc->resnorm = rn;
        if (conv) {
          a.sc->iter = a.verdict;
          a.sc->done = 1;
        }
        if (a.hostOut) *a.hostOut = *a.sc;
      }
      if (conv) return;
    }
    if (a.iter > 0) {
      const double* parts = a.partials + (1 + ((a.iter + 1) & 1) * 4) * (long)wg.blocks();
      double t[4];
      blockTotals<4, FT>(wg.blocks(), parts, red, t);
      dNew = t[0];
      beta = dNew / deltaOld;
      const double apq = (t[1] + (2.0 * beta) * t[2]) + (beta * beta) * t[3];
      alpha = (fabs(apq) > 0.0) ? dNew / apq : apq;
    } else {
      alpha = a.sc->alpha;
      beta = a.sc->beta;
    }
    if (wg.block() == 0 && threadIdx.x == 0) a.delta[a.iter & 1] = dNew;
  }
  if (MODE == M_PCG) {
    const double rz = blockTotal<FT>(a.dir.nb, a.dir.parts, red);
    const int now = a.dir.iter & 1;
    if (a.dir.iter > 0) beta = rz / a.dir.rz[1 - now];
    if (wg.block() == 0 && threadIdx.x == 0) a.dir.rz[now] = rz;
  }

#pragma unroll
  for (int u = 0; u < FHPT; u++) {
    const int h = threadIdx.x + FT * u;
    if (h < FHALO) {
      const int hx = h % FHX, hy = (h / FHX) % FHY, hz = h / (FHX * FHY);
      const int gx = x0 + hx - 1, gy = y0 + hy - 1, gz = z0 + hz - 1;
      double v = hin[u];
      if (MODE == M_UPDATE) {
        const double apn = hap[u] * beta + hs[u];
        const double qq = apn * hd[u];
        v = hin[u] - alpha * qq;
        // the block's own cells' operands, for the cell stage
        const int lx = hx - 1, ly = hy - 1, lz = hz - 1;
        if (lx >= 0 && lx < FX && ly >= 0 && ly < FY && lz >= 0 && lz < FZ) {
          const int t = lx + FX * (ly + FY * lz);
          os[0][t] = apn;
          os[1][t] = hd[u];
          os[2][t] = hin[u];
        }
      } else if (MODE == M_PCG) {
        v = a.dir.iter > 0 ? (double)he[u] + beta * hin[u] : (double)he[u];
      }
      const bool in = gx >= 0 && gx < d.CX && gy >= 0 && gy < d.CY && gz >= 0 && gz < d.CZ;
      xs[h] = in ? v : 0.0;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < FNPT; u++) {
    const int n = threadIdx.x + FT * u;
    if (n < FNODES) {
      const int nx = n % FNX, ny = (n / FNX) % FNY, nz = n / (FNX * FNY);
      const double* L = xs + nx + FHX * (ny + FHY * nz);
      double m0 = 0, m1 = 0, m2 = 0;
#pragma unroll
      for (int q = 0; q < 8; q++) {
        const double v = L[(q & 1) + FHX * ((q >> 1) & 1) + FHX * FHY * (q >> 2)];
        m0 += (q & 1) == 0 ? v : -v;
        m1 += ((q >> 1) & 1) == 0 ? v : -v;
        m2 += (q >> 2) == 0 ? v : -v;
      }
      const int i = x0 + nx, j = y0 + ny, k = z0 + nz;
      const bool interior =
          i >= 1 && i <= d.X - 2 && j >= 1 && j <= d.Y - 2 && k >= 1 && k <= d.Z - 2;
      ws[0][n] = interior ? m0 * mi[u] : 0.0;
      ws[1][n] = interior ? m1 * mi[u] : 0.0;
      ws[2][n] = interior ? m2 * mi[u] : 0.0;
    }
  }
  __syncthreads();
  double part0 = 0, part1 = 0, part2 = 0, part3 = 0;
#pragma unroll
  for (int u = 0; u < FCPT; u++) {
    const int t = threadIdx.x + FT * u;
    const int lx = t % FX, ly = (t / FX) % FY, lz = t / (FX * FY);
    const int n0 = lx + FNX * (ly + FNY * lz);
    double acc = 0;
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const int n = n0 + (q & 1) + FNX * ((q >> 1) & 1) + FNX * FNY * (q >> 2);
      acc += (q & 1) ? ws[0][n] : -ws[0][n];
      acc += ((q >> 1) & 1) ? ws[1][n] : -ws[1][n];
      acc += (q >> 2) ? ws[2][n] : -ws[2][n];
    }
    if (own[u]) {
      const long c = oc[u];
      const double v = xs[lx + 1 + FHX * (ly + 1 + FHY * (lz + 1))];  // the cell's own input
      if (MODE == M_UPDATE) {
        const double apn = os[0][t], dinv = os[1][t];
        const double pn = oP[u] * beta + os[2][t];
        a.r[c] = v;
        a.ApOut[c] = apn;
        a.p[c] = pn;
        a.xOut[c] = oX[u] + alpha * pn;
        a.sOut[c] = acc;
        const double sq = acc * dinv;
        part0 += v * acc;
        part1 += acc * sq;
        part2 += apn * sq;
        part3 += apn * (apn * dinv);
      } else if (MODE == M_CHECK) {
        const double r = acc - oB[u];
        part0 += r * r;
      } else if (MODE == M_PCG) {
        a.p[c] = v;
        a.out[c] = acc;
        part0 += v * acc;
      } else if (MODE == M_PCG_RESID) {
        const double rr = oB[u] - acc;
        const int cx = x0 + lx, cy = y0 + ly, cz = z0 + lz;
        a.r[c] = rr;
        a.r32[(long)cz * a.pxy + cy * a.px + cx] = (float)rr;
        part0 += rr * rr;
        part1 += oB[u] * oB[u];
      } else {
        a.out[c] = acc;
      }
    }
  }
  if (MODE == M_APPLY) return;
  if (MODE == M_UPDATE) {
    double mine[4] = {part0, part1, part2, part3};
    // (behind a check's set, which is written between two updates)
    blockPartialsAt<4>(mine, a.partials + (1 + (a.iter & 1) * 4) * (long)wg.blocks(), red,
                       wg.blocks(), wg.block());
  } else if (MODE == M_PCG_RESID) {
    double mine[2] = {part0, part1};
    blockPartialsAt<2>(mine, a.partials, red, wg.blocks(), wg.block());
  } else {
    double mine[1] = {part0};
    blockPartialsAt<1>(mine, a.partials, red, wg.blocks(), wg.block());
  }
}

// FT threads a block
template <int MODE, int FT, class GridT>
__device__ __forceinline__ void kSpmvFlat(const GridT& wg, Dims d, SpmvArgs<double> a, int tilesX,
                                          int tilesY) {
  __shared__ double xs[FHALO];
  __shared__ double ws[3][FNODES];
  // M_UPDATE: Ap, 1 / D and the old r of the block's cells
  constexpr bool upd = MODE == M_UPDATE || MODE == M_UPDATE_CHECK;
  __shared__ double os[upd ? 3 : 1][FCELLS];
  __shared__ double red[4 * (FT / 64)];
  __shared__ int flag;
  if constexpr (MODE == M_UPDATE_CHECK) {
    const int nb = wg.blocks() / 2, b = wg.block();
    if (b < nb)
      spmvFlat<M_UPDATE, FT>(SceneGrid{b, nb}, d, a, tilesX, tilesY, xs, ws, os, red, &flag);
    else
      spmvFlat<M_CHECK, FT>(SceneGrid{b - nb, nb}, d, a, tilesX, tilesY, xs, ws, os, red, &flag);
  } else {
    spmvFlat<MODE, FT>(wg, d, a, tilesX, tilesY, xs, ws, os, red, &flag);
  }
}
ESF_BOUNDS(kSpmvFlat, 512);

// b = J v0 - c, c (boundary velocities), D = diag(S); also the FP32 copies
// used by the mixed solve.  COUPLED_INTEGRATOR_3D.cpp:286-325 (c),
// :694-709 (D, b).  D == nullptr: b and c only (the mixed step forms the
// diagonal with kPressureDiag when its inner solve first needs it).
template <class GridT>
__device__ __forceinline__ void kPressureRhs(const GridT& wg, Dims d, const double* __restrict__ v0,
                                             const double* __restrict__ vel,
                                             const double* __restrict__ minv, double* c, double* b,
                                             double* D, double* Dinv, float* D32, float* Dinv32,
                                             CrScalars* sc, double eps) {
  const int r = wg.block() * blockDim.x + threadIdx.x;
  if (sc && r == 0) initScalarBlock(sc, eps);
  if (r >= d.cells) return;
  const int q = r / d.CX, cx = r - q * d.CX, cy = q % d.CY, cz = q / d.CY;
  const long base = cx + (long)cy * d.X + (long)cz * d.slab;
  double tmp = 0, cc = 0, dd = 0;
  for (int k = 0; k < 8; k++) {
    const int ox = k & 1, oy = (k >> 1) & 1, oz = k >> 2;
    const long n = base + ox + (long)oy * d.X + (long)oz * d.slab;
    const int ni = cx + ox, nj = cy + oy, nk = cz + oz;
    const bool interior =
        ni >= 1 && ni <= d.X - 2 && nj >= 1 && nj <= d.Y - 2 && nk >= 1 && nk <= d.Z - 2;
    const double sx = ox ? 1.0 : -1.0, sy = oy ? 1.0 : -1.0, sz = oz ? 1.0 : -1.0;
    if (interior) {
      tmp += sx * v0[3 * n];
      tmp += sy * v0[3 * n + 1];
      tmp += sz * v0[3 * n + 2];
      if (D) {
        const double mi = minv[n];
        dd += mi * 1.0;
        dd += mi * 1.0;
        dd += mi * 1.0;
      }
    } else {
      cc -= sx * vel[3 * n];
      cc -= sy * vel[3 * n + 1];
      cc -= sz * vel[3 * n + 2];
    }
  }
  c[r] = cc;
  b[r] = tmp - cc;
  if (D) {
    D[r] = dd;
    Dinv[r] = 1.0 / dd;
    if (D32) {
      D32[r] = (float)dd;
      Dinv32[r] = (float)(1.0 / dd);
    }
  }
}
ESF_BOUNDS(kPressureRhs, 1024);

// D = diag(S), its reciprocals and their FP32 copies, and minv in FP32, for
// the mixed solve's inner CR: the sums of kPressureRhs in the same order
template <class GridT>
__device__ __forceinline__ void kPressureDiag(const GridT& wg, Dims d,
                                              const double* __restrict__ minv, double* D,
                                              double* Dinv, float* D32, float* Dinv32,
                                              float* minv32) {
  const int t = wg.block() * blockDim.x + threadIdx.x;
  if (t < d.nodes) minv32[t] = (float)minv[t];
  if (t >= d.cells) return;
  const int q = t / d.CX, cx = t - q * d.CX, cy = q % d.CY, cz = q / d.CY;
  const long base = cx + (long)cy * d.X + (long)cz * d.slab;
  double dd = 0;
  for (int k = 0; k < 8; k++) {
    const int ox = k & 1, oy = (k >> 1) & 1, oz = k >> 2;
    const int ni = cx + ox, nj = cy + oy, nk = cz + oz;
    if (ni >= 1 && ni <= d.X - 2 && nj >= 1 && nj <= d.Y - 2 && nk >= 1 && nk <= d.Z - 2) {
      const double mi = minv[base + ox + (long)oy * d.X + (long)oz * d.slab];
      dd += mi * 1.0;
      dd += mi * 1.0;
      dd += mi * 1.0;
    }
  }
  D[t] = dd;
  Dinv[t] = 1.0 / dd;
  D32[t] = (float)dd;
  Dinv32[t] = (float)(1.0 / dd);
}
ESF_BOUNDS(kPressureDiag, 1024);

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// The z-march's launch shape, fixed per context when it is created:
//  - cell layers per block: each block loads two layers of x and forms one
//    node layer beyond the ones it outputs, so deeper blocks waste less,
//    but fewer blocks hide less latency.  The FP64 CR update (the most
//    registers) takes 16 layers, shallower only so that at least 512
//    blocks run; the other launches (the FP32 kernels, the FP64 residual of
//    the refinement, the applies and checks) take at least 1024 blocks.
//    On MI355X at 128^3 that is 8 layers: FP32 update 20.5 vs 22.8 us and
//    refinement residual 23.3 vs 27.9 us against 16, while the FP64 update
//    measured 30.5 at 16 against 32.5 at 8.  ESF_SPMV_LAYERS (4..64)
//    overrides both choices;
//  - how many iterations ahead the loads run (1..3): two sets of loads in
//    flight hide more latency but hold more registers, so the CR update
//    (more operands) keeps one.  ESF_SPMV_DEPTH (1..3) overrides both.
// The overrides are for tuning and tests; they are read at context creation.
static int envInt(const char* name, int lo, int hi) {
  const char* e = getenv(name);
  const int v = e ? atoi(e) : 0;
  return v >= lo && v <= hi ? v : 0;
}

void spmvConfigure(esf_ctx* ctx) {
  const Dims& d = ctx->d;
  const long tilesXY = (long)cdiv(d.CX, TX) * cdiv(d.CY, TY);
  auto layersFor = [&](long minBlocks) {
    int layers = 16;
    while (layers > 4 && tilesXY * cdiv(d.CZ, layers) < minBlocks) layers /= 2;
    return layers;
  };
  const int forcedLayers = envInt("ESF_SPMV_LAYERS", 4, 64);
  ctx->spmvLayers = forcedLayers ? forcedLayers : layersFor(512);
  ctx->spmvLayersWide = forcedLayers ? forcedLayers : layersFor(1024);
  const int forcedDepth = envInt("ESF_SPMV_DEPTH", 1, 3);
  ctx->spmvDepthUpdate = forcedDepth ? forcedDepth : 1;
  ctx->spmvDepthOther = forcedDepth ? forcedDepth : 2;
  // a forced shape of the march is for the march
  ctx->spmvFlat = !forcedLayers && !forcedDepth;
}

// `deep`: the FP64 CR update's shape
static void tileShape(const esf_ctx* ctx, bool deep, int& tx, int& ty, int& tz, int& layers) {
  const Dims& d = ctx->d;
  tx = cdiv(d.CX, TX);
  ty = cdiv(d.CY, TY);
  layers = deep ? ctx->spmvLayers : ctx->spmvLayersWide;
  tz = cdiv(d.CZ, layers);
}

// Tiles up to which the flat kernel is taken, and up to which with 512 threads
// a block (its updates and checks need 9 partials a tile).  Measured, us per
// FP64 CR iteration with its share of the checks: march / flat 256 / flat 512
// threads at 16^3 16.4 / 9.5 / 8.6, 33^3 17.1 / 9.8 / 9.2, 48^3 (216 tiles)
// 16.8 / 10.1 / 9.8, 64^3 (512) 17.6 / 12.7 / 13.6, 80^3 (1000) 24.1 / 21.8 /
// 22.2, 96^3 (1728) 30.0 / 37.4 / -.
// A check beside an update shares its registers: at 33^3 (135 tiles) that is
// the better way (8.8 us per iteration against 9.1), at 48^3 (216) neither, at
// 64^3 the worse (14.3 against 13.2).
constexpr int kFlatBlocks = 1024, kFlatWide = 256, kFlatRide = 160;
static int flatBlocks(const Dims& d) {
  const long nb = (long)cdiv(d.CX, FX) * cdiv(d.CY, FY) * cdiv(d.CZ, FZ);
  return nb <= kFlatBlocks ? (int)nb : 0;
}

template <int MODE>
static esf_status launchFlat(esf_ctx* ctx, int nb, const SpmvArgs<double>& a) {
  const Dims& d = ctx->d;
  const int cls = MODE == M_UPDATE_CHECK ? M_UPDATE : MODE > M_IR_RESID ? -1 : MODE;
  const int blocks = MODE == M_UPDATE_CHECK ? 2 * nb : nb;
  if (nb <= kFlatWide)
    launchTimed<ESF_KT(kSpmvFlat, MODE, 512)>(ctx, cls, dim3(blocks), dim3(512), d, a,
                                              cdiv(d.CX, FX), cdiv(d.CY, FY));
  else
    launchTimed<ESF_KT(kSpmvFlat, MODE, 256)>(ctx, cls, dim3(blocks), dim3(256), d, a,
                                              cdiv(d.CX, FX), cdiv(d.CY, FY));
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) return ESF_OK;
  ctx->err = std::string("kSpmvFlat launch: ") + hipGetErrorString(e);
  return ESF_ERR_DEVICE;
}

template <typename T, int MODE>
esf_status launchSpmv(esf_ctx* ctx, const SpmvArgs<T>& a) {
  int tx, ty, tz, layers;
  // (the FP64 CR update's flat form is crFlat's)
  constexpr bool flat = sizeof(T) == 8 && (MODE == M_CHECK || MODE == M_PCG ||
                                           MODE == M_PCG_RESID || MODE == M_APPLY);
  if constexpr (flat) {
    if (const int nb = ctx->spmvFlat ? flatBlocks(ctx->d) : 0) {
      const esf_status st = launchFlat<MODE>(ctx, nb, a);
      if constexpr (MODE == M_CHECK)
        launchFinish<F_CHECK, 1>(ctx, nb, a.sc, a.iter, 0, nullptr, a.hostOut);
      if constexpr (MODE == M_PCG_RESID)
        launchFinish<F_IR, 2>(ctx, nb, a.sc, 0, a.first, nullptr, a.hostOut);
      return st;
    }
  }
  tileShape(ctx, sizeof(T) == 8 && MODE == M_UPDATE, tx, ty, tz, layers);
  const int nb = tx * ty * tz;
  const int depth = MODE == M_UPDATE ? ctx->spmvDepthUpdate : ctx->spmvDepthOther;
  const int cls = MODE > M_IR_RESID ? -1 : MODE + (sizeof(T) == 4 ? 6 : 0);
  if (depth == 3)
    launchTimed<ESF_KT(kSpmv, T, MODE, 3)>(ctx, cls, dim3(nb), dim3(256), ctx->d, a, tx, ty, tz,
                                           layers);
  else if (depth == 2)
    launchTimed<ESF_KT(kSpmv, T, MODE, 2)>(ctx, cls, dim3(nb), dim3(256), ctx->d, a, tx, ty, tz,
                                           layers);
  else
    launchTimed<ESF_KT(kSpmv, T, MODE, 1)>(ctx, cls, dim3(nb), dim3(256), ctx->d, a, tx, ty, tz,
                                           layers);
  // the grid-wide sums of the mode (kSpmv's epilogue partials)
  if constexpr (MODE == M_SETUP_R) launchFinish<F_BNORM, 1>(ctx, nb, a.sc);
  if constexpr (MODE == M_SETUP_S) launchFinish<F_SETUP_S, 2>(ctx, nb, a.sc);
  if constexpr (MODE == M_UPDATE)
    launchFinish<F_CR, 5>(ctx, nb, a.sc, a.iter, a.recursive, nullptr, a.hostOut);
  if constexpr (MODE == M_CHECK)
    launchFinish<F_CHECK, 1>(ctx, nb, a.sc, a.iter, 0, nullptr, a.hostOut);
  if constexpr (MODE == M_IR_RESID || MODE == M_PCG_RESID)
    launchFinish<F_IR, 2>(ctx, nb, a.sc, 0, a.first, nullptr, a.hostOut);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    ctx->err = std::string("kSpmv launch: ") + hipGetErrorString(e);
    return ESF_ERR_DEVICE;
  }
  return ESF_OK;
}

// the blocks of M_PCG's launch
int spmvPcgBlocks(const esf_ctx* ctx) {
  const int nb = ctx->spmvFlat ? flatBlocks(ctx->d) : 0;
  if (nb) return nb;
  int tx, ty, tz, layers;
  tileShape(ctx, false, tx, ty, tz, layers);
  return tx * ty * tz;
}

// the most blocks a launch takes (the partials buffer's size)
int spmvBlocks(const esf_ctx* ctx) {
  int nb = 2 * flatBlocks(ctx->d);  // two sets of partials
  for (bool deep : {true, false}) {
    int tx, ty, tz, layers;
    tileShape(ctx, deep, tx, ty, tz, layers);
    nb = std::max(nb, tx * ty * tz);
  }
  return nb;
}

// sc (may be null): a scalar block initialised with tolerance eps for the
// solve that follows
esf_status pressureRhs(esf_ctx* ctx, CrScalars* sc, double eps) {
  const Dims& d = ctx->d;
  const bool mixed = ctx->p.precision == ESF_MIXED;
  launch<ESF_K(kPressureRhs)>(ctx, dim3(cdiv(d.cells, 256)), dim3(256), d, ctx->v0, ctx->vel,
                              ctx->minv, ctx->c, ctx->b, ctx->D, ctx->Dinv,
                              mixed ? ctx->D32 : nullptr, ctx->Dinv32, sc, eps);
  ctx->diagPending = false;
  return hipGetLastError() == hipSuccess ? ESF_OK : ESF_ERR_DEVICE;
}

// the mixed step's right-hand side: b and c only.  The diagonal and minv in
// FP32 follow (pressureDiagFlush) only where an inner solve runs, or where
// a caller reads the diagonal.
// It also initialises scalar block `sc` with tolerance eps for the solve
// that follows (null: none).
esf_status pressureRhsDeferDiag(esf_ctx* ctx, CrScalars* sc, double eps) {
  const Dims& d = ctx->d;
  launch<ESF_K(kPressureRhs)>(ctx, dim3(cdiv(d.cells, 256)), dim3(256), d, ctx->v0, ctx->vel,
                              ctx->minv, ctx->c, ctx->b, (double*)nullptr, (double*)nullptr,
                              (float*)nullptr, (float*)nullptr, sc, eps);
  ctx->diagPending = true;
  return hipGetLastError() == hipSuccess ? ESF_OK : ESF_ERR_DEVICE;
}

esf_status pressureDiagFlush(esf_ctx* ctx) {
  if (!ctx->diagPending) return ESF_OK;
  const Dims& d = ctx->d;
  launch<ESF_K(kPressureDiag)>(ctx, dim3(cdiv(std::max(d.nodes, d.cells), 256)), dim3(256), d,
                               (const double*)ctx->minv, ctx->D, ctx->Dinv, ctx->D32,
                               ctx->Dinv32, ctx->minv32);
  ctx->diagPending = false;
  return hipGetLastError() == hipSuccess ? ESF_OK : ESF_ERR_DEVICE;
}

template <class GridT>
__device__ __forceinline__ void kToFloat(const GridT& wg, long n, const double* a, float* b) {
  for (long i = wg.block() * (long)blockDim.x + threadIdx.x; i < n;
       i += (long)wg.blocks() * blockDim.x)
    b[i] = (float)a[i];
}
ESF_BOUNDS(kToFloat, 1024);
// streaming copy of n doubles (calibration of the HBM byte counters and
// the box's copy bandwidth): 16-byte vector loads and stores
template <class GridT>
__device__ __forceinline__ void kCopy(const GridT& wg, long n2, const double2* __restrict__ a,
                                      double2* __restrict__ b) {
  for (long i = wg.block() * (long)blockDim.x + threadIdx.x; i < n2;
       i += (long)wg.blocks() * blockDim.x)
    b[i] = a[i];
}
ESF_BOUNDS(kCopy, 256);

esf_status benchCopy(esf_ctx* ctx, long bytes, int reps, double* avgMs) {
  const long n2 = bytes / 16;
  double2 *a = nullptr, *b = nullptr;
  if (hipMalloc(&a, n2 * 16) != hipSuccess) return ESF_ERR_OOM;
  if (hipMalloc(&b, n2 * 16) != hipSuccess) {
    hipFree(a);
    return ESF_ERR_OOM;
  }
  hipMemsetAsync(a, 0, n2 * 16, ctx->stream);
  const int blocks = 256 * 32;
  launch<ESF_K(kCopy)>(ctx, dim3(blocks), dim3(256), n2, (const double2*)a, b);
  hipEventRecord(ctx->ev[2], ctx->stream);
  for (int i = 0; i < reps; i++)
    launch<ESF_K(kCopy)>(ctx, dim3(blocks), dim3(256), n2, (const double2*)a, b);
  hipEventRecord(ctx->ev[3], ctx->stream);
  hipError_t e = eventSync(ctx, ctx->ev[3]);
  float ms = 0;
  hipEventElapsedTime(&ms, ctx->ev[2], ctx->ev[3]);
  *avgMs = ms / reps;
  hipFree(a);
  hipFree(b);
  return e == hipSuccess ? ESF_OK : ESF_ERR_DEVICE;
}

// back-to-back applies between two events on the context stream: the
// average launch duration of the pressure SpMV on the current masses
esf_status benchPressureApply(esf_ctx* ctx, int fp32, int reps, double* avgMs) {
  const Dims& d = ctx->d;
  if (fp32 && !ctx->minv32) {
    ctx->err = "FP32 apply needs a mixed-precision context";
    return ESF_ERR_INVALID;
  }
  esf_status st = ESF_OK;
  if (fp32)
    launch<ESF_K(kToFloat)>(ctx, dim3(1024), dim3(256), d.nodes, (const double*)ctx->minv,
                            ctx->minv32);
  hipEventRecord(ctx->ev[2], ctx->stream);
  for (int i = 0; i < reps && !st; i++) {
    if (fp32) {
      SpmvArgs<float> a{};
      a.in = ctx->e32;
      a.minv = ctx->minv32;
      a.out = ctx->s32;
      st = launchSpmv<float, M_APPLY>(ctx, a);
    } else {
      SpmvArgs<double> a{};
      a.in = ctx->lambda;
      a.minv = ctx->minv;
      a.out = ctx->s;
      st = launchSpmv<double, M_APPLY>(ctx, a);
    }
  }
  hipEventRecord(ctx->ev[3], ctx->stream);
  if (eventSync(ctx, ctx->ev[3]) != hipSuccess) return ESF_ERR_DEVICE;
  float ms = 0;
  hipEventElapsedTime(&ms, ctx->ev[2], ctx->ev[3]);
  *avgMs = reps > 0 ? ms / reps : 0;
  return st;
}

esf_status pressureApplyDevice(esf_ctx* ctx, const double* x, double* y) {
  SpmvArgs<double> a{};
  a.in = x;
  a.minv = ctx->minv;
  a.out = y;
  return launchSpmv<double, M_APPLY>(ctx, a);
}

static esf_status initScalars(esf_ctx* ctx, int which, double eps) {
  initScalarsAsync(ctx, &ctx->sc[which], eps);
  return ESF_OK;
}

// the scalar block a finisher queued into report slot 3, after a
// synchronisation
static esf_status waitSlot3(esf_ctx* ctx, CrScalars* out) {
  ESF_HIP(streamSync(ctx));
  *out = ctx->hostSc[3];
  return ESF_OK;
}

// crSolve's loop on the flat kernel, after the set-up.  The verdict of a check
// (every 5 iterations, CONJUGATE_RESIDUAL.inl:166-176) is found by the update
// behind it, which leaves x alone when it passes.  On up to kFlatRide tiles the
// check of iterate c rides beside update c + 1, which then writes x to the
// other of the two lambda buffers (the other updates work in place), and
// update c + 2 finds the verdict; on more it is a launch of its own before
// update c + 1.  ctx->lambda is the accepted iterate's buffer on return.
static esf_status crFlat(esf_ctx* ctx, int which, SpmvArgs<double> a, double* rA, double* rB,
                         double* sA, double* sB, double* apA, double* apB, double* x, int maxIt,
                         int slot, DonePoller& poll) {
  const int nb = flatBlocks(ctx->d);
  const bool ride = nb <= kFlatRide;
  const int behind = ride ? 2 : 1;  // updates from an iterate to its verdict
  double* xs[2] = {x, ctx->lambda2};
  esf_status st = ESF_OK;
  auto checked = [](int i) { return i > 0 && i % 5 == 0; };
  auto check = [&](int i, double* xi) {  // the sums alone
    a.iter = i;
    a.in = a.x = xi;
    return launchFlat<M_CHECK>(ctx, nb, a);
  };
  int n = 0;    // updates queued
  int cur = 0;  // the buffer of the iterate after them
  bool done = false;
  while (n < maxIt && !done) {
    const int i = n;
    if (!ride && checked(i - 1) && (st = check(i - 1, xs[cur]))) return st;
    a.iter = i;
    a.in = rA;
    a.r = rB;
    a.s = sA;
    a.sOut = sB;
    a.Ap = apA;
    a.ApOut = apB;
    a.x = xs[cur];
    if (ride && checked(i - 1)) cur ^= 1;
    a.xOut = xs[cur];
    a.verdict = checked(i - behind) ? i - behind : -1;
    a.hostOut = a.verdict >= 0 ? poll.slot() : nullptr;
    st = ride && checked(i - 1) ? launchFlat<M_UPDATE_CHECK>(ctx, nb, a)
                                : launchFlat<M_UPDATE>(ctx, nb, a);
    if (st) return st;
    if (a.verdict >= 0) poll.mark(i);
    std::swap(rA, rB);
    std::swap(sA, sB);
    std::swap(apA, apB);
    n++;
    done = poll.drain(i);
  }
  if (!done) {
    // checks that no later update is there for: of iterate n - 2, made
    // beside the last update, and of the last
    if (ride && checked(n - 2)) launchFinish<F_CHECK, 1>(ctx, nb, a.sc, n - 2);
    if (checked(n - 1)) {
      if ((st = check(n - 1, xs[cur]))) return st;
      launchFinish<F_CHECK, 1>(ctx, nb, a.sc, n - 1);
    }
  }
  ctx->crQueued = n;
  copyScalarsAsync(ctx, &ctx->sc[which], &ctx->hostSc[slot]);
  int accepted = done ? poll.doneIter : -1;
  if (!done) {
    ESF_HIP(streamSync(ctx));
    if (ctx->hostSc[slot].done) accepted = ctx->hostSc[slot].iter;
  }
  // iterate 5 m: the buffer before update 5 m + 1 moved on, m - 1 moves in
  if (ride && accepted >= 0) cur = (accepted / 5 - 1) & 1;
  if (cur) std::swap(ctx->lambda, ctx->lambda2);
  return ESF_OK;
}

// CONJUGATE_RESIDUAL::solvePCR (matrix-free) on S, FP64 or FP32 vectors.
// The update multiplies by Dinv = 1 / D where the reference divides by D
// (JACOBI_PRECONDITIONER.h:35-37): the iterates differ from the
// reference's in rounding, as alpha's evaluation already makes them.
// x is the start vector.  Scalar block `which`.  *iters receives the
// reference's iteration count; *relres the last checked |Sx-b|/|b|.
// recursive = false: the reference's test, the true residual every 5
// iterations (CONJUGATE_RESIDUAL.inl:166-176).  recursive = true (the FP32
// inner solve of the mixed form, whose result the FP64 outer residual
// checks): the finisher of every iteration tests the residual the
// recursion carries, and no check SpMV runs.
template <typename T>
esf_status crSolve(esf_ctx* ctx, int which, const T* minv, const T* b, const T* D,
                   const T* Dinv, T* x, T* r, T* r2, T* p, T* s, T* s2, T* Ap, T* Ap2,
                   double eps, int maxIt, int slot, bool recursive, bool scalarsReady) {
  // scalarsReady: the kernel before the solve initialised scalar block `which`
  esf_status st = scalarsReady ? ESF_OK : initScalars(ctx, which, eps);
  if (st) return st;
  const Dims& d = ctx->d;
  SpmvArgs<T> a{};
  a.minv = minv;
  a.b = b;
  a.D = D;
  a.Dinv = Dinv;
  a.x = x;
  a.r = r;
  a.p = p;
  a.s = s;
  a.Ap = Ap;
  a.sc = &ctx->sc[which];
  a.partials = ctx->partials;
  a.delta = ctx->crDelta;
  T* rA = r;
  T* rB = r2;
  a.in = x;
  a.r = rA;
  if ((st = launchSpmv<T, M_SETUP_R>(ctx, a))) return st;
  a.in = rA;
  if ((st = launchSpmv<T, M_SETUP_S>(ctx, a))) return st;
  // the FP32 inner solve of the mixed form stops when its residual
  // stagnates; a check is waited for once two iterations are queued behind it
  DonePoller poll(ctx, which, sizeof(T) == 4, 2, 4);
  // the recursive solve's finishers test convergence on the device at every
  // iteration (later launches exit at once); the host reads every third of
  // them, since each read leaves the stream idle for some microseconds
  // (measured at 128^3: mixed steps/s 893 reading every one, 914 every
  // third, 909 every fourth, 902 every sixth)
  constexpr int kPollEvery = 3;
  T *sA = s, *sB = s2, *apA = Ap, *apB = Ap2;
  a.recursive = recursive ? 1 : 0;
  // iteration `it`: the fused update and S r, then the buffers swap
  auto update = [&](int it, CrScalars* hostOut) {
    a.iter = it;
    a.in = rA;
    a.r = rB;
    a.s = sA;
    a.sOut = sB;
    a.Ap = apA;
    a.ApOut = apB;
    a.hostOut = hostOut;
    const esf_status e = launchSpmv<T, M_UPDATE>(ctx, a);
    std::swap(rA, rB);
    std::swap(sA, sB);
    std::swap(apA, apB);
    return e;
  };
  int i = 0;
  if constexpr (sizeof(T) == 8) {
    if (ctx->spmvFlat && flatBlocks(ctx->d))
      return crFlat(ctx, which, a, rA, rB, sA, sB, apA, apB, x, maxIt, slot, poll);
  }
  for (; i < maxIt; i++) {
    const bool read = recursive && i % kPollEvery == kPollEvery - 1;
    if ((st = update(i, read ? poll.slot() : nullptr))) return st;
    if (recursive) {
      if (read) poll.mark(i);
    } else if (i > 0 && i % 5 == 0) {
      a.in = x;
      a.hostOut = poll.slot();
      if ((st = launchSpmv<T, M_CHECK>(ctx, a))) return st;
      poll.mark(i);
    }
    if (poll.drain(i)) {
      // a solve that stagnated runs on to `lag` iterations past the check
      // that showed it, however early the host saw that check, so the
      // iterate it leaves does not depend on the timing of the polls (a
      // converged solve's further launches exit at once)
      while (poll.stagnated && i < poll.stopIt && i + 1 < maxIt)
        if ((st = update(++i, nullptr))) return st;
      i++;
      break;
    }
  }
  ctx->crQueued = i;
  // the report is written without waiting; the caller reads report slot
  // `slot` after its next synchronisation
  copyScalarsAsync(ctx, &ctx->sc[which], &ctx->hostSc[slot]);
  return ESF_OK;
}

template esf_status crSolve<double>(esf_ctx*, int, const double*, const double*,
                                    const double*, const double*, double*, double*, double*,
                                    double*, double*, double*, double*, double*, double, int,
                                    int, bool, bool);
template esf_status crSolve<float>(esf_ctx*, int, const float*, const float*, const float*,
                                   const float*, float*, float*, float*, float*, float*,
                                   float*, float*, float*, double, int, int, bool, bool);

// the inner solve's correction zeroed, and its scalar block initialised
template <class GridT>
__device__ __forceinline__ void kZeroF(const GridT& wg, long n, float* a, CrScalars* sc,
                                       double eps) {
  if (wg.block() == 0 && threadIdx.x == 0) initScalarBlock(sc, eps);
  for (long i = wg.block() * (long)blockDim.x + threadIdx.x; i < n;
       i += (long)wg.blocks() * blockDim.x)
    a[i] = 0.0f;
}
ESF_BOUNDS(kZeroF, 1024);

esf_status spmvPcg(esf_ctx* ctx, const double* pOld, const float* z, double* pNew, double* q,
                   CrScalars* sc, const PcgDir& dir, double* parts) {
  SpmvArgs<double> a{};
  a.in = pOld;
  a.e32 = z;
  a.p = pNew;
  a.out = q;
  a.minv = ctx->minv;
  a.sc = sc;
  a.dir = dir;
  a.partials = parts;
  return launchSpmv<double, M_PCG>(ctx, a);
}

// the residual b - S lambda for the iterations of fdSolve, and its norm
// against eps |b| in scalar block 0 (hostOut: that block, pinned)
static esf_status fdResidual(esf_ctx* ctx, int first, CrScalars* hostOut) {
  const FdGeom g = fdGeom(ctx->d);
  SpmvArgs<double> o{};
  o.minv = ctx->minv;
  o.b = ctx->b;
  o.in = ctx->lambda;
  o.r = ctx->r;
  o.r32 = ctx->fd.r32;
  o.px = g.PX;
  o.pxy = g.PX * g.PY;
  o.sc = &ctx->sc[0];
  o.partials = ctx->partials;
  o.first = first;
  o.hostOut = hostOut;
  return launchSpmv<double, M_PCG_RESID>(ctx, o);
}

// Conjugate gradients preconditioned by fast diagonalisation
// (esf_fastdiag.hip) from lambda, whose residual fdResidual has formed.
// *h: scalar block 0 as the last check of the true residual left it (on
// entry: not done, its residual infinite where the host has not looked); *made
// iterations in *rounds starts.  It gives up (h->done == 0) past
// kFdIterations, when the direction breaks down, or when a restart does not
// halve the residual; lambda then holds the last iterate.
static esf_status fdSolve(esf_ctx* ctx, double eps, int maxIt, CrScalars* h, int* made,
                          int* rounds) {
  // A bound on what a solve that does not fall can waste.  Balls of a thousand
  // times the fluid's density take 150-184 iterations to 1e-12 on 24^3, 48^3
  // and 64^3 grids, 1e4 to 1e6 times 211-280 if left to run, where the FP32 CR
  // alone takes 1400-7700 of its own (4-9 ms against 20-113); handed over at
  // 200 they end in 5-9.5 ms, some a fifth sooner and some a third later.
  constexpr int kFdIterations = 200;
  const int most = std::min(maxIt, kFdIterations);
  esf_status st;
  while (!h->done && *made < most) {
    const double before = h->resnorm;
    if (*rounds > 0 && (st = fdResidual(ctx, 0, nullptr))) return st;
    (*rounds)++;
    // as many iterations as the last solve took are queued before the host
    // looks, then one or a few at a time; where the residual passes its test
    // decides the last iteration, however many were queued
    int it = 0, chunk = std::max(1, ctx->fd.last);
    while (*made + it < most) {
      const int upTo = std::min(it + chunk, most - *made);
      for (; it < upTo; it++)
        if ((st = fdIteration(ctx, it, eps))) return st;
      fdTest(ctx, it, eps, &ctx->hostSc[4]);
      SpmvArgs<double> a{};
      a.in = ctx->lambda;
      a.x = ctx->lambda;
      a.minv = ctx->minv;
      a.b = ctx->b;
      a.sc = &ctx->sc[0];
      a.partials = ctx->partials;
      a.hostOut = &ctx->hostSc[3];
      if ((st = launchSpmv<double, M_CHECK>(ctx, a))) return st;
      if ((st = waitSlot3(ctx, h))) return st;  // also completes report slot 4
      // (the recursive residual passes a little below eps: the true one may
      // have passed before)
      if (h->done || ctx->hostSc[4].done) break;
      chunk = it < 8 ? 1 : 4;
    }
    if (ctx->hostSc[4].done == 1) it = ctx->hostSc[4].iter;
    if (it == 0) (*rounds)--;  // queued unseen, and it passed where it stood
    *made += it;
    ctx->fd.last = it;
    if (!(h->resnorm < 0.5 * before)) break;
  }
  return ESF_OK;
}

// Mixed-precision pressure solve: FP32 CR on S (FP32 minv, FP32 vectors,
// FP64 inner products) inside FP64 iterative refinement.  The outer
// residual b - S x, the correction x += e and |r| stay in FP64.
esf_status mixedSolve(esf_ctx* ctx, double eps, int maxIt, int* iters, bool* converged,
                      double* relres, int* refinements, int* innerIters, bool scalarsReady) {
  const Dims& d = ctx->d;
  // scalarsReady: the right-hand side's kernel initialised scalar block 0
  esf_status st = scalarsReady ? ESF_OK : initScalars(ctx, 0, eps);
  if (st) return st;
  SpmvArgs<double> o{};
  o.minv = ctx->minv;
  o.b = ctx->b;
  o.in = ctx->lambda;
  o.x = ctx->lambda2;
  o.r32 = ctx->rhs32;
  o.e32 = nullptr;
  o.sc = &ctx->sc[0];
  o.partials = ctx->partials;
  o.first = 1;
  o.hostOut = &ctx->hostSc[3];
  CrScalars h{};
  int outer = 0, inner = 0;
  bool residual = true;  // form the residual the refinement starts from
  if (ctx->fd.T) {
    if ((st = fdResidual(ctx, 1, &ctx->hostSc[3]))) return st;
    // where the last solve needed iterations this one's are queued unseen
    // (the wait leaves the device idle for some 20 us); a scene at rest, whose
    // solves end here, waits instead, and so does a solve allowed no iteration
    h.resnorm = std::numeric_limits<double>::infinity();
    if ((ctx->fd.last == 0 || maxIt < 1) && (st = waitSlot3(ctx, &h))) return st;
    if (!h.done && (st = fdSolve(ctx, eps, maxIt, &h, &inner, &outer))) return st;
    residual = !h.done && inner < maxIt;
  }
  if (residual) {
    if ((st = launchSpmv<double, M_IR_RESID>(ctx, o))) return st;
    if ((st = waitSlot3(ctx, &h))) return st;
  }
  bool operands = false;
  // refinement rounds: each gains roughly the FP32 solve's attainable
  // reduction (about eps32 * cond on the smooth modes), so an ill-conditioned
  // cold start needs many; the total FP32 iterations stay capped by maxIt
  const int maxOuter = 1000;
  while (!h.done && outer < maxOuter && inner < maxIt) {
    // inner tolerance: ask for the reduction the outer test still needs,
    // with a margin, bounded by what FP32 can deliver.  The residual a
    // converged step leaves sits in the slowly converging modes, and the
    // inner CR's iterations grow with the reduction asked of them, so the
    // margin is shallow: on the 128^3 ball falling from rest, margins
    // 0.9 / 0.7 / 0.5 measured 7.7 / 6.7 / 8.7 FP32 iterations per step over
    // 30 steps (777 / 792 / 772 steps/s), and on the ball thrown at
    // (0.5, -1.4, 0.3) 13209 / 13879 / 15214 (2.42 / 2.30 / 2.10 steps/s);
    // earlier, slower builds measured 0.3 / 0.1 / 0.03 well below 0.5.
    double need = h.resnorm > 0 ? 0.7 * eps * h.bnorm / h.resnorm : 1.0;
    double innerEps = std::min(0.5, std::max(need, ctx->p.inner_eps));
    if (!operands) {
      operands = true;
      // the inner solve's operands: minv in FP32, and the diagonal where
      // the step left it for here
      if (ctx->diagPending) {
        if ((st = pressureDiagFlush(ctx))) return st;
      } else {
        launch<ESF_K(kToFloat)>(ctx, dim3(1024), dim3(256), d.nodes, (const double*)ctx->minv,
                                ctx->minv32);
      }
    }
    launch<ESF_K(kZeroF)>(ctx, dim3(1024), dim3(256), d.cells, ctx->e32, &ctx->sc[1], innerEps);
    if ((st = crSolve<float>(ctx, 1, ctx->minv32, ctx->rhs32, ctx->D32, ctx->Dinv32, ctx->e32,
                             ctx->r32,
                             ctx->r32b, ctx->p32, ctx->s32, ctx->s32b, ctx->Ap32, ctx->Ap32b,
                             innerEps, maxIt - inner, 4, true, true)))
      return st;
    outer++;
    o.e32 = ctx->e32;
    o.first = 0;
    o.in = ctx->lambda;
    o.x = ctx->lambda2;
    if ((st = launchSpmv<double, M_IR_RESID>(ctx, o))) return st;
    std::swap(ctx->lambda, ctx->lambda2);
    if ((st = waitSlot3(ctx, &h))) return st;  // also completes report slot 4
    int it = 0;
    bool conv = false;
    double rr = 0;
    solveReport(ctx->hostSc[4], maxIt - inner, &it, &conv, &rr);
    // an inner solve that stopped on stagnation ran the iterations it queued
    if (!conv) it = ctx->crQueued;
    inner += it;
  }
  *converged = h.done == 1;
  *iters = inner;
  *relres = h.bnorm > 0 ? h.resnorm / h.bnorm : h.resnorm;
  *refinements = outer;
  *innerIters = inner;
  return ESF_OK;
}

}  // namespace esf
