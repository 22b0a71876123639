// esf_sweep.hip -- the solid's fast sweeping on the GPU, bitwise the
// reference's ordered Gauss-Seidel sweeps:
//   computeSDF (DEFOR_SOLID_3D.cpp:216-267): phi = -0.5 on nodes with mass,
//     a large distance elsewhere, the box of the massive nodes widened by the
//     tight border and the extrapolation cells, two rounds of sweepPhi;
//   sweepPhi / solveDistance (:369-454): eight ordered sweeps of the grid
//     Eikonal update over the box;
//   extendVectorField (:566-574): four rounds of sweepVectorField (:521-564),
//     eight sweepOnePass (:457-519) and the box faces copied inwards.
//
// A sweep visits the box in loop order and each node reads the three
// neighbours visited before it along i, j and k (or, for the faces, only
// what the previous loop nest wrote).  A node's new value therefore depends
// only on those three, so the nodes of one plane i' + j' + k' = p (primed:
// positions along the sweep's directions) are independent, and every node
// gets the reference's value by the reference's arithmetic whatever order
// respects the three.  kPencil lets one wave march along i' with 8 x 8 rows
// (j', k'), the waves passing their edge rows on through memory.
// sweepOnePass also carries three flags across the whole pass
// (solvableX/Y/Z: once cleared they stay cleared).  Whether a node clears
// one depends on phi and the mass only, never on the field being swept, so
// a parallel prepass finds, per flag, the first node in loop order that
// clears it (an integer atomic minimum); a node's flag is then "its loop
// position comes before that one".  The four rounds of a pass share its
// flags and coefficients, formed once.
//
// These are host-side stages of the reference's finalize that the step does
// not run; the entry points serve a host integrator that keeps them.
#include <climits>
#include <mutex>

#include "esf_internal.h"

namespace esf {

namespace {

struct SweepBox {
  int X, Y, Z;
  int x0, y0, z0, x1, y1, z1;
};

__device__ __host__ inline long nodeAt(const SweepBox& b, int i, int j, int k) {
  return i + (long)b.X * (j + (long)b.Y * k);
}

// one ordered sweep: n* nodes along each axis from (i0, j0, k0) in steps
// (di, dj, dk), loop order k outer, i inner
struct Sweep {
  int i0, j0, k0, di, dj, dk, ni, nj, nk;
};

// phi -> -0.5 / large, and the extent of the massive nodes
template <class GridT>
__device__ __forceinline__ void kSdfInit(const GridT& wg, long n, int X, int Y,
                                         const double* __restrict__ mass, double large, double* phi,
                                         int* ext) {
  for (long c = wg.block() * (long)blockDim.x + threadIdx.x; c < n;
       c += (long)wg.blocks() * blockDim.x) {
    const bool m = mass[c] > 0;
    phi[c] = m ? -0.5 : large;
    if (m) {
      const int x = (int)(c % X), y = (int)((c / X) % Y), z = (int)(c / ((long)X * Y));
      atomicMin(&ext[0], x);
      atomicMin(&ext[1], y);
      atomicMin(&ext[2], z);
      atomicMax(&ext[3], x);
      atomicMax(&ext[4], y);
      atomicMax(&ext[5], z);
    }
  }
}
ESF_BOUNDS(kSdfInit, 1024);

// solveDistance with its three candidates formed side by side (the sweep's
// time is this chain's latency) and chosen as the reference's loop does; a
// division by 3 is the rounded reciprocal's product corrected by one fused
// step (Markstein: correctly rounded for finite quotients), one by 2 or 1
// exact
__device__ __forceinline__ double solveDistance3(double p, double q, double r, double v) {
  const double d0 = fmin(p, fmin(q, r)), d2 = fmax(p, fmax(q, r));
  const double d1 = p + q + r - d0 - d2;
  const double c0 = d0 * d0 - 1.0, b1 = d1 + d0, c1 = d1 * d1 + c0;
  const double b2 = d2 + b1, c2 = d2 * d2 + c1;
  const double disc2 = b2 * b2 - 3.0 * c2, disc1 = b1 * b1 - 2.0 * c1, disc0 = d0 * d0 - c0;
  constexpr double third = 1.0 / 3.0;
  const double n2 = b2 + sqrt(disc2), q2 = n2 * third;
  double nd = fma(fma(-3.0, q2, n2), third, q2);
  const double nd1 = (b1 + sqrt(disc1)) * 0.5, nd0 = d0 + sqrt(disc0);
  if (disc2 < 0.0 || nd < d2) {
    if (disc1 > 0.0) nd = nd1;
    if (disc1 < 0.0 || nd < d1) {
      if (disc0 > 0.0) nd = nd0;
    }
  }
  return nd < v ? nd : v;
}

// One ordered sweep (phi: sweepPhi, else sweepOnePass) by blocks of 8 x 8
// rows: lane (j, k) of the block's first wave has row j' = 8 J + j,
// k' = 8 K + k of tile (J, K) and updates i' = step - j - k, so the rows
// before it along j' and k' are one step ahead and their values come from
// lanes l - 1 and l - 8.  Row j = 7 (k = 7) hands its values to tile (J + 1,
// K) ((J, K + 1)) in `edge`: each double as two words of 32 bits with a tag
// that only this sweep uses, stored and loaded at device scope, so a reader
// knows a word's value as soon as it sees it and no fence is needed.  A block
// takes its tile by a ticket, in an order in which tiles depend only on
// earlier ones: a tile that waits waits for tiles that are running.
//
// What bounds a sweep is the chain of its planes (i' + j' + k') and the
// tiles' hand-overs, so the updating wave must not wait for memory: the
// second wave reads the rows' old values and operands ahead, the third asks
// for the edge words, both through rings in LDS, and the first only stores.
// (One wave doing all three waits for its stores whenever it looks for an
// edge word: 319 us per sweep of phi over the box of two balls at 96^3
// cells, 160 us this way.  One workgroup walking the planes of the whole box
// with a barrier each took 2 us per plane, 540 us at 64^3 cells, where this
// takes 111 us.)
constexpr int kRows = 8;
constexpr int kRing = 16;
// tickets of the sweeps of one call, and the tags' epoch before them
constexpr int kSweepTickets = 32;

struct SweepSync {
  int* ints;           // epoch, then a ticket per sweep
  unsigned long long* edge;
  int slot;            // this sweep's ticket
};

template <class GridT>
__device__ __forceinline__ void kSweepStart(const GridT& wg, int* ints) {
  const int t = threadIdx.x;
  if (t < kSweepTickets) ints[1 + t] = 0;
  // (a fresh buffer is 0: the epoch steps over tag 0)
  if (t == kSweepTickets) {
    const unsigned e = (unsigned)ints[0] + kSweepTickets;
    ints[0] = (int)(e < (unsigned)kSweepTickets ? (unsigned)kSweepTickets : e);
  }
}
ESF_BOUNDS(kSweepStart, 64);

// a counter in LDS, and everything this wave wrote to LDS before it
__device__ __forceinline__ int ldsCount(const int* c) {
  const int v = __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  asm volatile("" ::: "memory");
  return __builtin_amdgcn_readfirstlane(v);
}
__device__ __forceinline__ void ldsPublish(int* c, int v) {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __hip_atomic_store(c, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// The first word of row `row` at i' of a tile's edge, and the distance between
// its words.  The eight rows are one step apart, so what one step reads (and
// writes) of them shares a slot i' + row: with the field's six words per value
// whole lines move, and the passes of an 80^3-cell call take 5.9 ms where
// [i'][row][q] took 8.1; phi's two words measured 5 % better the plain way.
template <int C>
__device__ __forceinline__ long edgeAt(int i, int row, int ni) {
  if (C == 1) return ((long)i * kRows + row) * 2;
  const int t = i + row, slot = t < ni ? t : ni >= kRows ? t - ni : t % ni;
  return (long)slot * 2 * C * kRows + row;
}
template <int C>
constexpr int kEdgeStep = C == 1 ? 1 : kRows;

template <int C, bool PHI, class GridT>
__device__ __forceinline__ void kPencil(const GridT& wg, SweepBox b, Sweep s,
                                        const double* __restrict__ mass,
                                        const double2* __restrict__ coef, double* f,
                                        SweepSync sync) {
  constexpr int E = PHI ? 2 : 5;  // values per node read ahead: field, mass / alpha, beta
  __shared__ double ring[kRing * E * 64];
  __shared__ double ering[kRing * 16 * C];
  __shared__ int cnt[4];  // steps of the ring filled, of the edges, done; the tile
  const int lane = threadIdx.x & 63;
  const int role = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (threadIdx.x < 3) cnt[threadIdx.x] = 0;
  if (threadIdx.x == 0) cnt[3] = atomicAdd(&sync.ints[1 + sync.slot], 1);
  __syncthreads();
  const int tile = __builtin_amdgcn_readfirstlane(cnt[3]);
  const int nJ = (s.nj + kRows - 1) / kRows, nK = (s.nk + kRows - 1) / kRows;
  if (tile >= nJ * nK) return;
  const unsigned long long tag = (unsigned long long)(unsigned)(sync.ints[0] + sync.slot) << 32;
  const int J = tile % nJ, K = tile / nJ;
  const long strideJ = (long)s.dj * b.X, strideK = (long)s.dk * b.X * b.Y;
  // the edge words, per tile with a next one along j', then along k'
  const long perTile = (long)s.ni * kRows * 2 * C;
  const int fromJ = K * (nJ - 1) + J - 1, fromK = (nJ - 1) * nK + (K - 1) * nJ + J;
  const int steps = s.ni + 2 * (kRows - 1);

  if (role == 2) {
    // edge streams: 0..7 row j' - 1 of lanes (0, k), 8..15 row k' - 1 of lanes
    // (j, 0), from the tile before or, at the box's edge, from the field,
    // where no node of this sweep lies; lane 16 u + stream looks at
    // step u beyond those handed on (four steps a look: eight took longer)
    const int str = lane & 15, u = lane >> 4;
    const bool forJ = str < kRows;
    const int q8 = str & 7, ej = forJ ? 0 : q8, ek = forJ ? q8 : 0;
    const bool mem = forJ ? J == 0 : K == 0;
    const bool row = kRows * J + ej < s.nj && kRows * K + ek < s.nk;
    const int eJ = min(kRows * J + ej, s.nj - 1), eK = min(kRows * K + ek, s.nk - 1);
    const long mAt = nodeAt(b, s.i0, s.j0 + s.dj * eJ, s.k0 + s.dk * eK) -
                     (forJ ? strideJ : strideK);
    const unsigned long long* const in =
        sync.edge + (forJ ? perTile * fromJ : perTile * fromK);
    int p = 0;
    while (p < steps) {
      const int room = ldsCount(&cnt[2]) + kRing - p;
      if (room <= 0) {
        __builtin_amdgcn_s_sleep(1);
        continue;
      }
      const int i = p + u - q8;
      const bool need = row && i >= 0 && i < s.ni;
      unsigned long long w[2 * C];
#pragma unroll
      for (int q = 0; q < 2 * C; q++) w[q] = tag;
      if (need && mem) {
        const long c = mAt + (long)s.di * i;
#pragma unroll
        for (int q = 0; q < C; q++) {
          const double v = f[C * c + q];
          w[2 * q] = tag | (unsigned)__double2loint(v);
          w[2 * q + 1] = tag | (unsigned)__double2hiint(v);
        }
      } else if (need) {
        const unsigned long long* e = in + edgeAt<C>(i, q8, s.ni);
#pragma unroll
        for (int q = 0; q < 2 * C; q++)
          w[q] = __hip_atomic_load(e + q * kEdgeStep<C>, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
      }
      bool ready = true;
#pragma unroll
      for (int q = 0; q < 2 * C; q++) ready = ready && (w[q] >> 32) == (tag >> 32);
      // the leading steps whose 16 streams are all there, as far as the ring
      // has room
      const unsigned long long m = __ballot(ready);
      int n = 0;
      while (n < 4 && ((m >> (16 * n)) & 0xffff) == 0xffff) n++;
      n = min(n, room);
      if (n == 0) continue;
      if (u < n) {
        double* o = ering + (((p + u) & (kRing - 1)) * 16 + str) * C;
#pragma unroll
        for (int q = 0; q < C; q++)
          o[q] = __hiloint2double((int)(unsigned)w[2 * q + 1], (int)(unsigned)w[2 * q]);
      }
      p += n;
      ldsPublish(&cnt[1], p);
    }
    return;
  }

  const int j = lane & 7, k = lane >> 3;
  const int jp = kRows * J + j, kp = kRows * K + k;
  const bool row = jp < s.nj && kp < s.nk;
  const int jc = min(jp, s.nj - 1), kc = min(kp, s.nk - 1);
  const long at = nodeAt(b, s.i0, s.j0 + s.dj * jc, s.k0 + s.dk * kc);

  if (role == 1) {
    const long cAt = ((long)kc * s.nj + jc) * s.ni;  // coef: loop position of the row
    constexpr int G = 4;
    double v[G][E];
    auto fetch = [&](int step) {
#pragma unroll
      for (int u = 0; u < G; u++) {
        const int ic = min(max(step + u - j - k, 0), s.ni - 1);
        const long c = at + (long)s.di * ic;
#pragma unroll
        for (int q = 0; q < C; q++) v[u][q] = f[C * c + q];
        if (PHI) {
          v[u][1] = mass[c];
        } else {
          const double2 ab = coef[cAt + ic];
          v[u][E - 2] = ab.x;
          v[u][E - 1] = ab.y;
        }
      }
    };
    for (int step = 0; step < steps; step += G) {
      // the old values must be read before the first wave overwrites them:
      // it does so only after this group is handed on
      fetch(step);
      while (ldsCount(&cnt[2]) + kRing < step + G) __builtin_amdgcn_s_sleep(1);
#pragma unroll
      for (int u = 0; u < G; u++)
#pragma unroll
        for (int e = 0; e < E; e++)
          ring[(((step + u) & (kRing - 1)) * E + e) * 64 + lane] = v[u][e];
      ldsPublish(&cnt[0], step + G);
    }
    return;
  }

  unsigned long long* const outJ = sync.edge + perTile * (fromJ + 1);
  unsigned long long* const outK = sync.edge + perTile * (fromK + nJ);
  const bool giveJ = j == kRows - 1 && J + 1 < nJ && row;
  const bool giveK = k == kRows - 1 && K + 1 < nK && row;
  double last[C], cur[C];  // the values at i' - 1 and of the last step
#pragma unroll
  for (int q = 0; q < C; q++) {
    last[q] = f[C * (at - s.di) + q];
    cur[q] = 0;
  }
  int have = 0;
  for (int step = 0; step < steps; step++) {
    while (have <= step) have = min(ldsCount(&cnt[0]), ldsCount(&cnt[1]));
    const double* o = ring + (step & (kRing - 1)) * E * 64 + lane;
    const double* e = ering + (step & (kRing - 1)) * 16 * C;
    double own[E], nj[C], nk[C];
#pragma unroll
    for (int q = 0; q < E; q++) own[q] = o[64 * q];
#pragma unroll
    for (int q = 0; q < C; q++) {
      const double ej = e[k * C + q], ek = e[(kRows + j) * C + q];
      const double sj = dppMov<0x111>(cur[q]), sk = __shfl_up(cur[q], kRows, 64);  // row_shr:1
      nj[q] = j == 0 ? ej : sj;
      nk[q] = k == 0 ? ek : sk;
    }
    const int i = step - j - k;
    const bool act = row && i >= 0 && i < s.ni;
    double nv[C];
    if (PHI) {
      nv[0] = own[1] == 0 ? solveDistance3(last[0], nj[0], nk[0], own[0]) : own[0];
    } else {
      const double alpha = own[E - 2], beta = own[E - 1], gamma = 1 - alpha - beta;
      const bool upd = !isnan(alpha);  // else not updated in this pass
#pragma unroll
      for (int q = 0; q < C; q++) {
        const double v = alpha * last[q] + beta * nj[q] + gamma * nk[q];
        nv[q] = upd ? v : own[q];
      }
    }
    if (act) {
      const long c = at + (long)s.di * i;
#pragma unroll
      for (int q = 0; q < C; q++) {
        f[C * c + q] = nv[q];
        last[q] = nv[q];
        cur[q] = nv[q];
      }
      if (giveJ || giveK) {
        unsigned long long* const oJ = outJ + edgeAt<C>(i, k, s.ni);
        unsigned long long* const oK = outK + edgeAt<C>(i, j, s.ni);
#pragma unroll
        for (int q = 0; q < C; q++) {
          const unsigned long long lo = tag | (unsigned)__double2loint(nv[q]);
          const unsigned long long hi = tag | (unsigned)__double2hiint(nv[q]);
          constexpr int d = kEdgeStep<C>;
          if (giveJ) {
            __hip_atomic_store(oJ + 2 * q * d, lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(oJ + (2 * q + 1) * d, hi, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
          }
          if (giveK) {
            __hip_atomic_store(oK + 2 * q * d, lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(oK + (2 * q + 1) * d, hi, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
          }
        }
      }
    }
    ldsPublish(&cnt[2], step + 1);
  }
}
ESF_BOUNDS(kPencil, 192);

// sweepOnePass's per-node decisions, from phi and the mass only:
// returns false where the node is not updated; clear* say whether the node
// clears that flag (it does so before any later axis may skip it)
struct PassNode {
  double dp, dq, dr;
  bool clearX, clearY, clearZ;
};
__device__ inline bool passNode(const SweepBox& b, const Sweep& s, const double* mass,
                                const double* phi, int i, int j, int k, PassNode& o) {
  o.clearX = o.clearY = o.clearZ = false;
  const long c = nodeAt(b, i, j, k);
  if (mass[c] != 0) return false;
  const double pc = phi[c];
  o.dp = pc - phi[nodeAt(b, i - s.di, j, k)];
  const double dpn = pc - phi[nodeAt(b, i + s.di, j, k)];
  o.dq = pc - phi[nodeAt(b, i, j - s.dj, k)];
  const double dqn = pc - phi[nodeAt(b, i, j + s.dj, k)];
  o.dr = pc - phi[nodeAt(b, i, j, k - s.dk)];
  const double drn = pc - phi[nodeAt(b, i, j, k + s.dk)];
  if (o.dp < 0) {
    if (dpn >= 0) return false;
    o.clearX = true;
  }
  if (o.dq < 0) {
    if (dqn >= 0) return false;
    o.clearY = true;
  }
  if (o.dr < 0) {
    if (drn >= 0) return false;
    o.clearZ = true;
  }
  return true;
}

// sweepVectorField's eight passes, all of the same lengths
struct Passes {
  Sweep s[8];
};

// per pass the first node, in loop order, that clears each flag; blocks
// [p per, (p + 1) per) take pass p
template <class GridT>
__device__ __forceinline__ void kPassFlags(const GridT& wg, SweepBox b, Passes ps, int per,
                                           const double* __restrict__ mass,
                                           const double* __restrict__ phi, int* first) {
  const int p = wg.block() / per;
  const Sweep s = ps.s[p];
  const int n = s.ni * s.nj * s.nk;
  int m[3] = {INT_MAX, INT_MAX, INT_MAX};
  for (int t = (wg.block() % per) * blockDim.x + threadIdx.x; t < n; t += per * blockDim.x) {
    const int q = t / s.ni, ip = t - q * s.ni, kp = q / s.nj, jp = q - kp * s.nj;
    PassNode o;
    passNode(b, s, mass, phi, s.i0 + s.di * ip, s.j0 + s.dj * jp, s.k0 + s.dk * kp, o);
    if (o.clearX) m[0] = min(m[0], t);
    if (o.clearY) m[1] = min(m[1], t);
    if (o.clearZ) m[2] = min(m[2], t);
  }
  // one atomic per wave and flag: with one per node the three words' atomics
  // alone took 24 us per pass over a 92^3 box
#pragma unroll
  for (int a = 0; a < 3; a++) {
    for (int off = 32; off; off >>= 1) m[a] = min(m[a], __shfl_xor(m[a], off, 64));
    if ((threadIdx.x & 63) == 0 && m[a] != INT_MAX) atomicMin(&first[3 * p + a], m[a]);
  }
}
ESF_BOUNDS(kPassFlags, 1024);

// every node's coefficients for each pass, from the flags' first clearing
// nodes: alpha and beta where the node is updated, NaN in alpha where it
// is not (indexed by loop position), so the pass reads them together with
// the neighbours' field values in one round of loads
template <class GridT>
__device__ __forceinline__ void kPassCoef(const GridT& wg, SweepBox b, Passes ps, int per,
                                          const double* __restrict__ mass,
                                          const double* __restrict__ phi,
                                          const int* __restrict__ first, double2* coef) {
  const int p = wg.block() / per;
  const Sweep s = ps.s[p];
  const int n = s.ni * s.nj * s.nk;
  coef += (long)p * n;
  const int fx = first[3 * p], fy = first[3 * p + 1], fz = first[3 * p + 2];
  for (int t = (wg.block() % per) * blockDim.x + threadIdx.x; t < n; t += per * blockDim.x) {
    const int q = t / s.ni, ip = t - q * s.ni, kp = q / s.nj, jp = q - kp * s.nj;
    PassNode o;
    double2 ab = make_double2(NAN, 0.0);
    if (passNode(b, s, mass, phi, s.i0 + s.di * ip, s.j0 + s.dj * jp, s.k0 + s.dk * kp, o)) {
      // a flag is cleared from its first clearing node on, that node included
      const double dp = t >= fx ? 0.0 : o.dp;
      const double dq = t >= fy ? 0.0 : o.dq;
      const double dr = t >= fz ? 0.0 : o.dr;
      if (dp + dq + dr < 1e-3) {
        ab = make_double2(0.333, 0.333);
      } else {
        ab = make_double2(dp / (dp + dq + dr), dq / (dp + dq + dr));
      }
    }
    coef[t] = ab;
  }
}
ESF_BOUNDS(kPassCoef, 1024);

// sweepVectorField's face copies, one axis per launch (z, then y, then x):
// each thread copies both faces of its line in the reference's order
template <class GridT>
__device__ __forceinline__ void kFaceCopy(const GridT& wg, SweepBox b, int axis,
                                          const double* __restrict__ mass, double* field) {
  const int lo[3] = {b.x0, b.y0, b.z0}, hi[3] = {b.x1, b.y1, b.z1};
  const int u = axis == 0 ? 1 : 0, w = axis == 2 ? 1 : 2;  // the two other axes
  const long nu = hi[u] - lo[u], nw = hi[w] - lo[w];
  const long t = wg.block() * (long)blockDim.x + threadIdx.x;
  if (t >= nu * nw) return;
  int pos[3];
  pos[u] = lo[u] + (int)(t / nw);
  pos[w] = lo[w] + (int)(t % nw);
  auto copy = [&](int to, int from) {
    pos[axis] = to;
    const long c = nodeAt(b, pos[0], pos[1], pos[2]);
    pos[axis] = from;
    const long f = nodeAt(b, pos[0], pos[1], pos[2]);
    if (mass[c] == 0)
      for (int q = 0; q < 3; q++) field[3 * c + q] = field[3 * f + q];
  };
  copy(lo[axis], lo[axis] + 1);
  copy(hi[axis] - 1, hi[axis] - 2);
}
ESF_BOUNDS(kFaceCopy, 1024);

template <class GridT>
__device__ __forceinline__ void kFillFirst(const GridT& wg, int* first) {
  if (threadIdx.x < 24) first[threadIdx.x] = INT_MAX;
}
ESF_BOUNDS(kFillFirst, 1024);

// a sweep from a to b exclusive (the reference's sweepOnePass bounds)
Sweep passRange(int i0, int i1, int j0, int j1, int k0, int k1) {
  Sweep s;
  s.i0 = i0;
  s.j0 = j0;
  s.k0 = k0;
  s.di = i0 < i1 ? 1 : -1;
  s.dj = j0 < j1 ? 1 : -1;
  s.dk = k0 < k1 ? 1 : -1;
  s.ni = std::max((i1 - i0) * s.di, 0);
  s.nj = std::max((j1 - j0) * s.dj, 0);
  s.nk = std::max((k1 - k0) * s.dk, 0);
  return s;
}

// the context's sweep integers: three first-clear flags of each of the eight
// passes (or the six extent counters of computeSDF), then from kSyncInts on
// the epoch and the tickets of kPencil
constexpr int kSyncInts = 32;
constexpr int kSweepInts = kSyncInts + 1 + kSweepTickets;

// words of kPencil's edge buffer for sweeps of C doubles
long edgeWords(int ni, int nj, int nk, int C) {
  const long nJ = cdiv(nj, kRows), nK = cdiv(nk, kRows);
  return ((nJ - 1) * nK + nJ * (nK - 1)) * ni * kRows * 2 * C;
}
// for the sweeps of a box (its last node along an axis is never one of them)
long edgeWordsOf(const int box[6], int C) {
  return edgeWords(box[3] - box[0] - 1, box[4] - box[1] - 1, box[5] - box[2] - 1, C);
}

int pencils(const Sweep& s) { return cdiv(s.nj, kRows) * cdiv(s.nk, kRows); }

esf_status growEdges(esf_ctx* ctx, long words) {
  esf_status st;
  if (!ctx->swFirst && (st = devAlloc(ctx, &ctx->swFirst, kSweepInts))) return st;
  if (words > ctx->swEdgeCap) {
    if ((st = devAlloc(ctx, &ctx->swEdge, words))) return st;
    ctx->swEdgeCap = words;
  }
  return ESF_OK;
}

esf_status checkBox(esf_ctx* ctx, const int box[6]) {
  const Dims& d = ctx->d;
  const int res[3] = {d.X, d.Y, d.Z};
  for (int a = 0; a < 3; a++)
    if (box[a] < 0 || box[3 + a] > res[a] || box[3 + a] - box[a] < 3) {
      ctx->err = "sweep box must lie in the grid and span at least 3 nodes per axis";
      return ESF_ERR_INVALID;
    }
  return ESF_OK;
}

// one round of sweepPhi; ints, edge: kPencil's (slots 8 round .. 8 round + 7)
esf_status sweepPhiDevice(esf_ctx* ctx, const SweepBox& b, const double* mass, double* phi,
                          int round, int* ints, unsigned long long* edge) {
  for (int s = 0; s < 8; s++) {
    const int dx = (s & 2) ? -1 : 1, dy = (s & 1) ? -1 : 1, dz = (s & 4) ? -1 : 1;
    // ascending from min + 1 to max - 1, descending from max - 2 to min
    Sweep w;
    w.di = dx;
    w.dj = dy;
    w.dk = dz;
    w.i0 = dx > 0 ? b.x0 + 1 : b.x1 - 2;
    w.j0 = dy > 0 ? b.y0 + 1 : b.y1 - 2;
    w.k0 = dz > 0 ? b.z0 + 1 : b.z1 - 2;
    w.ni = b.x1 - b.x0 - 1;
    w.nj = b.y1 - b.y0 - 1;
    w.nk = b.z1 - b.z0 - 1;
    if (w.ni <= 0 || w.nj <= 0 || w.nk <= 0) continue;
    launch<ESF_KT(kPencil, 1, true)>(ctx, dim3(pencils(w)), dim3(192), b, w, mass,
                                     (const double2*)nullptr, phi,
                                     SweepSync{ints, edge, 8 * round + s});
  }
  return hipGetLastError() == hipSuccess ? ESF_OK : ESF_ERR_DEVICE;
}

}  // namespace

esf_status sweepPhiRounds(esf_ctx* ctx, const int box[6], const double* mass, double* phi,
                          int rounds) {
  const Dims& d = ctx->d;
  if (!(box[3] > box[0] && box[4] > box[1] && box[5] > box[2])) return ESF_OK;
  const SweepBox b{d.X, d.Y, d.Z, box[0], box[1], box[2], box[3], box[4], box[5]};
  esf_status st = growEdges(ctx, edgeWordsOf(box, 1));
  if (st) return st;
  int* ints = ctx->swFirst + kSyncInts;
  for (int r = 0; r < rounds; r++) {
    const int slots = kSweepTickets / 8;
    if (r % slots == 0) launch<ESF_K(kSweepStart)>(ctx, dim3(1), dim3(64), ints);
    if ((st = sweepPhiDevice(ctx, b, mass, phi, r % slots, ints, ctx->swEdge))) return st;
  }
  return ESF_OK;
}

// extendVectorField (:566-574) on device fields; the passes' flags and
// coefficients in the context's scratch (grown with the box)
esf_status extendDevice(esf_ctx* ctx, const int box[6], const double* m, const double* ph,
                        double* f) {
  esf_status st = checkBox(ctx, box);
  if (st) return st;
  const Dims& d = ctx->d;
  // nodes of a pass: the box without its faces
  const long cells =
      (long)(box[3] - box[0] - 2) * (box[4] - box[1] - 2) * (box[5] - box[2] - 2);
  if ((st = growEdges(ctx, edgeWordsOf(box, 3)))) return st;
  if ((size_t)(8 * cells) > ctx->swCoefCap) {
    if ((st = devAlloc(ctx, &ctx->swCoef, 8 * cells))) return st;
    ctx->swCoefCap = 8 * cells;
  }
  const SweepBox b{d.X, d.Y, d.Z, box[0], box[1], box[2], box[3], box[4], box[5]};
  int* first = ctx->swFirst;
  int* ints = first + kSyncInts;
  const int x0 = b.x0, y0 = b.y0, z0 = b.z0, x1 = b.x1, y1 = b.y1, z1 = b.z1;
  // sweepVectorField's eight passes (:524-545)
  const Passes passes = {{
      passRange(x0 + 1, x1 - 1, y0 + 1, y1 - 1, z0 + 1, z1 - 1),
      passRange(x0 + 1, x1 - 1, y1 - 2, y0, z0 + 1, z1 - 1),
      passRange(x1 - 2, x0, y0 + 1, y1 - 1, z0 + 1, z1 - 1),
      passRange(x1 - 2, x0, y1 - 2, y0, z0 + 1, z1 - 1),
      passRange(x0 + 1, x1 - 1, y0 + 1, y1 - 1, z1 - 2, z0),
      passRange(x0 + 1, x1 - 1, y1 - 2, y0, z1 - 2, z0),
      passRange(x1 - 2, x0, y0 + 1, y1 - 1, z1 - 2, z0),
      passRange(x1 - 2, x0, y1 - 2, y0, z1 - 2, z0)}};
  // the flags and coefficients depend on phi and the mass, the same in all
  // four rounds
  launch<ESF_K(kFillFirst)>(ctx, dim3(1), dim3(64), first);
  const int per = std::min(cdiv(cells, 256), 256);
  launch<ESF_K(kPassFlags)>(ctx, dim3(8 * per), dim3(256), b, passes, per, m, ph, first);
  launch<ESF_K(kPassCoef)>(ctx, dim3(8 * per), dim3(256), b, passes, per, m, ph,
                           (const int*)first, ctx->swCoef);
  launch<ESF_K(kSweepStart)>(ctx, dim3(1), dim3(64), ints);
  for (int round = 0; round < 4; round++) {
    for (int p = 0; p < 8; p++)
      launch<ESF_KT(kPencil, 3, false)>(ctx, dim3(pencils(passes.s[p])), dim3(192), b, passes.s[p],
                                        m, (const double2*)(ctx->swCoef + p * cells), f,
                                        SweepSync{ints, ctx->swEdge, 8 * round + p});
    // the faces: z (:547-552), y (:554-558), x (:560-564)
    const long lines[3] = {(long)(y1 - y0) * (z1 - z0), (long)(x1 - x0) * (z1 - z0),
                           (long)(x1 - x0) * (y1 - y0)};
    for (int axis : {2, 1, 0})
      launch<ESF_K(kFaceCopy)>(ctx, dim3(cdiv(lines[axis], 256)), dim3(256), b, axis, m, f);
  }
  return hipGetLastError() == hipSuccess ? ESF_OK : ESF_ERR_DEVICE;
}

// the host-array entry points' device staging, allocated once per context
esf_status sweepStaging(esf_ctx* ctx) {
  const long n = ctx->d.nodes;
  esf_status st = ESF_OK;
  if (!ctx->swMass && (st = devAlloc(ctx, &ctx->swMass, n))) return st;
  if (!ctx->swPhi && (st = devAlloc(ctx, &ctx->swPhi, n))) return st;
  if (!ctx->swField && (st = devAlloc(ctx, &ctx->swField, 3 * n))) return st;
  if (!ctx->swFirst && (st = devAlloc(ctx, &ctx->swFirst, kSweepInts))) return st;
  return st;
}

}  // namespace esf

using namespace esf;

// The allocation-free computeSDF's device memory (esf_compute_sdf_noalloc):
// one array per GPU, resident while the process lives.  [0, 64) doubles hold
// the extent counters and kPencil's integers, then the mass and phi of up to
// kSdfScratchNodes nodes (the (128 + 1)^3 nodes of a 128^3-cell grid) and
// kPencil's edge words for any box of such a grid, 45.5 MB in all.  Host code
// never passes `scratch` itself to a kernel or a copy (on the host the name
// is only a stand-in): it uses the device address hipGetSymbolAddress
// returns, looked up once per device.
constexpr long kSdfScratchNodes = 129L * 129 * 129;
// kPencil's words: at most 0.64 per node over all shapes (rows of 9 x 9)
constexpr long kSdfScratchEdges = kSdfScratchNodes * 13 / 20;
constexpr long kSdfScratchHead = 64;  // doubles
static_assert(2 * kSdfScratchHead >= kSweepInts, "the integers fit the head");
constexpr long kSdfScratchDoubles = kSdfScratchHead + 2 * kSdfScratchNodes + kSdfScratchEdges;
static __device__ __align__(256) double scratch[kSdfScratchDoubles];

namespace esf {
namespace {

// the extent counters start at (X, Y, Z, 0, 0, 0), kPencil's tickets at 0:
// written by a kernel, so the call works from memory the host cannot address
template <class GridT>
__device__ __forceinline__ void kExtInit(const GridT& wg, int* ext, int X, int Y, int Z) {
  if (threadIdx.x < 6) ext[threadIdx.x] = threadIdx.x == 0 ? X : threadIdx.x == 1 ? Y
                                          : threadIdx.x == 2 ? Z : 0;
  kSweepStart(wg, ext + kSyncInts);
}
ESF_BOUNDS(kExtInit, 1024);

// computeSDF on the device buffers dm (the mass, n doubles), dphi (n
// doubles), dext (kSweepInts ints) and edge (kPencil's words for the grid;
// null: the context's, grown to the box), all the caller's: boxes to the
// host, phi back
esf_status computeSdfOn(esf_ctx* ctx, const double* mass, double* phi, int box[6], int tight[6],
                        double* dm, double* dphi, int* dext, unsigned long long* edge) {
  const Dims& d = ctx->d;
  const long n = d.nodes;
  // (the entry point that allocates nothing leaves the pinned slots alone too)
  const bool noalloc = edge != nullptr;
  ESF_HIP(hipMemcpyAsync(dm, mass, 8 * n, hipMemcpyHostToDevice, ctx->stream));
  launch<ESF_K(kExtInit)>(ctx, dim3(1), dim3(64), dext, d.X, d.Y, d.Z);
  launch<ESF_K(kSdfInit)>(ctx, dim3(std::min<long>(cdiv(n, 256), 4096)), dim3(256), n, d.X, d.Y,
                          (const double*)dm, (double)(d.X + d.Y + d.Z + 2), dphi, dext);
  int ext[6];
  ESF_HIP(hipMemcpyAsync(ext, dext, sizeof(ext), hipMemcpyDeviceToHost, ctx->stream));
  ESF_HIP(streamSync(ctx));
  const int res[3] = {d.X, d.Y, d.Z};
  const int tb = ctx->p.tight_border, ex = ctx->p.extrapolation_cells;
  for (int a = 0; a < 3; a++) {
    tight[a] = std::max(ext[a] - tb, 0);
    tight[3 + a] = std::min(ext[3 + a] + tb, res[a]);
    box[a] = std::max(ext[a] - ex, 0);
    box[3 + a] = std::min(ext[3 + a] + ex, res[a]);
  }
  // no node with mass: the box is empty and the reference's loops run empty
  const bool sweep = box[3] > box[0] && box[4] > box[1] && box[5] > box[2];
  if (sweep) {
    const SweepBox b{d.X, d.Y, d.Z, box[0], box[1], box[2], box[3], box[4], box[5]};
    esf_status st;
    if (edge && edgeWordsOf(box, 1) > kSdfScratchEdges) return ESF_ERR_INVALID;
    if (!edge) {
      if ((st = growEdges(ctx, edgeWordsOf(box, 1)))) return st;
      edge = ctx->swEdge;
    }
    for (int r = 0; r < 2; r++)
      if ((st = sweepPhiDevice(ctx, b, dm, dphi, r, dext + kSyncInts, edge))) return st;
  }
  if (!noalloc) return copyToHost(ctx, phi, dphi, 8 * n);
  ESF_HIP(hipMemcpyAsync(phi, dphi, 8 * n, hipMemcpyDeviceToHost, ctx->stream));
  ESF_HIP(streamSync(ctx));
  return ESF_OK;
}

constexpr int kScratchDevices = 64;
std::mutex gScratchLock;
double* gScratch[kScratchDevices] = {};
// held by a call while it uses a device's array: tiles of a running sweep wait
// for words with the epoch they started under, so a second call that reset the
// tickets and the epoch beneath them would have them wait for good
std::mutex gScratchUse[kScratchDevices];

// the scratch array's address on device `dev`, looked up with that device
// current on the first call there
esf_status scratchOn(esf_ctx* ctx, int dev, double** out) {
  if (dev < 0 || dev >= kScratchDevices) {
    ctx->err = "device ordinal out of range for the scratch table";
    return ESF_ERR_INVALID;
  }
  std::lock_guard<std::mutex> lock(gScratchLock);
  if (!gScratch[dev]) {
    int cur = 0;
    ESF_HIP(hipGetDevice(&cur));
    if (cur != dev) ESF_HIP(hipSetDevice(dev));
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    const hipError_t back = cur != dev ? hipSetDevice(cur) : hipSuccess;
    if (back != hipSuccess) {
      ctx->err = std::string("hipSetDevice back to the caller's device: ") +
                 hipGetErrorString(back);
      return ESF_ERR_DEVICE;
    }
    if (e != hipSuccess || !p) {
      ctx->err = std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
      return ESF_ERR_DEVICE;
    }
    gScratch[dev] = (double*)p;
  }
  *out = gScratch[dev];
  return ESF_OK;
}

}  // namespace
}  // namespace esf

esf_status esf_compute_sdf(esf_ctx* ctx, const double* mass, double* phi, int box[6],
                           int tight[6]) {
  if (!ctx || !mass || !phi || !box || !tight) return ESF_ERR_INVALID;
  // staging held by the context (allocated on the first call)
  esf_status st = sweepStaging(ctx);
  if (st) return st;
  return computeSdfOn(ctx, mass, phi, box, tight, ctx->swMass, ctx->swPhi, ctx->swFirst,
                      nullptr);
}

esf_status esf_compute_sdf_noalloc(esf_ctx* ctx, const double* mass, double* phi, int box[6],
                                   int tight[6]) {
  if (!ctx || !mass || !phi || !box || !tight) return ESF_ERR_INVALID;
  if (ctx->d.nodes > kSdfScratchNodes) {
    ctx->err = "compute_sdf_noalloc: the grid has " + std::to_string(ctx->d.nodes) +
               " nodes, more than the " + std::to_string(kSdfScratchNodes) +
               " its scratch holds";
    return ESF_ERR_INVALID;
  }
  double* base = nullptr;
  esf_status st = scratchOn(ctx, ctx->device, &base);
  if (st) return st;
  double* const dm = base + kSdfScratchHead;
  std::lock_guard<std::mutex> use(gScratchUse[ctx->device]);
  st = computeSdfOn(ctx, mass, phi, box, tight, dm, dm + kSdfScratchNodes, (int*)base,
                    (unsigned long long*)(dm + 2 * kSdfScratchNodes));
  // (a call that fails may have left sweeps running: they end under the lock)
  if (st) (void)streamSync(ctx);
  return st;
}

esf_status esf_extend_vector_field(esf_ctx* ctx, const int box[6], const double* mass,
                                   const double* phi, double* field) {
  if (!ctx || !box || !mass || !phi || !field) return ESF_ERR_INVALID;
  esf_status st = checkBox(ctx, box);
  if (st) return st;
  // staging held by the context (allocated on the first call)
  if ((st = sweepStaging(ctx))) return st;
  const long n = ctx->d.nodes;
  ESF_HIP(hipMemcpyAsync(ctx->swMass, mass, 8 * n, hipMemcpyHostToDevice, ctx->stream));
  ESF_HIP(hipMemcpyAsync(ctx->swPhi, phi, 8 * n, hipMemcpyHostToDevice, ctx->stream));
  ESF_HIP(hipMemcpyAsync(ctx->swField, field, 24 * n, hipMemcpyHostToDevice, ctx->stream));
  if ((st = extendDevice(ctx, box, ctx->swMass, ctx->swPhi, ctx->swField))) return st;
  return copyToHost(ctx, field, ctx->swField, 24 * n);
}
