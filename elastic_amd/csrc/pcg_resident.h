// PCG on a system held on the chip (resident.h): the iteration of pcg.hip
// (Iters.f:252-524, Jacobi or the node-block inverse, FP64 or the FP32
// operator with the flexible recurrences) as one cooperative kernel.
//
// A workgroup owns 1, 2 or 4 tiles.  Matrix values, the row nodes' x, r and the
// Jacobi scale stay in registers, p of the tile's local columns in LDS, for the
// whole call.  Per iteration:
//   product from LDS; partials of external columns to their owners
//   exchange 1: the sum p.q (and p.r), and the row nodes' partials
//   x += alpha p, r -= alpha q, z = M r to its readers
//   exchange 2: the sum r.z (and z.q), and z of the external columns
//   p = z + beta p on own rows and, from the readers' side, on the external
//   columns (every reader forms the owner's value from the same z and beta)
// The call ends when the iteration has converged, a true-residual replacement
// is due (the mixed method; on systems whose launch iteration looks for it
// after every second iteration, after even ones, so that iteration counts stay
// comparable) or maxit is reached, and leaves x, r, p and the
// scalars as the launch-per-phase iteration leaves them.  A batch (batch.hip)
// runs several systems side by side in one launch, a number of iterations at a time.
#pragma once
#include <cmath>

#include "device_util.h"
#include "resident.h"

namespace elastic {

template <typename TV, typename T, typename VT, typename XT>
struct ResPcg {
  BlkArgs a;
  const TV *vals, *diag;
  MergeArgs mg;
  u64* slots;
  T* epart;       // two rounds of next partials
  double* z;      // three rounds of z of every row node, for its readers
  XT* x;
  VT *r, *p;
  const VT* m;
  const double* bm;  // node-block inverse (null: Jacobi)
  double* dslots;
  SolveScalars* sc;
  int64_t next, n;  // partials and rows
  int ntiles, maxit, limit, merge_max;
  int every;       // a replacement is made after any iteration (1) or after even ones (2)
  int stride;      // > 0: the products of every stride-th iteration are timed
  int iters;       // round at which a batch step ends (STEP)
  size_t tile_lds;
};

// Tiles whose row and transposed products share one buffer: four FP64-sum
// tiles of up to 1,024 blocks on a CU
template <typename T, int PER, int TPW>
constexpr bool res_one() { return sizeof(T) == 8 && PER > 2 && TPW == 4; }
// four such tiles leave no registers for x, r and the Jacobi scale either: the
// lane that owns them reads them, and writes x and r, in every iteration
template <typename T, int PER, int TPW>
constexpr bool res_vec_mem() { return sizeof(T) == 8 && TPW == 4 && PER > 2; }

// The iterations of one system on workgroups bid = 0 .. G - 1.  STEP: those of a
// batch step, which end at round g.iters and book an iteration limit
// themselves.
template <typename TV, typename T, typename VT, typename XT, int NB, int PER, int TPW, bool STEP>
__device__ __forceinline__ void res_pcg(const ResPcg<TV, T, VT, XT>& g, int G, int bid,
                                        unsigned char* smem, ResShared& sh) {
  constexpr bool FLEX = sizeof(TV) == 4;  // FP32 operator: flexible recurrences
  constexpr int NL = 256 * TPW, NS = FLEX ? 2 : 1;
  int lane = threadIdx.x;
  // (what a step derives from it may not stay in registers from system to system)
  if constexpr (STEP) asm volatile("" : "+v"(lane));
  const int grp = __builtin_amdgcn_readfirstlane(lane >> 8);  // uniform: scalar registers
  SolveScalars* sc = g.sc;
  if (lane == 0) {
    sh.bad = 0;
    if constexpr (STEP) sh.late = 0;
  }
  typedef ResTile<TV, T, NB, PER, TPW == 4, res_one<T, PER, TPW>()> Tile;
  constexpr bool MEM = res_vec_mem<T, PER, TPW>();
  const int tid = Tile::lane_of_tile(lane);
  Tile t;
  t.load(g.a, bid * TPW + grp, g.ntiles, g.vals, g.diag, g.mg, g.merge_max,
         smem + grp * g.tile_lds, lane);
  const bool own = tid < t.nr;
  // row of the lane's node; vectors are addressed by 32-bit byte offsets from
  // scalar bases (a resident system is far below 2^32 bytes)
  uint32_t i0 = (uint32_t)(NB * (t.I0 + (own ? tid : 0)));
  auto at = [&](auto* v) { return at_byte(v, (uint32_t)sizeof(*v) * i0); };
  VT rv[NB], mv[NB];
  XT xv[NB];
  double apr = 0.0;
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    rv[c] = own ? at(g.r)[c] : VT(0);
    xv[c] = own && !MEM ? at(g.x)[c] : XT(0);
    mv[c] = own && !MEM && !g.bm ? at(g.m)[c] : VT(0);
    const VT pv = own ? at(g.p)[c] : VT(0);
    if (own) t.xs[tid * NB + c] = (T)pv;
    apr += (double)pv * (double)rv[c];
  }
  __syncthreads();  // the external nodes are in LDS
  const int ne = (t.ncols - t.nr) * NB;
  T* xe = t.xs + t.nr * NB;
  for (int e = tid; e < ne; e += 256)
    xe[e] = (T)g.p[(int64_t)NB * t.exn[e / NB] + e % NB];
  const int reliable = sc->reliable, last_upd = sc->last_upd;
  int iter = sc->iter;
  if (lane == 0) {  // (kept in LDS: every lane would hold them in registers)
    sh.keep[0] = sc->conv;
    sh.keep[1] = sc->delta * sc->rmax;
    sh.keep[2] = g.dslots[iter & 1];  // r.z of the last iteration
  }
  long long ticks = 0;    // of the timed products on this workgroup
  int samples = 0;
  bool asked = false;     // a replacement was asked for
  // iteration of this call; a batch step goes on where the words of the step
  // before it stopped
  int k3 = STEP ? sc->res_round : 0;
  int state = 0;          // 1 converged, 2 replacement, 3 maxit, 4 end of the step
  __syncthreads();
  while (true) {
    T* ep = g.epart + (k3 & 1) * g.next;
    double* zc = g.z + (k3 % 3) * g.n;
    // (words emptied since the last product)
    peer_drain();
    asm volatile("" : "+v"(i0));
    T qt[NB];
    double s1[NS];
    const bool timed = g.stride > 0 && lane == 0 && iter % g.stride == 0;
    if (timed) ticks -= (long long)wall_clock64();
    s1[0] = t.product(ep, qt, t.xs);
    if (timed) {
      ticks += (long long)wall_clock64();
      ++samples;
    }
    if constexpr (FLEX) s1[1] = apr;
    int pe = tid;
    if (!res_exchange<NL, NS>(s1, g.slots, lane, G, bid, 2 * k3, g.limit, sh,
                              [&]() { return t.look(ep, pe); }))
      break;
    const double pq = s1[0];
    const double alpha = (FLEX ? s1[NS - 1] : sh.keep[2]) / pq;
    double zv[NB], s2[NS];
#pragma unroll
    for (int c = 0; c < NB; ++c) zv[c] = 0.0;
#pragma unroll
    for (int k = 0; k < NS; ++k) s2[k] = 0.0;
    if (own) {
      double qv[NB];
#pragma unroll
      for (int c = 0; c < NB; ++c) qv[c] = (double)qt[c];
      t.add(qv);
      if constexpr (MEM) {
#pragma unroll
        for (int c = 0; c < NB; ++c) {
          xv[c] = at(g.x)[c];
          rv[c] = at(g.r)[c];
          mv[c] = g.bm ? VT(0) : at(g.m)[c];
        }
      }
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        xv[c] = (XT)((double)xv[c] + alpha * (double)t.xs[tid * NB + c]);
        rv[c] = (VT)((double)rv[c] - alpha * qv[c]);
        if constexpr (MEM) {
          at(g.x)[c] = xv[c];
          at(g.r)[c] = rv[c];
        }
        zv[c] = (double)rv[c] * (double)mv[c];
      }
      if (g.bm) {
        if constexpr (NB == 3) {
          const double* b = at_byte(g.bm, (uint32_t)(6 * sizeof(double) / NB) * i0);
          const double r0 = (double)rv[0], r1 = (double)rv[1], r2 = (double)rv[2];
          zv[0] = b[0] * r0 + b[3] * r1 + b[4] * r2;
          zv[1] = b[3] * r0 + b[1] * r1 + b[5] * r2;
          zv[2] = b[4] * r0 + b[5] * r1 + b[2] * r2;
        } else {
          const double* b = at_byte(g.bm, (uint32_t)(3 * sizeof(double) / NB) * i0);
          const double r0 = (double)rv[0], r1 = (double)rv[1];
          zv[0] = b[0] * r0 + b[2] * r1;
          zv[1] = b[2] * r0 + b[1] * r1;
        }
      }
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        peer_put(at(zc) + c, zv[c]);
        s2[0] += (double)rv[c] * zv[c];
        if constexpr (FLEX) s2[1] += zv[c] * qv[c];
      }
    }
    int e0 = tid;
    asm volatile("" : "+v"(e0));
    ResExternal E;
    if (!res_exchange<NL, NS>(s2, g.slots, lane, G, bid, 2 * k3 + 1, g.limit, sh,
                              [&]() { return t.ext_look(zc, e0, E); }))
      break;
    const double di = s2[0];
    const double beta = FLEX ? -s2[NS - 1] / pq : di / sh.keep[2];
    apr = 0.0;
    // every reader has z of the iteration before, and the partials of this one
    t.empty_rows(g.z + ((k3 + 2) % 3) * g.n);
    t.empty_partials(ep);
    if (own) {
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        const T pv = (T)fma(beta, (double)t.xs[tid * NB + c], zv[c]);
        t.xs[tid * NB + c] = pv;
        apr += (double)pv * (double)rv[c];
      }
    }
    // (in a batch told as sh.bad behind the barrier only: a wavefront that still reads
    // that for the exchange would leave alone, its barriers meeting those of the next
    // instance.  A single solve ends there, lost; the flag's read behind the barrier
    // would cost it 0.3 to 0.7%)
    if (!t.ext_each(zc, e0, E, g.limit,
                    [&](int e, double ze) { xe[e] = (T)fma(beta, (double)xe[e], ze); })) {
      if constexpr (STEP) sh.late = 1;
      else sh.bad = 1;
    }
    ++iter;
    ++k3;
    const double rn = sqrt(fabs(di)), conv = sh.keep[0];
    if (!reliable) {
      if (rn < conv) state = 1;
    } else if (asked || rn < sh.keep[1] || rn < conv || iter - last_upd >= kForceReplace) {
      asked = true;
      if (g.every == 1 || (iter & 1) == 0) state = 2;
    }
    if constexpr (STEP) {
      if (state != 1 && iter >= g.maxit) state = 3;  // (no replacement after the last one)
      else if (state == 0 && k3 >= g.iters) state = 4;
    } else if (state == 0 && iter >= g.maxit) {
      state = 3;
    }
    __syncthreads();  // p is staged, and everyone has used the last r.z
    if (lane == 0) {
      sh.keep[2] = di;
      if constexpr (STEP)
        if (sh.late) sh.bad = 1;
    }
    if (state) break;
  }
  __syncthreads();
  if (state == 0 || sh.bad) {  // a peer did not arrive: the host starts over without this kernel
    if (lane == 0) sc->lost = 1;
    return;
  }
  if (own) {
#pragma unroll
    for (int c = 0; c < NB; ++c) {
      if constexpr (!MEM) {
        at(g.x)[c] = xv[c];
        at(g.r)[c] = rv[c];
      }
      at(g.p)[c] = (VT)t.xs[tid * NB + c];
    }
  }
  if (bid == 0 && lane == 0) {
    g.dslots[iter & 1] = sh.keep[2];
    sc->di = sh.keep[2];
    sc->prod_ticks = ticks;
    sc->prod_samples = samples;
    sc->iter = iter;
    if (state == 1) sc->done = 1;
    if (STEP) sc->res_round = k3;
    if (STEP && state == 3) {
      sc->done = 1;
      sc->status = ELASTIC_MAXIT;
    }
    if (state == 2) {
      sc->upd = 1;
      sc->skip64 = 0;
    }
  }
}

}  // namespace elastic
