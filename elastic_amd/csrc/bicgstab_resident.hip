// BiCGSTAB on a system held on the chip (resident.h): the FP64 iteration of
// bicgstab_run (Iters.f:1079-1349, Jacobi or the 3x3 node-block inverse) as one
// cooperative kernel.  x, r, p, v, r0 and the Jacobi scale of a row node stay
// in registers, z and r0 of the tile's local columns in LDS.  Per iteration:
//   v = A z, v.r0 from the tiles' shares (r0 is staged)     exchange 1
//   x += alpha z, r -= alpha v, z = M r to its readers
//   r.r and z of the external columns                       exchange 2, test
//   t = A z, own rows merged (neighbours only)
//   t.r, t.t                                                exchange 3
//   x += omega z, r -= omega t
//   r.r, r.r0                                               exchange 4, test
//   p = r + beta (p - omega v), z = M p to its readers (neighbours only)
// The launch iteration's eleven dependent kernels take 49 us on hex8 24^3, this 17.8.
// Words are emptied as in pcg_resident.hip: a z once everyone has published a
// sum that needed it, and both products' partials have words of their own.
#include <algorithm>
#include <cmath>

#include "device_util.h"
#include "resident.h"

namespace elastic {

struct ResBi {
  BlkArgs a;
  const double *vals, *diag;
  MergeArgs mg;
  u64* slots;
  double* epart;   // partials of the two products
  double* z;       // z of every row node: of the first product, of the second
  double* x;
  const double *b, *z0, *m, *bm;
  const double* rr;  // r.r0 = b.b
  SolveScalars* sc;
  int64_t next, n;
  int ntiles, maxit, limit, merge_max;
  size_t tile_lds, prod_lds;  // LDS of a tile, and of its product
};

template <int NB, int PER, int TPW>
__global__ __launch_bounds__(256 * TPW) void k_bicgstab_resident(ResBi g) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ ResShared sh;
  constexpr int NL = 256 * TPW;
  const int grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  typedef ResTile<double, double, NB, PER, false, false> Tile;
  const int tid = Tile::lane_of_tile(threadIdx.x);
  SolveScalars* sc = g.sc;
  if (sc->done) return;  // (no workgroup writes it before all have passed here)
  if (threadIdx.x == 0) sh.bad = 0;
  Tile t;
  unsigned char* mem = smem + grp * g.tile_lds;
  t.load(g.a, blockIdx.x * TPW + grp, g.ntiles, g.vals, g.diag, g.mg, g.merge_max, mem,
         threadIdx.x);
  double* r0s = reinterpret_cast<double*>(mem + g.prod_lds);  // r0 of the local columns
  const bool own = tid < t.nr;
  uint32_t i0 = (uint32_t)(NB * (t.I0 + (own ? tid : 0)));
  auto at = [&](auto* v) { return at_byte(v, (uint32_t)sizeof(*v) * i0); };
  double xv[NB], rv[NB], pv[NB], vv[NB], r0[NB], mv[NB];
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    xv[c] = vv[c] = 0.0;
    rv[c] = pv[c] = r0[c] = own ? at(g.b)[c] : 0.0;
    mv[c] = own && !g.bm ? at(g.m)[c] : 0.0;
    if (own) {
      t.xs[tid * NB + c] = at(g.z0)[c];
      r0s[tid * NB + c] = r0[c];
    }
  }
  __syncthreads();  // the external nodes are in LDS
  const int ne = (t.ncols - t.nr) * NB;
  double *xe = t.xs + t.nr * NB, *re = r0s + t.nr * NB;
  for (int e = tid; e < ne; e += 256) {
    xe[e] = *at_byte(g.z0, t.ext_off(e));
    re[e] = *at_byte(g.b, t.ext_off(e));
  }
  auto apply = [&](const double (&y)[NB], double (&z)[NB]) {  // z = M y on the lane's node
#pragma unroll
    for (int c = 0; c < NB; ++c) z[c] = y[c] * mv[c];
    if constexpr (NB == 3)
      if (g.bm && own) {
        const double* k = at_byte(g.bm, 16u * i0);  // 6 doubles per 3 rows
        z[0] = k[0] * y[0] + k[3] * y[1] + k[4] * y[2];
        z[1] = k[3] * y[0] + k[1] * y[1] + k[5] * y[2];
        z[2] = k[4] * y[0] + k[5] * y[1] + k[2] * y[2];
      }
  };
  const double conv = sc->conv;
  double rr = g.rr[0];
  double *ep1 = g.epart, *ep2 = g.epart + g.next, *z1 = g.z, *z2 = g.z + g.n;
  int iter = 0, seq = 0, state = 0, status = 0;  // state: 1 done, 2 maxit
  __syncthreads();
  while (true) {
    peer_drain();  // (words emptied since the last product)
    asm volatile("" : "+v"(i0));
    double s[2];
    int pe = tid;
    s[0] = t.product(ep1, vv, r0s);
    double s1[1] = {s[0]};
    if (!res_exchange<NL, 1>(s1, g.slots, threadIdx.x, gridDim.x, blockIdx.x, seq++, g.limit, sh,
                             [&]() { return t.look(ep1, pe); }))
      break;
    const double vr0 = s1[0];
    // a zero or non-finite denominator, or a non-finite r.r0: every lane sees it
    if (vr0 == 0.0 || !isfinite(vr0) || !isfinite(rr)) {
      state = 1;
      status = ELASTIC_BREAKDOWN;
      break;
    }
    const double alpha = rr / vr0;
    double zv[NB];
    s1[0] = 0.0;
    if (own) {
      t.add(vv);
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        xv[c] = xv[c] + alpha * t.xs[tid * NB + c];
        rv[c] = rv[c] - alpha * vv[c];
        s1[0] += rv[c] * rv[c];
      }
    }
    apply(rv, zv);
    if (own)
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        peer_put(at(z2) + c, zv[c]);
      }
    if (iter > 0) t.empty_rows(z1);  // (everyone has formed v from it)
    int e0 = tid;
    asm volatile("" : "+v"(e0));
    ResExternal E;
    if (!res_exchange<NL, 1>(s1, g.slots, threadIdx.x, gridDim.x, blockIdx.x, seq++, g.limit, sh,
                             [&]() { return t.ext_look(z2, e0, E); }))
      break;
    t.empty_partials(ep1);
    ++iter;
    double d = s1[0];
    if (!isfinite(d)) {
      state = 1;
      status = ELASTIC_BREAKDOWN;
      break;
    }
    if (sqrt(fabs(d)) < conv) {
      state = 1;
      break;
    }
    if (own)
#pragma unroll
      for (int c = 0; c < NB; ++c) t.xs[tid * NB + c] = zv[c];
    if (!t.ext_each(z2, e0, E, g.limit, [&](int e, double ze) { xe[e] = ze; })) sh.bad = 1;
    peer_drain();
    __syncthreads();
    double tv[NB];
    (void)t.product(ep2, tv, nullptr);
    // the transposed products have been read before the partials replace them
    __syncthreads();
    pe = tid;
    if (!res_wait(g.limit, sh, [&]() { return t.look(ep2, pe); })) break;
    s[0] = s[1] = 0.0;
    if (own) {
      t.add(tv);
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        s[0] += tv[c] * rv[c];
        s[1] += tv[c] * tv[c];
      }
    }
    if (!res_exchange<NL, 2>(s, g.slots, threadIdx.x, gridDim.x, blockIdx.x, seq++, g.limit, sh,
                             []() { return true; }))
      break;
    if (s[1] == 0.0 || !isfinite(s[1]) || !isfinite(s[0])) {
      state = 1;
      status = ELASTIC_BREAKDOWN;
      break;
    }
    const double w = s[0] / s[1];
    s[0] = s[1] = 0.0;
    if (own)
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        xv[c] = xv[c] + w * zv[c];
        rv[c] = rv[c] - w * tv[c];
        s[0] += rv[c] * rv[c];
        s[1] += rv[c] * r0[c];
      }
    t.empty_rows(z2);  // (everyone has formed t from it)
    t.empty_partials(ep2);
    if (!res_exchange<NL, 2>(s, g.slots, threadIdx.x, gridDim.x, blockIdx.x, seq++, g.limit, sh,
                             []() { return true; }))
      break;
    d = s[0];
    if (!isfinite(d) || !isfinite(s[1])) {
      state = 1;
      status = ELASTIC_BREAKDOWN;
      break;
    }
    if (sqrt(fabs(d)) < conv) {
      state = 1;
      break;
    }
    if (iter >= g.maxit) {
      state = 2;
      break;
    }
    const double beta = (s[1] / rr) * (alpha / w);
    rr = s[1];
#pragma unroll
    for (int c = 0; c < NB; ++c) pv[c] = rv[c] + beta * (pv[c] - w * vv[c]);
    apply(pv, zv);
    if (own)
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        peer_put(at(z1) + c, zv[c]);
        t.xs[tid * NB + c] = zv[c];
      }
    if (!res_wait(g.limit, sh, [&]() { return t.ext_look(z1, e0, E); })) break;
    if (!t.ext_each(z1, e0, E, g.limit, [&](int e, double ze) { xe[e] = ze; })) sh.bad = 1;
    __syncthreads();
  }
  __syncthreads();
  if (state == 0 || sh.bad) {  // a peer did not arrive: the host starts over without this kernel
    if (threadIdx.x == 0) sc->lost = 1;
    return;
  }
  if (own)
#pragma unroll
    for (int c = 0; c < NB; ++c) at(g.x)[c] = xv[c];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    sc->iter = iter;
    sc->status = status;
    if (state == 1) sc->done = 1;
  }
}

int bicgstab_resident_plan(Context* c, bool bdiag) {
  const DevBlocks& b = c->blk;
  if (!resident_on(c) || (bdiag && b.nb != 3)) return 0;
  // six vectors per row node beside the values: two tiles per CU at most
  return resident_tpw(c, 8, 2, sizeof(double) * b.nb * (size_t)b.ncols_max);
}

hipError_t bicgstab_resident_launch(Context* c, const double* bm, const double* rr, int maxit,
                                    int tpw) {
  const DevBlocks& b = c->blk;
  const int64_t n = (int64_t)b.nn * b.nb, next = b.next_nodes * b.nb;
  double* z = c->res_x + kResSlotWords;
  const size_t prod = res_tile_lds(8, b.nb, b.ncols_max, b.nblk_max, c->res_merge, false);
  ResBi g{blk_args(b), b.v64, b.d64, merge_of(c, c->epart64), (u64*)c->res_x, z + 3 * n, z,
          c->v64[VX], c->v64[VB], c->v64[VU], c->A64.m, bm, rr, c->scal, next, n, b.ntiles, maxit,
          c->resident_looks, c->res_merge, prod + sizeof(double) * b.nb * (size_t)b.ncols_max, prod};
  resident_clear(c, 8);
#define ELASTIC_RES(N, P, W) \
  return resident_start(c, (const void*)k_bicgstab_resident<N, P, W>, W, W * g.tile_lds, &g)
  if (b.nb == 2) {
    if (tpw == 1) ELASTIC_RES(2, 2, 1);
    ELASTIC_RES(2, 2, 2);
  }
  if (b.nblk_max <= 512) {
    if (tpw == 1) ELASTIC_RES(3, 2, 1);
    ELASTIC_RES(3, 2, 2);
  }
  if (tpw == 1) ELASTIC_RES(3, 4, 1);
  ELASTIC_RES(3, 4, 2);
#undef ELASTIC_RES
}

}  // namespace elastic
