// PCG on a system held on the chip (resident.h): the iteration of pcg.hip
// (Iters.f:252-524, Jacobi or the 3x3 node-block inverse, FP64 or the FP32
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
// scalars as the launch-per-phase iteration leaves them.
#include <algorithm>
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
  const double* bm;  // 3x3 node-block inverse (null: Jacobi)
  double* dslots;
  SolveScalars* sc;
  int64_t next, n;  // partials and rows
  int ntiles, maxit, limit, merge_max;
  int every;       // a replacement is made after any iteration (1) or after even ones (2)
  int stride;      // > 0: the products of every stride-th iteration are timed
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

template <typename TV, typename T, typename VT, typename XT, int NB, int PER, int TPW>
__global__ __launch_bounds__(256 * TPW)
void k_pcg_resident(ResPcg<TV, T, VT, XT> g) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ ResShared sh;
  constexpr bool FLEX = sizeof(TV) == 4;  // FP32 operator: flexible recurrences
  constexpr int NL = 256 * TPW, NS = FLEX ? 2 : 1;
  const int grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);  // uniform: scalar registers
  SolveScalars* sc = g.sc;
  if (sc->done) return;  // (no workgroup writes it before all have passed here)
  if (threadIdx.x == 0) sh.bad = 0;
  typedef ResTile<TV, T, NB, PER, TPW == 4, res_one<T, PER, TPW>()> Tile;
  constexpr bool MEM = res_vec_mem<T, PER, TPW>();
  const int tid = Tile::lane_of_tile();
  Tile t;
  t.load(g.a, blockIdx.x * TPW + grp, g.ntiles, g.vals, g.diag, g.mg, g.merge_max,
         smem + grp * g.tile_lds);
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
  if (threadIdx.x == 0) {  // (kept in LDS: every lane would hold them in registers)
    sh.keep[0] = sc->conv;
    sh.keep[1] = sc->delta * sc->rmax;
    sh.keep[2] = g.dslots[iter & 1];  // r.z of the last iteration
  }
  long long ticks = 0;    // of the timed products on this workgroup
  int samples = 0;
  bool asked = false;     // a replacement was asked for
  int k3 = 0, state = 0;  // k3: iteration of this call; state: 1 converged, 2 replacement, 3 maxit
  __syncthreads();
  while (true) {
    T* ep = g.epart + (k3 & 1) * g.next;
    double* zc = g.z + (k3 % 3) * g.n;
    // (words emptied since the last product)
    peer_drain();
    asm volatile("" : "+v"(i0));
    T qt[NB];
    double s1[NS];
    const bool timed = g.stride > 0 && threadIdx.x == 0 && iter % g.stride == 0;
    if (timed) ticks -= (long long)wall_clock64();
    s1[0] = t.product(ep, qt, t.xs);
    if (timed) {
      ticks += (long long)wall_clock64();
      ++samples;
    }
    if constexpr (FLEX) s1[1] = apr;
    int pe = tid;
    if (!res_exchange<NL, NS>(s1, g.slots, 2 * k3, g.limit, sh,
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
      if constexpr (NB == 3)
        if (g.bm) {
          const double* b = at_byte(g.bm, (uint32_t)(6 * sizeof(double) / NB) * i0);
          const double r0 = (double)rv[0], r1 = (double)rv[1], r2 = (double)rv[2];
          zv[0] = b[0] * r0 + b[3] * r1 + b[4] * r2;
          zv[1] = b[3] * r0 + b[1] * r1 + b[5] * r2;
          zv[2] = b[4] * r0 + b[5] * r1 + b[2] * r2;
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
    if (!res_exchange<NL, NS>(s2, g.slots, 2 * k3 + 1, g.limit, sh,
                              [&]() { return t.ext_look(zc, e0, E); }))
      break;
    const double di = s2[0];
    const double beta = FLEX ? -s2[NS - 1] / pq : di / sh.keep[2];
    apr = 0.0;
    if (own) {
      // (every reader has z of the iteration before)
      double* zo = g.z + ((k3 + 2) % 3) * g.n;
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        const T pv = (T)fma(beta, (double)t.xs[tid * NB + c], zv[c]);
        t.xs[tid * NB + c] = pv;
        apr += (double)pv * (double)rv[c];
        peer_empty(at(zo) + c);
      }
    }
    if (!t.ext_each(zc, e0, E, g.limit,
                    [&](int e, double ze) { xe[e] = (T)fma(beta, (double)xe[e], ze); }))
      sh.bad = 1;
    ++iter;
    ++k3;
    const double rn = sqrt(fabs(di)), conv = sh.keep[0];
    if (!reliable) {
      if (rn < conv) state = 1;
    } else if (asked || rn < sh.keep[1] || rn < conv || iter - last_upd >= kForceReplace) {
      asked = true;
      if (g.every == 1 || (iter & 1) == 0) state = 2;
    }
    if (state == 0 && iter >= g.maxit) state = 3;
    __syncthreads();  // p is staged, and everyone has used the last r.z
    if (threadIdx.x == 0) sh.keep[2] = di;
    if (state) break;
  }
  __syncthreads();
  if (state == 0 || sh.bad) {  // a peer did not arrive: the host starts over without this kernel
    if (threadIdx.x == 0) sc->lost = 1;
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
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    g.dslots[iter & 1] = sh.keep[2];
    sc->di = sh.keep[2];
    sc->prod_ticks = ticks;
    sc->prod_samples = samples;
    sc->iter = iter;
    if (state == 1) sc->done = 1;
    if (state == 2) {
      sc->upd = 1;
      sc->skip64 = 0;
    }
  }
}

// every word that workgroups exchange says that it has not arrived
__global__ __launch_bounds__(256) void k_res_empty(u64* w64, int64_t n64, uint32_t* w32,
                                                   int64_t n32, SolveScalars* sc) {
  const int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x, st = (int64_t)gridDim.x * 256;
  for (int64_t k = i0; k < n64; k += st) w64[k] = kResEmpty;
  for (int64_t k = i0; k < n32; k += st) w32[k] = kResEmpty32;
  if (i0 == 0) {
    sc->lost = 0;
    sc->prod_samples = 0;
    sc->prod_ticks = 0;
  }
}

// Entries of the longest merge list of a tile.
static int res_merge_max(const BlockLayout& L) {
  int m = 0;
  for (int t = 0; t < L.ntiles; ++t)
    m = std::max(m, L.inc_ptr[L.row0[t] + L.nrows[t]] - L.inc_ptr[L.row0[t]]);
  return m;
}

// Words of a resident solve: the slots, three rounds of a vector of the
// system, two rounds of external partials.
static size_t res_words(const DevBlocks& b) {
  return kResSlotWords + 3 * (size_t)b.nn * b.nb + 2 * (size_t)b.next_nodes * b.nb;
}

// Fewest tiles per workgroup that fit, since the tiles of a CU share its LDS
// pipe: 205 tiles of 512 blocks (hex8 20^3, FP64) take 7.5 us per iteration one
// to a CU and 8.0 two to a CU.
int resident_tpw(const Context* c, size_t t_size, int most, size_t more) {
  const DevBlocks& b = c->blk;
  for (int tpw = 1; tpw <= most; tpw *= 2) {
    const size_t lds = tpw * (more + res_tile_lds(t_size, b.nb, b.ncols_max, b.nblk_max, c->res_merge,
                                                  res_one_buffer(t_size, b.nblk_max, tpw)));
    if ((b.ntiles + tpw - 1) / tpw <= std::min(c->ncu, kResGroups) &&
        lds + sizeof(ResShared) + 64 <= 160 * 1024)
      return tpw;
  }
  return 0;
}

size_t resident_words(Context* c) {
  if (c->layout_nb < 2 || (c->layout_nb == 2 && c->blk.nblk_max > 512)) return 0;
  c->res_merge = res_merge_max(c->blayout);
  return resident_tpw(c, 4, kResTiles) || resident_tpw(c, 8, kResTiles) ? res_words(c->blk) : 0;
}

void resident_clear(Context* c, size_t t_size) {
  const DevBlocks& b = c->blk;
  const int64_t n = (int64_t)b.nn * b.nb, next = b.next_nodes * b.nb;
  const int64_t n64 = kResSlotWords + 3 * n + (t_size == 8 ? 2 * next : 0);
  hipLaunchKernelGGL(k_res_empty, dim3((unsigned)std::min<int64_t>((n64 + 255) / 256, 1024)),
                     dim3(256), 0, c->stream, (u64*)c->res_x, n64,
                     (uint32_t*)(c->res_x + kResSlotWords + 3 * n),
                     t_size == 4 ? 2 * next : (int64_t)0, c->scal);
}

hipError_t resident_start(Context* c, const void* kernel, int tpw, size_t lds, void* args) {
  if (lds > 65536) {
    const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             160 * 1024 - sizeof(ResShared) - 64);
    if (e != hipSuccess) return e;
  }
  void* list[] = {args};
  return hipLaunchCooperativeKernel(kernel, dim3((c->blk.ntiles + tpw - 1) / tpw), dim3(256 * tpw),
                                    list, (unsigned)lds, c->stream);
}

template <typename TV, typename T, typename VT, typename XT, int NB>
static hipError_t res_dispatch(Context* c, ResPcg<TV, T, VT, XT>& g, int tpw) {
#define ELASTIC_RES(P, W) \
  return resident_start(c, (const void*)k_pcg_resident<TV, T, VT, XT, NB, P, W>, W, W * g.tile_lds, &g)
  if (c->blk.nblk_max <= 512) {
    if (tpw == 1) ELASTIC_RES(2, 1);
    if (tpw == 2) ELASTIC_RES(2, 2);
    ELASTIC_RES(2, 4);
  }
  if constexpr (NB == 3) {
    if (tpw == 1) ELASTIC_RES(4, 1);
    if (tpw == 2) ELASTIC_RES(4, 2);
    ELASTIC_RES(4, 4);
  }
#undef ELASTIC_RES
  return hipErrorInvalidValue;
}

template <typename TV, typename T, typename VT, typename XT>
static hipError_t res_run(Context* c, const PcgVecs& V, const TV* vals, const TV* diag, XT* x, VT* r,
                          VT* p, const VT* m, int maxit, double* dslots, int tpw, int limit) {
  const DevBlocks& b = c->blk;
  const int64_t n = (int64_t)b.nn * b.nb, next = b.next_nodes * b.nb;
  double* z = c->res_x + kResSlotWords;
  ResPcg<TV, T, VT, XT> g{blk_args(b), vals, diag, merge_of(c, V.epart), (u64*)c->res_x,
                          (T*)(z + 3 * n), z, x, r, p, m, V.bm, dslots, c->scal, next, n,
                          b.ntiles, maxit, limit, c->res_merge, n < kPredictRows ? 2 : 1, c->time_stride,
                          res_tile_lds(sizeof(T), b.nb, b.ncols_max, b.nblk_max, c->res_merge,
                                       res_one_buffer(sizeof(T), b.nblk_max, tpw))};
  resident_clear(c, sizeof(T));
  return b.nb == 3 ? res_dispatch<TV, T, VT, XT, 3>(c, g, tpw)
                   : res_dispatch<TV, T, VT, XT, 2>(c, g, tpw);
}

int pcg_resident_plan(Context* c, bool fp32_operator, bool bdiag, bool v32) {
  const DevBlocks& b = c->blk;
  if (!c->res_x || !c->resident) return 0;
  if (bdiag && b.nb != 3) return 0;  // equation triples that are not nodes
  // FP32 sums: only with the FP32 vectors
  const bool f32 = fp32_operator && c->accum32;
  if (f32 && (!v32 || b.nb != 3)) return 0;
  return resident_tpw(c, f32 ? 4 : 8, kResTiles);
}

hipError_t pcg_resident_launch(Context* c, const PcgVecs& V, bool fp32_operator, int maxit,
                               double* dslots, int tpw, float* p32, float* r32, float* m32,
                               float* dx32) {
  const DevBlocks& b = c->blk;
  const int limit = c->resident_looks;
  if (!fp32_operator)
    return res_run<double, double, double, double>(c, V, b.v64, b.d64, V.x, V.r, V.p, V.m, maxit,
                                                   dslots, tpw, limit);
  if (!p32)
    return res_run<float, double, double, double>(c, V, b.v32, b.d32, V.x, V.r, V.p, V.m, maxit,
                                                  dslots, tpw, limit);
  if (dx32)
    return res_run<float, float, float, float>(c, V, b.v32, b.d32, dx32, r32, p32, m32, maxit,
                                               dslots, tpw, limit);
  return res_run<float, float, float, double>(c, V, b.v32, b.d32, V.x, r32, p32, m32, maxit,
                                              dslots, tpw, limit);
}

}  // namespace elastic
