// GMRES cycles on a system held on the chip (resident.h): the inner steps of
// gmres_run (Iters.f:528-808, FP64, Jacobi or the 3x3 node-block inverse,
// classical Gram-Schmidt twice) of one cycle as one cooperative kernel.  The
// matrix stays in registers and the tile's rows of the basis in LDS (the last
// vectors of a tile with many rows: the first tiles of an order, whose nodes have
// few lower neighbours, are read from memory), so a step moves little but what
// crosses tiles:
//   w = M A g_i, the row nodes' partials from the neighbours
//   h1 = G.w                                            exchange 1
//   w -= G h1; h2 = G.w and w.w                         exchange 2
//   w -= G h2 to its readers
//   rotations and stop test in every workgroup, g_{i+1} = w / ||w||
// (a reader divides the w of its external columns itself).  The launch
// iteration's six kernels and the host's looks take 35.6 us per step on hex8 17^3,
// this 20.2: about 2 each for the product, the two exchanges and w's way to its
// readers, 2.5 to 5 for the dot products and 2 to 3 for the updates, both set by
// the tile with the most rows.  The basis, H, e and the step count are left as
// the launches leave them; the back substitution, x and the true residual of a
// restart stay there.
#include <algorithm>
#include <cmath>

#include "device_util.h"
#include "resident.h"

namespace elastic {

struct ResGm {
  BlkArgs a;
  const double *vals, *diag;
  MergeArgs mg;
  u64* hw;          // words of the sums (gm_exchange)
  double* epart;    // two rounds of next partials
  double* z;        // two rounds of w of every row node
  double* basis;    // k + 1 vectors of n
  const double *m, *bm;
  double *H, *e;    // (k + 1) x k, k + 1
  SolveScalars* sc;
  int64_t next, n;
  int ntiles, k, limit, merge_max;
  int room;  // doubles of LDS for w and basis vectors of a tile
  double econv;
  size_t tile_lds, prod_lds;  // LDS of a tile, and of its product
};

// rows of a vector in LDS: odd multiples of 16, so that the two groups of sixteen
// lanes of a half wavefront read different banks
__host__ __device__ inline int gm_ld(int rows) { return (rows + 15) / 32 * 32 + 16; }

// Words of one round of an exchange of np sums: every workgroup's shares, then
// the sums, one copy per XCD.
constexpr int kGmCopies = 8;
static_assert(kResRounds * (kResGroups + kGmCopies) <= kGmWords, "words of an exchange");

// h[j] = the sums over all workgroups of their shares dts[j] (j < np; TPW tiles
// k + 1 apart).  Sum j is formed by workgroup G - 1 - j (mod G; the first
// workgroups are the slow ones) and fetched by everyone: all shares read by all
// workgroups would be 6.4 MB per look for 126 of them and 50 sums.  Words are
// emptied one round later and reused three rounds later, as in res_exchange: so
// every workgroup drains its stores (peer_drain) between the round in which it
// empties words and its shares two rounds on.  A step has two rounds and a drain
// at its top; one that forms the norm again has three, and drains before the third.
template <int TPW, int NW>
__device__ __forceinline__ bool gm_exchange(const ResGm& g, int np, int seq, const double* dts,
                                            double* h, ResShared& sh) {
  constexpr int kC = kResGroups / 64;
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = gridDim.x, bid = blockIdx.x, K = g.k + 1;
  const size_t round = (size_t)K * (kResGroups + kGmCopies);
  double* cur = reinterpret_cast<double*>(g.hw) + (seq % kResRounds) * round;
  double* old = reinterpret_cast<double*>(g.hw) + ((seq + kResRounds - 1) % kResRounds) * round;
  double *res = cur + (size_t)K * kResGroups, *ores = old + (size_t)K * kResGroups;
  for (int j = tid; j < np; j += 64 * NW) {
    double s = dts[j];
#pragma unroll
    for (int t = 1; t < TPW; ++t) s += dts[t * K + j];
    peer_put(cur + (size_t)j * kResGroups + bid, s);
  }
  for (int j = G - 1 - bid + G * wid; j < np; j += G * NW) {
    u64 w[kC];
#pragma unroll
    for (int c = 0; c < kC; ++c) w[c] = lane + 64 * c < G ? kResEmpty : 0;
    for (int n = 0;; ++n) {
      bool ok = true;
#pragma unroll
      for (int c = 0; c < kC; ++c)
        if (w[c] == kResEmpty) w[c] = peer_get(cur + (size_t)j * kResGroups + lane + 64 * c);
#pragma unroll
      for (int c = 0; c < kC; ++c) ok &= w[c] != kResEmpty;
      if (ok) break;
      if (n > g.limit) {
        sh.bad = 1;
        break;
      }
    }
    double v = 0.0;
#pragma unroll
    for (int c = 0; c < kC; ++c) v += PeerWord<double>::value(w[c]);
    v = wave_sum(v);
    v = __shfl(v, 63);
    if (lane < kGmCopies) peer_put(res + lane * K + j, v);
  }
  for (int j = tid; j < np; j += 64 * NW) {
    u64 w;
    for (int n = 0; (w = peer_get(res + (bid % kGmCopies) * K + j)) == kResEmpty; ++n)
      if (n > g.limit) {
        sh.bad = 1;
        break;
      }
    h[j] = PeerWord<double>::value(w);
  }
  __syncthreads();
  // every workgroup has sent shares of exchange seq, so it has the sums of seq - 1
  if (seq > 0) {
    for (int j = tid; j < K; j += 64 * NW) peer_empty(old + (size_t)j * kResGroups + bid);
    if (tid < kGmCopies)
      for (int j = G - 1 - bid; j < K; j += G) peer_empty(ores + tid * K + j);
  }
  return sh.bad == 0;
}

// A tile's lanes for the basis: with one tile to a workgroup 256 more help (the
// passes over the basis are two thirds of a step, and a tile of 381 rows keeps
// all others waiting).
template <int TPW>
constexpr int gm_lanes() { return TPW == 1 ? 512 : 256; }
constexpr int kGmHalf = 384;  // partial sums of one tile's rows

template <int NB, int PER, int TPW>
__global__ __launch_bounds__(gm_lanes<TPW>() * TPW) void k_gmres_resident(ResGm g) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ ResShared sh;
  __shared__ double half[TPW][kGmHalf];
  constexpr int WL = gm_lanes<TPW>(), NL = WL * TPW, NW = NL / 64;
  typedef ResTile<double, double, NB, PER, false, false> Tile;
  const int lane = threadIdx.x, grp = __builtin_amdgcn_readfirstlane(lane >> 8);
  const int tid = Tile::lane_of_tile(lane);
  if (lane == 0) sh.bad = 0;
  Tile t;  // (helping lanes: none)
  const int slot = TPW == 1 ? 0 : grp, tile = blockIdx.x * TPW + slot;
  unsigned char* mem = smem + slot * g.tile_lds;
  t.load(g.a, grp < TPW ? tile : g.ntiles, g.ntiles, g.vals, g.diag, g.mg, g.merge_max, mem, lane);
  const bool own = tid < t.nr;
  double mv[NB];
#pragma unroll
  for (int c = 0; c < NB; ++c) mv[c] = own && !g.bm ? g.m[NB * (t.I0 + tid) + c] : 0.0;
  // the tile's rows of w and of the basis, for its WL lanes bl
  const int bl = TPW == 1 ? lane : tid;
  const int k = g.k, R = tile < g.ntiles ? NB * g.a.nrows[tile] : 0, ld = gm_ld(R);
  const int64_t row0 = tile < g.ntiles ? (int64_t)NB * g.a.row0[tile] : 0;
  double* W = reinterpret_cast<double*>(mem + g.prod_lds);
  double* B = W + ld;                      // vectors 0 .. kl - 1
  const int kl = min(k, g.room / ld - 1);
  double* gb = g.basis + row0;             // vector j: gb + j n
  double* xs = reinterpret_cast<double*>(mem);
  double* hs = reinterpret_cast<double*>(smem + TPW * g.tile_lds);  // column of H
  double *cs = hs + k, *ss = cs + k, *h = ss + k, *dts = h + k + 1;
  for (int r = bl; r < R; r += WL) B[r] = xs[r] = gb[r];
  __syncthreads();  // the external nodes are in LDS
  const int ne = (t.ncols - t.nr) * NB;
  double* xe = xs + R;
  for (int e = tid; e < ne; e += 256) xe[e] = *at_byte(g.basis, t.ext_off(e));
  double e0 = g.e[0];
  int i = 0, seq = 0, state = 0;  // state: 1 converged, 2 the cycle's last step
  __syncthreads();
  while (true) {
    ++i;
    peer_drain();  // (words emptied in the step before)
    double* ep = g.epart + (i & 1) * g.next;
    double q[NB];
    (void)t.product(ep, q, nullptr);
    // the transposed products have been read before the partials replace them
    __syncthreads();
    int pe = tid;
    if (!res_wait(g.limit, sh, [&]() { return t.look(ep, pe); })) break;
    if (own) {
      t.add(q);
      double w[NB];
#pragma unroll
      for (int c = 0; c < NB; ++c) w[c] = mv[c] * q[c];
      if constexpr (NB == 3)
        if (g.bm) {
          const double* b = g.bm + 6 * (int64_t)(t.I0 + tid);
          w[0] = b[0] * q[0] + b[3] * q[1] + b[4] * q[2];
          w[1] = b[3] * q[0] + b[1] * q[1] + b[5] * q[2];
          w[2] = b[4] * q[0] + b[5] * q[1] + b[2] * q[2];
        }
#pragma unroll
      for (int c = 0; c < NB; ++c) W[NB * tid + c] = w[c];
    }
    // shares of w.g_j, j0 <= j < np, g_i standing for w: sixteen lanes per
    // product, their rows of w in registers
    auto dots = [&](int j0, int np) {
      for (int jb = j0; jb < np; jb += WL / 8) {
        double s[2] = {0.0, 0.0};
        for (int r0 = bl & 15; r0 < R; r0 += 128) {
          double w[8];
          int r[8];
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            r[u] = min(r0 + 16 * u, R - 1);
            w[u] = r0 + 16 * u < R ? W[r[u]] : 0.0;
          }
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const int j = jb + (bl >> 4) + WL / 16 * q;
            if (j < np) {
              if (j < kl || j == i) {
                const double* v = j == i ? W : B + j * ld;
#pragma unroll
                for (int u = 0; u < 8; ++u) s[q] += w[u] * v[r[u]];
              } else {
                const double* v = gb + j * g.n;
#pragma unroll
                for (int u = 0; u < 8; ++u) s[q] += w[u] * v[r[u]];
              }
            }
          }
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int j = jb + (bl >> 4) + WL / 16 * q;
          if (jb + WL / 16 * q < np) {
            s[q] += dpp_move<0x111, 0xF>(s[q]);
            s[q] += dpp_move<0x112, 0xF>(s[q]);
            s[q] += dpp_move<0x114, 0xF>(s[q]);
            s[q] += dpp_move<0x118, 0xF>(s[q]);
            if ((bl & 15) == 15 && j < np) dts[slot * (k + 1) + j - j0] = s[q];
          }
        }
      }
    };
    // acc += sum of h_j v_j, ja <= j < jb, v_j = v + j st
    double acc = 0.0;
    auto combine = [&](const double* v, int64_t st, int ja, int jb) {
      int j = ja;
      for (; j + 8 <= jb; j += 8) {
        double b[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) b[u] = v[(j + u) * st];
#pragma unroll
        for (int u = 0; u < 8; ++u) acc += h[j + u] * b[u];
      }
      if (j < jb) {
        double b[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) b[u] = v[min(j + u, jb - 1) * st];
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (j + u < jb) acc += h[j + u] * b[u];
      }
    };
    bool bad = false;
    for (int pass = 0; pass < 2 && !bad; ++pass) {
      __syncthreads();
      dots(0, i + pass);
      __syncthreads();
      bad = !gm_exchange<TPW, NW>(g, i + pass, seq++, dts, h, sh);
      if (pass == 0) {
        // every workgroup has the partials of this step and w of the last one
        t.empty_partials(ep);
        if (i > 1) t.empty_rows(g.z + ((i - 1) & 1) * g.n);
      }
      for (int j = lane; j < i; j += NL) hs[j] = pass == 0 ? h[j] : hs[j] + h[j];
      // w -= G h: the lanes in as many parts as have room for the rows, a part
      // of the vectors each
      const int lr = R <= 128 ? 128 : R <= 256 || WL == 256 ? 256 : WL, parts = WL / lr;
      const int part = __builtin_amdgcn_readfirstlane(bl / lr), r0 = bl & (lr - 1);
      const int ja = i * part / parts, jb = i * (part + 1) / parts;
      for (int r = r0; r < R; r += lr) {
        acc = 0.0;
        combine(B + r, ld, ja, min(jb, kl));
        combine(gb + r, g.n, max(ja, kl), jb);
        if (parts == 1) W[r] -= acc;
        else if (part) half[slot][(part - 1) * lr + r] = acc;
      }
      if (parts > 1) {
        __syncthreads();
        if (part == 0 && r0 < R) {
          for (int q = 1; q < parts; ++q) acc += half[slot][(q - 1) * lr + r0];
          W[r0] -= acc;
        }
      } else if constexpr (TPW > 1) {
        __syncthreads();  // (the other tile's)
      }
    }
    if (bad) break;
    // ||w||^2 after the second pass: w.w - h2.h2 unless h2 is a large part of w
    double hh = 0.0;
    for (int j = lane & 63; j < i; j += 64) hh += h[j] * h[j];
    const double ww = h[i];
    double n2 = ww - __shfl(wave_sum(hh), 63);
    __syncthreads();  // w and hs are complete
    double* zc = g.z + (i & 1) * g.n;
    for (int r = bl; r < R; r += WL) peer_put(zc + row0 + r, W[r]);
    if (!(n2 > 0.5 * ww)) {
      dots(i, i + 1);
      peer_drain();  // (words emptied in the first round)
      __syncthreads();
      if (!gm_exchange<TPW, NW>(g, 1, seq++, dts, h, sh)) break;
      n2 = h[0];
    }
    int e1 = tid;
    ResExternal E;
    bool turned = lane != NL - 64;
    if (!res_wait(g.limit, sh, [&]() {
          if (!turned) {  // one lane turns the column while the words are on their way
            double hj = hs[0];
#pragma unroll 8
            for (int j = 1; j < i; ++j) {
              const double hn = hs[j], c = cs[j - 1], s = ss[j - 1];
              hs[j - 1] = c * hj + s * hn;
              hj = -s * hj + c * hn;
            }
            sh.keep[0] = hj;
            turned = true;
          }
          return t.ext_look(zc, e1, E);
        }))
      break;
    const double nrm = sqrt(n2), hj = sh.keep[0];
    const double rr = sqrt(hj * hj + nrm * nrm), ci = hj / rr, si = nrm / rr;
    const double en = -si * e0;
    if (lane == 0) {
      cs[i - 1] = ci;
      ss[i - 1] = si;
    }
    if (blockIdx.x == 0) {
      double* H = g.H + (size_t)(i - 1) * (k + 1);
      for (int j = lane; j < i - 1; j += NL) H[j] = hs[j];
      if (lane == 0) {
        H[i - 1] = rr;
        H[i] = 0.0;
        g.e[i - 1] = ci * e0;
        g.e[i] = en;
      }
    }
    for (int r = bl; r < R; r += WL) {
      const double v = nrm != 0.0 ? W[r] / nrm : W[r];
      xs[r] = v;
      if (i < kl) B[i * ld + r] = v;
      gb[i * g.n + r] = v;
    }
    if (!t.ext_each(zc, e1, E, g.limit,
                    [&](int e, double w) { xe[e] = nrm != 0.0 ? w / nrm : w; }))
      sh.bad = 1;
    e0 = en;
    if (fabs(en) <= g.econv) state = 1;
    else if (i == k) state = 2;
    __syncthreads();
    if (state) break;
  }
  __syncthreads();
  if (state == 0 || sh.bad) {  // a peer did not arrive: the host starts over without this kernel
    if (lane == 0) g.sc->lost = 1;
    return;
  }
  if (blockIdx.x == 0 && lane == 0) {
    g.sc->gm_ni = i;
    g.sc->gm_e = fabs(e0);
    g.sc->gm_done = state == 1;
  }
}

constexpr size_t kGmFixed = 2 * kGmHalf * sizeof(double);  // half[]
constexpr int64_t kLdsLeft = 160 * 1024 - 64 - sizeof(ResShared) - kGmFixed;
static size_t gm_shared(int k, int tpw) {
  return sizeof(double) * ((size_t)k * (4 + tpw) + 1 + tpw);
}
// Doubles of LDS for w and the basis of a tile: enough for its largest number of
// rows, or what tpw tiles leave each other (0: less than half a cycle).
static int gm_room(const Context* c, int k, int tpw) {
  const DevBlocks& b = c->blk;
  int rows = 1;
  for (int t = 0; t < b.ntiles; ++t) rows = std::max(rows, (int)c->blayout.nrows[t] * b.nb);
  const int64_t ld = gm_ld(rows);
  const int64_t left = (kLdsLeft - (int64_t)gm_shared(k, tpw)) / tpw -
                       (int64_t)res_tile_lds(8, b.nb, b.ncols_max, b.nblk_max, c->res_merge, false);
  const int64_t room = std::min(left / 16 * 2, (k + 1) * ld);
  return room >= (k / 2 + 2) * ld ? (int)room : 0;
}

int gmres_resident_plan(Context* c, bool bdiag, int k) {
  if (!resident_on(c) || (bdiag && c->blk.nb != 3) || k > 256) return 0;
  for (int tpw = 1; tpw <= 2; ++tpw)
    if ((c->blk.ntiles + tpw - 1) / tpw <= std::min(c->ncu, kResGroups) && gm_room(c, k, tpw))
      return tpw;
  return 0;
}

hipError_t gmres_resident_launch(Context* c, const double* bm, double* basis, double* H, double* e,
                                 double* words, int k, double econv, int tpw) {
  const DevBlocks& b = c->blk;
  const int64_t n = (int64_t)b.nn * b.nb, next = b.next_nodes * b.nb;
  double* z = c->res_x + kResSlotWords;
  const int room = gm_room(c, k, tpw);
  const size_t prod = res_tile_lds(8, b.nb, b.ncols_max, b.nblk_max, c->res_merge, false);
  ResGm g{blk_args(b), b.v64, b.d64, merge_of(c, c->epart64), (u64*)words,
          z + 3 * n, z, basis, c->A64.m, bm, H, e, c->scal, next, n, b.ntiles, k,
          c->resident_looks, c->res_merge, room, econv, prod + sizeof(double) * room, prod};
  resident_clear(c, 8);
  resident_empty(c, (u64*)words, (int64_t)gm_resident_words(k));
  const size_t lds = tpw * g.tile_lds + gm_shared(k, tpw);
#define ELASTIC_RES(N, P, W)                                                                  \
  return resident_start(c, (const void*)k_gmres_resident<N, P, W>, W, lds, &g, kGmFixed, \
                        gm_lanes<W>() * W)
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
