// Solves that stay on the chip (gfx950): one cooperative kernel holds a
// node-blocked system's matrix in registers, one tile of the layout per 256
// lanes, and runs the iterations of a Krylov method without leaving the
// device.  A launch-per-phase iteration on such systems is bound by its four
// dependent launches (about 5 us each, whatever they move); here an iteration
// is bound by two exchanges between the workgroups.  Per iteration, launches
// against resident: hex8 20^3 FP64 20.9 and 6.8 us, hex8 38^3 mixed 31 and 12.5,
// quad4 141^2 FP64 18.2 and 5.9, tet4 41^3 x 6 mixed 26.5 and 10.4.  Of the 6.8, the
// exchanges take 2.1 and 2.3, the product 1.8; with four tiles of 1,024 blocks per CU
// and FP64 sums (hex8 43^3, 19.6 us) they take 4.2, 5 and 7.5.
//
// Where 1,024 lanes share a CU a lane has 128 registers: five of the kernels keep some
// values in scratch then (bytes per lane in tests/test_resident_resources.py).  Only
// PCG with FP64 sums on four tiles of up to 1,024 blocks re-reads matrix values, 7 of a
// lane's 36 in each pass of the product; the others one or two doubles per iteration
// or what a batch needs between instances.
//
// Everything that crosses workgroups goes through relaxed agent-scope atomics
// (write-through stores, loads that do not take a line another XCD may hold
// newer), never through fences: a device-scope fence writes back and
// invalidates the XCD's L2 and costs 3 to 67 us per barrier for 64 to 1,024
// workgroups.  A word says itself whether it has arrived: until then it holds
// a NaN that no computation produces.  So partial sums, external partials and
// vector entries are all polled at once, one round trip per exchange, and no
// store is waited for before a flag.  Words are emptied by
// the side that wrote them, in whole lines (2 to 7% of an iteration against the
// readers doing it a node at a time), once every reader is known to have them,
// and reused only after a later exchange.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

#include "spmv_block.h"

namespace elastic {

typedef unsigned long long u64;

// One workgroup per CU at most, so that a workgroup may use the whole CU and
// 256 lanes can read every workgroup's sums at once.
constexpr int kResGroups = 256;
constexpr int kResTiles = 4;  // tiles per workgroup at most (1,024 lanes)
// Words that have not arrived (a computed NaN of this pattern is stored as
// another NaN).
constexpr u64 kResEmpty = 0x7ff8dead00000001ull;
constexpr uint32_t kResEmpty32 = 0x7fc0dead;
constexpr int kResRounds = 4;  // rounds of slots in rotation
static_assert(kResCopyWords >= kResRounds * 2 * kResGroups, "rounds of two sums per workgroup");

template <typename T>
struct PeerWord;
template <>
struct PeerWord<double> {
  typedef u64 W;
  static constexpr W kEmpty = kResEmpty, kOther = 0x7ff8000000000000ull;
  static __device__ __forceinline__ W bits(double v) { return (W)__double_as_longlong(v); }
  static __device__ __forceinline__ double value(W w) { return __longlong_as_double((long long)w); }
};
template <>
struct PeerWord<float> {
  typedef uint32_t W;
  static constexpr W kEmpty = kResEmpty32, kOther = 0x7fc00000u;
  static __device__ __forceinline__ W bits(float v) { return __float_as_uint(v); }
  static __device__ __forceinline__ float value(W w) { return __uint_as_float(w); }
};
template <typename T>
using peer_w = typename PeerWord<T>::W;
// p + byte offset: a uniform base stays in scalar registers
template <typename T>
__device__ __forceinline__ T* at_byte(T* p, uint32_t off) {
  return reinterpret_cast<T*>(reinterpret_cast<char*>(p) + off);
}
template <typename T>
__device__ __forceinline__ const T* at_byte(const T* p, uint32_t off) {
  return reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + off);
}
template <typename T>
__device__ __forceinline__ void peer_put(T* p, T v) {
  peer_w<T> w = PeerWord<T>::bits(v);
  if (w == PeerWord<T>::kEmpty) w = PeerWord<T>::kOther;
  __hip_atomic_store(reinterpret_cast<peer_w<T>*>(p), w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void peer_empty(T* p) {
  __hip_atomic_store(reinterpret_cast<peer_w<T>*>(p), PeerWord<T>::kEmpty, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ peer_w<T> peer_get(const T* p) {
  return __hip_atomic_load(reinterpret_cast<const peer_w<T>*>(p), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}
// this lane's stores have reached the point where every XCD sees them
__device__ __forceinline__ void peer_drain() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Sum of v over the wavefront, in lane 63 (DPP lane moves, fixed order).
__device__ __forceinline__ double wave_sum(double v) {
  v += dpp_move<0x111, 0xF>(v);
  v += dpp_move<0x112, 0xF>(v);
  v += dpp_move<0x114, 0xF>(v);
  v += dpp_move<0x118, 0xF>(v);
  v += dpp_move<0x142, 0xA>(v);
  v += dpp_move<0x143, 0xC>(v);
  return v;
}

struct ResShared {
  double red[2][4 * kResTiles];  // wavefront sums of this workgroup
  double sum[2][4];              // wavefront sums over the workgroups
  double keep[4];                // scalars of the method
  int bad;                       // a wait ran out: every workgroup gives up
  int late;                      // the same, outside of an exchange, in a batch's step (pcg_resident.h)
};

// v[k] = its sum over all lanes (this one tid) of the system's workgroups (this
// one bid of G), the same value everywhere
// (wavefronts, then workgroups, in a fixed order).  `pend` is called until it
// returns true, its loads in flight together with those of the sums; it
// fetches the words this lane waits for in the same exchange.  Round `seq`
// uses slots seq % kResRounds; a workgroup empties its slots of round seq - 1
// once it has all of round seq (nobody reads them any more).  They are reused
// in round seq + 3; the caller drains its stores (peer_drain) at least once in
// every two rounds, before it publishes, so a peer that polls round seq + 3
// has passed a round that was published after they were empty.  Every sum is
// stored in kResCopies copies and a workgroup looks at one of them: with one
// copy all workgroups poll the same few lines of one memory channel (an
// exchange of 205 workgroups took 3.3 to 3.7 us, with eight copies 2.0 to 2.8;
// sixteen gave no more).  Returns false when something did not arrive within `limit`
// looks.
template <int NL, int NS, typename Pend>
__device__ __forceinline__ bool res_exchange(double (&v)[NS], u64* slots, int tid, int G,
                                             int bid, int seq, int limit, ResShared& sh,
                                             Pend pend) {
  constexpr int NW = NL / 64;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
  for (int k = 0; k < NS; ++k) {
    const double w = wave_sum(v[k]);
    if (lane == 63) sh.red[k][wid] = w;
  }
  __syncthreads();
  u64* cur = slots + (size_t)(seq % kResRounds) * 2 * kResGroups;
  if (lane < kResCopies && wid < NS) {  // wavefront k publishes sum k, a copy per lane
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < NW; ++k) s += sh.red[wid][k];
    peer_put(reinterpret_cast<double*>(cur + lane * kResCopyWords + wid * kResGroups + bid),
             s);
  }
  cur += (bid % kResCopies) * kResCopyWords;
  u64 w[NS];
#pragma unroll
  for (int k = 0; k < NS; ++k) w[k] = 0;  // (+0.0: lanes without a workgroup)
  bool sums = tid >= G, rest = false;
  int n = 0;
  while (true) {
    if (!sums)
#pragma unroll
      for (int k = 0; k < NS; ++k)
        w[k] = peer_get(reinterpret_cast<const double*>(cur + k * kResGroups + tid));
    if (!rest) rest = pend();
    if (!sums) {
      sums = true;
#pragma unroll
      for (int k = 0; k < NS; ++k) sums &= w[k] != kResEmpty;
    }
    if (sums && rest) break;
    if (++n > limit) {
      sh.bad = 1;
      break;
    }
  }
  if (wid < kResGroups / 64) {
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      const double s = wave_sum(PeerWord<double>::value(w[k]));
      if (lane == 63) sh.sum[k][wid] = s;
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NS; ++k)
    v[k] = (sh.sum[k][0] + sh.sum[k][1]) + (sh.sum[k][2] + sh.sum[k][3]);
  if (lane < kResCopies && wid < 2)  // (the round before may have had two sums)
    peer_empty(reinterpret_cast<double*>(
        slots + (size_t)((seq + kResRounds - 1) % kResRounds) * 2 * kResGroups +
        lane * kResCopyWords + wid * kResGroups + bid));
  return sh.bad == 0;
}

// Waits for words of neighbours only: `pend` until it returns true, then a
// barrier of the workgroup.
template <typename Pend>
__device__ __forceinline__ bool res_wait(int limit, ResShared& sh, Pend pend) {
  for (int n = 0; !pend(); ++n)
    if (n > limit) {
      sh.bad = 1;
      break;
    }
  __syncthreads();
  return sh.bad == 0;
}

// A vector of the system as its rows' owners send it to the tiles that have
// them as external columns: entry e = tid + 256 j of the tile's external
// columns, the first kExt per lane in flight together.
constexpr int kResExt = 3;
struct ResExternal {
  u64 w[kResExt];
};

// Shared memory of one tile (bytes): x of its local columns, the blocks'
// transposed products, the pieces of row products (`one`: one buffer for both,
// one after the other), the diagonal blocks of the rows, the external nodes, the merge list
// (merge_max entries) and the row and segment pointers.
constexpr size_t kResPieces = 256 + kBlkRowsMax;
inline size_t res_tile_lds(size_t t_size, int nb, int ncols_max, int nblk_max, int merge_max,
                           bool one) {
  // (the partials of a merge list pass through the first buffer)
  const size_t buf = std::max(nblk_max, merge_max) + (one ? 0 : kResPieces);
  const size_t vals = t_size * (nb * ((size_t)ncols_max + buf) +
                                (kBlkRowsMax + 1) * (nb * (nb + 1) / 2));
  const size_t ptrs = sizeof(int32_t) * ((size_t)ncols_max + (size_t)merge_max) +
                      sizeof(uint16_t) * ((size_t)kBlkRowsMax + 1 + (size_t)ncols_max + 1);
  return (vals + ptrs + 15) & ~(size_t)15;
}

// One tile held by 256 lanes: lane tid owns blocks PER tid + i (in row order, so
// that a lane adds the row products of its consecutive blocks of one row before
// they go to LDS, about one store per row instead of one per block; lane l's
// piece of row r goes to place l + r, which makes the pieces of a row one run);
// the values
// are read once per call, so their order in memory does not matter) and, below
// the row count, row node tid.  The partials of the tile's row nodes are one
// run of the merge list: all lanes fetch them, one word at a time, into LDS,
// where the row's lane adds its own in list order.  TIGHT: four such tiles
// share a CU, which leaves 128 registers per lane; they keep fewer loads in
// flight, and ONE product buffer (res_tile_lds) where two do not fit.
template <typename TV, typename T, int NB, int PER, bool TIGHT, bool ONE>
struct ResTile {
  static constexpr int kMerge = TIGHT ? (PER > 2 ? 2 : 4) : 6;  // partial words of a lane in flight
  uint32_t wr[PER];
  TV vr[PER][NB * NB];
  int I0, nr, nbk, ncols, ext0;
  int nm;      // words of the tile's partials
  int m0, m1;  // those of the row node among them
  int lane;    // lane of the workgroup
  T *xs, *rw, *tr, *dg;
  int32_t *exn, *mls;
  uint16_t *rps, *sps;

  // Lane of the tile: the wavefronts of a workgroup's tiles are rotated
  // against each other, so that the wavefronts that own rows (the first two
  // of every tile) are spread over the CU's SIMDs.
  static __device__ __forceinline__ int lane_of_tile(int lane) {
    return (lane + 64 * (lane >> 8)) & 255;
  }

  __device__ __forceinline__ void load(const BlkArgs& a, int t, int ntiles, const TV* vals,
                                       const TV* diag, const MergeArgs& mg, int merge_max,
                                       unsigned char* smem, int lane_) {
    lane = lane_;
    const int tid = lane_of_tile(lane);
    xs = reinterpret_cast<T*>(smem);
    tr = xs + a.ncols_max * NB;
    const int first = max(a.nblk_max, merge_max) * NB;
    rw = ONE ? tr : tr + first;
    dg = ONE ? tr + first : rw + kResPieces * NB;
    exn = reinterpret_cast<int32_t*>(dg + (kBlkRowsMax + 1) * (NB * (NB + 1) / 2));
    mls = exn + a.ncols_max;
    rps = reinterpret_cast<uint16_t*>(mls + merge_max);
    sps = rps + kBlkRowsMax + 1;
    const bool on = t < ntiles;
    I0 = on ? a.row0[t] : 0;
    nr = on ? a.nrows[t] : 0;
    nbk = on ? a.nblk[t] : 0;
    ncols = on ? a.ncols[t] : 0;
    ext0 = on ? a.ext0[t] : 0;
    const int64_t base = on ? a.blk0[t] : 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int q = PER * tid + i;
      if (q < nbk) {
        wr[i] = a.word[base + q];
        Planes<TV, NB>::load(vals + base * (NB * NB), nbk, q, vr[i]);
      } else {
        wr[i] = 0xFFFFFFFFu;
#pragma unroll
        for (int p = 0; p < NB * NB; ++p) vr[i][p] = TV(0);
      }
    }
    const int mt = on ? mg.ptr[I0] : 0, ml = on ? mg.ptr[I0 + nr] - mt : 0;
    nm = NB * ml;
    for (int c = tid; c < ml; c += 256) mls[c] = mg.idx[mt + c];
    m0 = m1 = 0;
    if (tid < nr) {
#pragma unroll
      for (int k = 0; k < NB * (NB + 1) / 2; ++k)
        dg[k * (kBlkRowsMax + 1) + tid] = (T)diag[(int64_t)k * a.nn + I0 + tid];
      m0 = NB * (mg.ptr[I0 + tid] - mt);
      m1 = NB * (mg.ptr[I0 + tid + 1] - mt);
    }
    if (on) {
      const uint16_t* rp = a.rowptr + a.rp0[t];
      const uint16_t* sp = a.segptr + a.seg0[t];
      for (int c = tid; c <= nr; c += 256) rps[c] = rp[c];
      for (int c = tid; c <= ncols; c += 256) sps[c] = sp[c];
      for (int c = tid; c < ncols - nr; c += 256) exn[c] = a.ext[ext0 + c];
    }
  }

  // s += the NB-vectors buf[NB q ..], q0 <= q < q1, in order.  With ONE buffer a
  // short last batch is loaded whole (hex8 43^3 20.5 -> 19.6 us per iteration);
  // elsewhere the wider batches cost more registers than they give.
  static __device__ __forceinline__ void add_run(const T* buf, int q0, int q1, T (&s)[NB]) {
    if constexpr (ONE) {
      constexpr int kU = 2;
      for (int q = q0; q < q1; q += kU) {
        T v[kU][NB];
#pragma unroll
        for (int j = 0; j < kU; ++j) {
          const int k = min(q + j, q1 - 1);
#pragma unroll
          for (int r = 0; r < NB; ++r) v[j][r] = buf[k * NB + r];
        }
#pragma unroll
        for (int j = 0; j < kU; ++j)
          if (q + j < q1)
#pragma unroll
            for (int r = 0; r < NB; ++r) s[r] += v[j][r];
      }
    } else {
      constexpr int kU = TIGHT ? 2 : 4;
      int q = q0;
      for (; q + kU <= q1; q += kU) {
        T v[kU][NB];
#pragma unroll
        for (int j = 0; j < kU; ++j)
#pragma unroll
          for (int r = 0; r < NB; ++r) v[j][r] = buf[(q + j) * NB + r];
#pragma unroll
        for (int j = 0; j < kU; ++j)
#pragma unroll
          for (int r = 0; r < NB; ++r) s[r] += v[j][r];
      }
      for (; q < q1; ++q)
#pragma unroll
        for (int r = 0; r < NB; ++r) s[r] += buf[q * NB + r];
    }
  }

  // q = the row node's own-tile rows of A x, x staged in xs; the partials of
  // external columns go to their words for the owners; returns the lane's share
  // of w.(A x), w staged at ws for the tile's local columns (null: 0).  Pieces of
  // rows and transposed products go to LDS, row by row and column by column, and
  // one lane per row or column adds its run.
  // Barriers inside: every lane of the workgroup calls it.
  __device__ __forceinline__ double product(T* epart, T (&q)[NB], const T* ws) {
    int tid = lane_of_tile(lane);
    // the compiler may not keep what it derives from the lane number and the
    // words (LDS addresses, conditions) in registers from call to call: the
    // values need them
    asm volatile("" : "+v"(tid));
    auto blocks = [&](bool rows, bool cols) {
      T y[NB];        // row products of the lane's current row
      int cur = -1;
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int qb = PER * tid + i;
        asm volatile("" : "+v"(wr[i]));
        if constexpr (sizeof(TV) != sizeof(T))  // (nor the values widened)
#pragma unroll
          for (int p = 0; p < NB * NB; ++p) asm volatile("" : "+v"(vr[i][p]));
        const uint32_t w = wr[i];
        const int key = w >> 25, lc = (w >> 10) & 0x7FFF, tp = w & 0x3FF;
        if (qb < nbk) {
          if (rows) {
            T xc[NB];
#pragma unroll
            for (int r = 0; r < NB; ++r) xc[r] = xs[lc * NB + r];
            if (key != cur) {
              if (cur >= 0)
#pragma unroll
                for (int r = 0; r < NB; ++r) rw[(tid + cur) * NB + r] = y[r];
              cur = key;
#pragma unroll
              for (int r = 0; r < NB; ++r) y[r] = T(0);
            }
#pragma unroll
            for (int r = 0; r < NB; ++r) {
              T s = T(0);
#pragma unroll
              for (int cc = 0; cc < NB; ++cc) s += (T)vr[i][r * NB + cc] * xc[cc];
              y[r] += s;
            }
          }
          if (cols) {
            T xr[NB];
#pragma unroll
            for (int r = 0; r < NB; ++r) xr[r] = xs[key * NB + r];
#pragma unroll
            for (int cc = 0; cc < NB; ++cc) {
              T s = T(0);
#pragma unroll
              for (int r = 0; r < NB; ++r) s += (T)vr[i][r * NB + cc] * xr[r];
              tr[tp * NB + cc] = s;
            }
          }
        }
        if constexpr (TIGHT) __builtin_amdgcn_sched_barrier(0);
      }
      if (rows && cur >= 0)
#pragma unroll
        for (int r = 0; r < NB; ++r) rw[(tid + cur) * NB + r] = y[r];
    };
#pragma unroll
    for (int r = 0; r < NB; ++r) q[r] = T(0);
    auto row = [&]() {  // the diagonal block and the row's products
      if (tid >= nr) return;
      T d[NB * (NB + 1) / 2];
#pragma unroll
      for (int k = 0; k < NB * (NB + 1) / 2; ++k) d[k] = dg[k * (kBlkRowsMax + 1) + tid];
      const T* xi = xs + tid * NB;
      if constexpr (NB == 3) {
        q[0] = d[0] * xi[0] + d[3] * xi[1] + d[4] * xi[2];
        q[1] = d[3] * xi[0] + d[1] * xi[1] + d[5] * xi[2];
        q[2] = d[4] * xi[0] + d[5] * xi[1] + d[2] * xi[2];
      } else {
        q[0] = d[0] * xi[0] + d[2] * xi[1];
        q[1] = d[2] * xi[0] + d[1] * xi[1];
      }
      // one piece per lane that owns blocks of the row
      const int q0 = rps[tid], q1 = rps[tid + 1];
      if (q0 < q1) add_run(rw, tid + q0 / PER, tid + (q1 - 1) / PER + 1, q);
    };
    if constexpr (ONE) {
      blocks(true, false);
      __syncthreads();
      row();
      __syncthreads();
      blocks(false, true);
      __syncthreads();
    } else {
      blocks(true, true);
      __syncthreads();
      row();
    }
    double dacc = 0.0;
    for (int c = tid; c < ncols; c += 256) {
      T s[NB];
#pragma unroll
      for (int r = 0; r < NB; ++r) s[r] = c < nr ? q[r] : T(0);  // c < nr: c == tid
      add_run(tr, sps[c], sps[c + 1], s);
      if (c < nr) {
#pragma unroll
        for (int r = 0; r < NB; ++r) q[r] = s[r];
      } else {
#pragma unroll
        for (int r = 0; r < NB; ++r)
          peer_put(at_byte(epart, (uint32_t)(sizeof(T) * NB) * (uint32_t)(ext0 + c - nr)) + r,
                   s[r]);
      }
      if (ws)
#pragma unroll
        for (int r = 0; r < NB; ++r) dacc += (double)s[r] * (double)ws[c * NB + r];
    }
    return dacc;
  }

  // External entries of the vector z: ext_look() until it returns true, then
  // ext_each(f) calls f(entry, value) for the lane's entries (false: an entry
  // beyond the first kResExt did not arrive).
  __device__ __forceinline__ uint32_t ext_off(int e) const {
    return 8u * (uint32_t)(NB * exn[e / NB] + e % NB);
  }
  __device__ __forceinline__ bool ext_look(const double* z, int e0, ResExternal& E) const {
    const int ne = (ncols - nr) * NB;
    bool ok = true;
#pragma unroll
    for (int j = 0; j < kResExt; ++j)
      if (e0 + 256 * j < ne) E.w[j] = peer_get(at_byte(z, ext_off(e0 + 256 * j)));
#pragma unroll
    for (int j = 0; j < kResExt; ++j)
      if (e0 + 256 * j < ne) ok &= E.w[j] != kResEmpty;
    return ok;
  }
  template <typename F>
  __device__ __forceinline__ bool ext_each(const double* z, int e0, const ResExternal& E, int limit,
                                           F f) const {
    const int ne = (ncols - nr) * NB;
#pragma unroll
    for (int j = 0; j < kResExt; ++j)
      if (e0 + 256 * j < ne) f(e0 + 256 * j, PeerWord<double>::value(E.w[j]));
    for (int e = e0 + 256 * kResExt; e < ne; e += 256) {
      u64 w;
      for (int n = 0; (w = peer_get(at_byte(z, ext_off(e)))) == kResEmpty; ++n)
        if (n > limit) return false;
      f(e, PeerWord<double>::value(w));
    }
    return true;
  }

  // Empties the tile's row nodes of the vector z and the partials it sent: the
  // side that wrote them does, whose words are one run each, so that a store
  // instruction fills whole lines (a reader would empty them a node at a time;
  // every request of a line costs the fabric about the same).
  __device__ __forceinline__ void empty_rows(double* z) const {
    for (int e = lane_of_tile(lane); e < nr * NB; e += 256)
      peer_empty(at_byte(z, 8u * (uint32_t)(NB * I0 + e)));
  }
  __device__ __forceinline__ void empty_partials(T* epart) const {
    for (int e = lane_of_tile(lane); e < (ncols - nr) * NB; e += 256)
      peer_empty(at_byte(epart, (uint32_t)sizeof(T) * (uint32_t)(NB * ext0 + e)));
  }

  // The partials of the tile's row nodes.  look() fetches the lane's words,
  // kMerge at a time, into LDS (buffers of the product, free by then) as they
  // arrive; it is called until it returns true (e: the lane's next word).
  // After a barrier add() adds the row node's partials to q in list order.
  __device__ __forceinline__ bool look(T* epart, int& e) const {
    while (e < nm) {
      peer_w<T> w[kMerge];
      bool ok = true;
#pragma unroll
      for (int j = 0; j < kMerge; ++j)
        if (e + 256 * j < nm) {
          const int k = (e + 256 * j) / NB;
          w[j] = peer_get(at_byte(
              epart, (uint32_t)sizeof(T) * (uint32_t)(NB * mls[k] + (e + 256 * j - NB * k))));
        }
#pragma unroll
      for (int j = 0; j < kMerge; ++j)
        if (e + 256 * j < nm) ok &= w[j] != PeerWord<T>::kEmpty;
      if (!ok) return false;
#pragma unroll
      for (int j = 0; j < kMerge; ++j)
        if (e + 256 * j < nm) {
          tr[e + 256 * j] = PeerWord<T>::value(w[j]);
        }
      e += 256 * kMerge;
    }
    return true;
  }
  __device__ __forceinline__ void add(double (&q)[NB]) const {
    for (int k = m0; k < m1; k += NB)
#pragma unroll
      for (int r = 0; r < NB; ++r) q[r] += (double)tr[k + r];
  }
};

// Tiles per workgroup with which the layout's tiles are all held at once, `more`
// bytes of LDS per tile beside the product's; 0: they do not fit.
int resident_tpw(const Context* c, size_t t_size, int most, size_t more = 0);
// tiles whose row and transposed products share one buffer
inline bool res_one_buffer(size_t t_size, int nblk_max, int tpw) {
  return t_size == 8 && nblk_max > 512 && tpw == kResTiles;
}
// empties every word of Context::res_x that a solve with sums of t_size bytes
// exchanges, and the call's flags
void resident_clear(Context* c, size_t t_size);
// empties n more words
void resident_empty(Context* c, u64* words, int64_t n);
// raises the kernel's LDS limit where needed and launches it cooperatively
// (`fixed`: bytes of LDS the kernel declares beside ResShared; `lanes`: of a
// workgroup, if not 256 per tile)
hipError_t resident_start(Context* c, const void* kernel, int tpw, size_t lds, void* args,
                          size_t fixed = 0, int lanes = 0);

}  // namespace elastic
