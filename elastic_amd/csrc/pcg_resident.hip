// One PCG on the chip: the iteration of pcg_resident.h for a context's own solve.
#include <algorithm>

#include "pcg_resident.h"

namespace elastic {

template <typename TV, typename T, typename VT, typename XT, int NB, int PER, int TPW>
__global__ __launch_bounds__(256 * TPW)
void k_pcg_resident(ResPcg<TV, T, VT, XT> g) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ ResShared sh;
  if (g.sc->done) return;  // (no workgroup writes it before all have passed here)
  res_pcg<TV, T, VT, XT, NB, PER, TPW, false>(g, gridDim.x, blockIdx.x, smem, sh);
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

void resident_empty(Context* c, u64* words, int64_t n) {
  hipLaunchKernelGGL(k_res_empty, dim3((unsigned)std::min<int64_t>((n + 255) / 256, 1024)),
                     dim3(256), 0, c->stream, words, n, (uint32_t*)nullptr, (int64_t)0, c->scal);
}

hipError_t resident_start(Context* c, const void* kernel, int tpw, size_t lds, void* args,
                          size_t fixed, int lanes) {
  if (lds > 65536) {
    const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             160 * 1024 - sizeof(ResShared) - fixed - 64);
    if (e != hipSuccess) return e;
  }
  void* list[] = {args};
  return hipLaunchCooperativeKernel(kernel, dim3((c->blk.ntiles + tpw - 1) / tpw),
                                    dim3(lanes ? lanes : 256 * tpw), list, (unsigned)lds, c->stream);
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
                          b.ntiles, maxit, limit, c->res_merge, n < kPredictRows ? 2 : 1, c->time_stride, 0,
                          res_tile_lds(sizeof(T), b.nb, b.ncols_max, b.nblk_max, c->res_merge,
                                       res_one_buffer(sizeof(T), b.nblk_max, tpw))};
  resident_clear(c, sizeof(T));
  if constexpr (sizeof(T) == 8)  // (no plan for FP32 sums in 2-D)
    if (b.nb == 2) return res_dispatch<TV, T, VT, XT, 2>(c, g, tpw);
  return res_dispatch<TV, T, VT, XT, 3>(c, g, tpw);
}

int pcg_resident_plan(Context* c, bool fp32_operator, bool bdiag, bool v32) {
  const DevBlocks& b = c->blk;
  if (!resident_on(c)) return 0;
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
