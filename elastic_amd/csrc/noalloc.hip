// The symmetric CSRC product on caller-held device arrays, with no device
// allocation: for callers that cannot call hipMalloc (code under HIP graph
// capture, tight serving loops).  It computes what elastic_spmv computes
// (Matvec.f:528-621) without a context: the transposed lists of the pattern
// that the gather-only product walks (spmv_gather.hip) are built on every call
// in `scratch`, a file-scope device array of fixed size, instead of a layout
// built once at set-up.
//
// Per call, on the caller's stream:
//   1. column counts of the pattern (integer atomics into cnt, one for the
//      entries that three consecutive rows have at the same place; cleared first
//      by a fill kernel; no hipMemsetAsync, so the call can be captured);
//   2. colptr = exclusive scan of the counts (three launches: block scans,
//      the scan of the block totals, the offsets);
//   3. every stored entry placed in its column's list (as many atomics on a
//      cursor copied from colptr; 32 lanes per three rows, so that their atomics
//      are in flight together);
//   4. per row, one wavefront orders the column's list by CSRC position, so
//      the order, and the FP64 result, never depend on the atomics, and adds
//      y_i = ad_i x_i + row i in CSRC order + column i in ascending rows,
//      bit-identical to matvec_csrcsym1.
// On hex8 28^3 (neq 70,644, nad 2.6 M) a call takes 128 us: counts 16,
// placement 35, ordering and product 69.  The first two are bound by their
// atomics (26 and 54 with one atomic per entry; 178 with one lane per row).  The
// last replaces an insertion sort of every list by one lane (1,113 us: a serial
// chain of dependent global loads and stores) and a gather product with one lane
// per row (98 us, uncoalesced); the call took 1,403 us.
#include <mutex>

#include "elastic_internal.h"

namespace elastic {
namespace {

// 128 MiB of int32 words per GPU: cnt (neq), colptr (neq+1), colk (nad),
// colrow (nad), the block totals of the scan.
constexpr int64_t kScratchWords = int64_t(32) << 20;
constexpr int kScanBlock = 1024;  // entries per block of the scan (256 lanes x 4)
constexpr int kMaxDevices = 64;

static __device__ __align__(256) int32_t scratch[kScratchWords];

// device address of `scratch` on each device (hipGetSymbolAddress once per
// device, with that device current)
int32_t* g_scratch[kMaxDevices] = {nullptr};
std::once_flag g_once[kMaxDevices];
hipError_t g_status[kMaxDevices];

int64_t scratch_words(int64_t neq, int64_t nad) {
  const int64_t nblk = (neq + 1 + kScanBlock - 1) / kScanBlock;
  return 2 * neq + 1 + 2 * nad + nblk + 1;
}

__global__ __launch_bounds__(256) void k_fill(int64_t n, int32_t* __restrict__ p, int32_t v) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) p[i] = v;
}

// The entries of rows r = 3 g .. r + 2 by 32 lanes: f(r, c, j0, m, a, q) for every
// column c[j0] at place q of these rows, which m rows j >= j0 have there (entry
// a[j] + q).  The dofs of a node
// have the same columns in the same places of their rows, so that one atomic serves
// three entries; rows that do not match (other node sizes, restrained dofs)
// take one each.  A column outside the system is dropped.
template <typename F>
__device__ __forceinline__ void row_triples(int n, const int32_t* __restrict__ ia,
                                            const int32_t* __restrict__ ja, F f) {
  const int sub = threadIdx.x & 31;
  for (int64_t r = 3 * (blockIdx.x * 8ll + (threadIdx.x >> 5)); r < n;
       r += 3 * (int64_t)gridDim.x * 8) {
    int a[3], len[3], longest = 0;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      a[j] = r + j < n ? ia[r + j] - 1 : 0;
      len[j] = r + j < n ? ia[r + j + 1] - 1 - a[j] : 0;
      longest = max(longest, len[j]);
    }
    for (int q = sub; q < longest; q += 32) {
      int c[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        c[j] = q < len[j] ? ja[a[j] + q] - 1 : -1;
        if (c[j] >= n) c[j] = -1;
      }
#pragma unroll
      for (int j0 = 0; j0 < 3; ++j0) {
        bool seen = c[j0] < 0;
        int m = 0;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          seen |= j < j0 && c[j] == c[j0];
          m += j >= j0 && c[j] == c[j0];
        }
        if (!seen) f(r, c, j0, m, a, q);
      }
    }
  }
}

__global__ __launch_bounds__(256) void k_count_cols(int n, const int32_t* __restrict__ ia,
                                                     const int32_t* __restrict__ ja,
                                                     int32_t* __restrict__ cnt) {
  row_triples(n, ia, ja, [&](int64_t, const int (&c)[3], int j0, int m, const int (&)[3], int) {
    atomicAdd(&cnt[c[j0]], m);
  });
}

// exclusive scan of in[0..n) into out[0..n), one kScanBlock chunk per
// workgroup; the chunk's total goes to tot[block]
__global__ __launch_bounds__(256) void k_scan_blocks(int n, const int32_t* __restrict__ in,
                                                      int32_t* __restrict__ out,
                                                      int32_t* __restrict__ tot) {
  __shared__ int32_t sh[256];
  const int base = blockIdx.x * kScanBlock + threadIdx.x * 4;
  int v[4], s = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    v[j] = base + j < n ? in[base + j] : 0;
    s += v[j];
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int d = 1; d < 256; d <<= 1) {  // inclusive scan of the lane totals
    const int o = threadIdx.x >= d ? sh[threadIdx.x - d] : 0;
    __syncthreads();
    sh[threadIdx.x] += o;
    __syncthreads();
  }
  int run = sh[threadIdx.x] - s;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (base + j < n) out[base + j] = run;
    run += v[j];
  }
  if (threadIdx.x == 255) tot[blockIdx.x] = sh[255];
}

// exclusive scan of the nb block totals in place (one workgroup, sequential
// chunks of 256); total of all at tot[nb]
__global__ __launch_bounds__(256) void k_scan_totals(int nb, int32_t* __restrict__ tot) {
  __shared__ int32_t sh[256];
  __shared__ int32_t carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int b0 = 0; b0 < nb; b0 += 256) {
    const int i = b0 + threadIdx.x;
    const int v = i < nb ? tot[i] : 0;
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int d = 1; d < 256; d <<= 1) {
      const int o = threadIdx.x >= d ? sh[threadIdx.x - d] : 0;
      __syncthreads();
      sh[threadIdx.x] += o;
      __syncthreads();
    }
    if (i < nb) tot[i] = carry + sh[threadIdx.x] - v;
    __syncthreads();
    if (threadIdx.x == 255) carry += sh[255];
    __syncthreads();
  }
  if (threadIdx.x == 0) tot[nb] = carry;
}

// colptr[i] += offset of its block; colptr[n] = the total; cursor = colptr
__global__ __launch_bounds__(256) void k_scan_add(int n, int32_t* __restrict__ colptr,
                                                   const int32_t* __restrict__ tot, int nb,
                                                   int32_t* __restrict__ cursor) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) {
    const int v = colptr[i] + tot[i / kScanBlock];
    colptr[i] = v;
    cursor[i] = v;
  }
  if (i == n) colptr[n] = tot[nb];
}

// every stored entry into its column's list (any order inside a list)
__global__ __launch_bounds__(256) void k_place(int n, const int32_t* __restrict__ ia,
                                                const int32_t* __restrict__ ja,
                                                int32_t* __restrict__ cursor,
                                                int32_t* __restrict__ colk,
                                                int32_t* __restrict__ colrow) {
  row_triples(n, ia, ja,
              [&](int64_t r, const int (&c)[3], int j0, int m, const int (&a)[3], int q) {
                int p = atomicAdd(&cursor[c[j0]], m);
#pragma unroll
                for (int j = 0; j < 3; ++j)
                  if (j >= j0 && c[j] == c[j0]) {
                    colk[p] = a[j] + q;
                    colrow[p] = (int)r + j;
                    ++p;
                  }
              });
}

// The list colk[a..b) ordered in place by one wavefront, with its rows
// (positions ascend with rows): Batcher's merge exchange, valid for any
// length.  Only lists the register path below cannot hold come here.
__device__ void sort_list(int a, int b, int32_t* colk, int32_t* colrow) {
  const int lane = threadIdx.x & 63, len = b - a;
  for (int64_t p = 1; p < len; p <<= 1)
    for (int64_t d = p; d >= 1; d >>= 1) {
      // pairs (i, i + d), i = (d mod p) + 2 d j + (0..d-1), inside one 2p group
      const int64_t off = d % p;
      for (int64_t q = lane;; q += 64) {
        const int64_t i = off + 2 * d * (q / d) + q % d;
        if (i + d >= len) break;  // i grows with q
        if (i / (2 * p) == (i + d) / (2 * p)) {
          const int32_t k0 = colk[a + i], k1 = colk[a + i + d];
          if (k0 > k1) {
            const int32_t r0 = colrow[a + i];
            colk[a + i] = k1;
            colk[a + i + d] = k0;
            colrow[a + i] = colrow[a + i + d];
            colrow[a + i + d] = r0;
          }
        }
      }
      // the next step reads what other lanes of this wavefront stored
      __threadfence_block();
      __builtin_amdgcn_wave_barrier();
    }
}

// y = A x from the transposed lists in any order.  One wavefront takes kCols
// rows at a time.  Products are formed by all lanes (row entries and list
// entries are contiguous, so their loads coalesce) and land in LDS in the
// order of the sum: row entries first, then the list's entries at their rank,
// found by comparing every key of the list (a broadcast LDS read serves four
// keys).  One lane per row then adds its products one after the other, since
// the order of the reference's sums is kept.  Rows with more than kSlots
// products, or lists of more than 64 entries, are ordered in place and added
// in pieces of 64.  Eight rows per wavefront: 36 KiB of LDS per workgroup,
// four workgroups per CU.
constexpr int kCols = 8, kSlots = 128;
__global__ __launch_bounds__(256) void k_sort_gather(int n, const int32_t* __restrict__ ia,
                                                      const int32_t* __restrict__ ja,
                                                      const double* __restrict__ ad,
                                                      const double* __restrict__ al,
                                                      const int32_t* __restrict__ colptr,
                                                      int32_t* colk, int32_t* colrow,
                                                      const double* __restrict__ x,
                                                      double* __restrict__ y) {
#pragma clang fp contract(off)
  __shared__ double prod[4][kCols][kSlots + 1];  // (odd stride: the summing lanes' banks differ)
  __shared__ __align__(16) int32_t keys[4][kCols][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  double(*pr)[kSlots + 1] = prod[w];
  for (int64_t i0 = ((int64_t)blockIdx.x * 4 + w) * kCols; i0 < n;
       i0 += (int64_t)gridDim.x * 4 * kCols) {
    const int nc = (int)min((int64_t)kCols, n - i0);
    // lane c < nc holds the bounds of row i0 + c and of its list
    int k1 = 0, k2 = 0, c1 = 0, c2 = 0;
    if (lane < nc) {
      k1 = ia[i0 + lane] - 1;
      k2 = ia[i0 + lane + 1] - 1;
      c1 = colptr[i0 + lane];
      c2 = colptr[i0 + lane + 1];
    }
    const bool fits = (int64_t)(k2 - k1) + (c2 - c1) <= kSlots && k2 - k1 <= 64 && c2 - c1 <= 64;
    int key[kCols];
    double pc[kCols];
#pragma unroll
    for (int c = 0; c < kCols; ++c) {
      const bool f = __shfl((int)fits, c, 64) != 0 && c < nc;
      const int a1 = __shfl(k1, c, 64), a2 = f ? __shfl(k2, c, 64) : a1;
      const int b1 = __shfl(c1, c, 64), b2 = f ? __shfl(c2, c, 64) : b1;
      key[c] = INT32_MAX;
      pc[c] = 0.0;
      if (b1 + lane < b2) {
        key[c] = colk[b1 + lane];
        pc[c] = al[key[c]] * x[colrow[b1 + lane]];
      }
      keys[w][c][lane] = key[c];
      if (a1 + lane < a2) pr[c][lane] = al[a1 + lane] * x[ja[a1 + lane] - 1];
    }
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
#pragma unroll
    for (int c = 0; c < kCols; ++c) {
      const int a1 = __shfl(k1, c, 64), a2 = __shfl(k2, c, 64);
      const int b1 = __shfl(c1, c, 64), b2 = __shfl(c2, c, 64);
      if (!__shfl((int)fits, c, 64) || c >= nc) continue;
      int rank = 0;
      const int4* kv = reinterpret_cast<const int4*>(keys[w][c]);
      for (int q = 0; 4 * q < b2 - b1; ++q) {  // (entries past the end hold INT32_MAX)
        const int4 v = kv[q];
        rank += (v.x < key[c]) + (v.y < key[c]) + (v.z < key[c]) + (v.w < key[c]);
      }
      if (b1 + lane < b2) pr[c][a2 - a1 + rank] = pc[c];
    }
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
    if (lane < nc && fits) {
      const int m = (k2 - k1) + (c2 - c1);
      double t = ad[i0 + lane] * x[i0 + lane];
      int q = 0;
      for (; q + 8 <= m; q += 8) {  // eight LDS reads in flight, added in order
        double v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = pr[lane][q + j];
#pragma unroll
        for (int j = 0; j < 8; ++j) t = t + v[j];
      }
      for (; q < m; ++q) t = t + pr[lane][q];
      y[i0 + lane] = t;
    }
    __builtin_amdgcn_wave_barrier();
    for (int c = 0; c < nc; ++c) {  // rows and lists that do not fit
      if (__shfl((int)fits, c, 64)) continue;
      const int a1 = __shfl(k1, c, 64), a2 = __shfl(k2, c, 64);
      const int b1 = __shfl(c1, c, 64), b2 = __shfl(c2, c, 64);
      sort_list(b1, b2, colk, colrow);
      double t = ad[i0 + c] * x[i0 + c];
      for (int part = 0; part < 2; ++part) {
        const int s1 = part ? b1 : a1, s2 = part ? b2 : a2;
        for (int s = s1; s < s2; s += 64) {
          const int m = min(64, s2 - s);
          if (lane < m)
            pr[0][lane] = part ? al[colk[s + lane]] * x[colrow[s + lane]]
                               : al[s + lane] * x[ja[s + lane] - 1];
          __builtin_amdgcn_wave_barrier();
          __threadfence_block();
          for (int q = 0; q < m; ++q) t = t + pr[0][q];
          __builtin_amdgcn_wave_barrier();
          __threadfence_block();
        }
      }
      if (lane == 0) y[i0 + c] = t;
    }
  }
}

int grid_of(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 16384)); }

}  // namespace
}  // namespace elastic

extern "C" int elastic_spmv_csrc_noalloc(int32_t neq, int64_t nad, const int32_t* ia,
                                         const int32_t* ja, const double* ad, const double* al,
                                         const double* x, double* y, void* stream) {
  using namespace elastic;
  if (neq <= 0 || nad < 0 || !ia || (nad > 0 && (!ja || !al)) || !ad || !x || !y)
    return ELASTIC_BAD_ARG;
  if (nad > INT32_MAX - 1 || scratch_words(neq, nad) > kScratchWords) {
    fprintf(stderr,
            "elastic_spmv_csrc_noalloc: neq %d, nad %lld need %lld scratch words; the fixed "
            "scratch holds %lld (2 neq + 2 nad + neq/1024 + 2 <= %lld)\n",
            neq, (long long)nad, (long long)scratch_words(neq, nad), (long long)kScratchWords,
            (long long)kScratchWords);
    return ELASTIC_BAD_ARG;
  }
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return ELASTIC_HIP_ERROR;
  std::call_once(g_once[dev], [dev]() {
    void* p = nullptr;
    g_status[dev] = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (g_status[dev] == hipSuccess) g_scratch[dev] = static_cast<int32_t*>(p);
  });
  if (g_status[dev] != hipSuccess || !g_scratch[dev]) {
    fprintf(stderr, "elastic_spmv_csrc_noalloc: hipGetSymbolAddress(scratch): %s\n",
            hipGetErrorString(g_status[dev]));
    return ELASTIC_HIP_ERROR;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  int32_t* cnt = g_scratch[dev];  // later the placement cursor
  int32_t* colptr = cnt + neq;
  int32_t* colk = colptr + neq + 1;
  int32_t* colrow = colk + nad;
  int32_t* tot = colrow + nad;
  const int nb = (neq + kScanBlock - 1) / kScanBlock;
  hipLaunchKernelGGL(k_fill, dim3(grid_of(neq)), dim3(256), 0, s, (int64_t)neq, cnt, 0);
  if (nad > 0)
    hipLaunchKernelGGL(k_count_cols, dim3(grid_of(32 * (int64_t)(neq / 3 + 1))), dim3(256), 0, s,
                       (int)neq, ia, ja, cnt);
  hipLaunchKernelGGL(k_scan_blocks, dim3(nb), dim3(256), 0, s, neq, (const int32_t*)cnt, colptr,
                     tot);
  hipLaunchKernelGGL(k_scan_totals, dim3(1), dim3(256), 0, s, nb, tot);
  hipLaunchKernelGGL(k_scan_add, dim3((neq + 1 + 255) / 256), dim3(256), 0, s, neq, colptr,
                     (const int32_t*)tot, nb, cnt);
  if (nad > 0) {
    hipLaunchKernelGGL(k_place, dim3(grid_of(32 * (int64_t)(neq / 3 + 1))), dim3(256), 0, s, neq,
                       ia, ja, cnt, colk, colrow);
  }
  hipLaunchKernelGGL(k_sort_gather, dim3(grid_of(8 * (int64_t)neq)), dim3(256), 0, s, neq, ia, ja,
                     ad, al, (const int32_t*)colptr, colk, colrow, x, y);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    fprintf(stderr, "elastic_spmv_csrc_noalloc: %s\n", hipGetErrorString(e));
    return ELASTIC_HIP_ERROR;
  }
  return ELASTIC_OK;
}
