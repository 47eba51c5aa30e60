// Tile layout of a large SpMV direction: row sums accumulated in LDS.
//
// A direction (rows x cols) is cut into units of (row tile, column segment).
// One 1024-thread workgroup runs a unit: an FP64 accumulator per row of the
// tile stays in LDS, and the unit's nonzeros stream past in column order, so
// a wave's 64 gathers of x fall into a few cache lines.  Entries come in
// batches of 1024, one per thread, whose rows are all different: a batch's
// adds never meet in one accumulator, and a barrier orders the batches, so
// every row is summed in one fixed order (bit-identical run to run) with
// plain LDS adds and no pass over row pointers.
//
// What bounds it (2,000,000 x 1,000,000, 32M nonzeros, FP64, MI355X): the
// streams alone (12 bytes per nonzero, the gathers made coalesced) take 72 us,
// the gathers bring the kernel to 107 us: each unit requests every cache line
// of its segment of x from L2 once, (rows / tile rows) * cols / 16 lines in
// all, which is why the tiles are as tall as the LDS allows; the adds and the
// barriers hide behind the loads (with the adds left out 110-118 us).  The
// column-sorted layout with every panel in one launch, which stages products
// instead of sums in LDS (1/16 of the nonzeros per block), takes 183 us, and
// its combine reads eight row-sum arrays where this one reads two.
#include <rocprim/device/device_radix_sort.hpp>

#include <algorithm>
#include <cstdlib>
#include <vector>

#include "pk_internal.h"

namespace pk {

namespace {

constexpr int kTB = kTileThreads;
// word: (column - batch base) << kTileRowBits | row in tile; a padding entry
// carries kTilePad as its row and adds nothing
constexpr int kTileRowBits = 15;
constexpr unsigned kTilePad = (1u << kTileRowBits) - 1u;
constexpr unsigned kTileSpan = 1u << (32 - kTileRowBits);
static_assert(kTileRows <= static_cast<int>(kTilePad), "tile rows fit the word");
// groups of batches the kernel loads together divide a unit's batch count
constexpr int kTileBatchPad = 4;

int bits_for(long long n) {
  int b = 1;
  while ((1LL << b) < n) ++b;
  return b;
}

__device__ __forceinline__ void lds_add(double* p, double v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Orders the workgroup's LDS operations only: loads from global memory stay
// in flight across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Workgroup w runs unit w.  Streams and batch bases are loaded three groups of
// U batches ahead, x is gathered one group ahead, in four register stages of a
// loop unrolled by four (no stage is copied).  The gathers bound it: without
// them the 2M x 1M, FP64, 32M directions take 80 us instead of 123 and 111,
// 1M x 500k, FP32, 16M 25 and 35 instead of 51 and 43; without the adds
// instead 115 and 111, 45 and 48.  Streams two groups ahead and each base read
// beside its gather: 1 to 2% longer in FP64, FP32 51.5 and 43.4 us instead of
// 47.8 and 42.6; x two groups ahead: the same or longer.  U = 1 / 2 / 4 / 6
// (streams two ahead, first of these) 110 / 107 / 117 / 126 us; two 512-thread
// workgroups per CU on half the rows each 121-141 us.
// last: the unit is its rows' only segment; the epilogue y = T(sum - c yprev)
// and the partials follow.  Otherwise the sums go to ypart[segment].
template <typename VT, typename T, int U>
__global__ __launch_bounds__(kTB) void k_spmv_tile(
    const TileDesc* __restrict__ desc, const int* __restrict__ base,
    const unsigned* __restrict__ wd, const VT* __restrict__ va, const T* __restrict__ x,
    T* __restrict__ y, const T* __restrict__ yprev, Scal coef, double* __restrict__ part,
    double* __restrict__ ypart, long long rows, int last, Gate gate) {
  const TileDesc t = desc[blockIdx.x];
  const bool off = gate.off();
  ready(t.b0);
  if (off) return;
  extern __shared__ double acc[];
  __shared__ double lds[(kTB / kWave) * 2];
  const int ng = t.nb / U;  // groups of U batches; at least one
  const unsigned* __restrict__ w0 = wd + static_cast<long long>(t.b0) * kTB + threadIdx.x;
  const VT* __restrict__ v0 = va + static_cast<long long>(t.b0) * kTB + threadIdx.x;
  const int* __restrict__ bb = base + t.b0;
  struct Stage {
    unsigned w[U];
    VT v[U];
    T x[U];
    int n[U];
  };
  Stage a, b, c, d;
  // groups past the end load the last one again and are not added
  auto load = [&](int g, Stage& q) {
    const int gb = min(g, ng - 1) * U;
    const long long o = static_cast<long long>(gb) * kTB;
#pragma unroll
    for (int u = 0; u < U; ++u) q.w[u] = __builtin_nontemporal_load(w0 + o + u * kTB);
#pragma unroll
    for (int u = 0; u < U; ++u) q.v[u] = __builtin_nontemporal_load(v0 + o + u * kTB);
#pragma unroll
    for (int u = 0; u < U; ++u) q.n[u] = bb[gb + u];
  };
  auto gather = [&](Stage& q) {
#pragma unroll
    for (int u = 0; u < U; ++u) q.x[u] = x[q.n[u] + static_cast<int>(q.w[u] >> kTileRowBits)];
  };
  auto add = [&](const Stage& q) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const unsigned r = q.w[u] & kTilePad;
      if (r != kTilePad)
        lds_add(acc + r, static_cast<double>(q.v[u]) * static_cast<double>(q.x[u]));
      lds_barrier();
    }
  };
  load(0, a);
  load(1, b);
  load(2, c);
  for (int i = threadIdx.x; i < t.nrows; i += kTB) acc[i] = 0.0;
  gather(a);
  lds_barrier();
  for (int g = 0;;) {
    gather(b);
    load(g + 3, d);
    add(a);
    if (++g >= ng) break;
    gather(c);
    load(g + 3, a);
    add(b);
    if (++g >= ng) break;
    gather(d);
    load(g + 3, b);
    add(c);
    if (++g >= ng) break;
    gather(a);
    load(g + 3, c);
    add(d);
    if (++g >= ng) break;
  }
  if (!last) {
    double* __restrict__ out = ypart + static_cast<long long>(t.seg) * rows + t.row0;
    for (int i = threadIdx.x; i < t.nrows; i += kTB) out[i] = acc[i];
    return;
  }
  const double cf = coef.get();
  double s[2] = {0.0, 0.0};
  for (int i = threadIdx.x; i < t.nrows; i += kTB) {
    const double yp = yprev ? static_cast<double>(yprev[t.row0 + i]) : 0.0;
    const T yv = static_cast<T>(acc[i] - cf * yp);
    y[t.row0 + i] = yv;
    s[0] += static_cast<double>(yv) * static_cast<double>(yv);
    s[1] += yp * static_cast<double>(yv);
  }
  block_sum<2, kTB>(s, lds);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = s[0];
    part[gridDim.x + blockIdx.x] = s[1];
  }
}

// ---------------------------------------------------------------- build ----
// key = unit << cbits | column in segment, and the row in its tile, of every
// nonzero of one source CSR (a column panel, or the whole direction): one
// thread per nonzero, the row by binary search in rp, the tile in bound.
__global__ void k_tile_keys(int rows, long long nnz, const int* __restrict__ rp,
                            const int* __restrict__ ci, int ntile, const int* __restrict__ bound,
                            int nseg, int width, int cbits, long long off,
                            unsigned* __restrict__ key, int* __restrict__ pos,
                            unsigned short* __restrict__ trow) {
  for (long long p = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; p < nnz;
       p += static_cast<long long>(gridDim.x) * blockDim.x) {
    int lo = 0, hi = rows;  // rp[lo] <= p < rp[hi]
    while (hi - lo > 1) {
      const int mid = lo + (hi - lo) / 2;
      if (rp[mid] <= p)
        lo = mid;
      else
        hi = mid;
    }
    int t = 0, te = ntile;  // bound[t] <= row < bound[te]
    while (te - t > 1) {
      const int mid = t + (te - t) / 2;
      if (bound[mid] <= lo)
        t = mid;
      else
        te = mid;
    }
    const int col = ci[p], seg = col / width;
    const unsigned unit = static_cast<unsigned>(t * nseg + seg);
    key[off + p] = (unit << cbits) | static_cast<unsigned>(col - seg * width);
    pos[off + p] = static_cast<int>(off + p);
    trow[off + p] = static_cast<unsigned short>(lo - bound[t]);
  }
}

// uptr[u] = first sorted key of unit u (uptr[nunit] = nnz).
__global__ void k_tile_unit_ptr(long long nnz, const unsigned* __restrict__ key, int cbits,
                                int nunit, int* __restrict__ uptr) {
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u > nunit) return;
  long long lo = 0, hi = nnz;
  while (lo < hi) {
    const long long mid = lo + (hi - lo) / 2;
    if (static_cast<int>(key[mid] >> cbits) < u)
      lo = mid + 1;
    else
      hi = mid;
  }
  uptr[u] = static_cast<int>(lo);
}

// Batches of one unit.  The unit's entries are taken in column order through
// a window of 2048 candidates (those an earlier batch left over first): of
// the candidates with one row the first wins, the first 1024 winners within
// kTileSpan columns of the first candidate make the batch, the others stay.
// The first candidate always wins, so every batch makes progress; a unit that
// needs more batches than its room (desc.nb on entry) sets *full.
constexpr int kTileWindow = 2 * kTB;
constexpr int kTileOrderBits = 11;
static_assert((1 << kTileOrderBits) == kTileWindow, "the claim code holds a candidate's order");

template <typename VT>
__global__ __launch_bounds__(kTB) void k_tile_batches(
    TileDesc* __restrict__ desc, const int* __restrict__ uptr, const unsigned* __restrict__ key,
    const int* __restrict__ pos, const unsigned short* __restrict__ trow,
    const VT* __restrict__ va, int nseg, int width, int cbits, int* __restrict__ base,
    unsigned* __restrict__ wd, VT* __restrict__ tva, int* __restrict__ full) {
  extern __shared__ unsigned owner[];  // per row: lowest claim code so far
  __shared__ int cpos[kTileWindow], ccol[kTileWindow];
  __shared__ unsigned short crow[kTileWindow];
  __shared__ int wsum[kTB / kWave + 1];
  const int unit = blockIdx.x;
  const TileDesc t = desc[unit];
  const int col0 = (unit % nseg) * width;
  const unsigned cmask = (1u << cbits) - 1u;
  const int lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
  for (int i = threadIdx.x; i < t.nrows; i += kTB) owner[i] = 0xffffffffu;
  int next = uptr[unit];
  const int end = uptr[unit + 1];
  int npend = 0, nb = 0;
  const int room = t.nb;
  __syncthreads();
  while (npend > 0 || next < end) {
    if (nb >= room) {  // uniform
      if (threadIdx.x == 0) *full = 1;
      break;
    }
    const int nnew = min(kTileWindow - npend, end - next);
    const int nc = npend + nnew;
    // later batches claim with lower codes, so nothing is cleared in between
    const unsigned code0 = ((1u << (32 - kTileOrderBits)) - 2u - static_cast<unsigned>(nb))
                           << kTileOrderBits;
    int p[2], col[2], r[2];
    bool in[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int i = 2 * static_cast<int>(threadIdx.x) + k;
      in[k] = i < nc;
      p[k] = col[k] = r[k] = 0;
      if (i < npend) {
        p[k] = cpos[i];
        col[k] = ccol[i];
        r[k] = crow[i];
      } else if (in[k]) {
        const int q = next + i - npend;
        p[k] = pos[q];
        col[k] = col0 + static_cast<int>(key[q] & cmask);
        r[k] = trow[p[k]];
      }
      if (in[k]) atomicMin(owner + r[k], code0 | static_cast<unsigned>(i));
    }
    if (threadIdx.x == 0) wsum[kTB / kWave] = col[0];
    __syncthreads();
    const int first = wsum[kTB / kWave];
    bool win[2];
    int cnt = 0;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const unsigned i = 2u * threadIdx.x + static_cast<unsigned>(k);
      win[k] = in[k] && owner[r[k]] == (code0 | i) &&
               static_cast<unsigned>(col[k] - first) < kTileSpan;
      cnt += win[k] ? 1 : 0;
    }
    int incl = cnt;  // inclusive scan of the winners over the workgroup
    for (int o = 1; o < kWave; o <<= 1) {
      const int v = __shfl_up(incl, o, kWave);
      if (lane >= o) incl += v;
    }
    if (lane == kWave - 1) wsum[wid] = incl;
    __syncthreads();
    int before = 0, total = 0;
    for (int w = 0; w < kTB / kWave; ++w) {
      if (w < wid) before += wsum[w];
      total += wsum[w];
    }
    const int nemit = min(total, kTB);
    int rank = before + incl - cnt;
    const long long o0 = (static_cast<long long>(t.b0) + nb) * kTB;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int i = 2 * static_cast<int>(threadIdx.x) + k;
      const bool emit = win[k] && rank < kTB;
      if (emit) {
        wd[o0 + rank] = (static_cast<unsigned>(col[k] - first) << kTileRowBits) |
                        static_cast<unsigned>(r[k]);
        tva[o0 + rank] = va[p[k]];
      } else if (in[k]) {
        const int j = i - min(rank, kTB);  // order among those left
        cpos[j] = p[k];
        ccol[j] = col[k];
        crow[j] = static_cast<unsigned short>(r[k]);
      }
      rank += win[k] ? 1 : 0;
    }
    if (static_cast<int>(threadIdx.x) >= nemit) {
      wd[o0 + threadIdx.x] = kTilePad;
      tva[o0 + threadIdx.x] = VT(0);
    }
    if (threadIdx.x == 0) base[t.b0 + nb] = first;
    next += nnew;
    npend = nc - nemit;
    ++nb;
    __syncthreads();
  }
  // whole groups, at least one: empty batches of padding (the room is a
  // multiple of kTileBatchPad)
  const int npad = max((nb + kTileBatchPad - 1) / kTileBatchPad, 1) * kTileBatchPad;
  for (int q = nb; q < npad && q < room; ++q) {
    const long long o0 = (static_cast<long long>(t.b0) + q) * kTB;
    wd[o0 + threadIdx.x] = kTilePad;
    tva[o0 + threadIdx.x] = VT(0);
    if (threadIdx.x == 0) base[t.b0 + q] = 0;
  }
  if (threadIdx.x == 0) desc[unit].nb = min(npad, room);
}

// Segments and tiles of a direction: one unit per CU (the LDS holds one
// tile) in every round.  Taller tiles and more segments ask L2 for fewer
// lines of x ((rows / tile rows) * cols * xbytes / 64 requests, which cost
// about 1 us per 460,000 beyond the streams: 2,000,000 x 1,000,000 above), but
// every segment writes a row-sum array that the combine reads back (5 GB/ms,
// and a launch).  Measured (us, FP64): 1,000,000 x 2,000,000 with 32M
// nonzeros, 2 / 4 / 5 segments 153 / 117 / 115; 270,000 x 140,000 with 4.3M,
// 16 / 3 segments 42 / 25 (row-block layout 32).  Tiles of about 2100 rows or
// fewer cannot fill their batches of distinct rows (an eighth of them would be
// padding); three batches' rows are asked for.  Past 256 full tiles: one segment, whole rounds of 256 tiles.
constexpr int kTileCus = 256;

void tile_shape(int rows, int cols, size_t xbytes, int* nseg, int* ntile) {
  double best = 0.0;
  *nseg = 0;
  for (int s = 1; s <= kMaxTileSegs; ++s) {
    const int nt = kTileCus / s, r = (rows + nt - 1) / nt;
    if (r > kTileRows || (r < 3 * kTB && s < kMaxTileSegs)) continue;
    const double us = static_cast<double>(nt) * cols * xbytes / 64.0 / 460e3 +
                      (s > 1 ? 4.0 + s * 16.0 * rows / 5e6 : 0.0);
    if (*nseg == 0 || us < best) {
      best = us;
      *nseg = s;
      *ntile = nt;
    }
  }
  if (*nseg > 0) return;
  const long long per = static_cast<long long>(kTileCus) * kTileRows;
  *nseg = 1;
  *ntile = static_cast<int>((rows + per - 1) / per) * kTileCus;
}

// Row bounds of the tiles: equal shares of the nonzeros, at most kTileRows
// rows each (more tiles than asked for where rows are empty).
std::vector<int> tile_bounds(const std::vector<int>& rp, int rows, int ntile) {
  const double share = static_cast<double>(rp[rows]) / ntile;
  std::vector<int> b{0};
  while (b.back() < rows) {
    const int r0 = b.back();
    const double want = share * static_cast<double>(b.size());
    int r = static_cast<int>(std::lower_bound(rp.begin() + r0, rp.begin() + rows + 1, want,
                                              [](int v, double w) { return v < w; }) -
                             rp.begin());
    r = std::min(std::max(r, r0 + 1), rows);
    if (static_cast<int>(b.size()) >= ntile) r = rows;
    b.push_back(std::min(r, r0 + kTileRows));
  }
  return b;
}

}  // namespace

void tile_free(TileLayout& L) {
  (void)hipFree(L.desc);
  (void)hipFree(L.base);
  (void)hipFree(L.wd);
  (void)hipFree(L.va);
  (void)hipFree(L.ypart);
  L = TileLayout{};
}

// Builds L from the source CSRs (column panels of one direction, over all
// rows).  PK_ERR_NOTSUP where the layout does not suit the matrix (see
// tile_wanted and the checks below); L is then empty.
template <typename VT>
static int build(TileLayout& L, int rows, int cols, const TileSource* src, int nsrc,
                 hipStream_t s) {
  long long nnz = 0;
  for (int i = 0; i < nsrc; ++i) nnz += src[i].nnz;
  int nseg = 1, ntile = 1;
  tile_shape(rows, cols, sizeof(VT), &nseg, &ntile);
  std::vector<int> rp(static_cast<size_t>(rows) + 1), one;
  if (hipMemcpy(rp.data(), src[0].rp, sizeof(int) * rp.size(), hipMemcpyDeviceToHost) !=
      hipSuccess)
    return PK_ERR_HIP;
  for (int i = 1; i < nsrc; ++i) {
    one.resize(rp.size());
    if (hipMemcpy(one.data(), src[i].rp, sizeof(int) * one.size(), hipMemcpyDeviceToHost) !=
        hipSuccess)
      return PK_ERR_HIP;
    for (size_t r = 0; r < rp.size(); ++r) rp[r] += one[r];
  }
  const std::vector<int> bound = tile_bounds(rp, rows, ntile);
  ntile = static_cast<int>(bound.size()) - 1;
  const int nunit = ntile * nseg, width = (cols + nseg - 1) / nseg;
  const int cbits = bits_for(width);
  if (cbits + bits_for(nunit) > 32) return PK_ERR_NOTSUP;
  int maxrows = 0;
  for (int t = 0; t < ntile; ++t) maxrows = std::max(maxrows, bound[t + 1] - bound[t]);

  unsigned *key = nullptr, *key2 = nullptr;
  int *pos = nullptr, *pos2 = nullptr, *dbound = nullptr, *uptr = nullptr, *full = nullptr;
  unsigned short* trow = nullptr;
  void *tmp = nullptr, *vall = nullptr;
  size_t tmp_bytes = 0;
  int rc = PK_OK;
  long long off = 0, nbatch = 0;
  std::vector<int> up(static_cast<size_t>(nunit) + 1);
  std::vector<TileDesc> desc(nunit);
  const size_t nz = static_cast<size_t>(nnz);
  const void* vsrc = src[0].va;
  int hfull = 0, maxunit = 0;
#define PKT(x)             \
  if ((x) != hipSuccess) { \
    rc = PK_ERR_HIP;       \
    goto out;              \
  }
  PKT(hipMalloc(&key, sizeof(unsigned) * nz));
  PKT(hipMalloc(&key2, sizeof(unsigned) * nz));
  PKT(hipMalloc(&pos, sizeof(int) * nz));
  PKT(hipMalloc(&pos2, sizeof(int) * nz));
  PKT(hipMalloc(&trow, sizeof(unsigned short) * nz));
  PKT(hipMalloc(&dbound, sizeof(int) * bound.size()));
  PKT(hipMalloc(&uptr, sizeof(int) * up.size()));
  PKT(hipMalloc(&full, sizeof(int)));
  PKT(hipMemcpyAsync(dbound, bound.data(), sizeof(int) * bound.size(), hipMemcpyHostToDevice, s));
  PKT(hipMemcpyAsync(full, &hfull, sizeof(int), hipMemcpyHostToDevice, s));
  if (nsrc > 1) {
    PKT(hipMalloc(&vall, sizeof(VT) * nz));
    vsrc = vall;
  }
  for (int i = 0; i < nsrc; ++i) {
    if (src[i].nnz == 0) continue;
    hipLaunchKernelGGL(k_tile_keys, dim3(4096), dim3(256), 0, s, rows, src[i].nnz, src[i].rp,
                       src[i].ci, ntile, dbound, nseg, width, cbits, off, key, pos, trow);
    if (nsrc > 1)
      PKT(hipMemcpyAsync(static_cast<VT*>(vall) + off, src[i].va, sizeof(VT) * src[i].nnz,
                         hipMemcpyDeviceToDevice, s));
    off += src[i].nnz;
  }
  PKT(hipGetLastError());
  PKT(rocprim::radix_sort_pairs(nullptr, tmp_bytes, key, key2, pos, pos2, nz, 0,
                                cbits + bits_for(nunit), s));
  PKT(hipMalloc(&tmp, std::max<size_t>(tmp_bytes, 1)));
  PKT(rocprim::radix_sort_pairs(tmp, tmp_bytes, key, key2, pos, pos2, nz, 0,
                                cbits + bits_for(nunit), s));
  hipLaunchKernelGGL(k_tile_unit_ptr, dim3((nunit + 256) / 256), dim3(256), 0, s, nnz, key2,
                     cbits, nunit, uptr);
  PKT(hipGetLastError());
  PKT(hipMemcpyAsync(up.data(), uptr, sizeof(int) * up.size(), hipMemcpyDeviceToHost, s));
  PKT(hipStreamSynchronize(s));
  for (int u = 0; u < nunit; ++u) {
    const int n = up[u + 1] - up[u], t = u / nseg;
    maxunit = std::max(maxunit, n);
    // an eighth more batches than full ones would take, and a group of slack
    const long long need = (static_cast<long long>(n) + kTB - 1) / kTB;
    const long long room =
        (need + need / 8 + 2 * kTileBatchPad) / kTileBatchPad * kTileBatchPad;
    desc[u] = TileDesc{bound[t], bound[t + 1] - bound[t], static_cast<int>(nbatch),
                       static_cast<int>(room), u % nseg, 0, 0, 0};
    nbatch += room;
  }
  // one unit's workgroup holds the launch back: units must be alike (the
  // launch's rounds end with the largest unit)
  if (static_cast<double>(maxunit) * std::min(nunit, kTileCus) >
          kTileImbalance * static_cast<double>(nnz) ||
      nbatch >= (1LL << 31) / kTB * 2) {
    rc = PK_ERR_NOTSUP;
    goto out;
  }
  PKT(hipMalloc(&L.desc, sizeof(TileDesc) * nunit));
  PKT(hipMalloc(&L.base, sizeof(int) * nbatch));
  PKT(hipMalloc(&L.wd, sizeof(unsigned) * nbatch * kTB));
  PKT(hipMalloc(&L.va, sizeof(VT) * nbatch * kTB));
  if (nseg > 1) PKT(hipMalloc(&L.ypart, sizeof(double) * nseg * static_cast<size_t>(rows)));
  PKT(hipMemcpyAsync(L.desc, desc.data(), sizeof(TileDesc) * nunit, hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL((k_tile_batches<VT>), dim3(nunit), dim3(kTB), sizeof(unsigned) * maxrows, s,
                     L.desc, uptr, key2, pos2, trow, static_cast<const VT*>(vsrc), nseg, width,
                     cbits, L.base, L.wd, static_cast<VT*>(L.va), full);
  PKT(hipGetLastError());
  PKT(hipMemcpyAsync(&hfull, full, sizeof(int), hipMemcpyDeviceToHost, s));
  PKT(hipStreamSynchronize(s));
  if (hfull) {  // rows too long for their tile: more padding than the layout gains
    rc = PK_ERR_NOTSUP;
    goto out;
  }
  L.nunit = nunit;
  L.nseg = nseg;
  L.maxrows = maxrows;
out:
#undef PKT
  (void)hipStreamSynchronize(s);
  (void)hipFree(key);
  (void)hipFree(key2);
  (void)hipFree(pos);
  (void)hipFree(pos2);
  (void)hipFree(trow);
  (void)hipFree(dbound);
  (void)hipFree(uptr);
  (void)hipFree(full);
  (void)hipFree(tmp);
  (void)hipFree(vall);
  if (rc != PK_OK) {
    (void)hipGetLastError();
    tile_free(L);
  }
  return rc;
}

int tile_build(TileLayout& L, int rows, int cols, int val_prec, const TileSource* src, int nsrc,
               hipStream_t s) {
  tile_free(L);
  if (val_prec == PK_F64) return build<double>(L, rows, cols, src, nsrc, s);
  if (val_prec == PK_F32) return build<float>(L, rows, cols, src, nsrc, s);
  return PK_ERR_NOTSUP;
}

template <typename VT, typename T>
int launch_spmv_tile(hipStream_t s, const TileLayout& L, long long rows, const T* x, T* y,
                     const T* yprev, Scal coef, double* part, double* ypart, Gate gate) {
  if (L.nunit <= 0 || (L.nseg > 1 && !ypart)) return -1;
  const size_t shm = sizeof(double) * static_cast<size_t>(L.maxrows);
  hipLaunchKernelGGL((k_spmv_tile<VT, T, 2>), dim3(L.nunit), dim3(kTB), shm, s, L.desc, L.base,
                     L.wd, static_cast<const VT*>(L.va), x, y, yprev, coef, part, ypart, rows,
                     L.nseg == 1 ? 1 : 0, gate);
  if (hipGetLastError() != hipSuccess) return -1;
  if (L.nseg == 1) return L.nunit;
  return launch_spmv_combine<T>(s, rows, L.nseg, ypart, yprev, coef, y, part, gate);
}

#define PK_INST_TILE(VT, T)                                                                   \
  template int launch_spmv_tile<VT, T>(hipStream_t, const TileLayout&, long long, const T*, T*, \
                                       const T*, Scal, double*, double*, Gate);
PK_INST_TILE(double, double)
PK_INST_TILE(float, float)
PK_INST_TILE(double, float)
PK_INST_TILE(float, double)
#undef PK_INST_TILE

}  // namespace pk
