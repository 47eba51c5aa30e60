// Lanczos steps of a small problem in one launch.
//
// The step chains (Impl::enqueue_step) cost about 4.5 us per launch and 18
// launches per step, most of them gated off: on a 1850 x 712 matrix 83 us a
// step, of which the kernels' own work is a few.  Here a few workgroups stay
// resident for the whole DLANBPRO call.  Every workgroup keeps its own copy of
// the control state in LDS and runs every control stage itself, on the same
// partial sums and with the same code, so all of them take the same decisions
// and a step needs a grid barrier only where vectors or partial sums cross
// workgroups: after the pending scaling, the operator, an ELR update, and the
// two halves of a Gram-Schmidt pass.  Phases that do not run cost nothing.
//
// The bodies are the chain kernels' (pk_bodies.h) on the same slices, slots
// and orders: the results are bit for bit the chains' and the host executor's.
//
// The operator's nonzeros stay in LDS for the whole launch, so an application
// is one gather of x from memory and the row sums.  A half-step without ELR or
// reorthogonalization takes about 11 us on 110 workgroups (12007 x 5003, 112,000
// nonzeros): gather 2.0, rows 1.5, barrier 4, reduction 1.5, control stage 2.9;
// the chains took 33.
//
// The barrier is one device-scope counter: 1.3 / 1.5 / 1.9 / 3.1 / 5.7 / 8.2 us
// over 8 / 16 / 32 / 64 / 128 / 256 workgroups, with the release and acquire of
// the XCDs' L2s; meeting in eight groups first 4.5 / 6.3 us over 128 / 256 (2.9
// over 64).  The launch is cooperative (all workgroups resident, or refused:
// then the chains run), and every wait is bounded.
#include <algorithm>

#include "pk_bodies.h"
#include "pk_internal.h"

namespace pk {

namespace {

constexpr unsigned kSpinLimit = 1u << 26;  // about a minute

// All workgroups of the grid; epoch counts the barriers of the launch.  Past
// 64 workgroups they meet in eight groups first (those of one XCD, by the
// dispatch order; only speed depends on that).  False if the wait ran out
// (uniform over the workgroup).
__device__ bool grid_barrier(ResidentBar* bar, unsigned& epoch, int* flag) {
  __builtin_amdgcn_s_waitcnt(0);  // this wave's stores have reached the L2
  __syncthreads();
  ++epoch;
  if (threadIdx.x == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    const unsigned n = gridDim.x;
    unsigned* at = &bar->count;
    unsigned want = epoch * n;
    if (n > 64) {
      const unsigned g = blockIdx.x % 8, members = (n + 7 - g) / 8;
      const unsigned a = __hip_atomic_fetch_add(&bar->group[g * 32], 1u, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
      if (a + 1 == epoch * members) {
        const unsigned r =
            __hip_atomic_fetch_add(&bar->count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (r + 1 == epoch * 8)
          __hip_atomic_store(&bar->passed, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      at = &bar->passed;
      want = epoch;
    } else {
      __hip_atomic_fetch_add(&bar->count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    unsigned spin = 0;
    while (__hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < want &&
           ++spin < kSpinLimit)
      __builtin_amdgcn_s_sleep(1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    *flag = spin < kSpinLimit;
    if (spin >= kSpinLimit) bar->failed = 1;
  }
  __syncthreads();
  return *flag != 0;
}

// A workgroup's row blocks of both directions, held in LDS for the whole
// launch: nonzeros (columns, values) and row bounds.  Slots [0, kResSlots) are
// A's, the rest A^T's.
template <typename T>
struct ResidentSlot {
  T val[kSpmvCap];
  int idx[kSpmvCap];
  int rp[kSpmvRows + 1];
  int r0, r1, nz;
};

// Row sums and epilogue of a slot (spmv_rows with g lanes per row).
template <typename T>
__device__ __forceinline__ void resident_rows(int g, const ResidentSlot<T>& S, const double* prod,
                                              T* y, const T* yprev, double c, double* q_s2,
                                              double* q_sd, double* lds) {
  const int* rp = S.rp - S.r0;
  const T* yp = yprev ? yprev - S.r0 : nullptr;
  switch (g) {
#define PK_RES_CASE(G)                                                                      \
  case G:                                                                                   \
    spmv_rows<T, G, kBlock>(S.r0, S.r1, 0, rp, prod, y, yp, c, q_s2, q_sd, nullptr, nullptr, \
                            1, lds);                                                        \
    break;
    PK_RES_CASE(2)
    PK_RES_CASE(4)
    PK_RES_CASE(8)
    PK_RES_CASE(16)
    PK_RES_CASE(32)
    default:
      spmv_rows<T, 64, kBlock>(S.r0, S.r1, 0, rp, prod, y, yp, c, q_s2, q_sd, nullptr, nullptr, 1,
                               lds);
#undef PK_RES_CASE
  }
}

// Sum of n partials by one wave, in reduce_partials' order (thread t of 256
// adds p[t], p[t + 256], ...; the wave sums; the four waves in turn).
__device__ __forceinline__ double wave_reduce_partials(const double* p, int n, int lane) {
  double v[kBlock / kWave] = {};
  for (int i = 0; i < n; i += kBlock)
#pragma unroll
    for (int w = 0; w < kBlock / kWave; ++w) {
      const int q = i + w * kWave + lane;
      const double t = p[min(q, n - 1)];
      if (q < n) v[w] += t;
    }
  double s = 0.0;
#pragma unroll
  for (int w = 0; w < kBlock / kWave; ++w) s += wave_sum(v[w]);
  return s;
}

// Dynamic LDS: the slots, then per slot of one direction the products and the
// rows' previous vector.
template <typename T>
struct ResidentLds {
  ResidentSlot<T> slot[2 * kResSlots];
  double prod[kResSlots][kSpmvCap];
  T yp[kResSlots][kSpmvRows];
};

template <typename T>
__global__ __launch_bounds__(kBlock) void k_resident(ResidentArgs A) {
  extern __shared__ __align__(16) char dyn[];
  ResidentLds<T>& S = *reinterpret_cast<ResidentLds<T>*>(dyn);
  __shared__ LbdCtlLds c;
  __shared__ int cols[kCtlLdsJ + 4];
  __shared__ double sh[kCtlLdsJ + 4];
  __shared__ double lds[(kBlock / kWave) * 2];
  __shared__ double tile[2][(kBlock / kWave) * kCT];
  __shared__ int flag;
  const int t = static_cast<int>(threadIdx.x), lane = t % kWave, wid = t / kWave;
  const int grid = static_cast<int>(gridDim.x), me = static_cast<int>(blockIdx.x);
  T* const U = static_cast<T*>(A.U);
  T* const V = static_cast<T*>(A.V);
  unsigned epoch = 0;
  int buf = 0;
  // A vector's pending 1/alpha or 1/beta is applied as it is read (as x by
  // the other side's operator, then as the previous vector of its own side,
  // rounded to T as the stored scaling rounds it) and stored only when its
  // last unscaled reader is past a barrier: no barrier of its own.
  struct Pending {
    int has;
    double f;
    T* col;
  } pu{0, 1.0, nullptr}, pv{0, 1.0, nullptr};
  bool stored = false;  // scaled slices of a basis column not yet behind a barrier
  auto store_scaled = [&](Pending& p, long long L) {
    if (p.has) {
      for (long long s = me; s * kRowsPerBlock < L; s += grid) scale_body<T>(s, L, p.col, p.f);
      stored = true;
    }
    p.has = 0;
  };

  // this workgroup's row blocks, blocks me, me + grid, ... of each direction
#pragma unroll 1
  for (int q = 0; q < 2 * kResSlots; ++q) {
    const ResidentDir& D = q < kResSlots ? A.da : A.dt;
    const int d = me + (q % kResSlots) * grid;
    ResidentSlot<T>& R = S.slot[q];
    if (d >= D.ndesc) {
      if (t == 0) R.r0 = R.r1 = R.nz = -1;
      continue;
    }
    const int4 de = D.desc[d];
    const int p0 = D.rp[de.x], nz = D.rp[de.y] - p0;
    for (int i = t; i < nz; i += kBlock) {
      R.val[i] = static_cast<const T*>(D.va)[p0 + i];
      R.idx[i] = D.ci[p0 + i];
    }
    for (int i = t; i <= de.y - de.x; i += kBlock) R.rp[i] = D.rp[de.x + i] - p0;
    if (t == 0) {
      R.r0 = de.x;
      R.r1 = de.y;
      R.nz = nz;
    }
  }
  // the state: scalars, and the arrays' windows of the steps up to kCtlLdsJ
  const int nd = min(CtlArrays::dlen(A.cap), kCtlWinD), ni = min(CtlArrays::ilen(A.cap), kCtlWinI);
  {
    const int4* src = reinterpret_cast<const int4*>(A.ctl);
    int4* dst = reinterpret_cast<int4*>(static_cast<LbdCtl*>(&c));
    for (int i = t; i < kCtlHdrWords; i += kBlock) dst[i] = src[i];
    for (int i = t; i < nd; i += kBlock) {
      c.mu[i] = CtlArrays::mu(A.arrays, A.cap)[i];
      c.nu[i] = CtlArrays::nu(A.arrays, A.cap)[i];
      c.B1[i] = CtlArrays::B1(A.arrays, A.cap)[i];
      c.B2[i] = CtlArrays::B2(A.arrays, A.cap)[i];
    }
    for (int i = t; i < ni; i += kBlock) c.index[i] = CtlArrays::index(A.arrays, A.cap)[i];
    if (t == 0) c.cols = cols;
  }
  __syncthreads();

  for (;;) {
    const int phase = c.phase, j = c.j;  // the same in every workgroup
    if (phase < PH_V_SPMV || phase > PH_U_REO || j > kCtlLdsJ) break;
    const bool vside = phase <= PH_V_REO;
    const long long L = vside ? A.n : A.m;       // length of the vector of this side
    T* const basis = vside ? V : U;
    const long long ld = vside ? A.ldv : A.ldu;
    T* const w = basis + static_cast<long long>(vside ? j - 1 : j) * ld;
    const T* const wprev = vside && j == 1 ? nullptr : w - ld;
    double* part = A.part + buf * A.half;
    buf ^= 1;
    int nb, kind;
    double a, b = 0.0;
    if (phase == PH_V_SPMV || phase == PH_U_SPMV) {
      const T* const x = vside ? U + static_cast<long long>(j - 1) * A.ldu
                               : V + static_cast<long long>(j - 1) * A.ldv;
      const int sx = vside ? c.uscale : c.vscale;
      const double fx = vside ? c.uscale_f : c.vscale_f;
      const Pending py = vside ? pv : pu;  // of wprev
      const ResidentDir& D = vside ? A.dt : A.da;
      const ResidentSlot<T>* slot = S.slot + (vside ? kResSlots : 0);
      nb = D.ndesc;
      constexpr int kPer = kSpmvCap / kBlock;
      T xv[kResSlots][kPer], yv[kResSlots][kPer];
      // every gather and previous row in flight together
#pragma unroll
      for (int q = 0; q < kResSlots; ++q)
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
          const int i = t + k * kBlock;
          xv[q][k] = i < slot[q].nz ? x[slot[q].idx[i]] : T(0);
          yv[q][k] = wprev && i < slot[q].r1 - slot[q].r0 ? wprev[slot[q].r0 + i] : T(0);
        }
#pragma unroll
      for (int q = 0; q < kResSlots; ++q)
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
          const int i = t + k * kBlock;
          if (i < slot[q].nz) {
            const T xs = sx ? static_cast<T>(fx * static_cast<double>(xv[q][k])) : xv[q][k];
            S.prod[q][i] = static_cast<double>(slot[q].val[i]) * static_cast<double>(xs);
          }
          if (i < slot[q].r1 - slot[q].r0)
            S.yp[q][i] =
                py.has ? static_cast<T>(py.f * static_cast<double>(yv[q][k])) : yv[q][k];
        }
      __syncthreads();
      const double coef = vside ? c.beta : c.alpha;
#pragma unroll 1
      for (int q = 0; q < kResSlots; ++q) {
        const int d = me + q * grid;
        if (d < nb)
          resident_rows<T>(D.g, slot[q], S.prod[q], w, wprev ? S.yp[q] : nullptr, coef, part + d,
                           part + nb + d, lds);
      }
      if (!grid_barrier(A.bar, epoch, &flag)) return;
      stored = false;
      // x keeps its factor until it has been the previous vector; wprev has
      // been, and takes it now
      if (vside) {
        store_scaled(pv, A.n);
        pu = Pending{sx, fx, U + static_cast<long long>(j - 1) * A.ldu};
      } else {
        store_scaled(pu, A.m);
        pv = Pending{sx, fx, V + static_cast<long long>(j - 1) * A.ldv};
      }
      kind = vside ? CTL_V_SPMV : CTL_U_SPMV;
    } else if (phase == PH_V_ELR || phase == PH_U_ELR) {
      nb = static_cast<int>((L + kRowsPerBlock - 1) / kRowsPerBlock);
      for (int s = me; s < nb; s += grid)
        axpy_norm_dot_body<T>(s, L, w, wprev, c.elr_s, part + s, part + nb + s, lds);
      if (!grid_barrier(A.bar, epoch, &flag)) return;
      stored = false;
      kind = vside ? CTL_V_ELR : CTL_U_ELR;
    } else {
      // (ELR reads the scaled rows its own threads stored; the projection
      // reads others')
      if (stored && !grid_barrier(A.bar, epoch, &flag)) return;
      const int ncols = c.reo_ncols;
      nb = static_cast<int>((L + kCgsRows - 1) / kCgsRows);
      if (ncols > 0) {
        // the projection's slices times groups of its column tiles (every
        // column's partial is a sum of its own)
        const int groups = max(1, min((ncols + kCT - 1) / kCT, grid / nb));
        const int per = ((ncols + groups - 1) / groups + kCT - 1) / kCT * kCT;
        for (int u = me; u < nb * groups; u += grid) {
          const int s = u % nb, c0 = u / nb * per;
          if (c0 < ncols)
            gemvt_body<T>(s, L, basis, ld, cols + c0, min(per, ncols - c0), w,
                          part + static_cast<long long>(c0) * nb, nb, s, tile);
          __syncthreads();
        }
        if (!grid_barrier(A.bar, epoch, &flag)) return;
        for (int q = wid; q < ncols; q += kBlock / kWave) {
          const double h = wave_reduce_partials(part + static_cast<long long>(q) * nb, nb, lane);
          if (lane == 0) sh[q] = h;
        }
        __syncthreads();
        part = A.part + buf * A.half;
        buf ^= 1;
      }
      for (int s = me; s < nb; s += grid)
        gemv_update_body<T>(s, L, basis, ld, cols, sh, ncols, w, part + s, lds);
      if (!grid_barrier(A.bar, epoch, &flag)) return;
      stored = false;
      kind = vside ? CTL_V_REO : CTL_U_REO;
    }
    if (kind == CTL_V_REO || kind == CTL_U_REO) {
      a = reduce_partials(part, nb, lds);
    } else {
      const double* const q[2] = {part, part + nb};
      double v[2];
      reduce_partials_n<2>(q, nb, v, lds);
      a = v[0];
      b = v[1];
    }
    ctl_run(c, kind, a, b, lds);
  }
  store_scaled(pu, A.m);
  store_scaled(pv, A.n);
  if (me != 0) return;
  __syncthreads();
  {
    int4* dst = reinterpret_cast<int4*>(A.ctl);
    const int4* src = reinterpret_cast<const int4*>(static_cast<LbdCtl*>(&c));
    for (int i = t; i < kCtlHdrWords; i += kBlock) dst[i] = src[i];
    for (int i = t; i < nd; i += kBlock) {
      CtlArrays::mu(A.arrays, A.cap)[i] = c.mu[i];
      CtlArrays::nu(A.arrays, A.cap)[i] = c.nu[i];
      CtlArrays::B1(A.arrays, A.cap)[i] = c.B1[i];
      CtlArrays::B2(A.arrays, A.cap)[i] = c.B2[i];
    }
    for (int i = t; i < ni; i += kBlock) CtlArrays::index(A.arrays, A.cap)[i] = c.index[i];
    // a pass left to the host reads the column list
    for (int i = t; i < c.reo_ncols && i < kCtlLdsJ + 4; i += kBlock)
      CtlArrays::cols(A.arrays, A.cap)[i] = cols[i];
  }
}

}  // namespace

// Workgroups for an operator: one row block of each direction per workgroup up
// to 128 blocks, two up to 512.  Measured solves (ms; 64 / 96 / 128 / 256
// workgroups, then the chains): 110 blocks 3.14 / 3.03 / 2.87 (110) / -, 4.61;
// 200 blocks 2.75 / 2.74 / 1.94 / 1.98 (200), 2.89; 420 blocks (256) 2.25, 2.82.
static int resident_grid(const CsrOp* op) {
  const int blocks = std::max(op->da.pan[0].part.ndesc, op->dt.pan[0].part.ndesc);
  if (blocks <= 128) return std::max(8, blocks);
  return std::max(128, (blocks + kResSlots - 1) / kResSlots);
}

bool resident_fits(const Engine* e) {
  const CsrOp* op = e->op;
  // (an engine without an operator runs the host executor, complex bases their
  // chains)
  if (!op || !e->rbar || (e->prec != PK_F64 && e->prec != PK_F32)) return false;
  for (const CsrOp::Dir* D : {&op->da, &op->dt})
    if (D->sorted || D->tile.nunit > 0 || D->np != 1 || D->pan[0].part.nlong > 0 ||
        D->pan[0].part.ndesc > kResSlots * kResGrid)
      return false;
  return true;
}

template <typename T>
int launch_resident(Engine* e, hipStream_t s) {
  const CsrOp* op = e->op;
  ResidentArgs A{};
  for (int tr = 0; tr < 2; ++tr) {
    const CsrOp::Panel& P = (tr ? op->dt : op->da).pan[0];
    (tr ? A.dt : A.da) = ResidentDir{P.part.desc, P.rp, P.ci, P.va, P.part.ndesc, P.g};
  }
  A.ctl = e->dctl;
  A.arrays = static_cast<char*>(e->darr);
  A.cap = e->kmax;
  A.U = e->u();
  A.V = e->v();
  A.ldu = e->ldu;
  A.ldv = e->ldv;
  A.m = e->m;
  A.n = e->n;
  A.part = e->part;
  A.half = static_cast<long long>(e->part_len / 2);
  A.bar = e->rbar;
  if (launch_fill_zero_bytes(s, e->rbar, sizeof(ResidentBar)) < 0) return -1;
  void* args[] = {&A};
  const hipError_t r = hipLaunchCooperativeKernel(
      reinterpret_cast<const void*>(&k_resident<T>), dim3(resident_grid(op)), dim3(kBlock), args,
      sizeof(ResidentLds<T>), s);
  if (r == hipSuccess) return 0;
  (void)hipGetLastError();  // refused: the caller enqueues the chains
  return -1;
}
template int launch_resident<double>(Engine*, hipStream_t);
template int launch_resident<float>(Engine*, hipStream_t);

}  // namespace pk
