// eph_fdm.hip -- the T_e solve of one grid: every sub-step of EPH_FDM::solve
// (eph_fdm.h:267-400) with as few launches as the grid's size allows.
//
// A sub-step of these grids moves 58 B per cell that the caches hold and as a
// launch of its own takes 4 to 6 us below 100,000 cells, most of it launch and
// load latency.  The kernels here run several sub-steps on cells kept in LDS.
// Their arithmetic is fdm_advance, so the bits are those of one launch per
// sub-step.  Measured on an MI355X, a whole solve of 19 sub-steps (wall time,
// call and status read included) against one launch per sub-step:
//   10^3 cells 118 -> 35 us, 16^3 118 -> 66 (one workgroup)
//   20^3 117 -> 78, 40^3 119 -> 80 (8 x 8 x 4 tiles, 3 sub-steps a launch)
//   64^3 144 -> 117 (16 x 8 x 8 tiles, 2), 80^3 226 -> 148 (16 x 16 x 8, 2)
#include <cstring>

#include "eph_deposit.hpp"
#include "eph_fdm.hpp"

namespace eph {

// ---- the whole solve in one workgroup
// T (twice) and kappa of every cell in LDS, the cells' other values in
// registers, one barrier per sub-step.  Bound by one CU's FP64 issue, about
// 0.7 us per 1000 cells and sub-step.  It also clears dT_e and looks for
// non-finite values.
constexpr int kFdmThreads = 1024;

// the solve's constants: divisors by the spacings, and (MODE 0) the material
struct FdmArgs {
  Divisor d3[3];
  FdmCell uni;
  double inner_dt;
};

template <int MODE, int NC>
__device__ __forceinline__ void fdm_block(const GridView& g, const FdmArgs& u, double* __restrict__ T, int nsub,
                                          int G, int* nonfinite, double* s_fdm) {
  __shared__ int s_slow;
  double* cur = s_fdm;
  double* nxt = s_fdm + G;
  if (threadIdx.x == 0) s_slow = 0;
  __syncthreads();
  bool ok = fdm_range_grid(u.d3);
  const double* sk = MODE != 0 ? s_fdm + 2 * G : nullptr;
  FdmCell c[NC];
#pragma unroll
  for (int m = 0; m < NC; ++m) {
    const int r = threadIdx.x + kFdmThreads * m;
    if (MODE == 0) c[m] = u.uni;
    if (r < G) {
      cur[r] = T[r];
      fdm_load<MODE>(c[m], g, r);
      fdm_neighbours(r, g.nx, g.ny, g.nz, c[m].p, c[m].q);
      if (MODE != 0) {
        s_fdm[2 * G + r] = c[m].kr;
        fdm_walls(c[m], r, g.flag, g.kappa);
      }
      ok = ok && fdm_range_T(cur[r]) && fdm_range_cell(c[m]);
    }
  }
  if (!ok) s_slow = 1;
  __syncthreads();
  for (int n = 0; n < nsub; ++n) {
    const bool fast = s_slow == 0;
#pragma unroll
    for (int m = 0; m < NC; ++m) {
      const int r = threadIdx.x + kFdmThreads * m;
      if (r < G) {
        const double t = fdm_advance<MODE>(c[m], u.d3, g, cur, sk, r, u.inner_dt, fast);
        nxt[r] = t;
        ok = ok && fdm_range_T(t);
      }
    }
    // (a store here races only with stores of the same value and with reads
    // of this sub-step's flag by threads still in it, for which either value
    // gives the same bits)
    if (!ok) s_slow = 1;
    __syncthreads();
    double* t = cur;
    cur = nxt;
    nxt = t;
  }
  bool bad = false;
#pragma unroll
  for (int m = 0; m < NC; ++m) {
    const int r = threadIdx.x + kFdmThreads * m;
    if (r < G) {
      const double v = cur[r];
      T[r] = v;
      g.dT[r] = 0.0;
      bad = bad || !isfinite(v);
    }
  }
  if (bad) atomicOr(nonfinite, 2);
}

template <int MODE, int NC>
__global__ __launch_bounds__(kFdmThreads) void k_fdm_block(GridView g, FdmArgs u, double* __restrict__ T,
                                                           int nsub, int G, int* nonfinite,
                                                           DepositTail tail) {
  extern __shared__ double s_fdm[];
  if (tail.E_local) {  // the deposit's remainder, which completes dT_e
    __shared__ double sh[kFdmThreads];
    __shared__ QueueShared qs;
    energy_reduce(tail.d.partial, tail.nblocks, tail.E_local, tail.Ee, sh);
    const int nq = *tail.b.nqueue;
    if (threadIdx.x == 0 && nq > kQueueEach) *tail.b.state = 0;  // (a cell below may make it kCrowded)
    for (int q = 0; q < nq; ++q)
      queued_cell(tail.a, tail.d, tail.b, g, tail.b.queue[q], tail.b.queue[q], 0, tail.a.nlocal, qs);
    __syncthreads();
  }
  fdm_block<MODE, NC>(g, u, T, nsub, G, nonfinite, s_fdm);
}

// A workgroup per replica of a batch, in place of a launch per sub-step (5 us
// each) and two or three (4 us each) for the copy, the clearing of dT_e and
// the scan for non-finite values: 16 us against 30 for 32 replicas and 4
// sub-steps.
template <int MODE, int NC>
__global__ __launch_bounds__(kFdmThreads) void k_fdm_block_batch(const GridView* __restrict__ grids,
                                                                 const FdmArgs* __restrict__ args,
                                                                 const int* __restrict__ nsub,
                                                                 int* nonfinite) {
  extern __shared__ double s_fdm[];
  const GridView g = grids[blockIdx.x];
  const FdmArgs u = args[blockIdx.x];
  fdm_block<MODE, NC>(g, u, g.T, nsub[blockIdx.x], g.nx * g.ny * g.nz, nonfinite, s_fdm);
}

// ---- K sub-steps per launch on tiles, one material in every cell
// A block loads a tile of TX x TY x TZ cells and K cells around it (periodic
// images wrapped in), T and dT_e, and runs K sub-steps on the shrinking valid
// region, whose cells are dealt to consecutive threads.  The halo's cells are
// computed again by the neighbouring tiles, with the same operands and so the
// same bits.  Bound by launch and load latency on grids of a few tiles, by LDS
// and FP64 issue on large ones; T and dT_e are the only per-cell reads (58 B
// down to 24 B per cell and launch).
template <int TX, int TY, int TZ, int K>
__global__ __launch_bounds__(kFdmThreads) void k_fdm_tile(GridView g, FdmArgs u, const double* __restrict__ Tin,
                                                          double* __restrict__ Tout, int ntx, int nty) {
  constexpr int BX = TX + 2 * K, BY = TY + 2 * K, BZ = TZ + 2 * K, NB = BX * BY * BZ;
  extern __shared__ double s_fdm[];
  __shared__ int s_slow;
  double* cur = s_fdm;
  double* nxt = s_fdm + NB;
  double* sd = s_fdm + 2 * NB;
  if (threadIdx.x == 0) s_slow = 0;
  __syncthreads();
  bool ok = fdm_range_grid(u.d3) && fdm_range_cell(u.uni);
  const int bx = blockIdx.x % ntx, by = (blockIdx.x / ntx) % nty, bz = blockIdx.x / (ntx * nty);
  auto fold = [](int a, int n) {
    if (a >= 0 && a < n) return a;
    a %= n;
    return a < 0 ? a + n : a;
  };
#pragma unroll
  for (int m = 0; m < (NB + kFdmThreads - 1) / kFdmThreads; ++m) {
    const int l = threadIdx.x + kFdmThreads * m;
    if (l < NB) {
      const int gx = fold(bx * TX + l % BX - K, g.nx), gy = fold(by * TY + (l / BX) % BY - K, g.ny),
                gz = fold(bz * TZ + l / (BX * BY) - K, g.nz);
      const int r = gx + g.nx * (gy + g.ny * gz);
      const double t = Tin[r], q = g.dT[r];
      cur[l] = t;
      sd[l] = q;
      ok = ok && fdm_range_T(t) && in_range(q, 500);
    }
  }
  FdmCell c = u.uni;
  if (!ok) s_slow = 1;
#pragma unroll
  for (int n = 1; n <= K; ++n) {
    __syncthreads();
    const bool fast = s_slow == 0;
    const int vx = BX - 2 * n, vy = BY - 2 * n, vz = BZ - 2 * n;
    for (int m = threadIdx.x; m < vx * vy * vz; m += kFdmThreads) {
      const int lx = m % vx, ly = (m / vx) % vy, lz = m / (vx * vy);
      const int l = lx + n + BX * (ly + n + BY * (lz + n));
      c.p[0] = l - 1; c.p[1] = l - BX; c.p[2] = l - BX * BY;
      c.q[0] = l + 1; c.q[1] = l + BX; c.q[2] = l + BX * BY;
      c.dT = sd[l];
      const double t = fdm_advance<0>(c, u.d3, g, cur, nullptr, l, u.inner_dt, fast);
      if (n < K) {
        nxt[l] = t;
        ok = ok && fdm_range_T(t);
      } else {
        const int gx = bx * TX + lx, gy = by * TY + ly, gz = bz * TZ + lz;
        if (gx < g.nx && gy < g.ny && gz < g.nz) Tout[gx + g.nx * (gy + g.ny * gz)] = t;
      }
    }
    if (!ok) s_slow = 1;
    double* t = cur;
    cur = nxt;
    nxt = t;
  }
}

// after the last sub-step: dT_e = 0 (eph_fdm.h:487), non-finite values flagged
__global__ __launch_bounds__(kBlock) void k_fdm_finish(const double* __restrict__ T, double* dT, int n,
                                                       int* nonfinite) {
  const int r = blockIdx.x * kBlock + threadIdx.x;
  if (r >= n) return;
  dT[r] = 0.0;
  if (!isfinite(T[r])) atomicOr(nonfinite, 2);
}

template <bool TDYN>
__global__ __launch_bounds__(kBlock) void k_fdm_substep(GridView g, const double* __restrict__ Tin,
                                                        double* __restrict__ Tout, double inner_dt) {
  const int r = blockIdx.x * kBlock + threadIdx.x;
  if (r >= g.nx * g.ny * g.nz) return;
  fdm_cell<TDYN>(g, Tin, Tout, r, inner_dt);
}

hipError_t launch_fdm_substep(const GridView& g, const double* Tin, double* Tout, double inner_dt,
                              bool any_tdyn, hipStream_t s) {
  const int n = g.nx * g.ny * g.nz;
  const int nb = (n + kBlock - 1) / kBlock;
  if (any_tdyn) k_fdm_substep<true><<<nb, kBlock, 0, s>>>(g, Tin, Tout, inner_dt);
  else k_fdm_substep<false><<<nb, kBlock, 0, s>>>(g, Tin, Tout, inner_dt);
  return hipGetLastError();
}

// more than 64 KB of dynamic LDS has to be asked for
template <typename Kern>
static hipError_t allow_lds(Kern k, size_t bytes) {
  if (bytes <= 65536) return hipSuccess;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                             static_cast<int>(bytes));
}

template <int MODE, int NC>
static hipError_t block_solve(const GridView& g, const FdmArgs& u, double* T, int nsub, int* nonfinite,
                              const DepositTail& tail, hipStream_t s) {
  const int G = g.nx * g.ny * g.nz;
  const size_t lds = static_cast<size_t>(G) * (MODE != 0 ? 24 : 16);
  auto k = k_fdm_block<MODE, NC>;
  if (hipError_t e = allow_lds(k, lds); e != hipSuccess) return e;
  k<<<1, kFdmThreads, lds, s>>>(g, u, T, nsub, G, nonfinite, tail);
  return hipGetLastError();
}

template <int TX, int TY, int TZ, int K>
static hipError_t tile_steps(const GridView& g, const FdmArgs& u, const double* Tin, double* Tout,
                             hipStream_t s) {
  const size_t lds = static_cast<size_t>(TX + 2 * K) * (TY + 2 * K) * (TZ + 2 * K) * 24;
  auto k = k_fdm_tile<TX, TY, TZ, K>;
  if (hipError_t e = allow_lds(k, lds); e != hipSuccess) return e;
  const int ntx = (g.nx + TX - 1) / TX, nty = (g.ny + TY - 1) / TY, ntz = (g.nz + TZ - 1) / TZ;
  k<<<ntx * nty * ntz, kFdmThreads, lds, s>>>(g, u, Tin, Tout, ntx, nty);
  return hipGetLastError();
}

// nsub sub-steps in launches of K (then 2, 1)
template <int TX, int TY, int TZ, int K>
static hipError_t tile_solve(const GridView& g, const FdmArgs& u, double*& T, double*& Tn, int nsub,
                             hipStream_t s) {
  hipError_t e = hipSuccess;
  for (int left = nsub; left > 0 && e == hipSuccess;) {
    const int k = left >= K ? K : left >= 2 ? 2 : 1;
    e = k == K ? tile_steps<TX, TY, TZ, K>(g, u, T, Tn, s)
        : k == 2 ? tile_steps<TX, TY, TZ, 2>(g, u, T, Tn, s)
                 : tile_steps<TX, TY, TZ, 1>(g, u, T, Tn, s);
    std::swap(T, Tn);
    left -= k;
  }
  return e;
}

// One workgroup up to here: at 16^3 cells of one material it takes 66 us
// against 78 in tiles, at 20^3 108 against 78.  Per-cell materials hold 20
// registers a cell, so two cells a thread.
constexpr int kFdmBlockUniform = 4096, kFdmBlockCells = 2048;
// The larger tile where it still gives most CUs one: 64^3 cells in 16 x 16 x 8
// tiles (128 of them) take 133 us, in 16 x 8 x 8 tiles 117.
constexpr int kFdmMinTiles = 200;

template <int MODE>
static hipError_t solve_any(const GridView& g, const FdmArgs& u, double*& T, double*& Tn, int nsub,
                            int* nonfinite, const DepositTail& tail, hipStream_t s) {
  const int G = g.nx * g.ny * g.nz;
  if (G <= (MODE == 0 ? kFdmBlockUniform : kFdmBlockCells)) {
    if (G <= kFdmThreads) return block_solve<MODE, 1>(g, u, T, nsub, nonfinite, tail, s);
    if (G <= 2 * kFdmThreads) return block_solve<MODE, 2>(g, u, T, nsub, nonfinite, tail, s);
    if constexpr (MODE == 0) return block_solve<MODE, 4>(g, u, T, nsub, nonfinite, tail, s);
  }
  hipError_t e = tail.E_local ? launch_deposit_tail(g, tail, s) : hipSuccess;
  if (e != hipSuccess) return e;
  if constexpr (MODE == 0) {
    if (G >= kFdmMinTiles * 2048) e = tile_solve<16, 16, 8, 2>(g, u, T, Tn, nsub, s);
    else if (G >= kFdmMinTiles * 1024) e = tile_solve<16, 8, 8, 2>(g, u, T, Tn, nsub, s);
    else e = tile_solve<8, 8, 4, 3>(g, u, T, Tn, nsub, s);
  } else {
    for (int n = 0; n < nsub && e == hipSuccess; ++n) {
      e = launch_fdm_substep(g, T, Tn, u.inner_dt, MODE == 2, s);
      std::swap(T, Tn);
    }
  }
  if (e != hipSuccess) return e;
  k_fdm_finish<<<(G + kBlock - 1) / kBlock, kBlock, 0, s>>>(T, g.dT, G, nonfinite);
  return hipGetLastError();
}

static FdmArgs fdm_args(const GridView& g, double inner_dt, const FdmMaterial* uniform) {
  FdmArgs u;
  u.inner_dt = inner_dt;
  u.d3[0] = divisor(g.dx); u.d3[1] = divisor(g.dy); u.d3[2] = divisor(g.dz);
  u.uni = FdmCell{};
  if (uniform) {
    u.uni.kr = uniform->kappa;
    u.uni.S = uniform->S;
    u.uni.div = divisor(uniform->rho * uniform->C);
    u.uni.flag = kCellDynamic;
    u.uni.flat = true;
  }
  return u;
}

size_t fdm_batch_args_size() { return sizeof(FdmArgs); }

void fdm_batch_args(void* entry, const GridView& g, double inner_dt, const FdmMaterial* uniform) {
  const FdmArgs u = fdm_args(g, inner_dt, uniform);
  std::memcpy(entry, &u, sizeof u);
}

bool fdm_batch_fits(int max_cells, bool uniform) {
  return max_cells <= (uniform ? kFdmBlockUniform : kFdmBlockCells);
}

template <int MODE, int NC>
static hipError_t block_batch(const GridView* grids, const void* args, const int* nsub, int nrep, int max_cells,
                              int* nonfinite, hipStream_t s) {
  const size_t lds = static_cast<size_t>(max_cells) * (MODE != 0 ? 24 : 16);
  auto k = k_fdm_block_batch<MODE, NC>;
  if (hipError_t e = allow_lds(k, lds); e != hipSuccess) return e;
  k<<<nrep, kFdmThreads, lds, s>>>(grids, static_cast<const FdmArgs*>(args), nsub, nonfinite);
  return hipGetLastError();
}

hipError_t launch_fdm_batch(const GridView* grids, const void* args, const int* nsub, int nrep, int max_cells,
                            bool uniform, int* nonfinite, hipStream_t s) {
  if (nrep == 0) return hipSuccess;
  if (!fdm_batch_fits(max_cells, uniform)) return hipErrorInvalidValue;
  const int nc = (max_cells + kFdmThreads - 1) / kFdmThreads;
  if (uniform)
    return nc <= 1 ? block_batch<0, 1>(grids, args, nsub, nrep, max_cells, nonfinite, s)
           : nc == 2 ? block_batch<0, 2>(grids, args, nsub, nrep, max_cells, nonfinite, s)
                     : block_batch<0, 4>(grids, args, nsub, nrep, max_cells, nonfinite, s);
  return nc <= 1 ? block_batch<1, 1>(grids, args, nsub, nrep, max_cells, nonfinite, s)
                 : block_batch<1, 2>(grids, args, nsub, nrep, max_cells, nonfinite, s);
}

hipError_t launch_fdm_solve(const GridView& g, double*& T, double*& Tn, double inner_dt, int nsub,
                            const FdmMaterial* uniform, bool any_tdyn, int* nonfinite, hipStream_t s,
                            const DepositTail* tail) {
  const DepositTail rest = tail ? *tail : DepositTail();
  const FdmArgs u = fdm_args(g, inner_dt, uniform);
  if (uniform) return solve_any<0>(g, u, T, Tn, nsub, nonfinite, rest, s);
  return any_tdyn ? solve_any<2>(g, u, T, Tn, nsub, nonfinite, rest, s)
                  : solve_any<1>(g, u, T, Tn, nsub, nonfinite, rest, s);
}

}  // namespace eph
