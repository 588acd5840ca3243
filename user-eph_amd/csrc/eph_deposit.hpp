// eph_deposit.hpp -- the end of the deposit: the tally and the overfull cells,
// as a kernel of its own or at the start of a one-workgroup T_e solve.
#pragma once

#include "eph_devfn.hpp"

namespace eph {

// E_local = sum of friction then random energies; Ee += E_local
__device__ __forceinline__ void energy_reduce(const double* partial, int nb, double* E_local,
                                              double* Ee, double* sh) {
  double sF = 0.0, sR = 0.0;
  for (int b = threadIdx.x; b < nb; b += 1024) {
    sF += partial[2 * b];
    sR += partial[2 * b + 1];
  }
  sF = block_sum(sF, sh);
  sR = block_sum(sR, sh);
  if (threadIdx.x == 0) {
    const double E = sF + sR;
    *E_local = E;
    *Ee += E;
  }
}

// acc += the first n lanes' v, in lane order: every lane keeps the same sum
static __device__ __forceinline__ double add_lanes(double acc, double v, int n) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  for (int k = 0; k < n; ++k)
    acc += __hiloint2double(__builtin_amdgcn_readlane(hi, k), __builtin_amdgcn_readlane(lo, k));
  return acc;
}

// A queued cell by a block of 1024 threads: its atoms from the bucket and the
// chain, sorted in LDS, their values added in ascending order by one wave.  A
// chain is walked by one thread, 0.5 us a link, so beyond 64 links and one for
// every 512 atoms (or beyond the LDS) an ordered scan over the atoms [i0, i1) is
// the faster: every wave ballots the atoms of the cell among its 64, and
// thread 0 adds their values.  32,000 atoms in an eighth of 24^3 cells, some 900
// cells queued: 0.6 ms a step with its host calls, 9.7 with a scan each.
// A scan of more than kQueueScan atoms (3 us per 1024) costs as much as the counted
// form does.
constexpr int kQueueItems = 4096, kQueueScan = 16384;
static __device__ __forceinline__ bool queue_walks(const int n, const int cap, const int atoms) {
  return n <= kQueueItems && (n - cap <= 64 || n - cap <= atoms / 512);
}
struct QueueShared {
  int key[kQueueItems];
  unsigned long long hits[16];
};

// c: the cell in its grid g; cb: its index in b
__device__ __forceinline__ void queued_cell(const AtomsView& a, const DepositView& d, const BucketView& b,
                                            const GridView& g, const int c, const int cb, const int i0,
                                            const int i1, QueueShared& sh) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int n = b.count[cb], held = min(n, b.cap);
  const bool walk = queue_walks(n, b.cap, i1 - i0);
  __syncthreads();  // count read by all, and the last cell's LDS
  if (threadIdx.x == 0) {
    int j = b.head[cb];
    b.count[cb] = 0;
    b.head[cb] = 0;
    if (walk)
      for (int k = held; k < n; ++k) {
        sh.key[k] = j - 1;
        j = b.next[j - 1];
      }
  }
  if (walk) {
    const int* items = b.items + static_cast<size_t>(cb) * b.cap;
    int m = 1;
    while (m < n) m <<= 1;
    for (int k = threadIdx.x; k < m; k += 1024)
      if (k < held || k >= n) sh.key[k] = k < held ? items[k] : 0x7fffffff;
    __syncthreads();
    for (int size = 2; size <= m; size <<= 1)
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
        for (int k = threadIdx.x; k < m; k += 1024) {
          const int l = k ^ stride;
          if (l > k) {
            const int x = sh.key[k], y = sh.key[l];
            if ((x > y) == ((k & size) == 0)) {
              sh.key[k] = y;
              sh.key[l] = x;
            }
          }
        }
        __syncthreads();
      }
    if (wv == 0) {
      double acc = g.dT[c];
      for (int pass = 0; pass < 2; ++pass) {
        const double* v = pass == 0 ? d.v1 : d.v2;
        if (!v) continue;
        for (int k = 0; k < n; k += 64)
          acc = add_lanes(acc, k + lane < n ? v[sh.key[k + lane]] : 0.0, min(n - k, 64));
      }
      if (lane == 0) g.dT[c] = acc;
    }
    return;
  }
  if (threadIdx.x == 0 && i1 - i0 > kQueueScan) *b.state = kCrowded;
  double acc = g.dT[c];  // meaningful in thread 0 only
  for (int pass = 0; pass < 2; ++pass) {
    const double* v = pass == 0 ? d.v1 : d.v2;
    if (!v) continue;
    for (int base = i0; base < i1; base += 1024) {
      const int i = base + threadIdx.x;
      bool in = false;
      if (i < i1 && (a.mask[i] & a.groupbit)) {
        const double4 x = a.pos[i];
        in = cell_of(g, x.x, x.y, x.z) == c;
      }
      const unsigned long long m = __ballot(in);
      if (lane == 0) sh.hits[wv] = m;
      __syncthreads();
      if (threadIdx.x == 0)
        for (int w2 = 0; w2 < 16; ++w2)
          for (unsigned long long bits = sh.hits[w2]; bits; bits &= bits - 1)
            acc += v[base + 64 * w2 + __builtin_ctzll(bits)];
      __syncthreads();
    }
  }
  if (threadIdx.x == 0) g.dT[c] = acc;
}

}  // namespace eph
