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

// The queued cells q0, q0 + step, ...: each by an ordered scan over all atoms
// by a block of 1024 threads; every wave ballots the atoms of the cell among
// its 64, and thread 0 adds their values in ascending order.
__device__ __forceinline__ void deposit_queued(const DepositTail& t, const GridView& g, const int q0,
                                               const int step, unsigned long long* hits) {
  const int n_items = t.a.nlocal;
  const int nq = *t.b.nqueue;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (int q = q0; q < nq; q += step) {
    const int c = t.b.queue[q];
    double acc = g.dT[c];  // meaningful in thread 0 only
    for (int pass = 0; pass < 2; ++pass) {
      const double* v = pass == 0 ? t.d.v1 : t.d.v2;
      if (!v) continue;
      for (int base = 0; base < n_items; base += 1024) {
        const int i = base + threadIdx.x;
        bool in = false;
        if (i < n_items && (t.a.mask[i] & t.a.groupbit)) {
          const double4 x = t.a.pos[i];
          in = cell_of(g, x.x, x.y, x.z) == c;
        }
        const unsigned long long m = __ballot(in);
        if (lane == 0) hits[wv] = m;
        __syncthreads();
        if (threadIdx.x == 0)
          for (int w2 = 0; w2 < 16; ++w2)
            for (unsigned long long bits = hits[w2]; bits; bits &= bits - 1)
              acc += v[base + 64 * w2 + __builtin_ctzll(bits)];
        __syncthreads();
      }
    }
    if (threadIdx.x == 0) g.dT[c] = acc;
  }
}

}  // namespace eph
