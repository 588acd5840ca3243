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

// One overfull cell c of grid g: dT_e plus the values of its atoms among
// [i0, i1), by an ordered scan of a block of 1024 threads; every wave ballots
// the atoms of the cell among its 64, and thread 0 adds their values in
// ascending order.
__device__ __forceinline__ void queued_cell(const AtomsView& a, const DepositView& d, const GridView& g,
                                            const int c, const int i0, const int i1,
                                            unsigned long long* hits) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
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

// the queued cells q0, q0 + step, ... of a single grid
__device__ __forceinline__ void deposit_queued(const DepositTail& t, const GridView& g, const int q0,
                                               const int step, unsigned long long* hits) {
  const int nq = *t.b.nqueue;
  for (int q = q0; q < nq; q += step) queued_cell(t.a, t.d, g, t.b.queue[q], 0, t.a.nlocal, hits);
}

}  // namespace eph
