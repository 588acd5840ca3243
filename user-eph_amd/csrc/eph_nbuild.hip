// eph_nbuild.hip -- device rebuild of ghosts and neighbour lists for the MD
// harness (the LAMMPS stand-in), bit-identical to the host build in eph_md.cpp:
//   * locals remapped into the box,
//   * periodic images made dimension by dimension (x, y, z), each pass
//     imaging every atom present before it, images in source order and
//     lower image first,
//   * atoms binned on bins of half the larger list cutoff, each bin holding
//     its atoms in ascending index,
//   * full lists found in stencil order (z outer, then y, then x, offsets
//     -2..2) and ascending index within a bin; the pair list keeps that
//     order, the fix list is then sorted by list_sort_key (distance, index).
// Several independent systems ("replicas") can be built at once: atom i of
// replica rep[i] only images and neighbours atoms of its own replica.
// The host launches the sequence when the check of the lists asks for it.
#include "eph_nbuild.hpp"

#include "eph_devfn.hpp"

namespace eph {

namespace {

__device__ __forceinline__ int bin_coord(double x, double glo, double bs, int nb) {
  int b = static_cast<int>(floor((x - glo) / bs));
  return b < 0 ? 0 : (b > nb - 1 ? nb - 1 : b);
}

__device__ __forceinline__ double comp(const double4& p, int d) {
  return d == 0 ? p.x : (d == 1 ? p.y : p.z);
}

}  // namespace

// Domain::remap of the locals
__global__ __launch_bounds__(kBlock) void k_nb_wrap(int nlocal, double4* pos, PosVel* pv,
                                                    const int* rep, NbBoxes b) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= nlocal) return;
  const int r = rep[i];
  double4 p = pos[i];
  double c[3] = {p.x, p.y, p.z};
  for (int d = 0; d < 3; ++d) {
    const double lo = b.lo[3 * r + d], hi = b.hi[3 * r + d], L = b.L[3 * r + d];
    if (c[d] < lo) c[d] += L;
    if (c[d] >= hi) c[d] -= L;
    if (c[d] < lo) c[d] = lo;
  }
  if (c[0] == p.x && c[1] == p.y && c[2] == p.z) return;
  p.x = c[0]; p.y = c[1]; p.z = c[2];
  pos[i] = p;
  if (pv) pv[i].p = p;
}

// images of source s in dimension d: count (0..2)
__global__ __launch_bounds__(kBlock) void k_nb_ghost_count(int d, int cap, int nlocal,
                                                           const int* nghost_in,
                                                           const double4* __restrict__ pos,
                                                           const int* __restrict__ rep, NbBoxes b,
                                                           int* cnt) {
  const int s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= cap) return;
  const int nsrc = nlocal + *nghost_in;
  int c = 0;
  if (s < nsrc) {
    const int r = rep[s];
    const double x = comp(pos[s], d);
    const double lo = b.lo[3 * r + d] - b.cg, hi = b.hi[3 * r + d] + b.cg, L = b.L[3 * r + d];
    for (int sgn = -1; sgn <= 1; sgn += 2) {
      const double img = x + sgn * L;
      if (img >= lo && img < hi) ++c;
    }
  }
  cnt[s] = c;
}

// write the images of pass d after the ghosts already present
__global__ __launch_bounds__(kBlock) void k_nb_ghost_write(int d, int cap, int nlocal,
                                                           const int* nghost_in, int* nghost_out,
                                                           const int* __restrict__ cnt,
                                                           const int* __restrict__ start,
                                                           NbAtoms at, NbBoxes b, int ghost_cap,
                                                           int* overflow) {
  const int s = blockIdx.x * kBlock + threadIdx.x;
  const int ng0 = *nghost_in;
  const int nsrc = nlocal + ng0;
  if (s >= nsrc || s >= cap) return;
  if (s == nsrc - 1) {
    const int total = ng0 + start[s] + cnt[s];
    *nghost_out = total <= ghost_cap ? total : ghost_cap;
    if (total > ghost_cap) atomicOr(overflow, 1);
  }
  if (cnt[s] == 0) return;
  const int r = at.rep[s];
  const double x = comp(at.pos[s], d);
  const double lo = b.lo[3 * r + d] - b.cg, hi = b.hi[3 * r + d] + b.cg, L = b.L[3 * r + d];
  const int o = s < nlocal ? s : at.owner[s - nlocal];
  const double4 sh0 = s < nlocal ? make_double4(0.0, 0.0, 0.0, 0.0) : at.shift[s - nlocal];
  int c = 0;
  for (int sgn = -1; sgn <= 1; sgn += 2) {
    const double img = x + sgn * L;
    if (!(img >= lo && img < hi)) continue;
    const int g = ng0 + start[s] + c;
    ++c;
    if (g >= ghost_cap) continue;
    double4 sh = sh0;
    if (d == 0) sh.x += sgn * L; else if (d == 1) sh.y += sgn * L; else sh.z += sgn * L;
    at.owner[g] = o;
    at.shift[g] = sh;
    const double4 po = at.pos[o];
    const int gi = nlocal + g;
    at.pos[gi] = make_double4(po.x + sh.x, po.y + sh.y, po.z + sh.z, po.w);
    at.vel[gi] = at.vel[o];
    at.type[gi] = at.type[o];
    at.mask[gi] = at.mask[o];
    at.tag[gi] = at.tag[o];
    at.rep[gi] = at.rep[o];
  }
}

__global__ __launch_bounds__(kBlock) void k_nb_bin(int cap, int nlocal, const int* nghost,
                                                    const double4* __restrict__ pos,
                                                    const int* __restrict__ rep, NbBoxes b,
                                                    int* bin_of, int* bcount) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= cap || i >= nlocal + *nghost) return;
  const int r = rep[i];
  const double4 p = pos[i];
  const int* nb = b.nb + 3 * r;
  const double* glo = b.glo + 3 * r;
  const int bx = bin_coord(p.x, glo[0], b.bs, nb[0]);
  const int by = bin_coord(p.y, glo[1], b.bs, nb[1]);
  const int bz = bin_coord(p.z, glo[2], b.bs, nb[2]);
  const int bin = b.bin_base[r] + bx + nb[0] * (by + nb[1] * bz);
  bin_of[i] = bin;
  atomicAdd(&bcount[bin], 1);
}

__global__ __launch_bounds__(kBlock) void k_nb_bin_scatter(int cap, int nlocal, const int* nghost,
                                                           const int* __restrict__ bin_of,
                                                           const int* __restrict__ bstart,
                                                           int* bfill, int* items) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= cap || i >= nlocal + *nghost) return;
  const int bin = bin_of[i];
  items[bstart[bin] + atomicAdd(&bfill[bin], 1)] = i;
}

// atoms of each bin in ascending index (insertion sort; bins hold few atoms)
__global__ __launch_bounds__(kBlock) void k_nb_bin_sort(int nbins, const int* __restrict__ bstart,
                                                        int* items) {
  const int bin = blockIdx.x * kBlock + threadIdx.x;
  if (bin >= nbins) return;
  int* it = items + bstart[bin];
  const int n = bstart[bin + 1] - bstart[bin];
  for (int k = 1; k < n; ++k) {
    const int v = it[k];
    int m = k - 1;
    while (m >= 0 && it[m] > v) {
      it[m + 1] = it[m];
      --m;
    }
    it[m + 1] = v;
  }
}

// both full lists of every local atom, transposed ELL
__global__ __launch_bounds__(kBlock) void k_nb_lists(int nlocal, const double4* __restrict__ pos,
                                                     const int* __restrict__ rep, NbBoxes b,
                                                     const int* __restrict__ bstart,
                                                     const int* __restrict__ items, NbLists l,
                                                     int* overflow) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= nlocal) return;
  const int r = rep[i];
  const double4 pi = pos[i];
  const int* nb = b.nb + 3 * r;
  const double* glo = b.glo + 3 * r;
  const int bx = bin_coord(pi.x, glo[0], b.bs, nb[0]);
  const int by = bin_coord(pi.y, glo[1], b.bs, nb[1]);
  const int bz = bin_coord(pi.z, glo[2], b.bs, nb[2]);
  // Squared distance from the atom to each bin slab of the 5 x 5 x 5 stencil,
  // per dimension.  A bin whose box lies farther than the larger cutoff
  // holds no atom of either list and is skipped, which leaves the lists (and
  // their order) unchanged.  Edge bins also hold the atoms clamped into them,
  // so they are never skipped; the margin covers the rounding of the slab
  // bounds.
  double sx[5], sy[5], sz[5];
  {
    const double pc[3] = {pi.x, pi.y, pi.z};
    const int bc[3] = {bx, by, bz};
    double* sd[3] = {sx, sy, sz};
    for (int d = 0; d < 3; ++d) {
      for (int o = 0; o < 5; ++o) {
        const int c = bc[d] + o - 2;
        const double lo = glo[d] + c * b.bs, hi = lo + b.bs;
        const double g = (c <= 0 || c >= nb[d] - 1) ? 0.0 : (pc[d] < lo ? lo - pc[d] : (pc[d] > hi ? pc[d] - hi : 0.0));
        sd[d][o] = g * g;
      }
    }
  }
  const double reach2 = b.cg * b.cg * (1.0 + 1e-9);
  int nf = 0, nl = 0, nc = 0;
  for (int dz = -2; dz <= 2; ++dz) {
    const int z = bz + dz;
    if (z < 0 || z >= nb[2]) continue;
    for (int dy = -2; dy <= 2; ++dy) {
      const int y = by + dy;
      if (y < 0 || y >= nb[1]) continue;
      for (int dx = -2; dx <= 2; ++dx) {
        const int x = bx + dx;
        if (x < 0 || x >= nb[0]) continue;
        if (sx[dx + 2] + sy[dy + 2] + sz[dz + 2] > reach2) continue;
        const int bin = b.bin_base[r] + x + nb[0] * (y + nb[1] * z);
        for (int k = bstart[bin]; k < bstart[bin + 1]; ++k) {
          const int j = items[k];
          if (j == i) continue;
          const double4 pj = pos[j];
          const double ex = pj.x - pi.x, ey = pj.y - pi.y, ez = pj.z - pi.z;
          const double r2 = ex * ex + ey * ey + ez * ez;
          if (r2 < l.cf2) {
            if (nf < l.cap_f) l.nbr_f[nf * l.stride + i] = j;
            ++nf;
            if (l.cand && r2 < l.cand2) {
              if (nc < l.cap_f) l.cand[nc * l.stride + i] = j;
              ++nc;
            }
          }
          if (r2 < l.cl2) {
            if (nl < l.cap_l) l.nbr_l[nl * l.stride + i] = j;
            ++nl;
          }
        }
      }
    }
  }
  if (nf > l.cap_f || nl > l.cap_l) atomicOr(overflow, 2);
  l.nn_f[i] = nf < l.cap_f ? nf : l.cap_f;
  l.nn_l[i] = nl < l.cap_l ? nl : l.cap_l;
  if (l.cand) l.ncand[i] = nc < l.cap_f ? nc : l.cap_f;
}

// bitonic sort of one wave's 64 E keys, ascending: element n = lane E + s
template <int E>
__device__ __forceinline__ void bitonic_wave(uint32_t (&key)[E], const int lane) {
  constexpr int N = 64 * E;
#pragma unroll
  for (int k = 2; k <= N; k <<= 1) {
#pragma unroll
    for (int d = k >> 1; d > 0; d >>= 1) {
      if (d < E) {
#pragma unroll
        for (int s = 0; s < E; ++s) {
          const int ps = s ^ d;
          if (ps > s) {
            const bool up = ((lane * E + s) & k) == 0;
            const uint32_t lo = min(key[s], key[ps]), hi = max(key[s], key[ps]);
            key[s] = up ? lo : hi;
            key[ps] = up ? hi : lo;
          }
        }
      } else {
#pragma unroll
        for (int s = 0; s < E; ++s) {
          const int n = lane * E + s;
          const uint32_t mine = key[s];
          const uint32_t other = static_cast<uint32_t>(__shfl_xor(static_cast<int>(mine), d / E));
          const bool keep_min = ((n & d) == 0) == ((n & k) == 0);
          key[s] = keep_min ? min(mine, other) : max(mine, other);
        }
      }
    }
  }
}

// Each atom's fix list into (q(r^2), found position) order, and its
// candidates (the entries with r^2 < cand2, in list order) rewritten to
// match: one wave per atom, a bitonic sort of N = 64 E 32-bit keys q x 2^9 + t
// (element n = lane E + s; padding keys ~0 sort last; nn_f <= cap_f <= N).
// The found position t in a key gives the entry's index, read back before the
// sorted list is written over the found one.  A fixed grid of waves walks the
// atoms.
template <int E>
__device__ __forceinline__ void nb_sort_atom(const int i, const int lane, const double4* __restrict__ pos,
                                             const NbLists& l) {
  const int nf = l.nn_f[i];
  const double4 pi = pos[i];
  uint32_t key[E];
#pragma unroll
  for (int s = 0; s < E; ++s) {
    const int n = lane * E + s;
    key[s] = ~0u;
    if (n < nf) {
      const double4 pj = pos[l.nbr_f[n * l.stride + i]];
      const double ex = pj.x - pi.x, ey = pj.y - pi.y, ez = pj.z - pi.z;
      key[s] = (list_sort_q(ex * ex + ey * ey + ez * ez, l.sort_scale) << 9) | static_cast<uint32_t>(n);
    }
  }
  bitonic_wave<E>(key, lane);
  // the indices of the sorted entries, all read before any is written
  int jv[E];
#pragma unroll
  for (int s = 0; s < E; ++s)
    jv[s] = lane * E + s < nf ? l.nbr_f[static_cast<int>(key[s] & 511u) * l.stride + i] : 0;
  __builtin_amdgcn_wave_barrier();
  int mine = 0;  // candidates among this lane's entries
#pragma unroll
  for (int s = 0; s < E; ++s) {
    const int n = lane * E + s;
    bool c = false;
    if (n < nf) {
      l.nbr_f[n * l.stride + i] = jv[s];
      if (l.cand) {
        const double4 pj = pos[jv[s]];
        const double ex = pj.x - pi.x, ey = pj.y - pi.y, ez = pj.z - pi.z;
        c = ex * ex + ey * ey + ez * ez < l.cand2;
      }
    }
    mine |= (c ? 1 : 0) << s;
  }
  if (!l.cand) return;
  // exclusive prefix of the candidate counts over the lanes
  const int cnt = __builtin_popcount(mine);
  int incl = cnt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(incl, o);
    if (lane >= o) incl += v;
  }
  int at = incl - cnt;
#pragma unroll
  for (int s = 0; s < E; ++s) {
    if ((mine >> s) & 1) {
      if (at < l.cap_f) l.cand[at * l.stride + i] = jv[s];
      ++at;
    }
  }
  if (lane == 63) l.ncand[i] = incl < l.cap_f ? incl : l.cap_f;
}

constexpr int kSortBlocks = 2048;
template <int E>
__global__ __launch_bounds__(kBlock) void k_nb_sort(int nlocal, const double4* __restrict__ pos, NbLists l) {
  const int lane = threadIdx.x & 63;
  const int nw = gridDim.x * (kBlock / 64);
  for (int i = blockIdx.x * (kBlock / 64) + static_cast<int>(threadIdx.x >> 6); i < nlocal; i += nw)
    nb_sort_atom<E>(i, lane, pos, l);  // i is the same for the whole wave
}

__global__ __launch_bounds__(kBlock) void k_nb_finish(int nlocal, const int* ng,
                                                      const double4* __restrict__ pos,
                                                      double4* ref, int* nreb,
                                                      int* cand_valid, double4* cref,
                                                      bool cand_written) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < nlocal) ref[i] = pos[i];
  // the candidates of the new lists, if written, are valid at the positions
  // of this rebuild (locals and the ghosts just made); otherwise the next
  // density sweep retakes them
  if (cand_written && i < nlocal + *ng) cref[i] = pos[i];
  if (i == 0 && cand_valid) {
    cand_valid[0] = cand_written ? 1 : 0;
    cand_valid[2] = 0;  // atoms that a check before this rebuild found moved
    cand_valid[6] = cand_written ? 2 : 0;  // the pair force's: to be taken in this step
    cand_valid[7] = 0;
  }
  if (i == 0) atomicAdd(nreb, 1);
}

__global__ __launch_bounds__(kBlock) void k_nb_zero(int* p, int n) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) p[i] = 0;
}

// ------------------------------------------------------------------ scan
constexpr int kSB = 1024, kSI = 4;
__global__ __launch_bounds__(kSB) void k_nb_scan_reduce(const int* in, int n, int* bsum) {
  __shared__ int sh[kSB];
  const int base = blockIdx.x * kSB * kSI;
  int s = 0;
  for (int k = 0; k < kSI; ++k) {
    const int idx = base + k * kSB + threadIdx.x;
    if (idx < n) s += in[idx];
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int st = kSB / 2; st > 0; st >>= 1) {
    if (threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) bsum[blockIdx.x] = sh[0];
}

__global__ __launch_bounds__(kSB) void k_nb_scan_blocks(int* bsum, int nb) {
  __shared__ int sh[kSB];
  int carry = 0;
  for (int base = 0; base < nb; base += kSB) {
    const int idx = base + threadIdx.x;
    const int v = idx < nb ? bsum[idx] : 0;
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int off = 1; off < kSB; off <<= 1) {
      const int add = threadIdx.x >= off ? sh[threadIdx.x - off] : 0;
      __syncthreads();
      sh[threadIdx.x] += add;
      __syncthreads();
    }
    if (idx < nb) bsum[idx] = carry + sh[threadIdx.x] - v;
    const int total = sh[kSB - 1];
    __syncthreads();
    carry += total;
  }
}

__global__ __launch_bounds__(kSB) void k_nb_scan_apply(const int* in, int n, const int* boff,
                                                       int* out) {
  __shared__ int sh[kSB];
  const int base = blockIdx.x * kSB * kSI;
  int carry = boff[blockIdx.x];
  for (int k = 0; k < kSI; ++k) {
    const int idx = base + k * kSB + threadIdx.x;
    const int v = idx < n ? in[idx] : 0;
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int off = 1; off < kSB; off <<= 1) {
      const int add = threadIdx.x >= off ? sh[threadIdx.x - off] : 0;
      __syncthreads();
      sh[threadIdx.x] += add;
      __syncthreads();
    }
    if (idx < n) out[idx] = carry + sh[threadIdx.x] - v;
    if (idx == n - 1) out[n] = carry + sh[threadIdx.x];
    const int total = sh[kSB - 1];
    __syncthreads();
    carry += total;
  }
}

// the atoms' positions in bin order, the index in .w
__global__ __launch_bounds__(kBlock) void k_nb_bin_pos(int cap, int nlocal, const int* nghost,
                                                       const double4* __restrict__ pos,
                                                       const int* __restrict__ items,
                                                       double4* __restrict__ bpos) {
  const int k = blockIdx.x * kBlock + threadIdx.x;
  if (k >= cap || k >= nlocal + *nghost) return;
  const int j = items[k];
  const double4 p = pos[j];
  bpos[k] = make_double4(p.x, p.y, p.z, __longlong_as_double(j));
}

// Both lists of TA atoms per block, the fix lists sorted, candidates and all:
// a wave takes one atom at a time.  The atom's 5 x 5 x 5 stencil is 25 runs of
// bins that are adjacent in x and so adjacent in bpos; the lanes take the runs'
// atoms 64 at a time (in the found order of the serial scan), and ballots give
// each entry its place.  The fix entries' keys are sorted in registers, the
// rows are collected in LDS and written whole.  (One thread per atom walked
// the bins' scattered positions and stored one row per lane, and a sort read
// and wrote the fix rows again.)  A whole rebuild, before and after: 2048
// atoms 0.60 -> 0.17 ms, 32,000 0.63 -> 0.23, 256,000 1.44 -> 0.77, 2,048,000
// 9.2 -> 5.0.  Bound by instruction issue: 992 VALU and 128 LDS instructions
// per atom (counters), 4.6 ms of the 5.0; tiles of 32 atoms, with twice the
// waves per CU, take the same time.
// LDS: rows of the pair list, the fix list and the candidates per atom (padded
// to an odd length), and per wave the keys, their indices and the runs.
constexpr int kTileWaves = 16, kTileKeys = 256, kTileBlocks = 512;
struct NbTile {
  int rl, rf;  // row lengths
};
__host__ __device__ inline NbTile nb_tile(const NbLists& l) { return {l.cap_l | 1, l.cap_f | 1}; }
static size_t nb_tile_lds(const NbLists& l, int ta) {
  const NbTile t = nb_tile(l);
  return sizeof(int) * (static_cast<size_t>(ta) * (t.rl + 2 * t.rf + 3) + kTileWaves * (2 * l.cap_f + 64));
}

template <int E>
__device__ __forceinline__ int nb_tile_sort(const int nf, const int lane, const uint32_t* key_in,
                                            const int* jt, int* row_f, int* row_c) {
  uint32_t key[E];
#pragma unroll
  for (int s = 0; s < E; ++s) {
    const int n = lane * E + s;
    key[s] = n < nf ? key_in[n] : ~0u;
  }
  bitonic_wave<E>(key, lane);
  int jv[E], mine = 0;
#pragma unroll
  for (int s = 0; s < E; ++s) {
    const bool in = lane * E + s < nf;
    jv[s] = in ? jt[key[s] & 511u] : 0;
    mine |= (jv[s] < 0 ? 1 : 0) << s;  // the top bit marks a candidate
    jv[s] &= 0x7fffffff;
    if (in) row_f[lane * E + s] = jv[s];
  }
  const int cnt = __builtin_popcount(mine);
  int incl = cnt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(incl, o);
    if (lane >= o) incl += v;
  }
  int at = incl - cnt;
#pragma unroll
  for (int s = 0; s < E; ++s)
    if ((mine >> s) & 1) row_c[at++] = jv[s];
  return __shfl(incl, 63);
}

template <int TA>
__global__ __launch_bounds__(64 * kTileWaves) void k_nb_lists_tile(
    int nlocal, const double4* __restrict__ pos, const int* __restrict__ rep, NbBoxes b,
    const int* __restrict__ bstart, const double4* __restrict__ bpos, NbLists l, int* overflow) {
  extern __shared__ int s_nb[];
  const NbTile tl = nb_tile(l);
  int* s_l = s_nb;
  int* s_f = s_l + TA * tl.rl;
  int* s_c = s_f + TA * tl.rf;
  int* s_n = s_c + TA * tl.rf;  // [3][TA] row counts: pair, fix, candidates
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  int* mine = s_n + 3 * TA + wv * (2 * l.cap_f + 64);
  uint32_t* s_key = reinterpret_cast<uint32_t*>(mine);
  int* s_jt = mine + l.cap_f;
  int* s_pre = s_jt + l.cap_f;  // [32] atoms before each run, [32] where the run starts less that
  int* s_beg = s_pre + 32;
  const double reach2 = b.cg * b.cg * (1.0 + 1e-9);
  // a fixed grid walks the tiles; those of XCD x form one range
  const int ntiles = (nlocal + TA - 1) / TA, x8 = blockIdx.x % 8;
  const int last = static_cast<int>(static_cast<long>(ntiles) * (x8 + 1) / 8);
  for (int tile = static_cast<int>(static_cast<long>(ntiles) * x8 / 8) + blockIdx.x / 8; tile < last;
       tile += gridDim.x / 8) {
    const int i0 = tile * TA;
    for (int a = wv; a < TA; a += kTileWaves) {
      const int i = i0 + a;
      int nf = 0, nl = 0, nc = 0;
      if (i < nlocal) {
        const int r = rep[i];
        const double4 pi = pos[i];
        const int* nb = b.nb + 3 * r;
        const double* glo = b.glo + 3 * r;
        const int bc[3] = {bin_coord(pi.x, glo[0], b.bs, nb[0]), bin_coord(pi.y, glo[1], b.bs, nb[1]),
                           bin_coord(pi.z, glo[2], b.bs, nb[2])};
        // Squared distance from the atom to a bin slab; edge bins also hold the
        // atoms clamped into them and count as near.
        auto slab2 = [&](double x, int d, int c) {
          const double lo = glo[d] + c * b.bs, hi = lo + b.bs;
          const double g = (c <= 0 || c >= nb[d] - 1) ? 0.0 : (x < lo ? lo - x : (x > hi ? x - hi : 0.0));
          return g * g;
        };
        // lane 5 (dz + 2) + (dy + 2): the run of x bins within reach (between
        // the first and the last of them; bins farther than reach hold no entry)
        int beg = 0, len = 0;
        const int z = bc[2] + lane / 5 - 2, y = bc[1] + lane % 5 - 2;
        if (lane < 25 && z >= 0 && z < nb[2] && y >= 0 && y < nb[1]) {
          const double yz = slab2(pi.y, 1, y) + slab2(pi.z, 2, z);
          int x0 = 1 << 30, x1 = -1;
          for (int x = max(bc[0] - 2, 0); x <= min(bc[0] + 2, nb[0] - 1); ++x)
            if (slab2(pi.x, 0, x) + yz <= reach2) {
              x0 = min(x0, x);
              x1 = x;
            }
          if (x1 >= 0) {
            const int bin = b.bin_base[r] + nb[0] * (y + nb[1] * z);
            beg = bstart[bin + x0];
            len = bstart[bin + x1 + 1] - beg;
          }
        }
        int incl = len;
#pragma unroll
        for (int o = 1; o < 32; o <<= 1) {
          const int v = __shfl_up(incl, o);
          if (lane >= o) incl += v;
        }
        const int total = __shfl(incl, 31);
        if (lane < 32) {
          s_pre[lane] = incl - len;
          s_beg[lane] = beg - (incl - len);
        }
        wave_lds_sync();
        int* row_l = s_l + a * tl.rl;
        // four rounds of 64 atoms at a time: their loads travel together
        constexpr int U = 4;
        for (int f0 = 0; f0 < total; f0 += 64 * U) {
          int run[U];
#pragma unroll
          for (int u = 0; u < U; ++u) run[u] = 0;
#pragma unroll
          for (int step = 16; step > 0; step >>= 1)
#pragma unroll
            for (int u = 0; u < U; ++u)
              if (s_pre[run[u] + step] <= f0 + 64 * u + lane) run[u] += step;
          double4 q[U];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int f = f0 + 64 * u + lane;
            q[u] = bpos[f < total ? s_beg[run[u]] + f : 0];
          }
#pragma unroll
          for (int u = 0; u < U; ++u) {
            if (f0 + 64 * u >= total) break;
            const int j = static_cast<int>(__double_as_longlong(q[u].w));
            const double ex = q[u].x - pi.x, ey = q[u].y - pi.y, ez = q[u].z - pi.z;
            const double r2 = ex * ex + ey * ey + ez * ez;
            const bool other = f0 + 64 * u + lane < total && j != i;
            const bool inl = other && r2 < l.cl2, inf = other && r2 < l.cf2;
            const unsigned long long bl = __ballot(inl), bf = __ballot(inf);
            const unsigned long long below = (1ull << lane) - 1ull;
            if (inl) {
              const int k = nl + __popcll(bl & below);
              if (k < l.cap_l) row_l[k] = j;
            }
            if (inf) {
              const int k = nf + __popcll(bf & below);
              if (k < l.cap_f) {
                s_key[k] = (list_sort_q(r2, l.sort_scale) << 9) | static_cast<uint32_t>(k);
                s_jt[k] = j | (r2 < l.cand2 ? 0x80000000 : 0);
              }
            }
            nl += __popcll(bl);
            nf += __popcll(bf);
          }
        }
        if ((nf > l.cap_f || nl > l.cap_l) && lane == 0) atomicOr(overflow, 2);
        nf = min(nf, l.cap_f);
        nl = min(nl, l.cap_l);
        wave_lds_sync();
        nc = nf <= 128 ? nb_tile_sort<2>(nf, lane, s_key, s_jt, s_f + a * tl.rf, s_c + a * tl.rf)
                       : nb_tile_sort<4>(nf, lane, s_key, s_jt, s_f + a * tl.rf, s_c + a * tl.rf);
        wave_lds_sync();
      }
      if (lane == 0) {
        s_n[a] = nl;
        s_n[TA + a] = nf;
        s_n[2 * TA + a] = nc;
      }
    }
    __syncthreads();
    // whole rows: entry k of the block's atoms by consecutive lanes
    constexpr int kRows = 64 * kTileWaves / TA;
    const int at = threadIdx.x % TA, k0 = threadIdx.x / TA;
    const int i = i0 + at;
    const int nl = s_n[at], nf = s_n[TA + at], nc = s_n[2 * TA + at];
    for (int k = k0; k < nl; k += kRows) l.nbr_l[k * l.stride + i] = s_l[at * tl.rl + k];
    for (int k = k0; k < nf; k += kRows) l.nbr_f[k * l.stride + i] = s_f[at * tl.rf + k];
    if (l.cand)
      for (int k = k0; k < nc; k += kRows) l.cand[k * l.stride + i] = s_c[at * tl.rf + k];
    if (k0 == 0 && i < nlocal) {
      l.nn_l[i] = nl;
      l.nn_f[i] = nf;
      if (l.cand) l.ncand[i] = nc;
    }
    __syncthreads();
  }
}

static inline int nbk(long n, int b = kBlock) { return static_cast<int>((n + b - 1) / b); }

static hipError_t scan(const int* in, int n, int* out, int* tmp, hipStream_t s) {
  const int per = kSB * kSI;
  const int nb = (n + per - 1) / per;
  k_nb_scan_reduce<<<nb, kSB, 0, s>>>(in, n, tmp);
  k_nb_scan_blocks<<<1, kSB, 0, s>>>(tmp, nb);
  k_nb_scan_apply<<<nb, kSB, 0, s>>>(in, n, tmp, out);
  return hipGetLastError();
}

hipError_t launch_nb_build(const NbBuild& w, hipStream_t s) {
  const int cap = w.nlocal + w.ghost_cap;
  k_nb_wrap<<<nbk(w.nlocal), kBlock, 0, s>>>(w.nlocal, w.at.pos, w.at.pv, w.at.rep, w.box);
  // ghost passes: nghost[0] = 0, nghost[d + 1] = after pass d
  k_nb_zero<<<1, 64, 0, s>>>(w.nghost, 4);
  for (int d = 0; d < 3; ++d) {
    k_nb_ghost_count<<<nbk(cap), kBlock, 0, s>>>(d, cap, w.nlocal, w.nghost + d, w.at.pos, w.at.rep,
                                                 w.box, w.cnt);
    (void)scan(w.cnt, cap, w.start, w.scan_tmp, s);
    k_nb_ghost_write<<<nbk(cap), kBlock, 0, s>>>(d, cap, w.nlocal, w.nghost + d, w.nghost + d + 1,
                                                 w.cnt, w.start, w.at, w.box, w.ghost_cap,
                                                 w.overflow);
  }
  const int* ng = w.nghost + 3;
  k_nb_zero<<<nbk(w.nbins + 1), kBlock, 0, s>>>(w.bcount, w.nbins + 1);
  k_nb_zero<<<nbk(w.nbins + 1), kBlock, 0, s>>>(w.bfill, w.nbins + 1);
  k_nb_bin<<<nbk(cap), kBlock, 0, s>>>(cap, w.nlocal, ng, w.at.pos, w.at.rep, w.box, w.bin_of,
                                       w.bcount);
  (void)scan(w.bcount, w.nbins, w.bstart, w.scan_tmp, s);
  k_nb_bin_scatter<<<nbk(cap), kBlock, 0, s>>>(cap, w.nlocal, ng, w.bin_of, w.bstart, w.bfill,
                                               w.items);
  k_nb_bin_sort<<<nbk(w.nbins), kBlock, 0, s>>>(w.nbins, w.bstart, w.items);
  // lists of at most kTileKeys fix entries whose rows fit the LDS: the tiled
  // build, 64 atoms per block where they do
  constexpr size_t kLdsMax = 160 * 1024 - 1024;
  const int ta = w.lists.cap_f > kTileKeys ? 0 : nb_tile_lds(w.lists, 64) <= kLdsMax ? 64
               : nb_tile_lds(w.lists, 32) <= kLdsMax ? 32 : 0;
  if (ta) {
    k_nb_bin_pos<<<nbk(cap), kBlock, 0, s>>>(cap, w.nlocal, ng, w.at.pos, w.items, w.bpos);
    const size_t lds = nb_tile_lds(w.lists, ta);
    auto kern = ta == 64 ? k_nb_lists_tile<64> : k_nb_lists_tile<32>;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    if (e != hipSuccess) return e;
    kern<<<std::min((nbk(w.nlocal, ta) + 7) / 8 * 8, kTileBlocks), 64 * kTileWaves, lds, s>>>(w.nlocal, w.at.pos, w.at.rep, w.box, w.bstart,
                                                         w.bpos, w.lists, w.overflow);
  } else {
    if (w.lists.cap_f > kListSortMax) return hipErrorInvalidValue;  // more fix-list entries per atom than the sort takes
    NbLists found = w.lists;
    found.cand = nullptr;  // the candidates are written in the sorted order by k_nb_sort
    k_nb_lists<<<nbk(w.nlocal), kBlock, 0, s>>>(w.nlocal, w.at.pos, w.at.rep, w.box, w.bstart,
                                                w.items, found, w.overflow);
    const int sb = std::min(kSortBlocks, nbk(w.nlocal, kBlock / 64));
    k_nb_sort<8><<<sb, kBlock, 0, s>>>(w.nlocal, w.at.pos, w.lists);
  }
  const bool cw = w.lists.cand && w.cref && w.cand_valid;
  k_nb_finish<<<nbk(cw ? cap : w.nlocal), kBlock, 0, s>>>(w.nlocal, ng, w.at.pos, w.xref,
                                                          w.nrebuild, w.cand_valid, w.cref, cw);
  return hipGetLastError();
}

}  // namespace eph
