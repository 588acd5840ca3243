// eph_shares.hpp -- how the harness's step divides the time of a kernel that
// serves the fix and the harness: by the bytes that each side moves.
#pragma once

namespace eph {

// The initial kick (224 B an atom) with the check of the lists (32): the fix's
// part.  check: both in one kernel (lists rebuilt on the device), the kick alone
// otherwise; moves: the kick moves atoms (EPH_NOINT off, the harness's atoms in
// the fix's group), else there is only the check.
inline double kick_share(bool check, bool moves) {
  if (!check) return 1.0;
  return moves ? 224.0 / 256.0 : 0.0;
}

// The ghost update (228 B a ghost) with the density sweep's candidate check (64
// an atom, ghosts too), which is the fix's
inline double ghosts_share(bool check, double nlocal, double nghost) {
  const double c = check ? 64.0 * (nlocal + nghost) : 0.0;
  return c > 0.0 ? c / (c + 228.0 * nghost) : 0.0;
}

}  // namespace eph
