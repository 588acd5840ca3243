"""CPU: the division of the harness's shared kernels between the fix's time and its own."""
import os
import subprocess

SRC = r"""
#include <cstdio>
#include "eph_shares.hpp"
int main() {
  using namespace eph;
  std::printf("%.17g %.17g %.17g %.17g ", kick_share(true, true), kick_share(false, true), kick_share(true, false),
              kick_share(false, false));
  std::printf("%.17g %.17g %.17g\n", ghosts_share(true, 1000, 500), ghosts_share(false, 1000, 500),
              ghosts_share(true, 0, 0));
}
"""


def test_shares(tmp_path):
    (tmp_path / "s.cpp").write_text(SRC)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    exe = str(tmp_path / "s")
    subprocess.check_call(["g++", "-std=c++17", "-I", os.path.join(root, "user-eph_amd", "csrc"), "-o", exe,
                           str(tmp_path / "s.cpp")])
    got = [float(v) for v in subprocess.check_output([exe], text=True).split()]
    # a kick that moves nothing (EPH_NOINT, or no atom in the group) is the harness's check alone
    assert got == [0.875, 1.0, 0.0, 1.0, 64 * 1500 / (64 * 1500 + 228 * 500), 0.0, 0.0]
