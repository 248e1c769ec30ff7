"""The rules by which a context chooses its launches, on the host: a program built against
the library's headers asks a context object (no device) what it would do."""
import os
import subprocess

import pytest

from conftest import PKG, ROOT

HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "fluid.hpp"
using namespace pbd;
static uint32_t arg(char** v, int i) { return (uint32_t)std::strtoul(v[i], nullptr, 10); }
int main(int, char** v) {
  const char* what = v[1];
  Fluid f;
  if (what[0] == 's') {  // shape: particles, then the small tiles by default, after get -> set, after the skin alone
    f.n_ = arg(v, 2);
    const uint32_t before = f.small_tiles(), reported = f.launch_shape().small_max;
    Fluid::LaunchShape s = f.launch_shape();
    int rc = f.set_launch_shape(s);
    const uint32_t same = f.small_tiles();
    s.skin_pct = 5;
    rc |= f.set_launch_shape(s);
    std::printf("%d %u %u %u %u %u\n", rc, reported, f.launch_shape().small_max, before, same, f.small_tiles());
  } else {  // grid: blocks, particles
    std::printf("%d %u\n", capped_grid(arg(v, 2), arg(v, 3)) ? 1 : 0, direct_grid(arg(v, 2), arg(v, 3)));
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(PROGRAM)
    # the rules are private members: the program reads them, the library's layout is unchanged
    subprocess.run([HIPCC, "-O0", "-std=c++17", "-x", "hip", "--cuda-host-only", "-fno-access-control",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(PKG, "csrc"), str(d / "rules.cpp"),
                    "-o", str(d / "rules"), "-L" + PKG, "-lpbd", "-Wl,-rpath," + PKG], check=True)

    def run(*args):
        out = subprocess.run([str(d / "rules"), *map(str, args)], check=True, capture_output=True, text=True).stdout
        return [int(x) for x in out.split()]

    return run


@pytest.mark.parametrize("n,small,tiles", [(1, 0, 0), (1 << 16, 0, 0), ((1 << 16) + 1, 32, 64), (1 << 20, 32, 64),
                                           ((1 << 21) - 1, 32, 64), (1 << 21, 64, 64)])
def test_a_shape_read_and_set_again_launches_the_same_step(ask, n, small, tiles):
    rc, reported, after, default, same, skin = ask("shape", n)
    assert rc == 0 and reported == small and after == small
    assert default == tiles and same == tiles and skin == tiles


# around 2^20 items, where a step leaves the direct grid (and a phased one its tiles), by
# blocks and by particles; few blocks; one
@pytest.mark.parametrize("blocks,n,capped", [(1 << 22, 1 << 20, 0), (1 << 22, (1 << 20) + 1, 1), (1 << 20, 1 << 24, 0),
                                             ((1 << 20) + 1, 1 << 24, 1), (1 << 22, 1042411, 0), (1 << 22, 1047000, 0),
                                             (40960, 1 << 20, 0), (1, 5000, 0), (16, 1, 0)])
def test_split_blocks_do_not_decide_the_grid(ask, blocks, n, capped):
    is_capped, grid = ask("grid", blocks, n)
    assert is_capped == capped
    # every block, and as many halves more as there can be: a halo of more than 1528
    # particles, each particle in at most 8 halos
    items = min(blocks, n) + min(blocks, n // 191)
    assert grid >= items and grid % 32 == 0 and grid < items + 64
