"""Grids near the limits of the context's index types, on the CPU: the stage
kernel's byte offsets over the whole range of k that a context accepts, and the
grids that edus_create refuses before it reads a table."""
import os
import subprocess

import pytest

import helpers as Hh
from helpers import N

PROBE = r"""
#include <cstdio>
#include "offsets.hpp"
template <int NB> int wrong() {
    const long long most = kMaxStateElems / (NB * NB) / 256 * 256;  // padded k of the largest state
    int bad = 0;
    const long long ks[] = {0LL, 1LL, 255LL, (1LL << 28) - 1, 1LL << 28, (1LL << 29) - 1, 1LL << 29, (1LL << 29) + 1, most / 2 + 1, most - 1};
    for (long long k : ks)
        if (k < most) bad += (unsigned long long)small_offset<NB>((int)k) != 8ULL * (unsigned long long)k;
    return bad;
}
int main() { std::printf("%d %d %d %d\n", wrong<1>(), wrong<2>(), wrong<3>(), wrong<4>()); }
"""


def test_small_kernel_offsets_reach_every_k(tmp_path):
    src, exe = tmp_path / "probe.cpp", tmp_path / "probe"
    src.write_text(PROBE)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(Hh.ROOT, "edus_amd", "csrc", "hip"), str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split() == ["0"] * 4


@pytest.mark.parametrize("nb,nk", [(1, 2 ** 31 - 200), (2, 2 ** 29), (2, 2 ** 30), (3, 2 ** 28), (4, 2 ** 27), (5, 2 ** 31 // 25 + 1), (32, 2 ** 21),
                                   (32, 2 ** 22)])
def test_states_beyond_the_index_type_are_refused(nb, nk):
    p = N.Problem()
    p.nk, p.nb = nk, nb
    with pytest.raises(N.EdusError, match="grid too large"):
        N.Engine(p)
    p.nk = 2 ** 31 // (nb * nb) - 256  # fits: the next check is reached
    with pytest.raises(N.EdusError, match="missing table"):
        N.Engine(p)
