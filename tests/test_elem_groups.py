"""The work list of the HEX20 element pass (csrc/elem_groups.hpp) on the CPU: every element of
every domain group once, in as many workgroups as the groups need and no more, whatever
their sizes and number."""
import os
import subprocess

import pytest

from conftest import PKG

MAIN = r"""
#include "elem_groups.hpp"
#include <cstdio>
#include <cstdlib>
int main(int argc, char** argv) {
    const int em = atoi(argv[1]);
    std::vector<int64_t> base(1, 0);
    for (int i = 2; i < argc; ++i) base.push_back(base.back() + atoll(argv[i]));
    for (const int4& w : dtc::elem_groups(base, em)) printf("%d %d %d %d\n", w.x, w.y, w.z, w.w);
}
"""


@pytest.fixture(scope="module")
def groups(tmp_path_factory):
    d = tmp_path_factory.mktemp("groups")
    (d / "m.cpp").write_text(MAIN)
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I",
                    os.path.join(PKG, "csrc"), str(d / "m.cpp"), "-o", str(d / "m")], check=True)
    return lambda em, ne: [tuple(map(int, line.split())) for line in subprocess.run(
        [str(d / "m"), str(em), *map(str, ne)], capture_output=True, text=True, check=True).stdout.splitlines()]


@pytest.mark.parametrize("em", [4, 8])
@pytest.mark.parametrize("ne", [[], [0], [1], [4], [5], [8], [9], [0, 3, 0, 17, 8, 0], [5800] + [100] * 40, [1] * 2000])
def test_every_element_once(groups, em, ne):
    w = groups(em, ne)
    assert len(w) == sum(-(-n // em) for n in ne)
    seen = set()
    for g, e0, n, base in w:
        assert n == ne[g] and base == sum(ne[:g]) and e0 % em == 0 and e0 < n
        seen |= {base + e for e in range(e0, min(e0 + em, n))}
    assert len(seen) == sum(ne)
