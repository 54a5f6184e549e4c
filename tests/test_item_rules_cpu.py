"""CPU checks of the rules by which the work items of the pair kernel are made and laid out.

The rules are the inline functions of csrc/nbabfs_kernels.h that the device and host code call; a small host program
compiled from that header evaluates them.
"""

import os
import re
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HARNESS = r"""
#include "nbabfs_kernels.h"
#include <iostream>
#include <string>
int main()
{
    std::string what;
    while (std::cin >> what) {
        if (what == "group") {
            std::cout << NB_TILED_WPG << "\n";
        } else if (what == "padded") {
            int n;
            std::cin >> n;
            std::cout << padded_items(n) << "\n";
        } else if (what == "waves") {
            int full_fp64, images, queue;
            std::cin >> full_fp64 >> images >> queue;
            std::cout << tiled_waves(full_fp64 != 0, images != 0, queue != 0) << "\n";
        }
    }
}
"""


@pytest.fixture(scope="session")
def rules(tmp_path_factory):
    """rules(lines) -> one list of ints per line."""
    from pdynamo_amd import build
    d = tmp_path_factory.mktemp("rules")
    src, exe = d / "rules.cpp", d / "rules"
    src.write_text(HARNESS)
    r = subprocess.run([build.HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-I" + build.INCLUDE,
                        "-I" + build.CSRC, str(src), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]

    def ask(lines):
        out = subprocess.run([str(exe)], input="\n".join(lines) + "\n", capture_output=True, text=True, check=True).stdout
        return [[int(v) for v in line.split()] for line in out.splitlines()]
    return ask


def test_batch_groups_hold_one_system(rules):
    """A workgroup of the pair launch evaluates the items of one system (they share its staged LJ rows): in a batch's
    layout every group of consecutive items carries one system, whatever the systems' item counts."""
    group = rules(["group"])[0][0]
    rng = np.random.default_rng(2)
    for counts in ([1], [0, 3, 0, 5], list(range(40)), rng.integers(0, 5000, 64).tolist()):
        padded = [v[0] for v in rules(["padded %d" % n for n in counts])]
        assert all(n <= p < n + group for n, p in zip(counts, padded))
        owner = np.repeat(np.arange(len(counts)), padded)
        assert owner.size % group == 0
        assert (owner.reshape(-1, group) == owner.reshape(-1, group)[:, :1]).all()


def test_lists_are_cut_for_the_waves_the_kernel_holds(rules, tmp_path):
    """tiled_waves, for which a list is cut to whole rounds of waves, is what the registers of the built kernel's
    instances allow (512 per lane and SIMD, in steps of 8)."""
    from pdynamo_amd import build
    if not os.path.exists(build.LIB):
        build.build()
    lib = shutil.copy(build.LIB, tmp_path)
    llvm = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(build.HIPCC))), "llvm", "bin")
    subprocess.run([os.path.join(llvm, "llvm-objdump"), "--offloading", lib], cwd=tmp_path, capture_output=True, check=True)
    notes = "".join(subprocess.run([os.path.join(llvm, "llvm-readelf"), "--notes", str(f)], capture_output=True, text=True,
                                   check=True).stdout for f in sorted(tmp_path.glob("*gfx950*")))
    found = 0
    # Template arguments: rows in LDS, images, full FP64, waves per workgroup.
    for img, full, wpg, rest in re.findall(r"\.name: +_Z13k_force_tiledILb[01]ELb([01])ELb([01])ELi(\d)E"
                                           r"(.*?)\.vgpr_spill_count", notes, re.S):
        vgprs = int(re.search(r"\.vgpr_count: +(\d+)", rest).group(1))
        queue = int(wpg == "1")
        assert rules(["waves %s %s %d" % (full, img, queue)]) == [[512 // ((vgprs + 7) // 8 * 8)]], (img, full, wpg, vgprs)
        found += 1
    assert found == 10
