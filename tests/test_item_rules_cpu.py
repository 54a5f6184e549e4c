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
#include <vector>
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
        } else if (what == "entry_costs") {
            for (int cbits = 0; cbits < 256; cbits++) std::cout << entry_cost(cbits) << " ";
            std::cout << NB_MIN_ITEM_COST << "\n";
        } else if (what == "item_cost") {
            ItemCut c;
            long long total;
            int nsc;
            std::cin >> c.most >> c.held >> total >> nsc;
            std::cout << item_cost(c, total, nsc) << "\n";
        } else if (what == "cut") {         // the entries of a block: the items' first entries
            int per_item, m, total = 0, p = 0;
            std::cin >> per_item >> m;
            std::vector<int> cost(m);
            for (int &c : cost) {
                std::cin >> c;
                total += c;
            }
            const int n = items_of(total, per_item);
            std::cout << n;
            for (int k = 0; k < m; k++) {
                const int q = item_of(p, n, total), before = k > 0 ? item_of(p - cost[k - 1], n, total) : -1;
                if (q != before) std::cout << " " << q << " " << k;
                p += cost[k];
            }
            std::cout << "\n";
        } else if (what == "bins") {
            int per_item, m, c;
            std::cin >> per_item >> m;
            for (int k = 0; k < m; k++) {
                std::cin >> c;
                const int n = items_of(c, per_item);
                std::cout << n << " " << (n > 0 ? item_bin(c, n, per_item) : -1) << " ";
            }
            std::cout << NB_IORDER_BINS << "\n";
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


def test_no_work_item_is_empty(rules):
    """The cut of a block's entries at equal steps of their cost: every item of the block starts at exactly one entry, in
    order, the first at the first entry, and no item costs more than a step and an entry; for costs of every kind, the
    smallest cost per item, and totals just above a whole number of items."""
    costs = rules(["entry_costs"])[0]
    least = costs.pop()
    top, some = max(costs), sorted(set(costs) - {0})
    assert costs[0] == 0 and least == 2 * top
    rng = np.random.default_rng(4)
    blocks = [[top] * m for m in range(1, 300)] + [[some[0]] * m for m in range(1, 300)]
    blocks += [rng.choice(some, rng.integers(1, 700)).tolist() for _ in range(300)]
    blocks += [[top] * m + [some[0]] * r for m in (2, 4, 64) for r in range(1, 13)]
    blocks += [[some[0]] * r + [top] * m for m in (2, 4, 64) for r in range(1, 13)]
    cases = [(per, b) for b in blocks for per in (least, least + 1, 44, 176, 1408)]
    for (per, b), got in zip(cases, rules(["cut %d %d %s" % (per, len(b), " ".join(map(str, b))) for per, b in cases])):
        n, q, first = got[0], got[1::2], got[2::2]
        assert n == -(-sum(b) // per) and q == list(range(n)) and first[0] == 0
        ends = first[1:] + [len(b)]
        assert all(0 < e - f for f, e in zip(first, ends))
        assert all(sum(b[f:e]) <= sum(b) / n + top for f, e in zip(first, ends))


def test_cost_per_item_follows_its_rules(rules):
    """item_cost: the nominal cost without a limit of waves; from a quarter of it for short lists; whole rounds of waves for
    long ones, half an item per block included; never below the smallest cost."""
    least = rules(["entry_costs"])[0][-1]
    rng = np.random.default_rng(5)
    cases = [(int(m), int(h), int(t), int(b)) for m, h, t, b in
             zip(rng.choice([11, 44, 176, 352, 1408], 4000), rng.choice([0, 3072, 4096, 5120], 4000),
                 np.exp(rng.uniform(0.0, 20.0, 4000)), rng.integers(1, 4000, 4000))]
    for (most, held, total, nsc), (got,) in zip(cases, rules(["item_cost %d %d %d %d" % c for c in cases])):
        nominal = max(most, least)
        assert got >= least
        if held == 0:
            assert got == nominal
        elif total < most * (held // 16):
            assert max(most // 4, least) <= got <= nominal
        elif total < most * held // 2:
            assert got == nominal
        elif got > least and got != most:
            rounds = (total + most * held // 2) // (most * held)
            assert total / got + nsc // 2 <= rounds * held
            assert got <= 3 * most + 1


def test_image_items_tile_their_list_by_falling_cost(rules):
    """The image lists' layout: the blocks of a step of cost follow those of the steps above it, so the offsets made from
    the steps' totals give every item one place."""
    rng = np.random.default_rng(6)
    for per in (34, 66, 96, 768):
        c = np.concatenate([rng.integers(0, 20 * per, 3000), np.arange(0, 3 * per)])
        got = rules(["bins %d %d %s" % (per, c.size, " ".join(map(str, c)))])[0]
        bins = got.pop()
        n, step = np.array(got[0::2]), np.array(got[1::2])
        assert (n == -(-c // per)).all()
        used = n > 0
        assert (step[used] >= 0).all() and (step[used] < bins).all()
        each = c[used] // n[used]
        order = np.argsort(each, kind="stable")
        assert (np.diff(step[used][order]) <= 0).all()
        start = np.concatenate([[0], np.cumsum(np.bincount(step[used], weights=n[used], minlength=bins))]).astype(int)
        place, cursor = [], start[:-1].copy()
        for k in rng.permutation(np.flatnonzero(used)):
            place.extend(range(cursor[step[k]], cursor[step[k]] + n[k]))
            cursor[step[k]] += n[k]
        assert np.array_equal(np.sort(place), np.arange(n.sum()))
        assert (cursor == start[1:]).all()
