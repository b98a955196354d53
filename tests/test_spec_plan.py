"""How a verify call is cut into workgroups (tms_spec_plan.h), on the host: the
launch arithmetic over batches, drafts, vocabularies and element types, compiled
by itself with the host compiler."""
from __future__ import annotations

import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NAMES = ("P", "Lp", "n2", "wait", "claim_parts", "S", "pv", "ns", "n1", "lazy", "claim_rows", "words")
MAIN = r"""
#include <stdio.h>
#include "tms_spec_plan.h"
int main() {
    int B, k, V, vec, cap1, cap2;
    while (scanf("%d %d %d %d %d %d", &B, &k, &V, &vec, &cap1, &cap2) == 6) {
        const tms::SpecPlan s = tms::spec_plan(B, k, V, vec, cap1, cap2);
        printf("%d %d %d %d %d %d %d %d %d %d %d %zu\n", s.P, s.Lp, s.n2, (int)s.wait, (int)s.claim_parts, s.S, s.pv,
               s.ns, s.n1, (int)s.lazy, (int)s.claim_rows, tms::spec_rpart_words(B, V));
    }
}
"""
# Workgroups resident at once on 256 compute units in 8 XCDs: the row kernel
# (two 1024-thread workgroups a CU) and the waiting resolve (256 threads).
CAP1, CAP2, XCDS = 512, 1024, 8
VOCABS = sorted({v + d for v in (1, 8, 2048, 4096, 8192, 16384, 32000, 32768, 65536, 98304, 128256, 131072, 151936,
                                 196608, 256000, 262144, 393216, 524288, 786432, 1048576)
                 for d in (-1, 0, 1) if 1 <= v + d <= 1048576})


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    """Every plan: the inputs and the fields, as columns."""
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("plan")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run([cxx, "-std=c++17", "-O1", "-I", os.path.join(ROOT, "tensormark_amd", "csrc"), "-o", d / "plan",
                    d / "main.cpp"], check=True)
    batches = [1, 2, 3, 4, 5, 7, 8, 9, 12, 16, 17, 24, 31, 32, 33, 64, 72, 96, 128, 257, 1024]
    cases = np.array([(B, k, V, vec, CAP1, CAP2) for B in batches for k in range(1, 17) for V in VOCABS
                      for vec in (4, 8)])
    text = "\n".join(" ".join(map(str, c)) for c in cases)
    out = subprocess.run([d / "plan"], input=text, capture_output=True, text=True, check=True).stdout
    got = np.array([line.split() for line in out.splitlines()], dtype=np.int64)
    assert len(got) == len(cases)
    return dict(zip(("B", "k", "V", "vec", "cap1", "cap2") + NAMES, np.concatenate([cases, got], axis=1).T))


def _first(p, bad):
    """The first case for which `bad` holds, for a failure's message."""
    i = int(np.flatnonzero(bad)[0])
    return {n: int(v[i]) for n, v in p.items()}


def test_every_row_is_covered_once(plans):
    p = plans
    nv = -(-p["V"] // p["vec"])
    bad = (p["S"] * p["pv"] < nv) | ((p["S"] - 1) * p["pv"] >= nv) | (p["pv"] > p["ns"] * 1024)
    assert not bad.any(), _first(p, bad)
    bad = (p["P"] * p["Lp"] < p["V"]) | ((p["P"] - 1) * p["Lp"] >= p["V"]) | (p["P"] > 64)
    assert not bad.any(), _first(p, bad)
    w = p["wait"] == 1
    bad = w & ((p["Lp"] > 16 * 256) | (p["Lp"] % (256 * p["vec"]) != 0))
    assert not bad.any(), _first(p, bad)
    rows = p["B"] * (2 * p["k"] + 1 - p["lazy"])
    bad = (p["n1"] < rows * p["S"]) | (p["n1"] % np.where(p["S"] > 1, 8 * p["S"], 1) != 0)
    assert not bad.any(), _first(p, bad)
    bad = (p["n2"] < p["B"] * p["P"]) | (p["n2"] % (8 * p["P"]) != 0)
    assert not bad.any(), _first(p, bad)
    # the maxima's and sums' words (two a part), the bonus rows' included
    bad = 2 * p["B"] * (2 * p["k"] + 1) * p["S"] > p["words"]
    assert not bad.any(), _first(p, bad)


def test_a_rows_parts_leave_room(plans):
    """A row's parts run on one XCD (a workgroup's index modulo 8 names both)
    and wait for each other: they have to fit it at once.  Beside them, three
    other contexts' parts: so a quarter of it, where the parts' length is a
    choice and not the registers' limit (V above 524288)."""
    p = plans
    bad = (p["S"] > 1) & (p["S"] > CAP1 // XCDS)
    assert not bad.any(), _first(p, bad)
    least = -(-p["V"] // 32768)
    bad = p["S"] > np.maximum(least, CAP1 // XCDS // 4)
    assert not bad.any(), _first(p, bad)


def test_places_are_claimed_where_the_grid_is_not_resident(plans):
    """The grids are padded to whole counters: it is the padded grid whose
    workgroups have to be resident at once, on every XCD."""
    p = plans
    bad = (p["S"] > 1) & (p["n1"] > CAP1) & (p["claim_rows"] == 0)
    assert not bad.any(), _first(p, bad)
    bad = (p["wait"] == 1) & (p["n2"] > CAP2) & (p["claim_parts"] == 0)
    assert not bad.any(), _first(p, bad)
