"""The cut of a panel leaf into workgroups (scalapack_amd/csrc/sla_panel_plan.h), by
arithmetic on the host: its workgroups hold all rows, and those that wait for one
another find room together whatever other leaves run.

A SIMD has 512 registers a lane, so a workgroup of four waves with 128 registers takes
a quarter of its CU.  On one XCD (32 CUs) four leaves have to fit at once, or the leaf
gives way; dealt over the eight XCDs, at least eight of at most 32 workgroups, and two
of any.
"""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "scalapack_amd" / "csrc"

PROGRAM = r"""
#include "sla_panel_plan.h"
#include <cstdio>
using namespace sla;
int main()
{
    const int heights[] = {1, 2, 16, 63, 511, 512, 513, 1024, 1025, 2048, 2049, 4096, 4097, 8192, 8193,
                           12000, 16384, 16385, 20011, 30011, 32768, 32769, 50001, 65536, 65537,
                           100000, 131072, 131073, 262144, 262145, 524288, 524289};
    for (int m : heights)
        for (int wa = 1; wa <= 32; wa++)
            for (int wgs : {1, 8, 32, 64, 128})
                for (int beside = 0; beside < 2; beside++)
                    for (int xcds = 0; xcds < 2; xcds++) {
                        const LeafPlan p = leaf_plan(m, wa, wgs, beside, xcds);
                        std::printf("%d %d %d %d %d %d %d %d %d %d %d\n", m, wa, wgs, beside, xcds, p.values,
                                    p.waves, p.wgs, (int)p.place, leaf_quarters(p), leaf_nc(wa));
                    }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not found")
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(d / "plan.cpp"), "-o",
                    str(d / "plan")], check=True)
    out = subprocess.run([str(d / "plan")], check=True, capture_output=True, text=True).stdout
    keys = "m wa panel_wgs beside xcds values waves wgs place quarters nc".split()
    return [dict(zip(keys, map(int, line.split()))) for line in out.splitlines()]


SPREAD, ONE_XCD, ONE_XCD_YIELDS = range(3)
GMAX, XCDS, XCD_CUS = 128, 8, 32


def test_rows_are_held(plans):
    for p in plans:
        rows = 16 * (p["values"] // p["nc"]) * p["waves"]
        assert p["wgs"] * rows >= p["m"], p
        assert (p["wgs"] - 1) * rows < p["m"], p
        assert 1 <= p["waves"] <= 8 and p["values"] in (16, 32, 64), p
        # the tallest leaf that 64 values a thread hold in 128 workgroups of 512
        assert (p["wgs"] <= GMAX) == (p["m"] <= GMAX * 16 * (64 // p["nc"]) * 8), p


def test_waiting_workgroups_find_room(plans):
    for p in plans:
        if p["wgs"] == 1 or p["wgs"] > GMAX:
            assert p["place"] == SPREAD, p
            continue
        if p["place"] == ONE_XCD:
            assert p["xcds"] and 4 * p["wgs"] * p["quarters"] <= 4 * XCD_CUS, p
        elif p["place"] == ONE_XCD_YIELDS:
            # alone it fits; a leaf of one column ends before it could give way
            assert p["xcds"] and p["wa"] > 1 and p["nc"] == 8 and p["waves"] == 8 and p["wgs"] * p["quarters"] <= 4 * XCD_CUS, p
        else:
            leaves = 8 if p["wgs"] <= 32 else 2
            per_xcd = -(-p["wgs"] // XCDS)
            assert leaves * per_xcd * p["quarters"] <= 4 * XCD_CUS, p


def test_narrow_leaves_hold_few_rows_a_quad(plans):
    """At most 16 columns: 64 values a thread only where nothing else holds the rows."""
    for p in plans:
        if p["nc"] < 8 and p["m"] <= GMAX * 16 * ((16 if p["nc"] == 2 else 32) // p["nc"]) * 8:
            assert p["values"] < 64, p


def test_preferred_workgroups(plans):
    """panel_wgs over its whole range, wide leaves with no update beside them: at most
    that many where a kind allows it, and more of them where the caller asks for more
    than one die runs."""
    by = {(p["m"], p["wa"], p["panel_wgs"]): p for p in plans if not p["beside"] and p["xcds"]}
    for (m, wa, wgs), p in by.items():
        if p["nc"] == 8 and m <= wgs * 16 * 8 * 8:
            assert p["wgs"] <= wgs, p
    assert [by[30011, 32, w]["wgs"] for w in (8, 32, 64, 128)] == [30, 30, 59, 118]
