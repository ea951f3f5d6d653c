"""The solver's launches at the sizes where their dispatch changes, against
the oracle: one workgroup's worth of atoms, all workgroups of a field launch
resident together or not (spread and field workgroups in order or
alternating), partial sums read by their consumers or collapsed beside the
spread (more than 2,048 workgroups), brick edges of unequal length, grids with
plane, compile-time and runtime-size transforms."""
import numpy as np
import pytest

from forcefieldx_amd import ffi
from forcefieldx_amd.forcefield import NonbondedParams
from forcefieldx_amd.systems import water_box

pytestmark = pytest.mark.gpu

DENSITY = 6912 / 59.1 ** 3
CASES = {
    # name: (waters, grid)
    "648": (216, (24, 24, 24)),
    "711-runtime-size": (237, (21, 28, 35)),
    # x lines assembled by a launch of their own (FP64; a point every 0.011 A is
    # no grid for the mixed form: second differences of FP32 values lose 1e4)
    "711-longest-lines": (237, (1701, 9, 14)),
    "3003": (1001, (40, 40, 40)),
    "9000-unequal-edges": (3000, (60, 48, 72)),
    "66003-collapsed": (22001, (96, 96, 96)),
}


def solve(name, precision, graph=False):
    waters, grid = CASES[name]
    xyz, box, top = water_box(waters, (waters / DENSITY) ** (1.0 / 3.0), seed=5)
    p = NonbondedParams(vdw_cutoff=9.0, grid=grid, polar_eps=1e-6)
    h = ffi.Handle(ffi.params_from(p, grid, precision), top)
    try:
        h.set_cell(box)
        h.set_positions(xyz)
        h.set_graph(graph)
        out = []
        for _ in range(3 if graph else 1):
            e, _ = h.evaluate(ffi.NB_GRAD)
            out.append((e, h.gradient().copy(), h.induced()[0].copy()))
        return out, xyz, box, top, p
    finally:
        h.close()


@pytest.mark.parametrize("name", list(CASES))
def test_fp64_equals_oracle(oracle, name):
    [(e, g, u)], xyz, box, top, p = solve(name, ffi.NB_PREC_FP64)
    eo, go, uo, _ = oracle.evaluate(oracle.System(xyz, box, top), p)
    assert e["pcg_iters"] == eo["pcg_iters"]
    for k in ("perm", "pol", "vdw"):
        assert abs(e[k] - eo[k]) <= 1e-8 * abs(eo[k]), k
    assert np.linalg.norm(g - go) <= 1e-8 * np.linalg.norm(go)
    assert np.linalg.norm(u - uo) <= 1e-8 * np.linalg.norm(uo)


@pytest.mark.parametrize("name", [c for c in CASES if c != "711-longest-lines"])
def test_mixed_and_replays(name):
    """The mixed form within the 1e-5 bar of FP64, and graph replays equal to
    the recorded evaluation (the energy sums are atomic: 1e-12)."""
    [(e64, g64, u64)], *_ = solve(name, ffi.NB_PREC_FP64)
    runs, *_ = solve(name, ffi.NB_PREC_MIXED, graph=True)
    for e, g, u in runs:
        assert np.linalg.norm(g - g64) <= 1e-5 * np.linalg.norm(g64)
        assert np.linalg.norm(u - u64) <= 1e-5 * np.linalg.norm(u64)
        assert abs(e["total"] - runs[0][0]["total"]) <= 1e-11 * abs(e["perm"])
        assert np.linalg.norm(g - runs[0][1]) <= 1e-12 * np.linalg.norm(g)
