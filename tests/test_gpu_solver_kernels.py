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


def system(name):
    waters, grid = CASES[name]
    xyz, box, top = water_box(waters, (waters / DENSITY) ** (1.0 / 3.0), seed=5)
    return xyz, box, top, NonbondedParams(vdw_cutoff=9.0, grid=grid, polar_eps=1e-6)


def solve(name, precision, graph=False):
    """Evaluations of frames displaced a little from one another (the first as
    built), and how many were graph replays."""
    xyz, box, top, p = system(name)
    h = ffi.Handle(ffi.params_from(p, p.grid, precision), top)
    rng = np.random.default_rng(3)
    try:
        h.set_cell(box)
        h.set_graph(graph)
        out = []
        for step in range(4):
            h.set_positions(xyz + (rng.normal(0.0, 0.002, xyz.shape) if step else 0.0))
            e, _ = h.evaluate(ffi.NB_GRAD)
            out.append((e, h.gradient().copy(), h.induced()[0].copy()))
        return out, h.graph_replays()
    finally:
        h.close()


@pytest.mark.parametrize("name", list(CASES))
def test_fp64_equals_oracle(oracle, name):
    (e, g, u), *_ = solve(name, ffi.NB_PREC_FP64)[0]
    xyz, box, top, p = system(name)
    eo, go, uo, _ = oracle.evaluate(oracle.System(xyz, box, top), p)
    assert e["pcg_iters"] == eo["pcg_iters"]
    for k in ("perm", "pol", "vdw"):
        assert abs(e[k] - eo[k]) <= 1e-8 * abs(eo[k]), k
    assert np.linalg.norm(g - go) <= 1e-8 * np.linalg.norm(go)
    assert np.linalg.norm(u - uo) <= 1e-8 * np.linalg.norm(uo)


@pytest.mark.parametrize("name", [c for c in CASES if c != "711-longest-lines"])
def test_mixed(name):
    """The mixed form within the 1e-5 bar of FP64, on every frame."""
    for (_, g64, u64), (_, g, u) in zip(solve(name, ffi.NB_PREC_FP64)[0], solve(name, ffi.NB_PREC_MIXED)[0]):
        assert np.linalg.norm(g - g64) <= 1e-5 * np.linalg.norm(g64)
        assert np.linalg.norm(u - u64) <= 1e-5 * np.linalg.norm(u64)


@pytest.mark.parametrize("name", [c for c in CASES if c != "711-longest-lines"])
@pytest.mark.parametrize("precision", [ffi.NB_PREC_FP64, ffi.NB_PREC_MIXED], ids=["fp64", "mixed"])
def test_replays_equal_regular_evaluations(name, precision):
    """Graph replays on displaced frames (a recorded solve with its radial factors
    stored and read in FP64, its r.z totals collapsed in the largest case) against
    a handle that records nothing: the same iterations, gradients and dipoles (the
    energy sums are atomic: 1e-11 of the permanent energy)."""
    regular, none = solve(name, precision)
    replayed, replays = solve(name, precision, graph=True)
    print(f"{name}: {replays} replays, iterations {[e['pcg_iters'] for e, _, _ in replayed]}", flush=True)
    assert none == 0 and replays >= 2
    for (e, g, u), (eg, gg, ug) in zip(regular, replayed):
        assert eg["pcg_iters"] == e["pcg_iters"]
        assert abs(eg["total"] - e["total"]) <= 1e-11 * abs(e["perm"])
        assert np.linalg.norm(gg - g) <= 1e-12 * np.linalg.norm(g)
        assert np.linalg.norm(ug - u) <= 1e-12 * np.linalg.norm(u)
