"""Grids of the batch kernel at the edges of its LDS buffers.

A cell's grid goes through LDS in slabs of whole z planes while a plane fits a
buffer (1792 complex points in FP64, 3584 in FP32), and through memory
otherwise: planes of exactly the buffer, just above it, a single slab, and a
last slab that is smaller than the others.  FP64 against the oracle as in the
other batch tests (1e-8), the mixed form against FP64 at its 1e-5."""
import dataclasses

import numpy as np
import pytest

from forcefieldx_amd import ffi
from forcefieldx_amd.forcefield import NonbondedParams
from forcefieldx_amd.systems import crystal_batch

PARAMS = NonbondedParams(ewald_cutoff=6.0, vdw_cutoff=6.0, polar_eps=1e-8)
FFT_CAP = {"float": 28672 // 8, "double": 28672 // 16}
EDGES = {
    "double": [(42, 42, 15), (64, 28, 21), (40, 45, 18), (12, 10, 14), (28, 30, 27), (64, 64, 9)],
    "float": [(56, 64, 15), (60, 60, 18), (40, 45, 21), (12, 16, 14), (24, 25, 28), (64, 64, 9)],
}


def rel(a, b):
    a, b = np.asarray(a, float), np.asarray(b, float)
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def evaluate(systems, precision, params, shape=None):
    hs = []
    for xyz, box, top, grid in systems:
        h = ffi.Handle(ffi.params_from(params, grid, precision), top)
        h.set_cell(box)
        h.set_positions(xyz)
        hs.append(h)
    try:
        e, rc = ffi.evaluate_batch(hs, ffi.NB_GRAD) if shape is None else ffi.test_batch_shape(hs, shape)
        assert rc == ffi.NB_OK and ffi.batch_config()["systems"] == len(systems)
        return e, [h.gradient().reshape(-1, 3) for h in hs], [h.induced()[0] for h in hs]
    finally:
        for h in hs:
            h.close()


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["double", "float"])
def test_batch_grids_at_the_buffer_edges(oracle, form):
    grids = EDGES[form]
    systems = [(x, b, t, grids[k]) for k, (x, b, t, _) in enumerate(crystal_batch(len(grids), seed=9))]
    print("batch grids", form, grids, flush=True)
    if form == "double":
        e, g, u = evaluate(systems, ffi.NB_PREC_FP64, PARAMS)
        for k, (xyz, box, top, grid) in enumerate(systems):
            eo, go, uo, _ = oracle.evaluate(oracle.System(xyz, box, top), dataclasses.replace(PARAMS, grid=grid))
            scale = max(abs(eo[q]) for q in ("perm", "pol", "vdw"))
            for q in ("perm_recip", "pol", "total"):
                assert abs(e[k][q] - eo[q]) <= 1e-8 * scale, (grid, q, e[k][q], eo[q])
            assert rel(g[k], go) <= 1e-8 and rel(u[k], uo) <= 1e-8, grid
            assert e[k]["pcg_iters"] == eo["pcg_iters"], grid
    else:
        p = dataclasses.replace(PARAMS, polar_eps=1e-6)
        e, g, u = evaluate(systems, ffi.NB_PREC_MIXED, p)
        ed, gd, ud = evaluate(systems, ffi.NB_PREC_FP64, p)
        for k, (_, _, _, grid) in enumerate(systems):
            scale = max(abs(ed[k][q]) for q in ("perm", "pol", "vdw"))
            assert abs(e[k]["total"] - ed[k]["total"]) <= 1e-5 * scale, grid
            assert rel(g[k], gd[k]) <= 1e-5 and rel(u[k], ud[k]) <= 1e-5, grid


SHAPES = [(256, 8), (256, 16), (512, 8), (512, 16), (256, 4)]   # threads, lanes per atom
# factors 7 and 5, odd edges, a pass of 6 beside 5 and 7 and alone, planes above the buffer
MIXES = [(14, 30, 21), (42, 28, 35), (36, 50, 9), (24, 18, 48), (60, 42, 10), (64, 63, 49), (45, 15, 27), (6 * 7, 6 * 5, 54)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", range(len(SHAPES)), ids=["x".join(map(str, s)) for s in SHAPES])
def test_every_shape_on_mixed_radices(oracle, shape):
    """Each shape of the batch kernel by itself, FP64 against the oracle and the
    mixed form against FP64, so that none depends on what the tuner picks."""
    systems = [(x, b, t, MIXES[k]) for k, (x, b, t, _) in enumerate(crystal_batch(len(MIXES), seed=11))]
    print("batch shape", SHAPES[shape], flush=True)
    e, g, u = evaluate(systems, ffi.NB_PREC_FP64, PARAMS, shape)
    cfg = ffi.batch_config()
    assert (cfg["threads"], cfg["lanes"]) == SHAPES[shape]
    for k, (xyz, box, top, grid) in enumerate(systems):
        eo, go, uo, _ = oracle.evaluate(oracle.System(xyz, box, top), dataclasses.replace(PARAMS, grid=grid))
        scale = max(abs(eo[q]) for q in ("perm", "pol", "vdw"))
        for q in ("perm_recip", "perm_real", "pol", "vdw", "total"):
            assert abs(e[k][q] - eo[q]) <= 1e-8 * scale, (grid, q, e[k][q], eo[q])
        assert rel(g[k], go) <= 1e-8 and rel(u[k], uo) <= 1e-8, grid
        assert e[k]["pcg_iters"] == eo["pcg_iters"], grid
    p = dataclasses.replace(PARAMS, polar_eps=1e-6)
    e, g, u = evaluate(systems, ffi.NB_PREC_MIXED, p, shape)
    ed, gd, ud = evaluate(systems, ffi.NB_PREC_FP64, p, shape)
    for k, (_, _, _, grid) in enumerate(systems):
        scale = max(abs(ed[k][q]) for q in ("perm", "pol", "vdw"))
        for q in ("perm", "pol", "vdw", "total"):
            assert abs(e[k][q] - ed[k][q]) <= 1e-5 * scale, (grid, q)
        assert rel(g[k], gd[k]) <= 1e-5 and rel(u[k], ud[k]) <= 1e-5, grid


@pytest.mark.gpu
def test_shape_past_the_last():
    (xyz, box, top, grid), = crystal_batch(1, seed=11)
    h = ffi.Handle(ffi.params_from(PARAMS, grid, ffi.NB_PREC_FP64), top)
    h.set_cell(box)
    h.set_positions(xyz)
    assert ffi.test_batch_shape([h], len(SHAPES))[1] == -1 and ffi.test_batch_shape([h], -1)[1] == -1
    h.close()


def test_slab_transforms_stay_in_the_buffer():
    """A model of a slab's x and y passes, independent of the library's code
    (which test_batch_lds_bounds.py walks): for every plane of admitted edges that
    fits, each pass reads and writes every point exactly once, and magic numbers
    as the library makes them divide exactly."""
    def radices(n):
        r = []
        for p in (4, 2, 3, 5, 7):
            while n % p == 0:
                r.append(p)
                n //= p
        if 2 in r and 3 in r:  # one pass of 6
            r[r.index(2)] = 6
            r.remove(3)
        return r if n == 1 else None

    def div(n, d):
        m = (2**32 + d - 1) // d if d > 1 else 0
        return (n.astype(np.uint64) * np.uint64(m) >> np.uint64(32)).astype(np.int64) if m else n

    n = np.arange(4096)
    for d in range(1, 4097):
        assert (div(n, d) == n // d).all(), d
    edges = [k for k in range(2, 65) if radices(k)]
    for cap in FFT_CAP.values():
        for K0 in edges:
            for K1 in edges:
                pl = K0 * K1
                if pl > cap:
                    continue
                for planes in {1, cap // pl}:
                    for N, inner, so, se, lines in ((K0, 1, K0, 1, planes * K1), (K1, K0, pl, K0, planes * K0)):
                        Ns = 1
                        for R in radices(N):
                            nb = N // R
                            b = np.arange(lines * nb)
                            q = div(b, inner)
                            i = b - q * inner
                            o = div(q, nb)
                            j = q - o * nb
                            jq = div(j, Ns)
                            jm = j - jq * Ns
                            k = np.arange(R)[:, None]
                            for place in (i + o * so + (j + k * nb) * se, i + o * so + (jq * Ns * R + jm + k * Ns) * se):
                                seen = np.zeros(planes * pl, int)
                                np.add.at(seen, place.ravel(), 1)
                                assert (seen == 1).all(), (K0, K1, planes, N, R)
                            assert (jm * (R - 1) * (nb // Ns)).max() < N
                            Ns *= R
