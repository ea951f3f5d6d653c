"""What the library's host code asks the HIP runtime for, on a runtime without
a device (host_stub): graphs, streams, events and memory are used within the
runtime's rules, and dynamics records no graph."""
import ctypes

import numpy as np
import pytest

import host_stub
from forcefieldx_amd import ffi
from forcefieldx_amd.forcefield import NonbondedParams
from forcefieldx_amd.systems import crystal_batch, water_box

PARAMS = NonbondedParams(vdw_cutoff=9.0, ewald_cutoff=7.0, grid=(24, 24, 24), polar_eps=1e-4)
FORMS = pytest.mark.parametrize("precision", [ffi.NB_PREC_FP64, ffi.NB_PREC_MIXED], ids=["fp64", "mixed"])


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    return host_stub.build(str(tmp_path_factory.mktemp("host")))


@pytest.fixture
def stub(library, monkeypatch):
    monkeypatch.setattr(ffi, "_lib", None)
    s = host_stub.Stub(library)
    s.set()
    s.reset()
    s.kept = s.counts()["live"]   # what the batch kernel's pool keeps for the process
    yield s
    s.set()
    assert s.faults() == [] and s.counts()["live"] == s.kept


def handle(precision, grid=PARAMS.grid, waters=216):
    xyz, box, top = water_box(waters, 18.643 * (waters / 216) ** (1.0 / 3.0), seed=1)
    h = ffi.Handle(ffi.params_from(PARAMS, grid, precision), top)
    h.set_cell(box)
    h.set_positions(xyz)
    return h, xyz, np.ones(top.n)


def test_misuse_is_found(stub):
    """The runtime's model by itself: what the other tests rely on it to report."""
    L, v = stub.L, ctypes.c_void_p
    for f in ("hipMemcpyAsync", "hipMemsetAsync", "hipStreamWaitEvent", "hipEventRecord", "hipStreamBeginCapture",
              "hipStreamEndCapture", "hipGraphInstantiate", "hipGraphLaunch", "hipGraphExecDestroy", "hipGraphDestroy",
              "hipStreamSynchronize", "hipStreamDestroy", "hipEventDestroy", "hipFree", "hipMalloc"):
        getattr(L, f).argtypes = None
    a, b, e, p, g, x = v(), v(), v(), v(), v(), v()
    L.hipStreamCreate(ctypes.byref(a)), L.hipStreamCreate(ctypes.byref(b)), L.hipEventCreate(ctypes.byref(e))
    L.hipMalloc(ctypes.byref(p), ctypes.c_size_t(64))

    def work(stream, nbytes=32):
        L.hipMemcpyAsync(p, v(p.value + 32), ctypes.c_size_t(nbytes), 3, stream)   # device to device

    def record(joined=True, body=None):
        L.hipStreamBeginCapture(a, 0)
        work(a)
        L.hipEventRecord(e, a), L.hipStreamWaitEvent(b, e, 0)
        work(b)
        if body:
            body()
        if joined:
            L.hipEventRecord(e, b), L.hipStreamWaitEvent(a, e, 0)
        L.hipStreamEndCapture(a, ctypes.byref(g))
        return stub.taken_faults()

    assert record() == []
    L.hipGraphInstantiate(ctypes.byref(x), g, None, None, ctypes.c_size_t(0))
    L.hipGraphLaunch(x, a)
    L.hipGraphExecDestroy(x)
    assert stub.taken_faults() == ["a graph destroyed while a launch of it is outstanding"]
    L.hipStreamWaitEvent(b, e, 0)
    assert stub.taken_faults() == ["a wait for an event of a capture that has ended"]
    L.hipGraphDestroy(g)
    for joined, body, found in ((False, None, "a captured stream is not joined"),
                                (True, lambda: L.hipStreamSynchronize(a), "hipStreamSynchronize inside a capture"),
                                (True, lambda: L.hipMemsetAsync(p, 0, ctypes.c_size_t(8), a), "hipMemsetAsync in a captured graph")):
        assert found in record(joined, body), found
        L.hipGraphDestroy(g)
    work(a, 64)
    assert stub.taken_faults() == ["copy past the end of a device allocation (read)"]
    L.hipGraphDestroy(g)
    assert stub.taken_faults() == ["a graph destroyed that does not exist"]
    L.hipFree(p), L.hipEventDestroy(e), L.hipStreamDestroy(a), L.hipStreamDestroy(b)


@FORMS
def test_recorded_evaluations(stub, precision):
    """Replays with rejections (a list to rebuild) and budgets that shrink:
    every capture is joined, no graph is destroyed with a launch outstanding,
    nothing is left behind."""
    h, _, _ = handle(precision)
    h.set_graph(True)
    stub.reset()
    for step in range(30):
        bad = int(step % 9 == 8)
        stub.set(moved=bad, reject=bad, iterations=4 if step % 5 else 1)
        h.evaluate(ffi.NB_GRAD)
    c = stub.counts()
    assert h.graph_replays() >= 15 and c["instantiated"] == c["captures"] >= 4
    h.close()


@FORMS
def test_dynamics_records_no_graph(stub, precision):
    """Runs of a graph-mode handle, each with a new predictor, with list
    rebuilds between steps: neither a capture nor a graph."""
    h, xyz, mass = handle(precision)
    h.set_graph(True)
    h.evaluate(ffi.NB_GRAD)
    for run in range(3):
        h.set_scf_predictor(ffi.NB_PRED_ASPC)
        h.set_positions(xyz)
        h.md_init(mass, np.zeros(3 * len(mass)))
        stub.reset()
        for step in range(12):
            stub.set(moved=int(step % 5 == 4))
            assert h.md_step(2, 0.001)["steps"] == 2
        c = stub.counts()
        assert c["captures"] == c["instantiated"] == c["replays"] == c["destroyed"] == 0 and c["launches"] > 0
    h.close()


@FORMS
def test_strain_derivatives_leave_no_memory(stub, precision):
    """A handle that computed the virial frees the grid it kept for it."""
    h, _, _ = handle(precision)
    h.evaluate(ffi.NB_GRAD | ffi.NB_VIRIAL)
    h.close()


@FORMS
@pytest.mark.parametrize("edge", [1620, 1680, 2048])
def test_lds_of_the_longest_lines(stub, precision, edge):
    """The longest lines a grid may have: no launch asks for more than the
    64 KB of LDS that the kernels' layouts are kept to."""
    for grid in ((edge, 9, 14), (9, edge, 14), (9, 14, edge)):
        h, _, _ = handle(precision, grid)
        stub.reset()
        h.evaluate(ffi.NB_GRAD | ffi.NB_VIRIAL)
        assert 0 < stub.counts()["lds"] <= 65536
        h.close()


def test_radial_factors_are_an_option(stub):
    """The FP64 form's stored radial factors (16 bytes a row entry, its largest
    allocation here) are tried once per row capacity and left out when they
    fail or, from 64 MB on, would take more than a quarter of the free memory."""
    for waters in (216, 6912):
        h, _, _ = handle(ffi.NB_PREC_FP64, waters=waters)
        stub.reset()
        h.evaluate(ffi.NB_GRAD)   # the rows' capacities
        h.close()
        size = max(stub.allocations())
        assert size % (16 * h.n) == 0 and (size >= 64 << 20) == (waters == 6912)
        for kw, tries, held in ((dict(fail_bytes=size), 1, False),
                                (dict(free_bytes=4 * size - 1), 0, waters == 216)):
            h, _, _ = handle(ffi.NB_PREC_FP64, waters=waters)
            stub.set(**kw)
            stub.reset()
            for _ in range(3):
                h.evaluate(ffi.NB_GRAD)
            assert stub.counts()["failed"] == tries and (size in stub.allocations()) == held
            h.close()
            stub.set()


@FORMS
def test_batches(stub, precision):
    """Batches through the batch kernel, from the static scratch and through
    recorded graphs: what the pool keeps does not grow with the calls."""
    for _ in range(2):
        stub.kept = stub.counts()["live"]
        hs = []
        for xyz, box, top, grid in crystal_batch(6, seed=3):
            h = ffi.Handle(ffi.params_from(NonbondedParams(ewald_cutoff=6.0, vdw_cutoff=6.0), grid, precision), top)
            h.set_cell(box)
            h.set_positions(xyz)
            h.set_graph(True)
            hs.append(h)
        assert ffi.evaluate_batch(hs)[1] == ffi.evaluate_batch_static(hs)[1] == ffi.NB_OK
        for _ in range(3):
            assert ffi.evaluate_batch(hs, ffi.NB_GRAD | ffi.NB_BATCH_SEPARATE)[1] == ffi.NB_OK
        assert all(h.graph_replays() == 2 for h in hs)
        for h in hs:
            h.close()
