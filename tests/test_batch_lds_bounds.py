"""LDS index bounds of the batch kernel's grid transforms, checked on the CPU.

The batch kernel transforms each cell's grid through two LDS buffers (28672 B
each: 3584 FP32 or 1792 FP64 complex entries) and a twiddle table of 3 x 64
entries.  The library walks a grid on the host with the schedule it hands to
the kernel and the index functions the kernel is compiled from
(nb_test_batch_walk): every step (slabs of whole planes, rows and columns of
planes that exceed a buffer, columns along z) and every butterfly of every
pass.  Each LDS read, write and twiddle index stays inside its buffer, each
element is read and written once in a pass, each grid point is taken once in
each direction.  The tuner's workgroup sizes change only the thread stride of
the same index set.  The sum of a workgroup's static LDS (63,288 B at most) is
asserted where the kernel is compiled."""
import ctypes

import numpy as np
import pytest

from forcefieldx_amd import ffi


def radices(n):
    """The prime factors of n among 2, 3, 5 and 7; None when it has another."""
    r = []
    for p in (2, 3, 5, 7):
        while n % p == 0:
            r.append(p)
            n //= p
    return r if n == 1 else None


# the edges the batch path admits (at least 8 for any grid, at most 64 for this kernel)
ADMITTED = [k for k in range(8, 65) if radices(k) is not None]
TW_CAP = 3 * 64


def walk(grid, precision, slip=0):
    why = ctypes.create_string_buffer(200)
    rc = ffi.load().nb_test_batch_walk(*map(int, grid), precision, slip, why, len(why))
    return rc, why.value.decode()


def test_admitted_edges():
    assert 64 in ADMITTED and 49 in ADMITTED and 11 not in ADMITTED and 22 not in ADMITTED


@pytest.mark.parametrize("precision", [ffi.NB_PREC_FP64, ffi.NB_PREC_MIXED], ids=["fp64", "mixed"])
def test_every_lds_index_of_the_batch_transforms_is_in_bounds(precision):
    # every plane, with the z edges taken in turn, and every z edge on the smallest and largest planes
    grids = [(a, b, ADMITTED[(7 * i + j) % len(ADMITTED)]) for i, a in enumerate(ADMITTED) for j, b in enumerate(ADMITTED)]
    grids += [(a, b, c) for c in ADMITTED for a, b in ((8, 8), (8, 64), (64, 8), (64, 64), (42, 42), (42, 45))]
    for grid in grids:
        assert walk(grid, precision) == (0, ""), grid


@pytest.mark.parametrize("precision", [ffi.NB_PREC_FP64, ffi.NB_PREC_MIXED], ids=["fp64", "mixed"])
def test_the_walk_finds_mistakes(precision):
    """A plane too many in a slab, a wrong magic number, edges no grid has."""
    for grid in ((32, 28, 63), (24, 18, 48)):
        assert walk(grid, precision, 1)[0] == walk(grid, precision, 2)[0] == 1, grid
    assert walk((22, 16, 16), precision)[0] == walk((7, 16, 16), precision)[0] == walk((16, 70, 16), precision)[0] == 1


def test_twiddle_tables_of_three_axes_fit():
    # the three axes' tables are stored one after the other: K0 + K1 + K2 <= 3 x 64
    assert 3 * max(ADMITTED) <= TW_CAP and np.prod(radices(max(ADMITTED))) == 64
