"""Element tables of the device set-up against the host's where rows outgrow
the 32 lanes that read them: a fan of prisms (or tetrahedra) around an edge
couples the edge's nodes to all others, up to the 256 entries a compact table
can address; element counts around the 32 of a lane group."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import modfem_amd as mf  # noqa: E402

pytestmark = pytest.mark.gpu


def fan(kind, m):
    """m elements around the edge of nodes 0 and 1; ring points below (and
    above) at growing angles"""
    t = np.linspace(0.1, 3.0, m + 1)
    ring = np.stack([np.cos(t), np.sin(t)], 1)
    low = np.c_[ring, np.zeros(m + 1)]
    coor = [np.array([[0, 0, 0], [0, 0, 1.0]]), low]
    en = np.full((m, 6), -1, np.int32)
    k = np.arange(m)
    if kind == "prism":
        coor.append(low + [0, 0, 1.0])
        up = 2 + m + 1 + k
        en[:] = np.stack([0 * k, 2 + k, 3 + k, 0 * k + 1, up, up + 1], 1)
    else:
        en[:, :4] = np.stack([0 * k, 2 + k, 3 + k, 0 * k + 1], 1)
    none = np.zeros(0, np.int32)
    return mf.Mesh.from_arrays(np.concatenate(coor), np.full(
        m, mf.PRISM if kind == "prism" else mf.TETRA, np.int32), en, none, none, none)


@pytest.mark.parametrize("kind,m", [("prism", 1), ("prism", 14), ("prism", 15), ("prism", 32),
                                    ("prism", 33), ("prism", 126), ("tetra", 28), ("tetra", 31),
                                    ("tetra", 97), ("tetra", 253)])
def test_tables_of_long_rows(kind, m):
    print("fan", kind, m, flush=True)
    mesh = fan(kind, m)
    h, d = mf.Problem.from_mesh(mesh), mf.Problem.from_mesh(mesh, device_setup=True)
    assert np.diff(h.pattern()[0]).max() == (2 * m + 4 if kind == "prism" else m + 3)
    for a, b in zip(h.pattern(), d.pattern()):
        assert np.array_equal(a, b)
    for e in range(m):
        assert np.array_equal(h.table(e), d.table(e))
    h.free()
    d.free()
    mesh.free()
