"""Wall distance on the device for descriptors at the edges of what the call
takes: no node count (the nodes are those that the cells name)."""
import ctypes as C

import numpy as np
import pytest

from csu_amd import cases, native

pytestmark = pytest.mark.gpu


def _dist(mesh):
    out = np.empty(mesh.ncell)
    native.check(native.lib().csu_wall_distance_dev(C.byref(mesh), out.ctypes.data_as(C.POINTER(C.c_double))))
    return out


@pytest.mark.parametrize("nnode", [0, -1])
def test_wall_distance_without_a_node_count(tmpcase, nnode):
    d = tmpcase("wn")
    cases.write_case(d, cases.plate_mesh(nx=31, ny=9, seed=2), cases.plate_input(threads=1, nmax=1, laminar=0, sa=1))
    c = native.HostCase(d)
    m = native.MeshDesc.from_buffer_copy(c.mesh)
    m.nnode = nnode
    assert np.array_equal(_dist(m), c.arrays()["wall_dist"])


@pytest.mark.parametrize("length", [1e-160, 1e-156, 1e-150, 1e-3])
def test_wall_of_one_short_edge(length):
    """A wall of one edge, of lengths whose square is subnormal, and not."""
    xy = np.array([[0.0, 0.0], [length, 0.0], [0.3, 0.4], [-0.2, 0.7]])
    cells = np.array([[0, 1, 2, -1], [0, 2, 3, -1]], np.int32)
    bface, mark, kind = np.array([[0, 0, 1]], np.int32), np.zeros(1, np.int32), np.array([3], np.int32)
    p = lambda a, t: a.ctypes.data_as(C.POINTER(t))   # noqa: E731
    m = native.MeshDesc(ncell=2, nnode=4, nface=0, nbface=1, nmark=1, node_xy=p(xy, C.c_double),
                        cell_vert=p(cells, C.c_int32), bface=p(bface, C.c_int32), bface_mark=p(mark, C.c_int32),
                        mark_type=p(kind, C.c_int32))
    want = []
    for c in cells:
        x, y = (((xy[c[0], k] + xy[c[1], k]) + xy[c[2], k]) / 3 for k in (0, 1))
        t = min(max(length * x / (length * length), 0.0), 1.0)
        want.append(np.sqrt((length * t - x) ** 2 + (0.0 - y) ** 2))
    assert np.array_equal(_dist(m), want)
