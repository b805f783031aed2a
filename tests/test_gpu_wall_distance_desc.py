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
