"""csu_dev_footprint on a mesh described by its counts alone (an estimate
before the mesh is read): a number for every form of iteration, no less than
the mesh's own."""
import ctypes as C

import pytest

from csu_amd import cases, native


@pytest.mark.parametrize("over", [{}, {"order": 1}, {"precision": 1}, {"limiter": 1}, {"axisymmetric": 1},
                                  {"timeScheme": "LUSGS"}, {"timeScheme": "DPLUR"}],
                         ids=lambda o: "_".join(f"{k}{v}" for k, v in o.items()) or "rk")
def test_footprint_of_counts(tmpcase, over):
    d = tmpcase("fc")
    cases.ramp_case(d, nx=60, ny=30, threads=1, nmax=1, **over)
    c = native.HostCase(d)
    full = native.lib().csu_dev_footprint(C.byref(c.mesh), C.byref(c.params), 50)
    m = native.MeshDesc()
    for k in ("ncell", "nnode", "nface", "nbface", "nmark", "axi"):
        setattr(m, k, getattr(c.mesh, k))
    est = native.lib().csu_dev_footprint(C.byref(m), C.byref(c.params), 50)
    assert 0 < full <= est <= 1.5 * full
