"""The wall-distance kernel's groups of segments against the host restatement
of saCalcD, bit for bit, where the skipping can go wrong: fewer segments than
a group, a remainder group, cells equally far from two groups (a vertex they
share), far cells, walls in two places, no wall, a degenerate segment."""
import numpy as np
import pytest

from csu_amd import cases, native

pytestmark = pytest.mark.gpu


def _plate(nx, ny):
    return cases.plate_mesh(nx=nx, ny=ny, seed=2), cases.plate_input(threads=1, nmax=1, laminar=0, sa=1)


def _channel(nx, ny):
    i = cases.ramp_input(threads=1, nmax=1, sa=1, flux="AUSM")
    i["BC:top"] = "wall"
    return cases.ramp_mesh(nx=nx, ny=ny, seed=4), i


def _no_wall(nx, ny):
    i = cases.ramp_input(threads=1, nmax=1, sa=1, flux="AUSM")
    i["BC:ramp"] = "symmetry"
    return cases.ramp_mesh(nx=nx, ny=ny, seed=4), i


def _degenerate(nx, ny):
    m, i = _channel(nx, ny)
    m.nodes[[k for _, e in m.markers[2:3] for k in e[3]][1]] = m.nodes[m.markers[2][1][3][0]]
    return m, i


@pytest.mark.parametrize("mk", [lambda: _plate(7, 5), lambda: _plate(61, 12), lambda: _channel(100, 30),
                                lambda: _no_wall(9, 5), lambda: _degenerate(40, 8),
                                lambda: (cases.naca_mesh(ni=130, nwall=9, nfar=12, seed=1),
                                         cases.naca_input(threads=1, nmax=1))],
                         ids=["one_group", "remainder", "two_walls", "none", "degenerate", "airfoil"])
def test_wall_distance_equals_host(tmpcase, mk):
    d = tmpcase("wd")
    cases.write_case(d, *mk())
    c = native.HostCase(d)
    host = c.arrays()["wall_dist"]
    assert np.array_equal(native.wall_distance_dev(c), host)
