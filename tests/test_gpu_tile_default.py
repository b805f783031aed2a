"""The form an untuned inviscid second-order RK context starts in, by
precision and numbering, and through changes of precision: the results of the
same changes with the form set by hand, bit for bit."""
import numpy as np
import pytest

from csu_amd import cases, native, renumber

pytestmark = pytest.mark.gpu


def _case(tmpcase, nx, ny, order, **inp):
    d = tmpcase("td")
    m = cases.ramp_mesh(nx=nx, ny=ny, seed=3)
    if order == "morton":
        m.cells = [m.cells[k] for k in renumber.morton_order(m.nodes, np.array([c + (-1,) for c in m.cells]))]
    elif order == "scattered":
        m.cells = [m.cells[k] for k in np.random.default_rng(2).permutation(len(m.cells))]
    cases.write_case(d, m, cases.ramp_input(threads=1, nmax=1, **inp))
    return native.HostCase(d)


# halo cells per cell 1.0 (columns longer than a tile), 0.27, 0.24 and 2.7: the
# form in FP64, mixed precision, long double sums; mixed precision with tiles
# that run all at once (117; 528: Roe on triangles only) and not (801)
@pytest.mark.parametrize("nx,ny,order,flux,forms", [
    (410, 250, "column", "ROE", (1, 0, 0)), (270, 250, "column", "ROE", (1, 1, 0)),
    (270, 250, "column", "AUSMDV", (1, 0, 0)), (270, 250, "morton", "AUSMDV", (1, 1, 1)),
    (100, 150, "column", "AUSMDV", (1, 1, 0)), (50, 50, "morton", "ROE", (1, 1, 1)),
    (50, 50, "scattered", "ROE", (0, 0, 0))])
def test_default_form(tmpcase, nx, ny, order, flux, forms):
    for precision, tile in enumerate(forms):
        dev = native.Device(_case(tmpcase, nx, ny, order, flux=flux, precision=precision))
        sh = dev.launch_shape()
        dev.close()
        assert sh["tuned"] or sh["tile"] == tile, precision


def test_form_follows_the_precision(tmpcase):
    c = _case(tmpcase, 270, 250, "column", flux="AUSMDV")
    U0 = c.initial_state() * (1 + 0.02 * np.random.default_rng(5).standard_normal((c.nvar, c.ncell)))
    out = []
    for tile in (None, 0, 1):
        dev = native.Device(c)
        if tile is not None:
            dev.set_launch_shape(64, 64, 1, tile)
        dev.set_state(U0)
        rows, forms = [], []
        for precision in (0, 1, 2, 0):
            dev.set_precision(precision)
            forms.append(dev.launch_shape()["tile"])
            rows += [x for n in (1, 3) for x in dev.iterate(n)]
        assert forms == ([1, 0, 0, 1] if tile is None else [tile] * 4)
        out.append(rows + [dev.get_state()])
        dev.close()
    for a, b, e in zip(*out):
        assert np.array_equal(a, b) and np.array_equal(a, e)
