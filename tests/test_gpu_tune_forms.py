"""What the autotuner remembers for a bucket, where runs of one kind and size
differ in the forms they have: contexts without a tile form, with it as their
default, and with halos that make it none, keep apart."""
import numpy as np
import pytest

from csu_amd import cases, native

pytestmark = pytest.mark.gpu


def _case(tmpcase, scattered=False, **inp):
    d = tmpcase("tf")
    m = cases.ramp_mesh(nx=101, ny=49, seed=3)
    if scattered:
        m.cells = [m.cells[k] for k in np.random.default_rng(2).permutation(len(m.cells))]
    cases.write_case(d, m, cases.ramp_input(threads=1, nmax=1, **inp))
    return native.HostCase(d)


def _shape(c):
    dev = native.Device(c)
    sh = dev.launch_shape()
    dev.close()
    return sh


def test_choices_keep_to_their_form(tmpcase):
    plain, lim1 = _case(tmpcase), _case(tmpcase, limiter=1)
    axi, scattered = _case(tmpcase, axisymmetric=1), _case(tmpcase, scattered=True)
    default = {id(c): _shape(c) for c in (plain, lim1, axi, scattered)}
    assert not any(s["tuned"] for s in default.values())
    assert [default[id(c)]["tile"] for c in (plain, lim1, axi, scattered)] == [1, 0, 0, 0]
    # no tile form: its choice is not taken by a run that has one
    dev = native.Device(lim1)
    dev.autotune(2)
    dev.close()
    assert _shape(lim1)["tuned"] and _shape(axi)["tuned"]
    assert _shape(plain) == default[id(plain)] and _shape(scattered) == default[id(scattered)]
    # the tile form as the default: not taken by a scattered numbering
    dev = native.Device(plain)
    ch = dev.autotune(2)
    dev.close()
    assert _shape(plain)["tuned"] and _shape(scattered) == default[id(scattered)]
    if ch["tile"]:   # the split kernels' workgroups were not among its candidates
        assert ch["block"] == default[id(plain)]["block"]
    dev = native.Device(scattered)
    dev.autotune(2)
    dev.close()
    assert _shape(scattered)["tuned"] and _shape(plain)["tile"] == ch["tile"]
