"""csu_dev_residual: any of its outputs may be asked for alone; each comes as
it does beside the others, on both sides of the sizes up to which several come
in one copy."""
import ctypes as C

import numpy as np
import pytest

from csu_amd import cases, native

pytestmark = pytest.mark.gpu

NAMES = ("R", "dPx", "dPy", "phi", "P", "Pb")


def _call(dev, names):
    nv, nc, nb = dev.nvar, dev.ncell, dev.nbface
    shape = dict.fromkeys(NAMES, (nv, nc)) | {"P": (nc, nv + 1), "Pb": (nb, nv + 1)}
    out = {k: np.full(shape[k], np.nan) for k in names}
    native.check(native.lib().csu_dev_residual(
        dev._h, *[out[k].ctypes.data_as(C.POINTER(C.c_double)) if k in out else None for k in NAMES]))
    return out


@pytest.mark.parametrize("kind", ["ramp_small", "ramp", "ramp_large", "laminar", "sa"])
def test_residual_outputs_alone_and_together(tmpcase, kind):
    d = tmpcase("ro")
    if kind.startswith("ramp"):
        nx, ny = {"ramp_small": (9, 7), "ramp": (90, 50), "ramp_large": (150, 80)}[kind]
        cases.ramp_case(d, nx=nx, ny=ny, threads=1, nmax=1)
    else:
        cases.write_case(d, cases.plate_mesh(nx=80, ny=30, seed=2),
                         cases.plate_input(threads=1, nmax=1, **({} if kind == "laminar" else {"laminar": 0, "sa": 1})))
    c = native.HostCase(d)
    dev = native.Device(c)
    U = c.initial_state() * (1 + 0.01 * np.random.default_rng(1).standard_normal((c.nvar, c.ncell)))
    subsets = [[k for b, k in enumerate(NAMES) if (s >> b) & 1] for s in range(1 << len(NAMES))]
    dev.set_state(U)
    ref = _call(dev, NAMES)
    assert all(np.isfinite(v).all() for v in ref.values())
    for names in subsets:
        dev.set_state(U)
        out = _call(dev, names)
        for k in names:
            assert np.array_equal(out[k], ref[k]), (names, k)
    dev.close()
