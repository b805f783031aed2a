"""The one-kernel stage of the inviscid second-order runs (kern_stage.h)
against the split kernels, bit for bit, where its lists and dispatch can go
wrong: one short tile, tiles with a remainder, both workgroup sizes, quads
and triangles, every flux, stage count (buffer parity), time-step mode,
limiter and precision; and against the oracle."""
import numpy as np
import pytest

from csu_amd import cases, native

pytestmark = pytest.mark.gpu

# name: (nx, ny, split, input overrides)
FORMS = {
    "one_short_tile": (5, 4, True, {}),
    "remainder": (41, 13, True, {}),
    "quads_ausm_1": (37, 19, False, {"flux": "AUSM", "stages": 1}),
    "quads_ausmdv_barth": (40, 20, False, {"flux": "AUSMDV", "limiter": 2, "stages": 3}),
    "pup_4": (33, 16, True, {"flux": "AUSMpup", "stages": 4}),
    "pup2_global_dt": (33, 16, True, {"flux": "AUSMpup2", "dtLocal": 0}),
    "dt_switch": (30, 15, True, {"dtLocalN": 3}),
    "wide_tiles": (700, 100, True, {}),          # above the 512-thread form's size
}


@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_stage_tile_equals_split(tmpcase, form, precision):
    nx, ny, split, inp = FORMS[form]
    d = tmpcase("st")
    m = cases.ramp_mesh(nx=nx, ny=ny, seed=3, split=split)
    if form == "wide_tiles":
        from csu_amd import renumber
        c4 = np.array([list(c) + [-1] * (4 - len(c)) for c in m.cells])
        m.cells = [m.cells[k] for k in renumber.morton_order(m.nodes, c4)]
    cases.write_case(d, m, cases.ramp_input(threads=1, nmax=1, precision=precision, **inp))
    c = native.HostCase(d)
    rng = np.random.default_rng(5)
    U0 = c.initial_state() * (1 + 0.02 * rng.standard_normal((c.nvar, c.ncell)))
    got = []
    for tile in (0, 1):
        dev = native.Device(c)
        dev.set_launch_shape(64, 64, 1, tile)
        dev.set_state(U0)
        parts = [dev.iterate(n) for n in (1, 5, 4)]      # eager, graphs in both parities
        got.append((np.concatenate([p[0] for p in parts]), np.concatenate([p[1] for p in parts]), dev.get_state(),
                    dev.residual()["R"]))
        dev.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    assert np.isfinite(got[1][2]).all()
    if precision != 1 and c.ncell < 5000:
        from oracle import pyoracle as po
        o = po.Oracle(c)
        o.set_state(U0)
        res, _ = o.iterate(10)
        assert np.max(np.abs(got[1][0] / res - 1)) < 1e-10      # the suite's history bar


def test_stage_tile_clamps_and_holds(tmpcase):
    """A start state outside the physical range (density and temperature
    clamps) and a held solve of a batch: as the split kernels."""
    d = tmpcase("cl")
    cases.ramp_case(d, nx=24, ny=13, threads=1, nmax=1)
    c = native.HostCase(d)
    U0 = c.initial_state()
    U0[3, ::17] *= 0.2          # internal energy below zero: T clamped
    U0[0, ::29] = 1e-9          # density below rLim
    out = []
    for tile in (0, 1):
        b = native.Batch([c, c])
        b.set_launch_shape(64, 64, 1, tile)
        for q in range(2):
            b.set_state(q, U0 if q else c.initial_state())
        b.set_active(1, False)
        r1, _ = b.iterate(3)
        held = b.get_state(1)
        b.set_active(1, True)
        r2, _ = b.iterate(1)
        out.append((r1[:, 0], r2, held, b.get_state(0), b.get_state(1)))
        b.close()
    assert np.array_equal(out[1][2], U0)
    for x, y in zip(*out):
        assert np.array_equal(x, y, equal_nan=True)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("form", ["one_short_tile", "remainder", "quads_ausm_1", "wide_tiles", "tube"])
def test_first_order_tile_equals_split(tmpcase, monkeypatch, form, precision):
    """First-order runs (edge states = cell states) in one kernel per stage:
    the split kernels' results bit for bit, a time-accurate run past its
    last step included."""
    d = tmpcase("o1")
    if form == "tube":
        m = cases.tube_mesh(nx=90, ny=7, seed=0)
        cases.write_case(d, m, cases.tube_input(threads=1, tmax=0.004, precision=precision))
    else:
        nx, ny, split, inp = FORMS[form]
        m = cases.ramp_mesh(nx=nx, ny=ny, seed=3, split=split)
        cases.write_case(d, m, cases.ramp_input(threads=1, nmax=1, order=1, precision=precision, **inp))
    c = native.HostCase(d)
    U0 = c.initial_state() * (1 + 0.02 * np.random.default_rng(5).standard_normal((c.nvar, c.ncell)))
    got = []
    for stored in ("1", "0"):
        monkeypatch.setenv("CSU_STORED_PRIMITIVES", stored)
        dev = native.Device(c)
        dev.set_state(U0)
        if form == "tube":
            dev.advance_time(c.tmax)
        parts = [dev.iterate(n) for n in (1, 5, 4)]
        dev.set_profiling(True)
        dev.iterate(1)
        assert ("k_stage" in dev.kernel_times()) == (stored == "0")
        got.append((np.concatenate([p[0] for p in parts]), np.concatenate([p[1] for p in parts]), dev.get_state(),
                    dev.residual()["R"]))
        dev.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b, equal_nan=True)  # the tube's forces: 0/0, its free stream is at rest
    assert np.isfinite(got[1][2]).all()
