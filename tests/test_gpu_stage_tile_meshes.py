"""The one-kernel stage on the meshes whose lists differ most from a ramp in
column order, against the split kernels bit for bit: triangles and quads in
one tile, quads in the 256-thread form, scattered numberings (every face of a
tile an outer one: halos of several tiles, more than 64 KB of LDS)."""
import numpy as np
import pytest

from csu_amd import cases, native, renumber

pytestmark = pytest.mark.gpu


def _order(m, perm):
    m.cells = [m.cells[k] for k in perm]
    return m


def _hybrid():
    m = cases.ramp_mesh(nx=43, ny=21, seed=3, split=False)
    half = np.random.default_rng(1).random(len(m.cells)) < 0.5
    m.cells = [t for c, h in zip(m.cells, half)
               for t in ([(c[0], c[1], c[2]), (c[0], c[2], c[3])] if h else [c])]
    return m


def _scattered(nx, ny, split):
    m = cases.ramp_mesh(nx=nx, ny=ny, seed=3, split=split)
    return _order(m, np.random.default_rng(2).permutation(len(m.cells)))


def _quads_256():
    m = cases.ramp_mesh(nx=400, ny=340, seed=3, split=False)     # above the 512-thread form's size
    return _order(m, renumber.morton_order(m.nodes, np.array(m.cells)))


MESHES = {"hybrid": _hybrid, "quads_256": _quads_256, "scattered_quads": lambda: _scattered(60, 50, False),
          "scattered_triangles": lambda: _scattered(40, 33, True)}


def _runs(c, set_form):
    rng = np.random.default_rng(5)
    U0 = c.initial_state() * (1 + 0.02 * rng.standard_normal((c.nvar, c.ncell)))
    out = []
    for tile in (0, 1):
        dev = set_form(tile)
        dev.set_state(U0)
        parts = [dev.iterate(n) for n in (1, 4)]
        out.append((np.concatenate([p[0] for p in parts]), np.concatenate([p[1] for p in parts]), dev.get_state()))
        dev.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert np.isfinite(out[0][2]).all()


@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("mesh", sorted(MESHES))
def test_stage_tile_equals_split_on(tmpcase, mesh, precision):
    d = tmpcase("sm")
    cases.write_case(d, MESHES[mesh](), cases.ramp_input(threads=1, nmax=1, precision=precision, flux="AUSMDV"))
    c = native.HostCase(d)

    def form(tile):
        dev = native.Device(c)
        dev.set_launch_shape(64, 64, 1, tile)
        return dev
    _runs(c, form)


def test_batch_of_such_meshes(tmpcase):
    """The lists of a batch (each solve's tiles and ids offset)."""
    cs = []
    for k, mesh in enumerate(("scattered_quads", "hybrid", "scattered_triangles")):
        d = tmpcase("sb")
        cases.write_case(d, MESHES[mesh](), cases.ramp_input(threads=1, nmax=1, mach=str(2.0 + 0.2 * k)))
        cs.append(native.HostCase(d))
    out = []
    for tile in (0, 1):
        b = native.Batch(cs)
        b.set_launch_shape(64, 64, 1, tile)
        r, f = b.iterate(5)
        out.append([r, f] + [b.get_state(q) for q in range(3)])
        b.close()
    for x, y in zip(*out):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("precision", [0, 1])
def test_first_order_holds_no_lists_it_does_not_read(tmpcase, monkeypatch, precision):
    """A first-order run takes the form or not by its halos alone: on a
    scattered numbering it holds what the split form holds, not a byte of
    lists; where it takes the form, two buffers of primitives, its own cells'
    slots, its boundary faces, and its tiles' faces with their cells."""
    held = {}
    for mesh in ("scattered_triangles", "hybrid"):
        d = tmpcase("fo")
        cases.write_case(d, MESHES[mesh](), cases.ramp_input(threads=1, nmax=1, precision=precision, order=1))
        c = native.HostCase(d)
        for stored in ("1", "0"):
            monkeypatch.setenv("CSU_STORED_PRIMITIVES", stored)
            dev = native.Device(c)
            held[mesh, stored] = dev.bytes()
            dev.close()
    assert held["scattered_triangles", "0"] == held["scattered_triangles", "1"]
    nt = (c.ncell + 255) // 256
    e = c.arrays()["face"][:, :2] // 256
    entries = c.nface + int((e[:, 0] != e[:, 1]).sum())
    lists = 4 * (3 * (nt + 1) + nt + 3 * c.nbface) + entries * (24 + 8 + 12 * precision) + 8 * c.ncell
    assert held["hybrid", "0"] - held["hybrid", "1"] == lists + 64 * c.ncell


@pytest.mark.parametrize("precision", [0, 1])
def test_second_order_shares_the_edge_states_room(tmpcase, monkeypatch, precision):
    """The tile form's primitives lie where the split kernels keep edge
    states: a context holds its lists more than one without the form, and
    residual evaluations and precision changes between iterations (which
    write edge states, or allocate others) leave the results the split
    form's."""
    d = tmpcase("sh")
    cases.write_case(d, _hybrid(), cases.ramp_input(threads=1, nmax=1, precision=precision, stages=3))
    c = native.HostCase(d)
    out, held = [], []
    for stored in ("1", "0"):
        monkeypatch.setenv("CSU_STORED_PRIMITIVES", stored)
        dev = native.Device(c)
        held.append(dev.bytes())
        if stored == "0":
            dev.set_launch_shape(64, 64, 1, 1)
        rows = []
        for prec in (precision, 1 - precision, 2, precision):
            dev.set_precision(prec)
            rows += [dev.iterate(1)[0], *dev.residual().values(), dev.iterate(5)[0], dev.iterate(2)[0],
                     dev.primitives(), dev.iterate(4)[0], dev.get_state()]
        out.append(rows)
        dev.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    nt = (c.ncell + 255) // 256
    e = c.arrays()["face"][:, :2]
    t = e // 256
    cross = t[:, 0] != t[:, 1]
    halo = len(set(map(tuple, np.r_[np.c_[t[cross, 0], e[cross, 1]], np.c_[t[cross, 1], e[cross, 0]]])))
    lists = 4 * (3 * (nt + 1) + nt + halo) + (24 + 12 * precision) * (c.nface + cross.sum()) + 16 * (c.ncell + halo)
    entries = held[1] - held[0] - lists        # boundary faces, of own and halo cells: three numbers each
    assert entries % 12 == 0 and 12 * c.nbface <= entries <= 4 * 12 * c.nbface
