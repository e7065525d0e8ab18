"""The triangular sweeps by strips against the oracle and the row-by-row sweep.

One M^-1 r with a random right-hand side on grids whose sides sit at the edges
of a strip (eight rows per sub-level): one strip, one row more, ragged last
strips, long and short columns, several components, and a mesh with shuffled
vertex numbers (its strips import most of their rows, or the mesh does not fit
strips at all).  Each operation is one IEEE rounding in the reference's order,
so the comparison is exact."""
import numpy as np
import pytest

from cloth_sim_self_collision_amd import scene

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sim_mod():
    from cloth_sim_self_collision_amd import _lib, sim
    if _lib.device_count() < 1:
        pytest.skip("no HIP device")
    return sim


def _grid(nx, ny):
    return scene.drop_on_obstacle(nx, 0.4, scene.sphere((0.0, 0.0, 0.0), 0.3), ny=ny, seed=nx + ny)


def _shuffled(n):
    """A square grid with its vertices renumbered at random."""
    cl = _grid(n, n)
    perm = np.random.default_rng(n).permutation(cl.np_).astype(np.int32)
    inv = np.empty_like(perm)
    inv[perm] = np.arange(cl.np_, dtype=np.int32)
    cl.xyz0 = cl.xyz0.reshape(-1, 3)[perm].reshape(-1).copy()
    cl.xyz = cl.xyz.reshape(-1, 3)[perm].reshape(-1).copy()
    cl.tri = inv[cl.tri]
    cl.quad = scene.bending_quads(cl.tri)
    return cl


def _tube(m, n, copies=1, closed=False):
    """Tubes of m vertices around and n along (closed: tori), side by side.
    Four around: rows with 35 factor updates; 3 x 3 tori, where every vertex
    couples to all others: 36.  A lane of the factorisation keeps updates 1 to
    32 of a row in registers."""
    cl = _grid(m, n * copies)
    a, c = np.meshgrid(np.arange(m), np.arange(n if closed else n - 1))
    p, q = c * m + a, c * m + (a + 1) % m
    r, s = (c + 1) % n * m + a, (c + 1) % n * m + (a + 1) % m
    tri = np.stack([p, q, s, p, s, r], -1).reshape(-1)
    cl.tri = np.concatenate([tri + k * m * n for k in range(copies)]).astype(np.int32)
    v = np.arange(m * n * copies)
    t, u, k = 2 * np.pi * (v % m) / m, v // m % n, v // (m * n)
    u = 2 * np.pi * u / n if closed else 0.02 * u
    xyz = [0.05 * np.cos(t) + (0.1 * np.cos(u) if closed else u) + 0.4 * k,
           0.05 * np.sin(t) + 0.3, 0.1 * np.sin(u) if closed else 0.05 * np.cos(t)]
    cl.xyz = np.stack(xyz, -1).reshape(-1)
    cl.xyz0 = cl.xyz.copy()
    cl.quad = scene.bending_quads(cl.tri)
    return cl


MESHES = {
    "2x3": lambda: _grid(2, 3), "8x8": lambda: _grid(8, 8), "9x9": lambda: _grid(9, 9),
    "16x40": lambda: _grid(16, 40), "17x33": lambda: _grid(17, 33), "33x17": lambda: _grid(33, 17),
    "3x90": lambda: _grid(3, 90), "90x3": lambda: _grid(90, 3), "65x64": lambda: _grid(65, 64),
    "stack3x18": lambda: scene.stacked_sheets(3, 18), "shuffled20": lambda: _shuffled(20),
    "tube4x60": lambda: _tube(4, 60), "tori3x3": lambda: _tube(3, 3, 60, True),
}


@pytest.mark.parametrize("name", sorted(MESHES))
def test_solve_by_strips_bitwise(sim_mod, oracle_mod, name):
    cl = MESHES[name]()
    o = oracle_mod.Oracle(cl, "port")
    rng = np.random.default_rng(len(name))
    with sim_mod.DeviceCloth(cl) as d:
        dia, crs, b = d.assemble(cl.xyz, cl.uvw)
        d.ilu_factor()
        fd, fc = d.get_factor()
        for k in range(3):  # a repeated launch finds the state the one before left
            v = rng.standard_normal(3 * cl.np_)
            d.set_option(1, 0)
            strips = d.ilu_solve(v)
            d.set_option(1, 1)
            rows = d.ilu_solve(v)
            assert np.array_equal(strips, rows)
            assert np.array_equal(strips, o.ilu_solve(fd, fc, v))
        d.set_option(1, 0)
        # non-finite right-hand sides are results, not values still awaited
        v[3] = np.inf
        v[0] = np.nan
        strips = d.ilu_solve(v)
        d.set_option(1, 1)
        assert np.array_equal(strips, d.ilu_solve(v), equal_nan=True)


def test_solves_of_each_layout_alternate(sim_mod):
    """The packed copies of one factor follow the solve that needs them."""
    cl = _grid(20, 24)
    with sim_mod.DeviceCloth(cl) as d:
        _, _, b = d.assemble(cl.xyz, cl.uvw)
        d.ilu_factor()
        want = d.pcg_solve(b, 1e-6, 60)
        for pcg, sweep in ((2, 0), (0, 0), (0, 1), (2, 0), (0, 0)):
            d.set_option(1, sweep)
            d.set_option(2, pcg)
            got = d.pcg_solve(b, 1e-6, 60)
            assert all(np.array_equal(g, w) for g, w in zip(got, want))
        # a new factor invalidates both copies
        fd, fc = d.get_factor()
        d.set_factor(2.0 * fd, fc)
        d.set_option(1, 0)
        strips = d.ilu_solve(b)
        d.set_option(1, 1)
        assert np.isfinite(strips).all() and np.array_equal(strips, d.ilu_solve(b))


@pytest.mark.parametrize("name", sorted(MESHES))
def test_factor_by_strips_bitwise(sim_mod, oracle_mod, name):
    """The factorisation on the same meshes, on the assembled system and on a
    random one (other update patterns of magnitude), twice each."""
    cl = MESHES[name]()
    o = oracle_mod.Oracle(cl, "port")
    rng = np.random.default_rng(3)
    with sim_mod.DeviceCloth(cl) as d:
        dia, crs, b = d.assemble(cl.xyz, cl.uvw)
        rdia = rng.standard_normal(dia.shape) + np.tile(9.0 * np.eye(3).reshape(-1), cl.np_)
        rcrs = rng.standard_normal(crs.shape)
        for A, B in ((dia, crs), (rdia, rcrs), (dia, crs)):
            d.set_system(A, B, b)
            assert d.ilu_factor() == 0
            fd, fc = d.get_factor()
            wd, wc = o.ilu(A, B)
            assert np.array_equal(fd, wd) and np.array_equal(fc, wc)


def _states(devs):
    return [a for d in devs for a in d.get_state()]


def test_batch_steps_after_given_up_waits(sim_mod, monkeypatch):
    """A step whose waits are given up is an error; every member's strips are
    reset, so that the next step gives what it gives on new cloths."""
    from cloth_sim_self_collision_amd import _lib
    cls = [_grid(24, 24), _grid(33, 40), _grid(40, 24)]
    for c in cls:
        c.pcg_maxit = 40
    runs = []
    for fail in (False, True):
        devs = [sim_mod.DeviceCloth(c) for c in cls]
        try:
            with sim_mod.DeviceBatch(devs) as b:
                if fail:
                    monkeypatch.setenv("CLOTHSIM_STRIP_POLLS", "0")
                    with pytest.raises(_lib.ClothSimError, match="gave up waiting"):
                        b.step(1)
                    monkeypatch.delenv("CLOTHSIM_STRIP_POLLS")
                    for d, c in zip(devs, cls):
                        d.set_state(c.xyz, c.uvw)
                        d.time = 0.0
                b.step(2)
                runs.append(_states(devs))
        finally:
            for d in devs:
                d.close()
    assert all(np.array_equal(g, w) for g, w in zip(*runs))


def test_solve_ends_after_given_up_waits(sim_mod, monkeypatch):
    """The iterations stop at the first convergence poll (every eight) after a
    wait was given up, not at the cap."""
    from cloth_sim_self_collision_amd import _lib
    cl = _grid(33, 40)
    monkeypatch.setenv("CLOTHSIM_STRIP_POLLS", "0")
    with sim_mod.DeviceCloth(cl) as d, sim_mod.DeviceBatch([d]) as b:
        for who in (d, b):
            who.profile(True)
            with pytest.raises(_lib.ClothSimError, match="gave up waiting"):
                who.step(1)
            assert who.profile_read()["ilu_sweep"][1] == 9
            who.profile(False)


def test_one_cloth_steps_after_given_up_waits(sim_mod, monkeypatch):
    from cloth_sim_self_collision_amd import _lib
    cl = _grid(33, 40)
    cl.pcg_maxit = 40
    with sim_mod.DeviceCloth(cl) as d:
        d.step(2)
        want = _states([d])
    with sim_mod.DeviceCloth(cl) as d:
        monkeypatch.setenv("CLOTHSIM_STRIP_POLLS", "0")
        for call in (lambda: d.step(1), d.ilu_factor, lambda: d.ilu_solve(cl.xyz)):
            with pytest.raises(_lib.ClothSimError, match="gave up waiting"):
                call()
        monkeypatch.delenv("CLOTHSIM_STRIP_POLLS")
        d.set_state(cl.xyz, cl.uvw)
        d.step(2)
        got = _states([d])
    assert all(np.array_equal(g, w) for g, w in zip(got, want))
