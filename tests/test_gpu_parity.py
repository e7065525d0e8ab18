"""GPU parity: every stage of the HIP step against the CPU oracle, bit for bit.

The oracle (oracle/cloth_oracle.c) is itself pinned to the compiled
reference (tests/test_oracle.py), so equality here is equality with the
reference on the same inputs.  Float arrays are compared with
np.array_equal (exact; +0.0 and -0.0 compare equal), contact sets as int
arrays.
"""
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


def _scenes():
    return {
        "drape16": scene.drape_over_sphere(16),
        "drape32": scene.drape_over_sphere(32),
        "refdemo0": scene.reference_demo(0),
        "refdemo1": scene.reference_demo(1),
        "fold24": scene.fold_sweep(24, size=0.3),
        "box24": scene.drop_on_obstacle(24, 0.3, scene.box((0.0, 0.0, 0.0), (0.25, 0.25, 0.25)),
                                        seed=5),
        "bar24": scene.drop_on_obstacle(
            24, 0.2, scene.bar_over_ground((-0.6, 0.05, 0.0), (0.6, -0.05, 0.0), 0.05, -0.25),
            seed=6),
        "stack16": scene.stacked_sheets(2, 16, size=0.5, dt=0.005, seed=3),
    }


def _trajectory(oracle_mod, cl, steps, keep):
    """Oracle states (x, v, x_start) before each step index in `keep`."""
    o = oracle_mod.Oracle(cl, "port")
    x, v, t = cl.xyz.copy(), cl.uvw.copy(), 0.0
    out = {}
    for k in range(steps):
        scene.apply_sweep(cl, x, t + cl.dt)
        if k in keep:
            out[k] = (x.copy(), v.copy())
        x, v, *_ = o.step(x, v)
        t += cl.dt
    return o, out


def test_device_division_and_sqrt_are_correctly_rounded(sim_mod):
    rng = np.random.default_rng(1)
    n = 1 << 16
    a = rng.standard_normal(n) * np.exp2(rng.integers(-60, 60, n))
    b = rng.standard_normal(n) * np.exp2(rng.integers(-60, 60, n))
    a = np.concatenate([a, [1.0, 2.0, 3.0, 1e-310, 5e-324, 1e308, 0.0, 0.25]])
    b = np.concatenate([b, [3.0, 7.0, 1e-300, 3.0, 1.0, 1e-10, 1.0, 3.0]])
    q, s = sim_mod.selftest_divsqrt(a, b)
    assert np.array_equal(q, a / b)
    pos = a >= 0
    assert np.array_equal(s[pos], np.sqrt(a[pos]))


def _sequential(t):
    s = 0.0
    for x in t:
        s += x
    return s


def test_ordered_sum_is_the_sequential_sum(sim_mod):
    """The device reduction used by the PCG equals the left-to-right loop
    bit for bit on adversarial inputs: magnitudes over 2^+-60, exact halves
    (rounding ties), runs of zeros, subnormals, cancellation, infinities."""
    rng = np.random.default_rng(11)
    cases = []
    for n in (1, 17, 1000, 16384, 16385, 70000, 196608):
        cases.append(rng.standard_normal(n))
        cases.append(rng.standard_normal(n) ** 2 * np.exp2(rng.integers(-30, 30, n)))
        cases.append(np.round(rng.standard_normal(n) * 8) / 4)
        cases.append(np.concatenate([np.zeros(n // 2), rng.standard_normal(n - n // 2)]))
        t = rng.standard_normal(n)
        t[::7] *= -1e10
        cases.append(t)
        cases.append(np.exp2(rng.integers(-60, 60, n)).astype(float) * rng.choice([-1, 1], n))
        # mixed signs decaying over 600 binades: dense binade changes early,
        # then addends far below the running sum's ulp
        cases.append(rng.standard_normal(n) * np.exp2(np.linspace(300, -300, n)))
    # more than 1024 tiles (two windows of tile summaries)
    cases.append(rng.standard_normal(1_100_000))
    # a running sum crossing binades at every addend (alternating signs)
    n = 20000
    cases.append((1.0 + 1e-3 * rng.standard_normal(n)) * np.where(np.arange(n) % 2, -1.0, 1.0))
    # products of correlated vectors, as in the PCG reductions
    a = rng.standard_normal(70000) * np.exp2(rng.integers(-20, 20, 70000))
    cases.append(a * (a + 0.5 * rng.standard_normal(70000)))
    cases.append(rng.standard_normal(3000) * np.exp2(rng.integers(-1074, -1000, 3000)))
    t = rng.standard_normal(5000)
    t[100] = np.inf
    cases.append(t)
    t = t.copy()
    t[4000] = -np.inf
    cases.append(t)
    t = rng.standard_normal(9000)
    t[3000] = np.nan
    cases.append(t)
    cases.append(np.zeros(0))
    for t in cases:
        got = sim_mod.ordered_sum(t)
        want = _sequential(t)
        assert got == want or (np.isnan(got) and np.isnan(want)), (len(t), got, want)


def test_element_routines_bitwise(sim_mod, oracle_mod):
    rng = np.random.default_rng(2)
    n = 512
    C = rng.standard_normal((n, 9))
    c = C + 0.1 * rng.standard_normal((n, 9))
    dW, ddW = sim_mod.element_cst(C, c, 576.9, 384.6)
    for e in range(0, n, 37):
        _, g, h = oracle_mod.element_cst(C[e], c[e], 576.9, 384.6)
        assert np.array_equal(dW[e], g) and np.array_equal(ddW[e], h)
    Cq = rng.standard_normal((n, 12))
    cq = Cq + 0.1 * rng.standard_normal((n, 12))
    dWb, ddWb = sim_mod.element_bend(Cq, cq, 1e-3)
    for e in range(0, n, 37):
        g, h = oracle_mod.element_bend(Cq[e], cq[e], 1e-3)
        assert np.array_equal(dWb[e], g) and np.array_equal(ddWb[e], h)
    p = rng.standard_normal((n, 3)) * 0.4
    for ob in (scene.sphere((0.0, 0.0, 0.0), 0.3), scene.plane((0.0, 0.0, 1.0), -0.1),
               scene.Obstacle(scene.OBST_SPHERE_INV, (0.1, 0.0, 0.0, 0.35)),
               scene.box((0.05, 0.0, -0.1), (0.2, 0.25, 0.15)),
               scene.bar((-0.3, 0.1, 0.0), (0.4, -0.1, 0.05), 0.2),
               scene.bar_over_ground((-0.3, 0.1, 0.0), (0.4, -0.1, 0.05), 0.15, -0.2)):
        g, h = sim_mod.element_contact(p, 1e3, 0.01, ob)
        for e in range(0, n, 17):
            _, g0, h0 = oracle_mod.element_contact(p[e], 1e3, 0.01, ob.as_array())
            assert np.array_equal(g[e], g0) and np.array_equal(h[e], h0)
    # energies: W of WdWddW_CST, and WdWddW_Contact from callback values (a
    # sphere's depth and direction computed here as the C callback does)
    W = sim_mod.element_cst_energy(C, c, 576.9, 384.6)
    for e in range(0, n, 37):
        assert W[e] == oracle_mod.element_cst(C[e], c[e], 576.9, 384.6)[0]
    ob = scene.sphere((0.05, -0.02, 0.01), 0.3)
    d = p - np.array(ob.params[:3])
    ln = np.sqrt(d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2])
    nrm = d / ln[:, None]
    pd = ob.params[3] - ln
    Wc, gc, hc = sim_mod.element_contact_depth(pd, nrm, 1e3, 0.01)
    assert (pd + 0.01 >= 0).any() and (pd + 0.01 < 0).any()
    for e in range(n):
        w0, g0, h0 = oracle_mod.element_contact(p[e], 1e3, 0.01, ob.as_array())
        assert Wc[e] == w0 and np.array_equal(gc[e], g0) and np.array_equal(hc[e], h0), e


@pytest.mark.parametrize("name", ["drape16", "refdemo0", "fold24"])
def test_setup_products(sim_mod, oracle_mod, name):
    cl = _scenes()[name]
    o = oracle_mod.Oracle(cl, "port")
    with sim_mod.DeviceCloth(cl) as d:
        for a, b in zip(d.pattern(), o.pattern()):
            assert np.array_equal(a, b)
        assert np.array_equal(d.bvh(), o.bvh())


def test_sweep_shape_and_issue_probe(sim_mod):
    """The sweep shape the bench prices its issue floor with: one sub-level per
    level while levels are at most 128 rows, four lanes per row of the widest
    level, and the per-lane loads of the packed layout (metadata groups,
    coefficient pairs, then D^-1 pairs or the right-hand side)."""
    from cloth_sim_self_collision_amd import _lib
    cl = scene.fold_sweep(40, size=0.4)
    info = _lib.inspect_setup(cl)
    k = max(info["max_lower"], info["max_upper"])
    with sim_mod.DeviceCloth(cl) as d:
        sh = d.sweep_shape()
        assert sh["quad"] == 1 and sh["components"] == 1
        assert sh["fwd_sublevels"] == info["levels_forward"]
        assert sh["bwd_sublevels"] == info["levels_backward"]
        assert 1 <= sh["waves"] <= 8
        pairs, groups = (3 * k + 1) // 2, (k + 2 + 7) // 8
        assert (sh["loads_fwd"], sh["loads_bwd"]) == (groups + pairs + 2, groups + pairs + 1)
        # wave-load instructions: level widths from the pattern, then each
        # wave's load sets (three up front, three per group of three levels
        # unless the group and the one before it have no row of the wave's)
        rp, ci = info["rowptr"], info["colind"]
        n = len(rp) - 1
        lf, lb = np.zeros(n, int), np.zeros(n, int)
        for i in range(n):
            lo = ci[rp[i]:rp[i + 1]]
            lo = lo[lo < i]
            lf[i] = lf[lo].max() + 1 if len(lo) else 0
        for i in range(n - 1, -1, -1):
            hi = ci[rp[i]:rp[i + 1]]
            hi = hi[hi > i]
            lb[i] = lb[hi].max() + 1 if len(hi) else 0

        def sets(widths, w):
            q1 = len(widths)
            idle = [not (s < q1 and widths[s] > 16 * w) for s in range(q1 + 3)]
            total, g = 3, 0
            while g < q1:
                if all(idle[g:g + 3]):
                    while g + 3 < q1 and all(idle[g + 3:g + 6]):
                        g += 3
                total += 3
                g += 3
            return total

        wf, wb = np.bincount(lf), np.bincount(lb)
        assert max(wf.max(), wb.max()) <= 128  # one sub-level per level
        want = sum(sets(wf, w) * sh["loads_fwd"] + sets(wb, w) * sh["loads_bwd"]
                   for w in range(sh["waves"]))
        assert sh["wave_loads"] == want
        d.set_option(1, 1)  # the row-by-row sweep: no quad shape
        assert d.sweep_shape()["quad"] == 0
    ns = sim_mod.issue_probe(8, 300)
    assert 0.5 < ns < 100.0


def test_profile_modes(sim_mod):
    """Sweep-only profiling times the ILU sweeps and nothing else; full
    profiling times every class and counts the reductions."""
    cl = scene.fold_sweep(24, size=0.3)
    cl.pcg_maxit = 20
    with sim_mod.DeviceCloth(cl) as d:
        d.set_option(2, 1)  # one launch per PCG operation: each class has its launches
        d.profile(True, sweep_only=True)
        d.step(1)
        p = d.profile_read()
        assert p["ilu_sweep"][1] > 0 and p["ilu_sweep"][0] > 0.0
        assert all(n == 0 for k, (ms, n) in p.items() if k != "ilu_sweep")
        assert d.reduction_stats()["sums"] == 0
        d.profile(True)
        d.step(1)
        p = d.profile_read()
        assert p["ilu_sweep"][1] > 0 and p["pcg_reduce"][1] > 0 and p["spmv"][1] > 0
        assert d.reduction_stats()["sums"] > 0
        d.set_option(2, 2)  # the one-workgroup solve is timed as one class
        d.profile(True)
        d.step(1)
        p = d.profile_read()
        assert p["pcg_workgroup"][1] == 1 and p["ilu_sweep"][1] == 0 and p["pcg_reduce"][1] == 0
        d.profile(False)
        with pytest.raises(Exception):
            from cloth_sim_self_collision_amd import _lib
            sim_mod.check(_lib.load().cs_profile_enable(d.h, 3))


@pytest.mark.parametrize("pcg", [0, 2])
def test_profile_classes_are_the_same_alone_and_in_a_batch(sim_mod, pcg):
    """A step's launches fall into the same classes alone and in a batch (the
    packing of the factor counts as factorisation in both)."""
    cl = scene.fold_sweep(24, size=0.3)
    cl.pcg_maxit = 20
    with sim_mod.DeviceCloth(cl) as d:
        d.set_option(2, pcg)
        d.profile(True)
        d.step(1)
        alone = {k: n for k, (ms, n) in d.profile_read().items()}
        d.profile(False)
        d.set_state(cl.xyz, cl.uvw)
        d.time = 0.0
        with sim_mod.DeviceBatch([d]) as b:
            b.profile(True)
            b.step(1)
            batch = {k: n for k, (ms, n) in b.profile_read().items()}
    assert alone.pop("contact") == 1 and batch.pop("contact") == 0  # run per cloth, not shared
    assert alone == batch and alone["ilu_factor"] == 1


@pytest.mark.parametrize("nsing", [5, 14])
def test_ilu_singular_pivots(sim_mod, oracle_mod, nsing):
    """Exactly singular pivots: rows whose diagonal block and lower blocks are
    zero get no update that could restore them.  Up to 10 of them the
    factorisation goes on; past 10 the reference stops at the 11th singular
    row (ilu_sparse.cpp:507-569), which the re-run kernel reproduces.  The
    factor bit for bit against the oracle, the count of singular pivots as
    constructed."""
    cl = _scenes()["drape16"]
    o = oracle_mod.Oracle(cl, "port")
    with sim_mod.DeviceCloth(cl) as d:
        dia, crs, b = d.assemble(cl.xyz, cl.uvw)
        rp, ci, di = d.pattern()
        rows = np.sort(np.random.default_rng(7).choice(np.arange(10, cl.np_ - 10), nsing,
                                                       replace=False))
        dia, crs = dia.copy(), crs.copy()
        for i in rows:
            dia[9 * i:9 * i + 9] = 0.0
            for k in range(rp[i], di[i]):
                crs[9 * k:9 * k + 9] = 0.0
        d.set_system(dia, crs, b)
        assert d.ilu_factor() == nsing
        fd, fc = d.get_factor()
        ofd, ofc = o.ilu(dia, crs)
        assert np.array_equal(fd, ofd) and np.array_equal(fc, ofc)


def test_ilu_wide_row_factor(sim_mod, oracle_mod):
    """A fan of 40 triangles: the centre's row has 40 blocks, too wide for the
    LDS-staged factorisation, so the row-searching kernel runs; its factor
    bit for bit against the oracle."""
    n = 40
    ang = np.arange(n) * 2.0 * np.pi / n
    xyz = np.concatenate([[0.0, 0.0, 0.0],
                          np.stack([np.cos(ang), np.sin(ang), 0.01 * np.sin(3 * ang)], 1).ravel()])
    tri = np.array([[0, 1 + k, 1 + (k + 1) % n] for k in range(n)]).ravel()
    cl = scene.from_config({"scene": "mesh", "xyz": xyz.tolist(), "tri": tri.tolist(), "dt": 0.01})
    o = oracle_mod.Oracle(cl, "port")
    with sim_mod.DeviceCloth(cl) as d:
        rp, _, _ = d.pattern()
        assert int(np.diff(rp).max()) == n
        x = cl.xyz + 0.01 * np.sin(np.arange(3 * cl.np_))
        dia, crs, b = d.assemble(x, cl.uvw)
        odia, ocrs, ob = o.assemble(x, cl.uvw)
        assert np.array_equal(dia, odia) and np.array_equal(crs, ocrs)
        assert d.ilu_factor() == 0
        fd, fc = d.get_factor()
        ofd, ofc = o.ilu(odia, ocrs)
        assert np.array_equal(fd, ofd) and np.array_equal(fc, ofc)


@pytest.mark.parametrize("name,steps,keep", [
    ("drape32", 70, (0, 25, 50, 69)),
    ("refdemo1", 30, (0, 29)),
    ("fold24", 40, (10, 39)),
])
def test_stages_bitwise(sim_mod, oracle_mod, name, steps, keep):
    cl = _scenes()[name]
    o, states = _trajectory(oracle_mod, cl, steps, keep)
    with sim_mod.DeviceCloth(cl) as d:
        for k, (x, v) in states.items():
            dia, crs, b = d.assemble(x, v)
            odia, ocrs, ob = o.assemble(x, v)
            assert np.array_equal(dia, odia) and np.array_equal(crs, ocrs) and np.array_equal(b, ob), k
            ns = d.ilu_factor()
            fd, fc = d.get_factor()
            ofd, ofc = o.ilu(odia, ocrs)
            assert ns == 0
            assert np.array_equal(fd, ofd) and np.array_equal(fc, ofc), k
            vec = np.sin(np.arange(3 * cl.np_) * 0.37)
            assert np.array_equal(d.ilu_solve(vec), o.ilu_solve(ofd, ofc, vec)), k
            y = np.cos(np.arange(3 * cl.np_) * 0.11)
            assert np.array_equal(d.matvec(1.0, vec, 0.5, y), o.matvec(odia, ocrs, 1.0, vec, 0.5, y)), k
            oxs, ors, oconv, oit = o.pcg(odia, ocrs, ofd, ofc, ob, cl.pcg_tol, cl.pcg_maxit)
            for pcg in (1, 2):  # one launch per operation; the one-workgroup solve
                d.set_option(2, pcg)
                xs, rs, conv, it = d.pcg_solve(b, cl.pcg_tol, cl.pcg_maxit)
                assert it == oit and conv == oconv, (k, pcg)
                assert np.array_equal(xs, oxs) and np.array_equal(rs, ors), (k, pcg)
            d.set_option(2, 0)
            px = d.contacts_proximity(x, cl.clearance)
            assert np.array_equal(px, o.prox_set(x, cl.clearance)), k
            vv = v * 3.0
            cc = d.contacts_ccd(x, vv, cl.dt, cl.clearance)
            assert np.array_equal(cc, o.ccd_set(x, vv, cl.dt, cl.clearance)), k
            bbp = d.bvh_refit_prx(x, cl.clearance)
            assert np.array_equal(bbp, o.refit_prx(x, cl.clearance)), k
            bbc = d.bvh_refit_ccd(x, vv, cl.dt)
            assert np.array_equal(bbc, o.refit_ccd(x, vv, cl.dt)), k


def test_velocity_update_and_host_obstacle_values(sim_mod, oracle_mod):
    cl = _scenes()["drape32"]
    o, states = _trajectory(oracle_mod, cl, 40, (39,))
    x, v = states[39]
    with sim_mod.DeviceCloth(cl) as d:
        assert np.array_equal(d.update_velocity(v, x), o.update_velocity(v, x))
        dia0, crs0, b0 = d.assemble(x, v)
        # penetrationDepth evaluated on the host, as the reference's callback
        pd, n = cl.obstacle.depth(x)
        d.set_obstacle_values(pd, n.ravel())
        with pytest.raises(sim_mod._lib.ClothSimError):
            d.step(1)  # host values describe one state only
        dia1, crs1, b1 = d.assemble(x, v)
        d.set_obstacle_values()
        assert np.array_equal(dia0, dia1) and np.array_equal(crs0, crs1) and np.array_equal(b0, b1)
        assert (pd + cl.clearance > 0).any()  # the obstacle term is active


# (scene, steps, sweep variant, PCG variant): sweep 0 = automatic (these meshes:
# by strips), 1 = row-by-row; PCG 0 = automatic (one launch per PCG operation),
# 2 = the whole solve in one workgroup (packed one-workgroup sweeps)
@pytest.mark.parametrize("name,steps,variant,pcg", [
    ("drape32", 100, 0, 0), ("drape32", 100, 0, 2), ("refdemo0", 60, 0, 0),
    ("refdemo1", 60, 0, 2), ("fold24", 60, 0, 0), ("fold24", 60, 0, 2),
    ("drape32", 60, 1, 0), ("fold24", 40, 1, 0), ("box24", 60, 0, 0), ("bar24", 70, 0, 2),
    ("stack16", 60, 0, 0), ("stack16", 60, 0, 2)])
def test_trajectory_bitwise(sim_mod, oracle_mod, name, steps, variant, pcg):
    cl = _scenes()[name]
    o = oracle_mod.Oracle(cl, "port")
    x, v = cl.xyz.copy(), cl.uvw.copy()
    with sim_mod.DeviceCloth(cl) as d:
        d.set_option(1, variant)
        d.set_option(2, pcg)
        for k in range(steps):
            x_before = x.copy()
            scene.apply_sweep(cl, x, d.time + cl.dt)
            x, v, imp, it, conv = o.step(x, v)
            st = d.step(1)
            gx, gv = d.get_state()
            assert st["pcg_iters"] == it and st["impulse_applied"] == imp, (k, st)
            assert np.array_equal(gx, x) and np.array_equal(gv, v), (
                k, np.abs(gx - x).max(), np.abs(gv - v).max(), st)
            del x_before


@pytest.mark.parametrize("lds", [None, 100])
@pytest.mark.parametrize("n,clearance,gap,closing", [(96, 1.05, 0.9, 0.0), (64, 0.05, 0.5, 0.28)])
def test_wide_impulse_rounds(sim_mod, oracle_mod, monkeypatch, n, clearance, gap, closing, lds):
    """Two sheets with randomly numbered vertices: proximity rounds of up to
    605 contacts (more than the 512 that have a thread of their own and the
    384 whose data is fetched ahead) and continuous ones of up to 281, with
    every round's list in LDS or all but 100 of it in the global lists."""
    from _meshes import renumbered
    h = 1.0 / (n - 1)
    cl = scene.stacked_sheets(2, n, gap=gap * h, z0=1.0, jitter=0.05 * h, clearance=clearance * h)
    cl = renumbered(cl, np.random.default_rng(1).permutation(cl.np_))
    z = cl.xyz.reshape(-1, 3)[:, 2]
    cl.uvw.reshape(-1, 3)[:, 2] = np.where(z > z.mean(), -closing, closing) * h / cl.dt
    v, applied = oracle_mod.Oracle(cl, "port").contact_resolve(cl.xyz, cl.uvw)
    if lds:
        monkeypatch.setenv("CLOTHSIM_DRAIN_LDS", str(lds))
    with sim_mod.DeviceCloth(cl) as d:
        d.set_step_start(cl.xyz)
        got, st = d.intermediate_velocity_contact_resolved()
        assert got == applied
        assert st["n_prox"] == 81999 if n == 96 else st["n_ccd"][0] == 34218
        assert np.array_equal(d.get_state()[1], v)


def test_impulse_rounds_through_the_global_lists(sim_mod, oracle_mod, monkeypatch):
    """The impulse worklist keeps each round's list in LDS up to a capacity
    and the rest of a wider round in global memory; with the capacity cut to
    2 entries (CLOTHSIM_DRAIN_LDS) every round wider than that goes through
    the global lists, and drape32's impulse steps stay bit-identical."""
    monkeypatch.setenv("CLOTHSIM_DRAIN_LDS", "2")
    cl = _scenes()["drape32"]
    o = oracle_mod.Oracle(cl, "port")
    x, v = cl.xyz.copy(), cl.uvw.copy()
    impulses = 0
    with sim_mod.DeviceCloth(cl) as d:
        for k in range(70):
            x, v, imp, it, conv = o.step(x, v)
            st = d.step(1)
            gx, gv = d.get_state()
            impulses += int(imp)
            assert st["pcg_iters"] == it and st["impulse_applied"] == imp, (k, st)
            assert np.array_equal(gx, x) and np.array_equal(gv, v), k
    assert impulses > 0


def test_cpp_shim_step_loop_matches_reference(sim_mod, oracle_mod, tmp_path):
    """The reference's StepTime written against include/clothsim_ref.hpp
    (tests/shim/step_loop.cpp, a separate process) reproduces the oracle's
    trajectory bit for bit, obstacle given as a host penetrationDepth callback."""
    import os
    import subprocess
    exe = os.path.join(os.path.dirname(__file__), "shim", "bin", "step_loop")
    if not os.path.exists(exe):
        pytest.fail("tests/shim/bin/step_loop is not built (make -C tests/shim)")
    cl = _scenes()["drape16"]
    steps = 30
    m = cl.material
    hdr = np.array([cl.np_, cl.nt, cl.nq, steps, cl.pcg_maxit], np.int32)
    prm = np.array([cl.dt, m.lam, m.mu, m.stiff_bend, *m.gravity, cl.mass_point, m.stiff_contact,
                    cl.clearance, cl.pcg_tol, *cl.obstacle.params], np.float64)
    assert cl.obstacle.kind == scene.OBST_SPHERE and len(prm) == 15
    src = tmp_path / "in.bin"
    with open(src, "wb") as f:
        for a in (hdr, prm, cl.xyz0, cl.xyz, cl.uvw):
            f.write(np.ascontiguousarray(a).tobytes())
        for a in (cl.tri, cl.quad, cl.bc):
            f.write(np.ascontiguousarray(a, np.int32).tobytes())
    out = tmp_path / "out.bin"
    r = subprocess.run([exe, str(src), str(out)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    res = np.fromfile(out, np.float64)
    o = oracle_mod.Oracle(cl, "port")
    x, v = cl.xyz.copy(), cl.uvw.copy()
    for _ in range(steps):
        x, v, *_ = o.step(x, v)
    assert np.array_equal(res[:3 * cl.np_], x) and np.array_equal(res[3 * cl.np_:], v)


def _read_ops(path, np_, nnz):
    """The results tests/shim/ops_check.cpp writes, in its order."""
    raw = open(path, "rb").read()
    pos = 0

    def take(dtype, n):
        nonlocal pos
        a = np.frombuffer(raw, dtype, n, pos)
        pos += a.nbytes
        return a

    out = {}
    out["rejected"], out["accepted"], out["iteration"], out["n_singular"] = take(np.int32, 4)
    out["conv"], out["W"] = take(np.float64, 2)
    for k, n in (("dia", 9 * np_), ("crs", 9 * nnz), ("b", 3 * np_), ("fdia", 9 * np_),
                 ("fcrs", 9 * nnz)):
        out[k] = take(np.float64, n)
    out["diaind"] = take(np.int32, np_)
    for k in ("x", "r", "y", "z"):
        out[k] = take(np.float64, 3 * np_)
    nnode = int(take(np.int32, 1)[0])
    out["nodes"] = take(np.int32, 3 * nnode).reshape(-1, 3)
    out["bb_prx"] = take(np.float64, 6 * nnode).reshape(-1, 6)
    out["bb_ccd"] = take(np.float64, 6 * nnode).reshape(-1, 6)
    for k in ("prox", "ccd"):
        n = int(take(np.int32, 1)[0])
        out[k] = take(np.int32, 5 * n).reshape(-1, 5)
    assert pos == len(raw)
    return out


@pytest.mark.parametrize("name,steps", [("drape16", 40), ("fold20", 45), ("stack16", 34)])
def test_cpp_reference_named_operations_match_oracle(sim_mod, oracle_mod, tmp_path, name, steps):
    """The reference's lower-level classes and functions written against
    include/clothsim_ref_ops.hpp (tests/shim/ops_check.cpp, a separate
    process), at a state mid-trajectory (a drape over a sphere, a swept fold
    with pinned vertices, two sheets in contact): SetPattern takes the stencil pattern
    and rejects a different one; the system assembled element by element
    (WdWddW_CST/_Bend/_Contact, Mearge, the m_valDia mass poke,
    SetBoundaryCondition) equals the oracle's assembly; the ILU factor,
    m_diaInd, Solve_PCG (solution, residual, ratio, iteration), MatVec and
    CPreconditionerILU::Solve equal the oracle's; the BVH topology, both
    refits and both contact sets equal the oracle's."""
    import os
    import subprocess
    exe = os.path.join(os.path.dirname(__file__), "shim", "bin", "ops_check")
    if not os.path.exists(exe):
        pytest.fail("tests/shim/bin/ops_check is not built (make -C tests/shim)")
    cl = {"drape16": lambda: scene.drape_over_sphere(16),
          "fold20": lambda: scene.fold_sweep(20, size=0.3),
          "stack16": lambda: scene.stacked_sheets(2, 16, size=0.5, dt=0.005, seed=3,
                                                  obstacle=scene.sphere((0.0, 0.0, -0.3), 0.3))}[name]()
    o = oracle_mod.Oracle(cl, "port")
    x, v, t = cl.xyz.copy(), cl.uvw.copy(), 0.0
    for _ in range(steps):
        scene.apply_sweep(cl, x, t + cl.dt)
        x, v, *_ = o.step(x, v)
        t += cl.dt
    scene.apply_sweep(cl, x, t + cl.dt)
    m = cl.material
    sphere = cl.obstacle.kind == scene.OBST_SPHERE
    hdr = np.array([cl.np_, cl.nt, cl.nq, cl.pcg_maxit, 2 if sphere else 0], np.int32)
    ob = list(cl.obstacle.params[:4]) if sphere else [0.0] * 4
    prm = np.array([m.lam, m.mu, m.stiff_bend, *m.gravity, cl.mass_point, m.stiff_contact,
                    cl.clearance, cl.dt, cl.pcg_tol, *ob], np.float64)
    assert len(prm) == 15
    src = tmp_path / "in.bin"
    with open(src, "wb") as f:
        for a in (hdr, prm, cl.xyz0, cl.xyz, x, v):
            f.write(np.ascontiguousarray(a).tobytes())
        for a in (cl.tri, cl.quad, cl.bc):
            f.write(np.ascontiguousarray(a, np.int32).tobytes())
    out = tmp_path / "out.bin"
    r = subprocess.run([exe, str(src), str(out)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    rp, ci, di = o.pattern()
    g = _read_ops(out, cl.np_, len(ci))
    assert g["rejected"] == 1 and g["accepted"] == 1
    dia, crs, b = o.assemble(x, v)
    assert np.array_equal(g["dia"], dia) and np.array_equal(g["crs"], crs)
    assert np.array_equal(g["b"], b)
    fd, fc = o.ilu(dia, crs)
    assert np.array_equal(g["fdia"], fd) and np.array_equal(g["fcrs"], fc)
    assert np.array_equal(g["diaind"], di)
    xs, rr, conv, it = o.pcg(dia, crs, fd, fc, b, cl.pcg_tol, cl.pcg_maxit)
    assert np.array_equal(g["x"], xs) and np.array_equal(g["r"], rr)
    assert g["conv"] == conv and g["iteration"] == it
    assert np.array_equal(g["y"], o.matvec(dia, crs, 1.5, xs, 0.5, b))
    assert np.array_equal(g["z"], o.ilu_solve(fd, fc, b))
    assert np.array_equal(g["nodes"], o.bvh())
    vm = xs / cl.dt
    assert np.array_equal(g["bb_prx"], o.refit_prx(x, cl.clearance))
    assert np.array_equal(g["bb_ccd"], o.refit_ccd(x, vm, cl.dt))
    prox = o.prox_set(x, cl.clearance)
    assert np.array_equal(g["prox"], prox)
    assert np.array_equal(g["ccd"], o.ccd_set(x, vm, cl.dt, cl.clearance))
    if name == "stack16":
        assert len(prox) > 0  # sheet on sheet: the state has self-contact


@pytest.mark.parametrize("pcg", [0, 2])
def test_batch_matches_each_cloth_alone(sim_mod, oracle_mod, pcg):
    """Cloths of different sizes stepped together (cs_batch_step): every cloth
    follows its own oracle trajectory bit for bit, including a swept fold and
    PCG runs that stop at different iterations; with shared launches per PCG
    operation (pcg 0) and with the one-workgroup solve (one workgroup per
    cloth, pcg 2)."""
    cls = [scene.drape_over_sphere(16), scene.fold_sweep(24, size=0.3), scene.drape_over_sphere(32),
           scene.reference_demo(0)]
    for cl in cls:
        cl.pcg_tol, cl.pcg_maxit = 1e-6, 1000
    steps = 25
    devs = [sim_mod.DeviceCloth(cl) for cl in cls]
    for d in devs:
        d.set_option(2, pcg)
    try:
        with sim_mod.DeviceBatch(devs) as b:
            st = b.step(steps)
        for cl, d, s in zip(cls, devs, st):
            o = oracle_mod.Oracle(cl, "port")
            x, v, t = cl.xyz.copy(), cl.uvw.copy(), 0.0
            for k in range(steps):
                scene.apply_sweep(cl, x, t + cl.dt)
                x, v, imp, it, conv = o.step(x, v)
                t += cl.dt
            gx, gv = d.get_state()
            assert s["pcg_iters"] == it, (cl.name, s, it)
            assert np.array_equal(gx, x) and np.array_equal(gv, v), (
                cl.name, np.abs(gx - x).max(), np.abs(gv - v).max())
    finally:
        for d in devs:
            d.close()


def test_served_results_equal_alone(sim_mod, oracle_mod):
    """Continuous batching: requests of different sizes arriving while others
    run end bit-identical to the same simulations stepped alone, with a
    generous HBM budget (all overlap), a tight one (requests queue), and one
    lane whose PCG variant the autotuner changes from tick to tick."""
    from cloth_sim_self_collision_amd import serve
    sph = scene.sphere((0.0, 0.0, 0.0), 0.3)
    bx = scene.box((0.0, 0.0, 0.0), (0.25, 0.25, 0.25))
    reqs = [serve.Request(0, scene.drop_on_obstacle(20, 0.35, sph, seed=1), steps=12, arrival=0.0),
            serve.Request(1, scene.drop_on_obstacle(16, 0.32, bx, ny=24, seed=2), steps=8,
                          arrival=0.02),
            serve.Request(2, scene.drape_over_sphere(16), steps=10, arrival=0.04)]
    alone = {}
    for r in reqs:
        with sim_mod.DeviceCloth(r.cloth) as d:
            d.step(r.steps)
            alone[r.rid] = d.get_state()
    # absolute parity of one request against the oracle
    o = oracle_mod.Oracle(reqs[1].cloth, "port")
    x, v = reqs[1].cloth.xyz.copy(), reqs[1].cloth.uvw.copy()
    for _ in range(reqs[1].steps):
        x, v, *_ = o.step(x, v)
    assert np.array_equal(alone[1][0], x) and np.array_equal(alone[1][1], v)
    biggest = max(r.cloth.np_ for r in reqs) * serve.BYTES_PER_VERTEX_ESTIMATE
    for budget, realtime, tune in ((1 << 36, True, False), (biggest + 1, False, False),
                                   (1 << 36, False, True)):
        # the last run: one lane whose PCG variant the tuner switches between ticks
        kw = {"lanes": (), "autotune": True} if tune else {}
        out = serve.Server(budget, **kw).run(reqs, realtime=realtime)
        assert [r.rid for r in out["results"]] == [0, 1, 2]
        for res in out["results"]:
            assert len(res.step_ms) == reqs[res.rid].steps
            ax, av = alone[res.rid]
            assert np.array_equal(res.xyz, ax) and np.array_equal(res.uvw, av), (budget, res.rid)


@pytest.mark.parametrize("name,steps", [("drape32", 30), ("fold24", 60), ("stack16", 20)])
def test_mixed_precision_tracks_the_reference(sim_mod, oracle_mod, name, steps):
    """CS_OPT_PRECISION 1 (the packed ILU sweep reads the factor rounded to
    FP32; everything else FP64) on scenes whose ILU(0)-PCG converges: over
    trajectories up to the first contact impulse the positions stay within
    1e-5 m (the tolerance stated for the mixed mode) of the FP64 reference
    after every step, and every solve converges.  Past the first impulse the
    reference's own trajectory is chaotic (its contact decisions are
    thresholds): a 1e-13 m change of drape32's start grows to 2e-3 m by step
    100 in the oracle itself, so only a bit-identical step can follow it
    there; single steps are checked along such a trajectory below."""
    cl = _scenes()[name]
    o = oracle_mod.Oracle(cl, "port")
    x, v, t = cl.xyz.copy(), cl.uvw.copy(), 0.0
    worst = 0.0
    with sim_mod.DeviceCloth(cl) as d:
        d.set_option(sim_mod.DeviceCloth.OPT_PRECISION, 1)
        for k in range(steps):
            scene.apply_sweep(cl, x, t + cl.dt)
            x, v, imp, *_ = o.step(x, v)
            t += cl.dt
            assert not imp, f"step {k} applies an impulse: past the comparable range"
            st = d.step(1)
            gx, _ = d.get_state()
            worst = max(worst, float(np.abs(gx - x).max()))
            assert st["pcg_iters"] < cl.pcg_maxit, (k, st)
    print(f"{name}: max position error of the mixed mode over {steps} steps {worst:.3e} m")
    assert worst <= 1e-5, worst


def test_mixed_precision_single_steps_along_a_contact_trajectory(sim_mod, oracle_mod):
    """Along drape32's first 100 steps (impulses from step 36 on), each mixed
    step taken from the reference's own state ends within 1e-5 m of the
    reference's step."""
    cl = _scenes()["drape32"]
    o = oracle_mod.Oracle(cl, "port")
    x, v = cl.xyz.copy(), cl.uvw.copy()
    errs = []
    with sim_mod.DeviceCloth(cl) as d:
        d.set_option(sim_mod.DeviceCloth.OPT_PRECISION, 1)
        for k in range(100):
            d.set_state(x, v)
            d.step(1)
            gx, _ = d.get_state()
            x, v, *_ = o.step(x, v)
            errs.append(float(np.abs(gx - x).max()))
    e = np.array(errs)
    print(f"drape32 single mixed steps: median {np.median(e):.3e} m, max {e.max():.3e} m")
    assert e.max() <= 1e-5, (int(e.argmax()), e.max())


def test_mixed_batch_and_served_equal_mixed_alone(sim_mod):
    """Mixed-precision cloths stepped together (one FP32-coefficient sweep
    launch for all) or served end bit-identical to each stepped alone in
    mixed precision; a mixed request whose solve stops at the PCG cap gets
    an error record; a batch may not mix precisions."""
    from cloth_sim_self_collision_amd import _lib, serve
    cls = [scene.drape_over_sphere(16), scene.fold_sweep(24, size=0.3), scene.drape_over_sphere(32)]
    steps = 15
    alone = []
    for cl in cls:
        with sim_mod.DeviceCloth(cl) as d:
            d.set_option(sim_mod.DeviceCloth.OPT_PRECISION, 1)
            d.step(steps)
            alone.append(d.get_state())
    devs = [sim_mod.DeviceCloth(cl) for cl in cls]
    try:
        for d in devs:
            d.set_option(sim_mod.DeviceCloth.OPT_PRECISION, 1)
        with sim_mod.DeviceBatch(devs) as b:
            b.step(steps)
        for d, (ax, av) in zip(devs, alone):
            gx, gv = d.get_state()
            assert np.array_equal(gx, ax) and np.array_equal(gv, av)
        devs[1].set_option(sim_mod.DeviceCloth.OPT_PRECISION, 0)
        with sim_mod.DeviceBatch(devs) as b:
            with pytest.raises(_lib.ClothSimError, match="precision"):
                b.step(1)
    finally:
        for d in devs:
            d.close()
    stuck = scene.drop_on_obstacle(40, 0.4, scene.sphere((0.0, 0.0, 0.0), 0.3), seed=4)
    stuck.pcg_maxit = 5
    reqs = [serve.Request(k, cl, steps=steps, precision="mixed") for k, cl in enumerate(cls)]
    reqs.append(serve.Request(3, stuck, steps=2, precision="mixed"))
    out = serve.Server(1 << 36).run(reqs, realtime=False)
    fails = {f.rid: f.error for f in out["failures"]}
    assert set(fails) == {3} and "converges" in fails[3]
    for res in out["results"]:
        ax, av = alone[res.rid]
        assert np.array_equal(res.xyz, ax) and np.array_equal(res.uvw, av), res.rid


def test_cloth_from_setup_cache_steps_identically(sim_mod, tmp_path):
    """A cloth created from the on-disk setup cache (pattern, schedules,
    sweep slots, gather lists, BVH all loaded, none rebuilt) steps exactly
    like one whose setup was built."""
    from cloth_sim_self_collision_amd import _lib
    cl = scene.drape_over_sphere(32)
    steps = 20
    with sim_mod.DeviceCloth(cl) as d:
        d.step(steps)
        want = d.get_state()
    try:
        _lib.set_setup_cache(tmp_path)
        with sim_mod.DeviceCloth(cl):
            pass  # builds and writes the file
        s0 = _lib.setup_cache_stats()
        with sim_mod.DeviceCloth(cl) as d:
            assert _lib.setup_cache_stats()["hits"] == s0["hits"] + 1
            d.step(steps)
            got = d.get_state()
    finally:
        _lib.set_setup_cache(None)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


def test_wire_served_results_equal_alone(sim_mod, oracle_mod):
    """Serving over the JSON-lines wire format: each decoded final state equals
    stepping that request's cloth alone, bit for bit (a swept fold, a bar over
    the ground, a drape), and the drape's decoded state equals the oracle's;
    an unservable request gets an error record."""
    import io
    import json
    from cloth_sim_self_collision_amd import serve
    bar = {"kind": "bar_over_ground", "a": [-1, 0, 0], "b": [1, 0, 0], "radius": 0.05,
           "ground_z": -0.3}
    reqs = [
        {"id": "drape", "scene": {"scene": "drape", "n": 16}, "steps": 12, "return": ["x", "v"]},
        {"id": 7, "scene": {"scene": "drop", "n": 14, "height": 0.3, "seed": 1, "obstacle": bar},
         "steps": 9, "arrival": 0.02},
        {"id": "bad", "scene": {"scene": "drape", "n": 16}, "steps": 4, "precision": "bf16"},
        {"id": "fold", "scene": {"scene": "fold", "n": 20, "size": 0.3}, "steps": 6},
    ]
    out = io.StringIO()
    serve.serve_jsonl([json.dumps(r) for r in reqs], out, hbm_budget_bytes=4 << 30,
                      realtime=False)
    recs = {json.dumps(r["id"]): r for r in map(json.loads, out.getvalue().splitlines())}
    assert len(recs) == 4 and recs['"bad"']["status"] == "error"
    for r in reqs:
        if r["id"] == "bad":
            continue
        rec = recs[json.dumps(r["id"])]
        assert rec["status"] == "ok" and len(rec["step_ms"]) == r["steps"] == rec["steps"]
        cl = scene.from_config(r["scene"])
        with sim_mod.DeviceCloth(cl) as d:
            d.step(r["steps"])
            x, v = d.get_state()
        assert np.array_equal(serve.decode_array(rec["x"]).reshape(-1), x), r["id"]
        if "v" in r.get("return", []):
            assert np.array_equal(serve.decode_array(rec["v"]).reshape(-1), v), r["id"]
    # the decoded drape against the oracle itself
    cl = scene.from_config(reqs[0]["scene"])
    o = oracle_mod.Oracle(cl, "port")
    ox, ov = cl.xyz.copy(), cl.uvw.copy()
    for _ in range(reqs[0]["steps"]):
        ox, ov, *_ = o.step(ox, ov)
    rec = recs[json.dumps("drape")]
    assert np.array_equal(serve.decode_array(rec["x"]).reshape(-1), ox)
    assert np.array_equal(serve.decode_array(rec["v"]).reshape(-1), ov)


@pytest.mark.parametrize("name,maxit", [("fold256", 30), ("stack4x512", 3)])
def test_full_size_configs(sim_mod, oracle_mod, name, maxit):
    """The benchmark's single cloth (256^2, 65,536 vertices) and four stacked
    512^2 sheets (1,048,576 vertices, four components, each swept by its own
    workgroup) at full size, PCG capped so that the oracle finishes in
    seconds: the internal step (assembly, ILU(0), PCG) bit for bit, and for
    the 256^2 cloth a whole StepTime with its contact pass."""
    import os
    cfg = os.path.join(os.path.dirname(os.path.dirname(__file__)), "cloth_sim_self_collision_amd",
                       "configs", name + ".json")
    cl = scene.load_config(cfg)
    cl.pcg_maxit = maxit
    o = oracle_mod.Oracle(cl, "port")
    x0, v0 = cl.xyz.copy(), cl.uvw.copy()
    scene.apply_sweep(cl, x0, cl.dt)
    ox, ov, oconv, oit = o.step_internal(x0, v0)
    with sim_mod.DeviceCloth(cl) as d:
        d.set_state(x0, v0)
        conv, it = d.step_internal_dynamics_ilu()
        gx, gv = d.get_state()
        assert (it, conv) == (oit, oconv)
        assert np.array_equal(gx, ox) and np.array_equal(gv, ov)
    if name == "fold256":
        x, v, imp, it, conv = o.step(x0, v0)
        with sim_mod.DeviceCloth(cl) as d:
            st = d.step(1)
            gx, gv = d.get_state()
        assert st["pcg_iters"] == it and st["impulse_applied"] == imp
        assert np.array_equal(gx, x) and np.array_equal(gv, v)


def test_impact_zone_vertex_count_reported(sim_mod):
    """Steps that run rigid impact zones report how many vertices the zones
    hold (the drape over the sphere reaches them within 100 steps)."""
    cl = scene.drape_over_sphere(32)
    riz = []
    with sim_mod.DeviceCloth(cl) as d:
        for _ in range(100):
            st = d.step(1)
            if st["n_riz_pass"] > 0:
                riz.append((st["n_riz_pass"], st["n_riz_vertices"]))
    assert riz, "no step reached the impact zones"
    assert all(nv > 0 for _, nv in riz), riz


def test_nonfinite_solve_is_reported_not_stepped(sim_mod, oracle_mod):
    """A mesh on which the reference's ILU(0) overflows (489 x 151 vertices,
    the fast vertex index along the short side): the internal solve is NaN,
    as in the oracle, and the step returns CS_ERR_NONFINITE before its
    contact pass; in a batch only that cloth is flagged and the other steps
    exactly as alone."""
    from cloth_sim_self_collision_amd import _lib
    bad = scene.drop_on_obstacle(489, 0.5, scene.sphere((0, 0, 0), 0.3), ny=151, seed=3,
                                 pcg_maxit=3)
    o = oracle_mod.Oracle(bad, "port")
    _, ov, oconv, _ = o.step_internal(bad.xyz.copy(), bad.uvw.copy())
    assert not np.isfinite(ov).all() and np.isnan(oconv)
    o.close()
    with sim_mod.DeviceCloth(bad) as d:
        with pytest.raises(_lib.ClothSimError) as e:
            d.step(1)
        assert e.value.status == 6  # CS_ERR_NONFINITE
    good = scene.drape_over_sphere(16)
    good.pcg_maxit = bad.pcg_maxit = 20  # a batch shares the PCG settings
    with sim_mod.DeviceCloth(good) as d:
        d.step(2)
        want = d.get_state()
    devs = [sim_mod.DeviceCloth(good), sim_mod.DeviceCloth(bad)]
    try:
        with sim_mod.DeviceBatch(devs) as b:
            st = b.step(2)
        assert st[0]["status"] == 0 and st[1]["status"] == 6
        gx, gv = devs[0].get_state()
        assert np.array_equal(gx, want[0]) and np.array_equal(gv, want[1])
    finally:
        for dv in devs:
            dv.close()
