"""The work split of the step's kernels at the edges of their rules: every choice gives the
bits of the generic kernels (integer current, order-independent), so the comparisons are
exact; the FP64 energy sums are grouped differently and agree to round-off (1e-12)."""
import numpy as np
import pytest

import osiris_amd as oa

pytestmark = pytest.mark.gpu


def _run(dims, nx, order, steps, **kw):
    with oa.Simulation(dims, nx, (0.1,) * dims, 0.04, order, **kw) as sim:
        rng = np.random.default_rng(5)
        n = 3 * int(np.prod(nx))
        for rqm, drift in ((-1.0, 0.3), (1.0, -0.2)):
            sid = sim.add_species(rqm)
            ix = np.stack([rng.integers(1, m + 1, n) for m in nx], 1).astype(np.int32)
            x = (rng.random((n, dims), np.float32) - np.float32(0.5)).astype(np.float32)
            u = (rng.standard_normal((n, 3)) * 0.2).astype(np.float32)
            u[:, 0] += np.float32(drift)
            sim.set_particles(sid, ix, x, u, np.full(n, 0.05 * rqm, np.float32))
        sim.run(steps)
        return sim.get_fields(), sim.get_particles(0), sim.get_particles(1), sim.history()


def _same(a, b):
    for x, y in zip(a[0] + a[1] + a[2], b[0] + b[1] + b[2]):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
    for x, y in zip(a[3], b[3]):
        assert np.allclose(x, y, rtol=1e-12, atol=0)


@pytest.mark.parametrize("nx,tile,waves", [
    ((16, 16), (16, 16), 4), ((16, 40), (16, 16), 4), ((128, 256), (16, 16), 4),
    ((129, 256), (16, 16), 4), ((384, 256), (16, 16), 4), ((385, 250), (16, 16), 4),
    ((64, 33), (32, 16), 8), ((640, 512), (32, 16), 8), ((641, 512), (32, 16), 8),
    ((48, 40), (16, 16), 8), ((70, 30), (8, 8), 4)])
def test_push_workgroups_per_tile(nx, tile, waves):
    """1, 2 and 4 push workgroups per tile, on both sides of each limit, tiles cut by the
    grid's edge, 1 and 2 tiles per direction."""
    print(f"case nx={nx} tile={tile} waves={waves}", flush=True)
    _same(_run(2, nx, 2, 6, tile=tile, push_waves=waves), _run(2, nx, 2, 6, tile=tile, kernel=1))


@pytest.mark.parametrize("dims,order,pusher", [(2, 1, 0), (2, 2, 1), (2, 3, 0), (3, 1, 1), (3, 2, 0), (3, 3, 1)])
@pytest.mark.parametrize("case", ["all_cross", "none_cross", "one_cell"])
def test_push_crossing_queue(dims, order, pusher, case):
    """The queue of face-crossing particles: every particle of a wave crosses (up to all
    faces at once), none does, and thousands pile up in one cell; grids large enough for the
    raw fixed-point sums, against the generic kernel (bit for bit)."""
    print(f"case dims={dims} order={order} pusher={pusher} {case}", flush=True)
    nx = (256, 192) if dims == 2 else (48, 40, 24)
    out = []
    for kernel in (0, 1):
        with oa.Simulation(dims, nx, (0.1,) * dims, 0.055, order, kernel=kernel) as sim:
            rng = np.random.default_rng(3)
            n = 150_001
            ix = np.stack([rng.integers(1, m + 1, n) for m in nx], 1).astype(np.int32)
            if case == "one_cell":
                ix[:5000] = 17
            x = (rng.random((n, dims), np.float32) - np.float32(0.5)).astype(np.float32)
            u = (rng.standard_normal((n, 3)) * (1e-23 if case == "none_cross" else 0.1)).astype(np.float32)
            if case == "all_cross":
                u[:, :dims] = np.where(rng.random((n, dims)) < 0.5, -5.0, 5.0)
                x[:, :dims] = np.sign(u[:, :dims]) * np.float32(0.49)
            sid = sim.add_species(-1.0, pusher)
            sim.set_particles(sid, ix, x, u, np.full(n, -0.01, np.float32))
            sim.fill_fields(b0=(0.0, 0.0, 0.2) if case != "none_cross" else (0.0, 0.0, 0.0))
            sim.run(3)
            out.append((sim.get_fields(), sim.get_particles(0), (), sim.history()))
    _same(*out)


@pytest.mark.parametrize("nx,order", [((1, 1), 1), ((2, 3), 2), ((31, 7), 1), ((33, 9), 2), ((65, 17), 3),
                                      ((32, 8), 1), ((700, 600), 2), ((1024, 512), 1)])
def test_fused_field_step(nx, order):
    """The one-launch periodic 2D field step against the three-launch drop-in Yee step on
    the same fields and current-free plasma (bit for bit, both copies used in turn), and
    the history rows against the FP64 sums of the fields the steps began with; runs
    split over calls and fields set between them continue on the same rows."""
    print(f"case nx={nx} order={order}", flush=True)
    rng = np.random.default_rng(11)
    dx, dt = (0.1, 0.12), 0.06
    shape = (nx[1], nx[0], 3)
    e, b = (rng.standard_normal(shape).astype(np.float32) for _ in range(2))
    gcl, pad = (1, 1), (2, 2)

    def guarded(f):
        return np.ascontiguousarray(np.pad(f, ((gcl[1], pad[1]), (gcl[0], pad[0]), (0, 0)), "wrap"))

    ge, gb = guarded(e), guarded(b)
    rows = []
    with oa.Simulation(2, nx, dx, dt, order) as sim:
        sim.set_fields(e, b)
        for k in range(6):
            inner = (slice(1, 1 + nx[1]), slice(1, 1 + nx[0]))
            rows.append([(f[inner][..., m].astype(np.float64) ** 2).sum() for f in (gb, ge) for m in range(3)])
            oa.yee_advance(2, nx, gcl, dx, dt, ge, gb, np.zeros_like(ge))
            if k != 1:  # steps 1 and 2 in one call
                sim.run(2 if k == 2 else 1)
                se, sb = sim.get_fields()
                assert np.array_equal(se.view(np.uint32), ge[inner].view(np.uint32))
                assert np.array_equal(sb.view(np.uint32), gb[inner].view(np.uint32))
            if k == 3:
                ge, gb = guarded(e * np.float32(0.5)), guarded(b)
                sim.set_fields(e * np.float32(0.5), b)
        fld, _ = sim.history()
    want = 0.5 * dx[0] * dx[1] * np.array(rows)
    assert np.allclose(fld, want, rtol=1e-12, atol=0)


@pytest.mark.parametrize("nx,order", [((6, 5), (15, 15)), ((32, 16), (1, 2)), ((33, 17), (3, 3)), ((31, 70), (15, 0)),
                                      ((90, 15), (0, 15)), ((300, 200), (3, 3))])
def test_smoothed_current_2d(nx, order):
    """After one step from zero fields E = -dt J; with dt a power of two the product is
    exact, so the smoothed run's E is the filter (x before y, taps summed left to right with
    each product rounded) of the unsmoothed run's E bit for bit."""
    print(f"case nx={nx} order={order}", flush=True)
    rng = np.random.default_rng(3)
    n = 5 * nx[0] * nx[1]
    ix = np.stack([rng.integers(1, m + 1, n) for m in nx], 1).astype(np.int32)
    x = (rng.random((n, 2), np.float32) - np.float32(0.5)).astype(np.float32)
    u = (rng.standard_normal((n, 3)) * 0.5).astype(np.float32)
    q = (-rng.random(n)).astype(np.float32)
    coef = np.zeros((3, 31), np.float32)
    for d in range(2):
        coef[d, 15 - order[d]:16 + order[d]] = rng.standard_normal(2 * order[d] + 1)
    e = []
    for smooth in (False, True):
        with oa.Simulation(2, nx, (0.1, 0.1), 0.0625, 2) as sim:
            sim.set_particles(sim.add_species(-1.0), ix, x, u, q)
            if smooth:
                sim.set_smooth(order + (0,), coef)
            sim.run(1)
            e.append(sim.get_fields()[0])
    want = e[0]
    for d in range(2):
        if order[d]:
            k = order[d]
            taps = [np.roll(want, -m, 1 - d) * coef[d, 15 + m] for m in range(-k, k + 1)]
            want = taps[0]
            for t in taps[1:]:
                want = want + t
    assert np.array_equal(e[1], want)  # the sign of a zero sum is not the product's


@pytest.mark.parametrize("dims,n", [(2, 1), (2, 2047), (2, 200_000), (3, 70_000)])
def test_particles_come_back_in_upload_order(dims, n):
    """get_particles after absorbing walls removed some: the survivors in upload order (the
    charges number the particles), each with its own cell, position and momentum (free
    motion without charge-weighted forces is checked through u, which stays as given up to
    the tiny fields of 1e-12 charges)."""
    print(f"case dims={dims} n={n}", flush=True)
    rng = np.random.default_rng(9)
    nx = (64, 40, 24)[:dims]
    ix = np.stack([rng.integers(1, m + 1, n) for m in nx], 1).astype(np.int32)
    x = (rng.random((n, dims), np.float32) - np.float32(0.5)).astype(np.float32)
    u = (rng.standard_normal((n, 3)) * 3.0).astype(np.float32)
    q = (-(np.arange(n) + 1) * 1e-14).astype(np.float32)
    with oa.Simulation(dims, nx, (0.1,) * dims, 0.05, 2, xbnd="lindman") as sim:
        sid = sim.add_species(-1.0)
        sim.set_particles(sid, ix, x, u, q)
        got0 = sim.get_particles(sid)
        for a, b in zip(got0, (ix, x, u, q)):
            assert np.array_equal(a, b)
        sim.run(25)
        jx, jp, ju, jq = sim.get_particles(sid)
        assert len(jq) == sim.count(sid) and (n < 100 or len(jq) < n)
    k = np.searchsorted(-q, -jq)  # ascending and unique
    assert np.array_equal(q[k], jq) and np.all(np.diff(k) > 0)
    assert np.allclose(ju, u[k], rtol=0, atol=1e-5)
    v = u[k].astype(np.float64) / np.sqrt(1 + (u[k].astype(np.float64) ** 2).sum(1, keepdims=True))
    end = (ix[k] + x[k] + 25 * 0.5 * v[:, :dims])
    d = jx + jp - end
    for m in range(1, dims):
        d[:, m] -= nx[m] * np.round(d[:, m] / nx[m])
    assert np.abs(d).max() < 1e-3


@pytest.mark.parametrize("dims,xbnd", [(2, "lindman"), (2, "vpml"), (3, "lindman"), (3, "vpml")])
def test_laser_steps_in_one_call(dims, xbnd):
    """Steps of one call against calls of one step: inside a call the last field launch of a
    step adds the next step's laser values, the first step of a call has a launch of its
    own.  The drifting block overflows tiles, so steps also stop between the two."""
    print(f"case dims={dims} xbnd={xbnd}", flush=True)
    nx = (32, 30, 10)[:dims]
    rng = np.random.default_rng(21)
    n = 6000
    ix = np.stack([rng.integers(lo, hi, n) for lo, hi in ((17, 25), (1, 9), (1, 5))[:dims]], 1).astype(np.int32)
    x = (rng.random((n, dims), np.float32) - np.float32(0.5)).astype(np.float32)
    u = (rng.standard_normal((n, 3)) * 0.05 + (2.0, 1.5, 0.0)).astype(np.float32)
    out = []
    for calls in ((1,) * 23, (23,), (9, 2, 12)):
        with oa.Simulation(dims, nx, (0.1,) * dims, 0.05, 2, xbnd=xbnd, tile=(8, 8, 4)[:dims]) as sim:
            sim.set_particles(sim.add_species(-1.0), ix, x, u, np.full(n, -0.02, np.float32))
            for prop in ("forward", "backward"):
                sim.add_zpulse_wall(a0=0.7, omega0=5.0, pol=30.0, pol_type=1, propagation=prop,
                                    tenv_type="sin2", tenv_rise=0.4, tenv_flat=0.5, tenv_fall=0.3)
            for k in calls:
                sim.run(k)
            out.append((sim.get_fields(), sim.get_particles(0), (), sim.history()))
            rel = sim.relayouts
    assert rel >= 1
    for o in out[1:]:
        _same(out[0], o)


@pytest.mark.parametrize("dims,order", [(2, 1), (2, 2), (2, 3), (3, 1), (3, 2), (3, 3)])
@pytest.mark.parametrize("n", [1, 256, 257, 9000])
def test_dropin_current_in_any_particle_order(dims, order, n):
    """Particles in cell order, whose workgroups sum their current in LDS, and the same ones
    shuffled over the whole grid, whose workgroups add to memory: the integer sums agree, so
    the currents have the same bits; so have the particles."""
    print(f"case dims={dims} order={order} n={n}", flush=True)
    rng = np.random.default_rng(17)
    nx, lo, hi = (90, 70, 40)[:dims], 3, 4
    ix = np.stack([rng.integers(1, m + 1, n) for m in nx], 1).astype(np.int32)
    if dims == 3:  # dense enough for the sorted case to fit: 9000 in a 24 x 20 x 10 corner
        ix = np.stack([rng.integers(1, m + 1, n) for m in (24, 20, 10)], 1).astype(np.int32)
    ix = ix[np.lexsort(ix.T)]
    x = (rng.random((n, dims), np.float32) - np.float32(0.5)).astype(np.float32)
    u = (rng.standard_normal((n, 3)) * 2.0).astype(np.float32)
    q = np.full(n, -0.0173, np.float32)
    shape = tuple(m + lo + hi for m in reversed(nx)) + (3,)
    e, b = (rng.standard_normal(shape).astype(np.float32) for _ in range(2))
    out = []
    for p in (np.arange(n), rng.permutation(n)):
        j = np.zeros(shape, np.float32)
        r = oa.advance_deposit(dims, order, ix[p], x[p], u[p], q, -1.0, e, b, lo, j, lo,
                               (0.1,) * dims, 0.05)
        back = np.argsort(p)
        out.append([j] + [a[back] for a in r[:3]])
    for a, c in zip(*out):
        assert np.array_equal(a.view(np.uint32), c.view(np.uint32))


@pytest.mark.parametrize("n", [1, 4, 5, 64, 65, 700])
@pytest.mark.parametrize("cells", [1, 3, 40])
def test_cubic_deposit_lanes(n, cells):
    """The cubic 3D deposit permutes its lanes by their base node: few particles, full waves
    and remainders, all of a kind or of many kinds, against the generic kernel (bit for
    bit)."""
    print(f"case n={n} cells={cells}", flush=True)
    rng = np.random.default_rng(n + cells)
    nx = (24, 16, 12)
    at = np.stack([rng.integers(1, m + 1, cells) for m in nx], 1).astype(np.int32)
    ix = at[rng.integers(0, cells, n)]
    x = (rng.random((n, 3), np.float32) - np.float32(0.5)).astype(np.float32)
    u = (rng.standard_normal((n, 3)) * 0.3).astype(np.float32)
    out = []
    for kernel in (0, 1):
        with oa.Simulation(3, nx, (0.1,) * 3, 0.055, 3, kernel=kernel) as sim:
            sim.set_particles(sim.add_species(-1.0), ix, x, u, np.full(n, -0.01, np.float32))
            sim.run(5)
            out.append((sim.get_fields(), sim.get_particles(0), (), sim.history()))
    _same(*out)


@pytest.mark.parametrize("dims,nx,kw,smooth", [
    (2, (64, 48), {}, 0), (2, (64, 48), {}, 3), (2, (150, 90), dict(reorder=2), 0), (2, (1024, 512), {}, 0),
    (3, (24, 20, 12), {}, 0), (3, (24, 20, 12), dict(reorder=3), 1), (2, (64, 48), dict(xbnd="lindman"), 0),
    (3, (24, 20, 12), dict(xbnd="lindman"), 0), (2, (64, 48), dict(xbnd="vpml"), 0),
    (2, (64, 48), dict(xbnd="vpml", vpml_diffuse=(True, False)), 0), (3, (24, 20, 12), dict(xbnd="vpml"), 0)])
def test_field_work_beside_the_fill(dims, nx, kw, smooth):
    """A run, whose tile fill carries the first part of the field advance, against steps with
    every kernel in a launch of its own (the timed ones), bit for bit."""
    print(f"case nx={nx} {kw} smooth={smooth}", flush=True)
    rng = np.random.default_rng(29)
    n = 4 * int(np.prod(nx))
    out = []
    ix = np.stack([rng.integers(1, m + 1, n) for m in nx], 1).astype(np.int32)
    x = (rng.random((n, dims), np.float32) - np.float32(0.5)).astype(np.float32)
    u = (rng.standard_normal((n, 3)) * 0.2).astype(np.float32)
    e, b = (rng.standard_normal(tuple(reversed(nx)) + (3,)).astype(np.float32) * np.float32(0.1) for _ in range(2))
    for timed in (False, True):
        with oa.Simulation(dims, nx, (0.1,) * dims, 0.05, 2, **kw) as sim:
            for rqm in (-1.0, 100.0):
                sim.set_particles(sim.add_species(rqm), ix, x, u, np.full(n, 0.02 * np.sign(rqm), np.float32))
            sim.set_fields(e, b)
            if smooth:
                sim.set_smooth(*oa.smooth_setup(dims, ["compensated"] * dims, (smooth,) * dims, (0.1,) * dims))
            sim.time_kernels(9) if timed else sim.run(9)
            out.append((sim.get_fields(), sim.get_particles(0), sim.get_particles(1), sim.history()))
    _same(*out)


@pytest.mark.parametrize("n", [1, 4095, 4096, 4097, 16384, 16385, 33000])
def test_noalloc_sums(n):
    """The allocation-free drop-in sums |q| (which sets the current's scale) and the energy
    partials in the order of the host entry point; sizes at the remainders of its 16 x 256
    loads and 64 partials at a time.  Equal charges, so the scales agree and J too."""
    from test_zz_no_alloc import _noalloc

    print(f"case n={n}", flush=True)
    rng = np.random.default_rng(n)
    nx, lo, hi = (40, 30), 3, 4
    ix = np.stack([rng.integers(1, m + 1, n) for m in nx], 1).astype(np.int32)
    x = (rng.random((n, 2), np.float32) - np.float32(0.5)).astype(np.float32)
    u = rng.standard_normal((n, 3)).astype(np.float32)
    q = np.full(n, -0.25, np.float32)
    shape = tuple(m + lo + hi for m in reversed(nx)) + (3,)
    e, b = (rng.standard_normal(shape).astype(np.float32) for _ in range(2))
    j0 = np.zeros(shape, np.float32)
    jr = j0.copy()
    want = oa.advance_deposit(2, 2, ix.copy(), x.copy(), u.copy(), q, -1.0, e, b, lo, jr, lo, (0.1, 0.1), 0.05)
    got = _noalloc(2, 2, oa.OSR_BORIS, ix, x, u, q, e, b, lo, j0, (0.1, 0.1), 0.05)
    for a, c in zip(want[:3], got[:3]):
        assert np.array_equal(a.view(np.uint32), c.view(np.uint32))
    assert np.array_equal(jr.view(np.uint32), got[3].view(np.uint32)) and want[3] == got[4]
