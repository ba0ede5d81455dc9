"""A periodic 2D grid beyond 2^27 cells keeps one copy of its fields and advances them in three
launches, the first of them beside the tile fill."""
import numpy as np
import pytest

import osiris_amd as oa

pytestmark = pytest.mark.gpu


def test_large_grid_on_one_copy():
    """A cloud of particles on 12000x11200 cells against the same cloud on 240x192, which takes
    both copies and one launch: nothing reaches the small grid's edge in 6 steps, so the fields
    around the cloud and its particles have the same bits, and the fields are zero elsewhere."""
    rng = np.random.default_rng(8)
    n, at = 3000, (4800, 3200)
    ix = rng.integers(100, 130, (n, 2)).astype(np.int32)
    x = (rng.random((n, 2), np.float32) - np.float32(0.5)).astype(np.float32)
    u = (rng.standard_normal((n, 3)) * 0.5).astype(np.float32)
    q = np.full(n, -0.02, np.float32)
    out = []
    for nx, lo in (((240, 192), (0, 0)), ((12000, 11200), at)):
        print(f"case nx={nx}", flush=True)
        with oa.Simulation(2, nx, (0.1, 0.1), 0.06, 2, tile=(48, 32)) as sim:
            grid = 48 * nx[0] * nx[1]
            assert sim.footprint // grid == (2 if nx[0] == 240 else 1)
            sid = sim.add_species(-1.0)
            sim.set_particles(sid, ix + np.array(lo, np.int32), x, u, q)
            sim.run(6)
            px = sim.get_particles(sid)
            e, b = sim.get_fields()
            fld, par = sim.history()
        win = (slice(lo[1] + 80, lo[1] + 150), slice(lo[0] + 80, lo[0] + 150))
        for f in (e, b):
            assert np.count_nonzero(f) == np.count_nonzero(f[win]) > 0
        out.append([e[win].view(np.uint32), b[win].view(np.uint32), px[0] - np.array(lo, np.int32)] + list(px[1:]) +
                   [fld, par])
    for a, c in zip(out[0][:-2], out[1][:-2]):
        assert np.array_equal(a, c)
    for a, c in zip(out[0][-2:], out[1][-2:]):
        assert np.allclose(a, c, rtol=1e-12, atol=0)
