"""What a tile's fill takes without a re-layout of the species."""
import numpy as np
import pytest

import osiris_amd as oa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [32_768, 32_769, 40_000])
def test_any_number_may_leave_a_tile(n):
    """n particles leave a tile in one step, through an absorbing wall; the others close the gap
    behind them, whole and in the fill's order, in the step itself."""
    print(f"case n={n}", flush=True)
    rng = np.random.default_rng(n)
    stay = 3000
    ix = np.empty((n + stay, 2), np.int32)
    ix[:, 0], ix[:, 1] = 64, 20
    x = np.empty((n + stay, 2), np.float32)
    x[:, 0], x[:, 1] = 0.49, rng.random(n + stay, np.float32) * 0.5 - 0.25
    u = np.zeros((n + stay, 3), np.float32)
    go = np.zeros(n + stay, bool)
    go[rng.permutation(n + stay)[:n]] = True
    u[go, 0] = 5.0
    ix[~go, 0], x[~go, 0] = 60, 0.0
    q = (-(np.arange(n + stay) + 1) * 1e-14).astype(np.float32)
    with oa.Simulation(2, (64, 32), (0.1, 0.1), 0.05, 2, xbnd="lindman") as sim:
        sid = sim.add_species(-1.0)
        sim.set_particles(sid, ix, x, u, q)
        sim.run(1)
        assert sim.relayouts == 0
        got = sim.get_particles(sid)
        assert sim.count(sid) == stay
        sim.run(2)
        assert sim.count(sid) == stay and sim.relayouts == 0
    assert np.array_equal(got[0], ix[~go]) and np.array_equal(got[3], q[~go])
    assert np.allclose(got[1], x[~go], rtol=0, atol=1e-6)
