"""Several push workgroups per tile, chosen by the tiles and particles of a launch: every choice
gives the bits of the generic kernel (integer current)."""
import numpy as np
import pytest

import osiris_amd as oa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,tile,ppc,nsp", [
    ((192, 256), (16, 16), (4, 4), 1), ((193, 256), (16, 16), (4, 4), 1), ((384, 250), (16, 16), (4, 4), 1),
    ((385, 250), (16, 16), (4, 4), 1), ((100, 90), (16, 16), (2, 2), 1), ((256, 128), (16, 16), (4, 4), 3),
    ((256, 250), (32, 16), (4, 4), 1), ((257, 250), (32, 16), (4, 4), 1), ((64, 60), (8, 8), (4, 4), 2)])
def test_split_changes_no_bit(nx, tile, ppc, nsp):
    """Both sides of the limits; the particles are replaced between two runs, so that the choice
    changes with mover lists of the first run behind it."""
    print(f"case nx={nx} tile={tile} ppc={ppc} nsp={nsp}", flush=True)
    out = []
    for kernel in (0, 1):
        with oa.Simulation(2, nx, (0.1, 0.1), 0.05, 2, tile=tile, kernel=kernel) as sim:
            for k in range(nsp):
                sim.generate(sim.add_species(-1.0), (1, 1), uth=(0.3,) * 3, seed=3 + k)
            sim.run(4)
            for k in range(nsp):
                sim.generate(k, ppc, uth=(0.3,) * 3, ufl=(0.2, 0.1, 0.0), seed=13 + k)
            sim.run(4)
            got = sim.get_fields()
            for k in range(nsp):
                got = got + sim.get_particles(k)
            out.append(([a.view(np.uint32) for a in got], sim.history()))
    for a, b in zip(out[0][0], out[1][0]):
        assert np.array_equal(a, b)
    for a, b in zip(out[0][1], out[1][1]):
        assert np.allclose(a, b, rtol=1e-12, atol=0)


def test_split_changes_at_a_relayout():
    """Free particles of a block of 25 tiles meet in its middle one: tiles overflow, and with one
    tile at some 20 times the others' count the re-layouts find two workgroups per tile the better
    choice between steps of one run."""
    rng = np.random.default_rng(2)
    nx, steps = (512, 256), 240
    cells = np.stack(np.meshgrid(np.arange(1, nx[0] + 1), np.arange(1, nx[1] + 1), indexing="ij"), -1)
    ix = cells.reshape(-1, 2).astype(np.int32)
    n = len(ix)
    x = (rng.random((n, 2), np.float32) - np.float32(0.5)).astype(np.float32)
    off = np.array((272.5, 136.5)) - ix - x  # to the middle of tile (8, 8) of 32x16
    u = np.zeros((n, 3), np.float32)
    inside = (np.abs(off[:, 0]) < 80) & (np.abs(off[:, 1]) < 40)
    v = off[inside] / steps * 0.1 / 0.05  # c = 0.5 cells per step
    u[inside, :2] = v / np.sqrt(1 - (v ** 2).sum(1, keepdims=True))
    out = []
    for kernel in (0, 1):
        with oa.Simulation(2, nx, (0.1, 0.1), 0.05, 2, tile=(32, 16), kernel=kernel) as sim:
            sid = sim.add_species(-1.0)
            sim.set_particles(sid, ix, x, u, np.full(n, -1e-12, np.float32))
            for k in (steps - 20, 20, 20):
                sim.run(k)
            assert sim.relayouts >= 1
            got = sim.get_particles(sid)
            at = got[0] - 1
            most = np.bincount(at[:, 0] // 32 + 16 * (at[:, 1] // 16)).max()
            out.append(([a.view(np.uint32) for a in sim.get_fields() + got], sim.history()))
    assert most > 8000  # 15 times the 512 of a tile at the start
    for a, b in zip(out[0][0], out[1][0]):
        assert np.array_equal(a, b)
    for a, b in zip(out[0][1], out[1][1]):
        assert np.allclose(a, b, rtol=1e-12, atol=0)
