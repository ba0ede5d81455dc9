"""The compile-time push kernels add the current's fixed-point terms as raw FP64 bits where no
tile's sums can leave +-2^50, and convert each term elsewhere.  Both against the generic kernel,
bit for bit, for every order and pusher, and each test asserts which of the two ran."""
import numpy as np
import pytest

import osiris_amd as oa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,order,pusher", [(d, o, p) for d in (2, 3) for o in (1, 2, 3) for p in (0, 1)])
@pytest.mark.parametrize("pile,raw", [(600, True), (5000, False)])
def test_raw_and_converted_sums(dims, order, pusher, pile, raw):
    """`pile` fast particles in one cell: as many as the rule lets through (their sums come to
    a good part of 2^50), or several times more, which it must turn away."""
    print(f"case dims={dims} order={order} pusher={pusher} pile={pile}", flush=True)
    nx = (512, 384) if dims == 2 else (48, 40, 24)
    rng = np.random.default_rng(23)
    n = 150_001
    ix = np.stack([rng.integers(1, m + 1, n) for m in nx], 1).astype(np.int32)
    x = (rng.random((n, dims), np.float32) - np.float32(0.5)).astype(np.float32)
    u = (rng.standard_normal((n, 3)) * 0.5).astype(np.float32)
    ix[:pile] = 17
    x[:pile] = 0.0
    u[:pile] = (0.01, -0.02, 8.0)
    out = []
    for kernel in (0, 1):
        with oa.Simulation(dims, nx, (0.1,) * dims, 0.055, order, kernel=kernel) as sim:
            sid = sim.add_species(-1.0, pusher)
            sim.set_particles(sid, ix, x, u, np.full(n, -0.01, np.float32))
            sim.fill_fields(b0=(0.1, 0.0, 0.2))
            assert sim.raw_sums(sid) == (raw and kernel == 0)
            sim.run(3)
            assert sim.raw_sums(sid) == (raw and kernel == 0)
            out.append([a.view(np.uint32) for a in sim.get_fields() + sim.get_particles(sid)])
            hist = sim.history()
            if kernel == 0:
                first = hist
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    for a, b in zip(first, hist):  # FP64 sums, grouped by the kernels' waves
        assert np.allclose(a, b, rtol=1e-12, atol=0)
