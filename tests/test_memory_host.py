"""The library's use of device memory and the size of its push launches on the CPU, over the mock
runtime of tests/hostcheck with a device memory that fills up (capi_mock_mem.hip)."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HC = os.path.join(ROOT, "tests", "hostcheck")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def mem_lib():
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    out = os.path.join(HC, "_build", "libosiris_hostcheck_mem.so")
    os.makedirs(os.path.dirname(out), exist_ok=True)
    csrc = os.path.join(ROOT, "osiris_amd", "csrc")
    srcs = [os.path.join(HC, f) for f in os.listdir(HC) if f.endswith((".h", ".hip"))] + [
        os.path.join(csrc, f) for f in os.listdir(csrc)]
    if not os.path.exists(out) or os.path.getmtime(out) < max(os.path.getmtime(s) for s in srcs):
        # host code only: the device code, which the mock never runs, is named but not there
        tmp = f"{out}.{os.getpid()}.tmp"
        subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-O1", "-w", "-std=c++17",
                        "-fPIC", "-I", os.path.join(ROOT, "include"), "-c", "-o", tmp + ".o",
                        os.path.join(HC, "capi_mock_mem.hip")], check=True)
        syms = subprocess.run(["nm", "-u", tmp + ".o"], check=True, capture_output=True, text=True).stdout
        subprocess.run([HIPCC, "-shared", "-rdynamic", "-o", tmp, tmp + ".o"] + [
            f"-Wl,--defsym={s}=0" for s in syms.split() if s.startswith("__hip_fatbin")], check=True)
        os.remove(tmp + ".o")
        os.replace(tmp, out)
    return out


PRELUDE = """
import ctypes as C, json, sys
sys.path.insert(0, {root!r})
import numpy as np
import osiris_amd._lib as L
L.LIB_PATH = {lib!r}
L.lib()
raw = C.CDLL({lib!r})
for f in ("mock_errors", "mock_order_errors", "mock_live"):
    getattr(raw, f).restype = C.c_longlong
raw.mock_leave_free.argtypes = [C.c_longlong]
from osiris_amd.sim import Simulation
out = {{}}
"""


def _run(lib, body):
    """Result of `body` (which fills the dict `out`) in a process of its own."""
    code = PRELUDE.format(root=ROOT, lib=lib) + body + """
out["errors"] = raw.mock_errors() + raw.mock_order_errors()
out["live"] = raw.mock_live()
print(json.dumps(out))
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    res = json.loads(r.stdout.strip().splitlines()[-1])
    assert res.pop("errors") == 0 and res.pop("live") == 0, r.stderr[-3000:]
    return res


@pytest.mark.parametrize("dims,nx", [(2, (150, 110)), (3, (40, 30, 20))])
def test_read_back_without_device_memory(mem_lib, dims, nx):
    """Fields and particles come back when the device has no memory left for laying them out."""
    res = _run(mem_lib, f"""
dims, nx = {dims}, {nx}
rng = np.random.default_rng(4)
n = 20000
ix = np.stack([rng.integers(1, m + 1, n) for m in nx], 1).astype(np.int32)
x = (rng.random((n, dims), np.float32) - np.float32(0.5)).astype(np.float32)
u = rng.standard_normal((n, 3)).astype(np.float32)
q = (-rng.random(n)).astype(np.float32)
e, b = (rng.standard_normal(tuple(reversed(nx)) + (3,)).astype(np.float32) for _ in range(2))
with Simulation(dims, nx, (0.1,) * dims, 0.05, 2) as s:
    sid = s.add_species(-1.0)
    s.set_particles(sid, ix, x, u, q)
    s.set_fields(e, b)
    raw.mock_leave_free(0)
    out["particles"] = all(np.array_equal(a, c) for a, c in zip(s.get_particles(sid), (ix, x, u, q)))
    lo, up = [3, 1, 2][:dims], [2, 4, 1][:dims]
    pad = [(l, h) for l, h in zip(reversed(lo), reversed(up))] + [(0, 0)]
    out["fields"] = all(np.array_equal(a, np.pad(c, pad, "wrap")) for a, c in zip(s.get_fields(lo, up), (e, b)))
    raw.mock_leave_free(-1)
""")
    assert res == {"particles": True, "fields": True}


@pytest.mark.parametrize("nx,tile,nsp,ppc,split", [
    ((128, 128), (16, 16), 1, (4, 4), 4), ((256, 128), (16, 16), 1, (1, 1), 1), ((128, 128), (16, 16), 1, (2, 2), 4),
    ((256, 128), (16, 16), 8, (2, 2), 1), ((128, 128), (16, 16), 8, (4, 4), 1), ((256, 128), (16, 16), 1, (2, 2), 2),
    ((256, 192), (16, 16), 2, (4, 4), 2), ((256, 192), (16, 16), 1, (2, 2), 1), ((512, 256), (16, 16), 1, (4, 4), 1),
    ((256, 256), (32, 16), 1, (4, 4), 2), ((512, 256), (32, 16), 1, (4, 4), 1), ((640, 512), (32, 16), 2, (2, 2), 1)])
def test_push_workgroups_per_tile(mem_lib, nx, tile, nsp, ppc, split):
    """A push launch has several workgroups per tile where the tiles of all its species leave the
    chip idle and each wave still has iterations to share, and one elsewhere.  The points are
    measured ones: in each the number expected here was the fastest."""
    res = _run(mem_lib, f"""
with Simulation(2, {nx}, (0.1, 0.1), 0.05, 2, tile={tile}) as s:
    for k in range({nsp}):
        s.generate(s.add_species(-1.0), {ppc})
    s.run(1)
    out["wgs"] = raw.mock_push_workgroups()
""")
    tiles = -(-nx[0] // tile[0]) * -(-nx[1] // tile[1])
    assert res["wgs"] == tiles * nsp * split


def test_split_follows_the_particles(mem_lib):
    """The number of workgroups is chosen again when species or their particles change, also
    between runs; every tile table holds the largest number."""
    res = _run(mem_lib, """
out["wgs"] = []
with Simulation(2, (256, 128), (0.1, 0.1), 0.05, 2) as s:
    s.generate(s.add_species(-1.0), (1, 1))
    s.run(2)
    out["wgs"].append(raw.mock_push_workgroups())
    s.generate(0, (4, 4))
    s.time_kernels(1)
    out["wgs"].append(raw.mock_push_workgroups())
    s.run(3)
    for k in range(7):
        s.generate(s.add_species(1.0), (4, 4))
    s.run(3)
    out["wgs"].append(raw.mock_push_workgroups())
    s.get_particles(3)
""")
    assert res == {"wgs": [128, 512, 8 * 128]}


def test_one_copy_of_the_fields_where_two_do_not_fit(mem_lib):
    """A 2D grid whose fields and current fit the card once, but not twice, is simulated on one
    copy, and read back; with room for both it takes both."""
    res = _run(mem_lib, """
nx = (400, 350)
one = 48 * nx[0] * nx[1]
for name, free in (("one", one + one // 2), ("two", 3 * one)):
    raw.mock_leave_free(free)
    with Simulation(2, nx, (0.1, 0.1), 0.05, 2) as s:
        out[name] = s.footprint // one
        raw.mock_leave_free(-1)
        s.generate(s.add_species(-1.0), (1, 1))
        e = np.arange(3 * nx[0] * nx[1], dtype=np.float32).reshape(nx[1], nx[0], 3)
        s.set_fields(e, -e)
        raw.mock_leave_free(0)
        f = s.get_fields()
        raw.mock_leave_free(-1)
        out[name + " fields"] = bool(np.array_equal(f[0], e) and np.array_equal(f[1], -e))
        s.run(9)
        s.time_kernels(2)
        out[name + " steps"] = s.steps
""")
    assert res == {"one": 1, "one fields": True, "one steps": 11, "two": 2, "two fields": True, "two steps": 11}


@pytest.mark.parametrize("dims,order,tile,kernel", [
    (2, 2, (16, 16), 0), (2, 1, (32, 16), 0), (2, 3, (8, 8), 0), (2, 2, (16, 16), 1), (2, 2, (10, 10), 0),
    (3, 1, (8, 8, 4), 0), (3, 2, (8, 8, 4), 0), (3, 3, (8, 8, 4), 0), (3, 2, (8, 8, 4), 1), (3, 1, (4, 4, 4), 0)])
def test_reported_launch_configuration_is_accepted(mem_lib, dims, order, tile, kernel):
    """The waves that launch_config reports can be asked for and give the same configuration; in
    3D so can 4; another number than 4 and 8 or than the kernel's is refused."""
    res = _run(mem_lib, f"""
kw = dict(tile={tile}, kernel={kernel})
mk = lambda w: Simulation({dims}, (32,) * {dims}, (0.1,) * {dims}, 0.05, {order}, push_waves=w, **kw)
with mk(0) as s:
    cfg = s.launch_config
with mk(cfg["push_waves"]) as s:
    out["same"] = s.launch_config == cfg
for w in (2, 4, 8):
    try:
        with mk(w) as s:
            out[str(w)] = s.push_waves
    except L.OsrError:
        out[str(w)] = 0
out["own"] = cfg["push_waves"]
""")
    own = res["own"]
    assert res["same"] and res["2"] == 0
    either = dims == 2 and kernel == 0 and tile in ((16, 16), (32, 16))
    assert res["4"] == (4 if own == 4 or either else own if dims == 3 else 0)
    assert res["8"] == (8 if own == 8 or either else 0)


@pytest.mark.parametrize("dims,nx,buffers", [(2, (300, 250), 1), (3, (40, 36, 30), 2)])
def test_smoothing_buffers(mem_lib, dims, nx, buffers):
    """Smoothing in 2D takes one float copy of the current, in 3D two; a call that finds no room
    for them leaves the next one to try again."""
    res = _run(mem_lib, f"""
from osiris_amd.sim import smooth_setup
dims, nx = {dims}, {nx}
one = 12 * int(np.prod(nx))
filt = smooth_setup(dims, ["binomial"] * dims, (1,) * dims, (0.1,) * dims)
with Simulation(dims, nx, (0.1,) * dims, 0.05, 2) as s:
    s.generate(s.add_species(-1.0), (1,) * dims)
    out["fails"] = 0
    for room in (0, one + one // 2):
        raw.mock_leave_free(room)
        try:
            s.set_smooth(*filt)
        except L.OsrError:
            out["fails"] += 1
    raw.mock_leave_free(-1)
    s.set_smooth(*filt)
    s.run(5)
    out["steps"] = s.steps
""")
    assert res == {"fails": buffers, "steps": 5}
