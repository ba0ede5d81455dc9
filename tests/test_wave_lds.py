"""LDS that the lanes of one wave exchange without a barrier (the queues of face-crossing
particles, the ranks of the in-tile re-order) is ordered by wave_lds_sync in
osiris_amd/csrc/osr_device.hpp: each lane is a thread of its own to the compiler, which may
otherwise let a value that a lane has read stand for a second read after another lane's
store.  Which code the compiler makes today cannot show that, so this reads the sources."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "osiris_amd", "csrc")


def _src(name):
    txt = open(os.path.join(CSRC, name)).read()
    return re.sub(r"//[^\n]*", "", txt)


def test_wave_lds_sync_orders_both_ways():
    body = re.search(r"void wave_lds_sync\(\) \{(.*?)\n\}", _src("osr_device.hpp"), re.S).group(1)
    steps = [s.strip() for s in body.split(";") if s.strip()]
    assert [re.match(r"(\w+)", s).group(1) for s in steps] == [
        "__builtin_amdgcn_fence", "__builtin_amdgcn_wave_barrier", "__builtin_amdgcn_fence"]
    assert "__ATOMIC_RELEASE" in steps[0] and "__ATOMIC_ACQUIRE" in steps[2]


def test_queue_reads_lie_between_two_syncs():
    for name in ("k_push2d.hip", "k_push3d.hip"):
        txt = _src(name)
        reads = [m.start() for m in re.finditer(r"Q[01]\[lane\]", txt)]
        between = [m.span(1) for m in re.finditer(r"wave_lds_sync\(\);(\s*const f32x4 [^;]*;\s*)wave_lds_sync\(\);", txt)]
        assert reads, name
        for r in reads:
            assert any(a <= r < b for a, b in between), f"{name}: queue read without wave_lds_sync around it"


def test_generic_queue_and_reorder_are_ordered():
    txt = _src("k_tiles.hip")
    body = re.search(r"deposit_queue = \[&\]\(int head, int cnt\) \{(.*?)\n  \};", txt, re.S).group(1).strip()
    assert body.startswith("wave_lds_sync();") and body.endswith("wave_lds_sync();")
    update = txt.index("s_cnt[wave][lc] += before + 1")
    assert re.search(r"wave_lds_sync\(\);[^;]*$", txt[:update])
    assert re.match(r"[^;]*;\s*wave_lds_sync\(\);", txt[update:])


def test_no_bare_wave_barrier():
    for f in sorted(os.listdir(CSRC)):
        if f != "osr_device.hpp":
            assert "__builtin_amdgcn_wave_barrier" not in _src(f), f
