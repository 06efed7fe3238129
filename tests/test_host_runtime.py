"""Host code of the library on a runtime that keeps "device" memory on the heap
and reports launches instead of running them (host_runtime.cpp): what a call
leaves behind when an allocation fails, which kernels it launches and how many,
and what memory stays with a graph.  CPU only; each test body runs in a child
process with that runtime preloaded, its launch hook standing in for the kernels
whose results the host reads."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes, struct, sys
import numpy as np
sys.path.insert(0, {root!r})
rt = ctypes.CDLL({rt!r})
rt.rt_live.restype = ctypes.c_size_t
rt.rt_fail_at.argtypes = [ctypes.c_long]
HOOK = ctypes.CFUNCTYPE(None, ctypes.c_char_p, ctypes.c_uint, ctypes.POINTER(ctypes.c_void_p))
launched = []   # kernel names of the launches so far
effects = {{}}    # substring of a kernel's name -> function(args)

@HOOK
def hook(name, grid, args):
    name = name.decode()
    launched.append(name)
    for key, f in effects.items():
        if key in name:
            f(args)

def count(key):
    return sum(key in x for x in launched)

def u64(p):
    return ctypes.c_uint64.from_address(p)

def u32(p):
    return ctypes.c_uint32.from_address(p)

rt.rt_hook(hook)
import olive_amd
from olive_amd import _lib
from olive_amd._lib import lib
olive_amd.init()

def graph(n, m, weighted=True, transpose=False):
    # edges spread over the vertices, all to vertex 0; no kernel looks at them here
    rp = (np.arange(n + 1, dtype=np.uint64) * m // n).astype(np.uint32)
    w = np.ones(m, np.int32) if weighted else None
    return olive_amd.Graph(olive_amd.CsrGraph(rp, np.zeros(m, np.uint32), w), transpose=transpose)

def weights_of_one(args):  # wstat_kernel: minimum and sum of the weights
    out, m = u64(args[2]).value, u32(args[1]).value
    u64(out).value, u64(out + 8).value = 1, m
effects["wstat_kernel"] = weights_of_one
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    rt = str(tmp_path_factory.mktemp("rt") / "libhostrt.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "host_runtime.cpp"), "-o", rt], check=True, timeout=120)

    def go(body):
        env = dict(os.environ)
        env["LD_PRELOAD"] = " ".join(x for x in (rt, env.get("LD_PRELOAD")) if x)
        code = PRELUDE.format(root=ROOT, rt=rt) + textwrap.dedent(body)
        r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
        return r.stdout

    return go


# The binned SSSP rounds: their launch arguments are read back as the kernels
# would (FusedArgs: base at byte 56, ctl at 80, nparts at 104; ctl: done first).
BINNED = """
n, m = 1_300_000, 40
def caps(args):   # ssspf_cap_kernel: all edges go from the first slice to itself
    u32(u64(args[6]).value).value = u32(args[3]).value * m
bases = []
def round_(args):
    a = args[0]
    base, ctl, nparts = u64(a + 56).value, u64(a + 80).value, u32(a + 104).value
    bases.append((u32(base).value, u32(base + 4).value, u32(base + 4 * nparts * nparts).value))
    u32(ctl).value = 1
effects["ssspf_cap_kernel"] = caps
effects["ssspf_round_kernel"] = round_
out = olive_amd.DeviceBuffer(n, np.int32)
def call(g, flags=0):
    return lib().olv_sssp(g.h, 0, None, out.c, flags, None)
"""


def test_failed_sssp_bins_are_not_kept(run):
    """Whichever allocation of a first binned call fails, the call says so and
    the next one builds the bins anew: its rounds get the region offsets."""
    run(BINNED + """
g = graph(n, m)
rt.rt_fail_at(0)
assert call(g) == 0 and bases and set(bases) == {(0, m, m)}
allocs = rt.rt_allocs()
assert allocs > 8
for i in range(1, allocs + 1):
    g = graph(n, m)
    live = rt.rt_live()
    rt.rt_fail_at(i)
    del bases[:]
    assert call(g) != 0 and not bases, i
    rt.rt_fail_at(0)
    assert call(g) == 0 and bases and set(bases) == {(0, m, m)}, (i, bases[:1])
    g.close()
""")


def test_failed_allocation_is_reported_once(run):
    """The runtime keeps a failed allocation as its last error until asked; the
    call that failed takes it along, so the next call's launches are not blamed."""
    run(BINNED + """
g = graph(3000, 40)
def done(args):   # SSSP by direct relaxation: the control block says done
    u32(u64(args[0] + 64).value).value = 1
effects["sssp_compact_kernel"] = done
rt.rt_fail_at(0)
assert call(g) == 0
for i in range(1, rt.rt_allocs() + 1):
    g = graph(3000, 40)
    rt.rt_fail_at(i)
    assert call(g) in (2, 3), i   # OLV_ENOMEM, OLV_EHIP
    rt.rt_fail_at(0)
    assert call(g) == 0, lib().olv_last_error()
""")


# BFS: a traversal of `depth` levels.  A narrow launch runs what is left of it,
# a launch pair one level (BfsCtl: done, skip, level, level_e, pairs, nlevels,
# levels).
BFS = """
FLAGS = _lib.OLV_GRAPH_ORDER | _lib.OLV_NO_DIRECTION_OPT
n = 20_000
depth = 300
def ctl_of(args, at):
    return u64(args[at]).value
def reset(args):
    for i in range(7):
        u32(ctl_of(args, 7) + 4 * i).value = 0
def finish(c):
    u32(c + 24).value, u32(c).value = depth, 1
def narrow(args):
    c = ctl_of(args, 1)
    if not u32(c).value:
        u32(c + 20).value += depth - u32(c + 8).value
        finish(c)
def compact(args):
    c = ctl_of(args, 1)
    if u32(c).value:
        return
    u32(c + 8).value += 1
    u32(c + 16).value += 1
    if u32(c + 8).value == depth:
        finish(c)
effects.update(bfs_reset_kernel=reset, bfs_narrow_kernel=narrow, bfs_compact_kernel=compact)
out = olive_amd.DeviceBuffer(n, np.int32)
def call(g, flags=0):
    del launched[:]
    assert lib().olv_bfs(g.h, 0, out.c, FLAGS | flags, None) == 0, lib().olv_last_error()
    return count("bfs_compact"), count("bfs_narrow")
"""


@pytest.mark.parametrize("flags", [0, 0x8, 0x4])  # OLV_HOST_LOOP, OLV_FORCE_BOTTOM_UP
def test_history_leads_to_the_narrow_kernel(run, flags):
    """Whatever kind of call comes first on a graph of many small levels, plain
    calls run it in the narrow kernel, and enqueue no pairs for the others."""
    run(BFS + f"flags = {flags}" + """
if flags & _lib.OLV_FORCE_BOTTOM_UP:
    FLAGS = _lib.OLV_GRAPH_ORDER
g = graph(n, 40, weighted=False, transpose=True)
for _ in range(2):
    if flags:
        pairs, launches = call(g, flags)
        assert pairs >= depth and launches == 0
    for _ in range(3):
        pairs, launches = call(g)
        assert pairs <= 12 and launches, (pairs, launches)
# levels too wide for the narrow kernel, then the first again
effects["bfs_narrow_kernel"] = lambda args: None
for _ in range(5):
    call(g)
pairs, launches = call(g)
assert pairs == depth and launches   # no surplus
effects["bfs_narrow_kernel"] = narrow
for _ in range(5):
    call(g)
assert call(g)[0] <= 4
""")


def test_batched_groups_of_unlike_depth(run):
    """Groups of a batched BFS whose depths differ by a few levels: no group
    enqueues many launches past its end (MbfsParams: k at byte 44, ctl at 184;
    MbfsCtl: level, -, done, levels)."""
    run("""
depth = {256: 130, 44: 128}
def reset(args):
    c = u64(args[0] + 184).value
    for i in range(4):
        u32(c + 4 * i).value = 0
def compact(args):
    c, d = u64(args[0] + 184).value, depth[u32(args[0] + 44).value]
    if u32(c + 8).value:
        return
    u32(c).value += 1
    if u32(c).value == d:
        u32(c + 12).value, u32(c + 8).value = d, 1
effects.update(mbfs_reset_kernel=reset, mbfs_compact_kernel=compact)
n = 500
g = graph(n, 40, weighted=False, transpose=True)
srcs = np.zeros(300, np.uint32)
out = olive_amd.DeviceBuffer(300 * n, np.int32)
for i in range(4):
    del launched[:]
    assert lib().olv_bfs_batched(g.h, srcs.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)), 300, out.c,
                                 _lib.OLV_GRAPH_ORDER | _lib.OLV_NO_DIRECTION_OPT, None) == 0, lib().olv_last_error()
    if i:
        assert 258 <= count("mbfs_compact") <= 258 + 20, (i, count("mbfs_compact"))
""")


def test_sssp_work_kept(run):
    """Directly relaxed SSSP keeps its work for calls of as many sources or
    fewer, and only up to 4 GiB (SsspParams: ctl at byte 64)."""
    run("""
def done(args):
    u32(u64(args[0] + 64).value).value = 1
effects["sssp_compact_kernel"] = done
def call(g, k, out):
    srcs = np.zeros(k, np.uint32)
    rt.rt_fail_at(0)
    assert lib().olv_sssp_batched(g.h, srcs.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)), k, None, out.c,
                                  _lib.OLV_SSSP_DIRECT, None) == 0, lib().olv_last_error()
    return rt.rt_allocs()
g = graph(50_000, 40)
out = olive_amd.DeviceBuffer(64 * g.n, np.int32)
for k in (64, 1, 5):   # without candidate copies and with them
    call(g, k, out)
for k in (5, 64, 3, 1, 17):
    assert call(g, k, out) <= 1, (k, rt.rt_allocs())   # the copy of the sources
g = graph(9_000_000, 40)
out = olive_amd.DeviceBuffer(100 * g.n, np.int32)
call(g, 1, out)
live = rt.rt_live()
call(g, 100, out)   # 4.5 GB of queue and marks
assert rt.rt_live() < live + (1 << 20)
""")


@pytest.mark.parametrize("n,m,k,binned", [
    (1000, 5000, 899, 0), (1000, 5000, 900, 1), (1000, 5001, 900, 0),  # 900K vertices of at most 5 edges
    (1000, 6000, 1249, 0), (1000, 6000, 1250, 1),                      # 1.25M of any
    (1 << 24, 40, 1, 1), ((1 << 24) + 1, 40, 1, 0),                    # 1024 slices of 16K
    (1000, 6000, 20_000, 2)])                                          # 20M: in groups of as many as fit
def test_sssp_route(run, n, m, k, binned):
    """Graphs without hubs that go through the binned rounds."""
    run(f"n, m, k, binned = {n}, {m}, {k}, {binned}" + """
groups = []
def caps(args):   # (k at 3)
    groups.append(u32(args[3]).value)
    u32(u64(args[6]).value).value = u32(args[3]).value * m
def round_(args):
    u32(u64(args[0] + 80).value).value = 1
def done(args):
    u32(u64(args[0] + 64).value).value = 1
effects.update(ssspf_cap_kernel=caps, ssspf_round_kernel=round_, sssp_compact_kernel=done)
g = graph(n, m)
out = olive_amd.DeviceBuffer(k * n, np.int32)
srcs = np.zeros(k, np.uint32)
assert lib().olv_sssp_batched(g.h, srcs.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)), k, None, out.c, 0, None) == 0
assert len(groups) == binned and bool(count("ssspf_round")) == bool(binned), groups
assert bool(count("sssp_relax")) == (not binned)
assert not groups or sum(groups) == k
""")
