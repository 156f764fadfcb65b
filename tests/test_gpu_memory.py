"""Graphs and handles where device memory is short: the library's device
allocations go through a stand-in that keeps a budget, in a process of its own,
so nothing but the budget runs out.  Needs an MI355X."""
import shutil
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

BUDGET = r"""
#include <dlfcn.h>
#include <stddef.h>

/* hipMalloc and hipFree with a budget of live bytes (2 = hipErrorOutOfMemory) */
enum { N = 4096 };
static void *at[N];
static size_t size[N], live, limit = (size_t)-1;
static int (*real_malloc)(void **, size_t), (*real_free)(void *);

int budget_init(const char *hip) {
  void *h = dlopen(hip, RTLD_LAZY);
  if (!h) return 1;
  real_malloc = (int (*)(void **, size_t))dlsym(h, "hipMalloc");
  real_free = (int (*)(void *))dlsym(h, "hipFree");
  return !real_malloc || !real_free;
}
size_t budget_live(void) { return live; }
void budget_limit(size_t n) { limit = n; }

int hipMalloc(void **p, size_t n) {
  int i = 0, r;
  if (n > limit - live) return 2;
  while (i < N && at[i]) ++i;
  if (i == N || (r = real_malloc(p, n)) != 0) return 2;
  at[i] = *p;
  size[i] = n;
  live += n;
  return 0;
}
int hipFree(void *p) {
  for (int i = 0; p && i < N; ++i)
    if (at[i] == p) {
      at[i] = 0;
      live -= size[i];
    }
  return real_free(p);
}
"""

CHILD = r"""
import ctypes
import sys

budget = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
budget.budget_live.restype = ctypes.c_size_t
budget.budget_limit.argtypes = [ctypes.c_size_t]
import numpy as np

import ibfs_amd
import oracle
from test_gpu_levels import _degrees_graph

ibfs_amd._lib.lib()
hip = [l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l][0]
assert budget.budget_init(hip.encode()) == 0
FREE = (1 << 64) - 1


def say(*a):
    print("[gpu]", *a, file=sys.stderr, flush=True)


def nomem(make):
    try:
        make()
    except ibfs_amd.IbfsError as e:
        return e.code == ibfs_amd._lib.IBFS_ERR_NOMEM
    return False


def live():
    return budget.budget_live()


V = int(sys.argv[2])
beg, adj = _degrees_graph(V, seed=V)
host = ibfs_amd.HostCsr.from_arrays(beg, adj)
src = np.random.default_rng(1).integers(0, V, size=130).astype(np.int32)
want = oracle.bfs_many(beg, adj, src, threads=8)
vt = int(np.count_nonzero(np.diff(beg)))
heads = 32 * vt

for hubs in (None, 0, 16):
    base = live()
    g = ibfs_amd.DeviceGraph(host, hub_count=hubs)
    full = live() - base
    g.close()
    assert live() == base
    say(f"graph of V={V} hubs={hubs} within {full - heads} of {full} bytes")
    budget.budget_limit(base + full - heads)
    g = ibfs_amd.DeviceGraph(host, hub_count=hubs)
    assert live() == base + full - heads
    budget.budget_limit(FREE)
    for lanes in (64, 128, 256, 512):
        for pol in (ibfs_amd.POLICY_BU_ONLY, ibfs_amd.POLICY_HYBRID, ibfs_amd.POLICY_ALPHA_BETA):
            say(f"no heads, lanes={lanes} policy={pol}")
            for timing in (0, 1):
                e = ibfs_amd.Engine(g, lane_bits=lanes, policy=pol, hybrid_hubs=40, kernel_timing=timing)
                np.testing.assert_array_equal(e.run_groups(src), want)
                e.close()
            b = ibfs_amd.Batch(g, lane_bits=lanes, policy=pol, hybrid_hubs=40, split_cov=50)
            np.testing.assert_array_equal(b.run(src), want)
            b.close()
    s = ibfs_amd.Server(g, lane_bits=128)
    out = ibfs_amd.DeviceBuffer(4 * 128 * V)
    s.wait(s.submit(src[:128], out))
    np.testing.assert_array_equal(out.to_host().reshape(128, V), want[:128])
    s.close()
    g.traversal_noalloc(src[:128], out, ibfs_amd.default_config(policy=ibfs_amd.POLICY_BU_ONLY))
    np.testing.assert_array_equal(out.to_host().reshape(128, V), want[:128])
    out.free()
    g.close()

for name, make, run in (
        ("engine", lambda g: ibfs_amd.Engine(g), lambda e: e.run_groups(src)),
        ("batch", lambda g: ibfs_amd.Batch(g, contexts=2, burst=4), lambda b: b.run(src)),
        ("server", lambda g: ibfs_amd.Server(g, lane_bits=64), None)):
    say(f"heads given up for a first {name}, kept for a second")
    g = ibfs_amd.DeviceGraph(host)
    base = live()
    h = make(g)
    need = live() - base
    h.close()
    assert live() == base
    budget.budget_limit(base + need - heads)
    h = make(g)
    assert live() == base + need - heads
    budget.budget_limit(FREE)
    if run:
        np.testing.assert_array_equal(run(h), want)
    h.close()
    g.close()
    g = ibfs_amd.DeviceGraph(host)
    e = ibfs_amd.Engine(g)
    budget.budget_limit(live() + need - heads)
    assert nomem(lambda: make(g))
    budget.budget_limit(FREE)
    np.testing.assert_array_equal(e.run_groups(src), want)
    e.close()
    g.close()

say("heads given up for the rows of a host output")
g = ibfs_amd.DeviceGraph(host)
e = ibfs_amd.Engine(g, policy=ibfs_amd.POLICY_BU_ONLY)
budget.budget_limit(live() + 4 * V * 128 - heads)
np.testing.assert_array_equal(e.traversal(src[:128]), want[:128])
print("done")
"""


@pytest.mark.gpu
@pytest.mark.skipif(shutil.which("gcc") is None, reason="no host compiler")
@pytest.mark.parametrize("V", [513, 70_001])
def test_graphs_and_handles_without_memory_for_list_heads(tmp_path, V):
    """The heads of the adjacency lists (32 bytes per vertex) take no memory that
    a graph, an engine, a batch or a server of the graph cannot do without, and
    every form is exact without them."""
    lib = tmp_path / "libbudget.so"
    (tmp_path / "budget.c").write_text(BUDGET)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", str(tmp_path / "budget.c"), "-o", str(lib),
                    "-ldl"], check=True)
    r = subprocess.run([sys.executable, "-c", f"import sys; sys.path[:0] = {[str(ROOT), str(ROOT / 'tests')]!r}\n"
                        + CHILD, str(lib), str(V)], stdout=subprocess.PIPE, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.strip().endswith("done")
