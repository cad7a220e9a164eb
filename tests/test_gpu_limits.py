"""What the library does when an allocation fails.  Each case runs in a child
process that loads limits.c ahead of the library, so that HIP's memory calls
end with out-of-memory where the case says; nothing is exhausted."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

HEAD = """
import ctypes, sys, threading
sys.path.insert(0, {root!r})
lim = ctypes.CDLL({lib!r}, ctypes.RTLD_GLOBAL)
lim.limits_used.restype = lim.limits_peak.restype = lim.limits_pins.restype = ctypes.c_size_t
lim.limits_set.argtypes = [ctypes.c_size_t, ctypes.c_size_t]
NONE = 2**64 - 1
import numpy as np
import beedrill_amd as bd
import oracle as orc

def searched(c):
    off, adj = c.csr()
    root = int(c.pick_roots(1)[0])
    c.bfs(root)
    depth, parent = c.fetch()
    np.testing.assert_array_equal(depth, orc.bfs_depth(off, adj, root))
    assert orc.check(off, adj, root, parent)
"""


@pytest.fixture(scope="module")
def limited(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("limits") / "limits.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", lib, os.path.join(HERE, "limits.c"),
                    "-ldl", "-lpthread"], check=True)

    def run(code):
        r = subprocess.run([sys.executable, "-c", HEAD.format(root=ROOT, lib=lib) + code],
                           capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout
    return run


def test_memory_kept_by_another_context(limited):
    """What a context keeps of its freed blocks goes back when another's
    allocation fails, and what it has in use stays."""
    limited("""
c = bd.Context(0)
before = lim.limits_used()
assert before > 0  # the calls go through the limits
lim.limits_peak()
c.generate_er(300000, 1500000, seed=2)
need = lim.limits_peak() - before
c.close()
a, b = bd.Context(0), bd.Context(0)
a.generate_er(1000000, 4000000, seed=1)
held = lim.limits_used()
a.generate_er(1000, 4000, seed=1)
a.components()
used = lim.limits_used()
assert used - before > need  # most of it kept
lim.limits_set(used + need // 4, NONE)
b.generate_er(300000, 1500000, seed=2)
searched(b)
searched(a)
assert a.component_labels().size == 1000
lim.limits_set(lim.limits_used(), NONE)
try:
    b.generate_er(3000000, 15000000, seed=2)
    raise SystemExit("over the limit")
except bd.BeedrillError as e:
    assert e.code == -2, e
lim.limits_set(NONE, NONE)
b.generate_er(1000, 3000, seed=2)
searched(b)
searched(a)
print("done")
""")


def test_memory_kept_by_contexts_of_several_threads(limited):
    """Contexts of three threads build and search graphs under a limit that
    holds what they have in use, but not what they keep as well."""
    limited("""
c = bd.Context(0)
before = lim.limits_used()
lim.limits_peak()
c.generate_er(200000, 1000000, seed=2)
need = lim.limits_peak() - before
c.close()
lim.limits_set(lim.limits_used() + 4 * need, NONE)
bad = []
def work(k):
    try:
        with bd.Context(0) as x:
            for i in range(6):
                x.generate_er(200000 // (1 + (i + k) % 3), 1000000 // (1 + (i + k) % 3), seed=i)
                searched(x)
    except BaseException as e:
        bad.append(e)
        raise
ts = [threading.Thread(target=work, args=(k,)) for k in range(3)]
[t.start() for t in ts]
[t.join() for t in ts]
assert not bad, bad
print("done")
""")


def test_results_where_nothing_can_be_pinned(limited):
    """Results and small inputs then go by plain copies: chunks of every form
    (bytes, ints, ids; short and in several pieces), batches, components and
    training; and again through pinned memory once there is some."""
    limited("""
def everything(c, deep):
    for nv, m in ((700, 3000), (300000, 900000), (1100003, 2500000)):
        c.generate_er(nv, m, seed=nv & 7)
        searched(c)
        off, adj = c.csr()
        r = c.components()
        labels, n, _ = orc.components(off, adj)
        assert r["num_components"] == n
        np.testing.assert_array_equal(c.component_labels(), labels)
        roots = [int(v) for v in c.pick_roots(3)]
        np.testing.assert_array_equal(c.multi_root(roots)[0],
                                      [orc.bfs_depth(off, adj, v) for v in roots])
    s = np.arange(deep - 1)
    c.from_edges(deep, s, s + 1)
    searched(c)  # past 250 levels: depths as ints
    depth, _ = c.multi_graph([0, deep], [0])
    np.testing.assert_array_equal(depth, np.arange(deep))
    rng = np.random.default_rng(1)
    x, t = rng.random((500, 8), np.float32), rng.random((500, 2), np.float32)
    p = rng.standard_normal(32 * 8 + 32 + 32 * 32 + 32 + 64 + 2).astype(np.float32) / 8
    c.mlp_set(p, 32, 32)
    loss = c.mlp_train(x, t, epochs=5, lr=3e-3)
    return loss, c.mlp_get()[0], c.mlp_infer(x, mfma=False), c.mlp_infer(x), c.mlp_loss_grad(x, t)[1]

free = bd.Context(0)
want = everything(free, 700)
c = bd.Context(0)
lim.limits_set(NONE, 0)
got = [everything(c, 700), everything(c, 700)]
lim.limits_set(NONE, NONE)
c.generate_er(2000, 9000, seed=1)
searched(c)  # a small ring
lim.limits_set(NONE, 0)
got.append(everything(c, 400000 // 1000))
lim.limits_set(NONE, NONE)
got.append(everything(c, 300))
for g in got:
    for a, b in zip(g, want):
        np.testing.assert_array_equal(a, b)
print("done")
""")


def test_a_context_pins_memory_once(limited):
    limited("""
for k in range(3):
    c = bd.Context(0)
    assert lim.limits_pins() == k + 1
    c.close()
""")
