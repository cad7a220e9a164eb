"""GPU parity for connected components (components.cc): the device labels,
called through the C ABI, equal the oracle's (each component labelled by its
smallest vertex id, whatever the pass order), with the same component count,
and the check passes."""
import os
import subprocess

import numpy as np
import pytest

from conftest import complete_graph, path_graph, star_graph, two_components

pytestmark = pytest.mark.gpu


def compare(ctx, orc, off, adj):
    st = ctx.components()
    lab = ctx.component_labels()
    ref, n, _ = orc.components(off, adj)
    np.testing.assert_array_equal(lab, ref)
    assert st["num_components"] == n
    assert st["num_iters"] >= 1 and st["ms"] > 0
    assert 0 < st["pass_ms"] <= st["ms"]
    # the first pass takes neighbour ids, later pulls read every label and
    # pushes the changed vertices' labels only
    nnz, nv = int(off[-1]), len(off) - 1
    assert 0 <= st["labels_read"] <= (st["num_iters"] - 1) * nnz
    assert st["edge_bytes"] >= 4 * nnz + 12 * nv + 8 * st["labels_read"]
    assert st["num_iters"] <= st["pass_launches"] <= 9 * st["num_iters"]
    assert ctx.components_check()
    return st


@pytest.mark.parametrize("g", [path_graph(300), star_graph(100), complete_graph(30),
                               two_components()])
def test_small_graphs(ctx, orc, g):
    nv, s, d = g
    ctx.from_edges(nv, s, d)
    off, adj = orc.build_csr(nv, s, d)
    compare(ctx, orc, off, adj)


def test_isolated_vertices_and_self_loops(ctx, orc):
    nv = 10
    s = np.array([2, 3, 7], np.int64)
    d = np.array([3, 4, 7], np.int64)
    ctx.from_edges(nv, s, d)
    off, adj = orc.build_csr(nv, s, d)
    compare(ctx, orc, off, adj)
    assert ctx.component_labels().tolist() == [0, 1, 2, 2, 2, 5, 6, 7, 8, 9]


def test_long_path_under_relabelling(ctx, orc):
    # one component whose smallest id sits in the middle of a 20000-vertex
    # path: labels travel both ways through the id space
    n = 20000
    perm = np.random.default_rng(3).permutation(n).astype(np.int64)
    ctx.from_edges(n, perm[:-1], perm[1:])
    off, adj = orc.build_csr(n, perm[:-1], perm[1:])
    st = compare(ctx, orc, off, adj)
    assert st["num_components"] == 1


@pytest.mark.parametrize("scale,ef,seed", [(16, 16, 0), (14, 2, 5), (12, 1, 9)])
def test_rmat(ctx, orc, scale, ef, seed):
    ctx.generate_rmat(scale, ef, seed=seed)
    off, adj = ctx.csr()
    compare(ctx, orc, off, adj)


def test_long_lists_and_slices(ctx, orc):
    # lists of 255 and 256 edges (either side of the long-list cut), hubs of
    # several 2048-edge slices, long and short lists in one 64-vertex group,
    # and a group whose vertices all have long lists
    rng = np.random.default_rng(11)
    nv = 40000
    src, dst = [], []
    for hub, deg in [(5, 255), (6, 256), (7, 257), (70, 5000), (71, 2048), (72, 2049),
                     (20000, 9000)] + [(128 + i, 300 + i) for i in range(64)]:
        nb = rng.choice(np.arange(30000, nv), deg, replace=False)
        src.append(np.full(deg, hub)); dst.append(nb)
    a = rng.integers(1000, 30000, 6000)
    src.append(a); dst.append(a + 1)  # short lists elsewhere
    s = np.concatenate(src).astype(np.int64)
    d = np.concatenate(dst).astype(np.int64)
    ctx.from_edges(nv, s, d)
    off, adj = orc.build_csr(nv, s, d)
    compare(ctx, orc, off, adj)
    compare(ctx, orc, off, adj)  # second run reuses the slices


def test_er_and_lattice(ctx, orc):
    ctx.generate_er(20000, 12000, seed=4)
    off, adj = ctx.csr()
    st = compare(ctx, orc, off, adj)
    assert st["num_components"] > 100
    ctx.generate_lattice(60, 70, seed=1)
    off, adj = ctx.csr()
    compare(ctx, orc, off, adj)


def test_cli_components_check():
    exe = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                       "beedrill_amd", "bin", "components")
    r = subprocess.run([exe, "--generate", "graph500-scale12", "--num_trials", "2",
                        "--check_results"], capture_output=True, text=True, timeout=120)
    out = r.stdout + r.stderr
    assert r.returncode == 0, out
    assert out.count("Found ") == 2 and "PASS" in out and "FAIL" not in out, out


@pytest.mark.parametrize("order", [2, 4])
def test_passes_that_skip_the_largest_label(ctx, orc, order):
    """From the second pass on, vertices carrying the label of the vertex of
    largest degree read nothing: components whose smallest ids lie on either
    side of that label, joined to it through short lists, through lists cut
    into slices, and through chains that need several passes, with components
    and isolated vertices it never meets; twice, to reuse the slices."""
    rng = np.random.default_rng(17)
    nv, hub = 60000, 30000
    near = rng.choice(np.arange(20000, 50000), 9000, replace=False)
    near = near[near != hub]
    src = [np.full(len(near), hub)]
    dst = [near]
    # a long list below the hub's labels, touching the hub's set at its end
    src.append(np.full(3000, 7))
    dst.append(np.concatenate([np.arange(100, 3099), near[:1]]))
    # chains that start low, wander through high ids, and end at the hub's set
    for k in range(8):
        chain = np.concatenate([[10 + k], rng.choice(np.arange(50000, 59000), 120, replace=False),
                                near[10 + k:11 + k]])
        src.append(chain[:-1])
        dst.append(chain[1:])
    # components of their own, below and above the hub
    src.append(np.arange(4000, 5000)); dst.append(np.arange(4001, 5001))
    src.append(np.arange(59100, 59900)); dst.append(np.arange(59101, 59901))
    s, d = np.concatenate(src).astype(np.int64), np.concatenate(dst).astype(np.int64)
    t0 = ctx.get_tuning()
    try:
        ctx.set_tuning(vertex_order=order)
        ctx.from_edges(nv, s, d)
        off, adj = orc.build_csr(nv, s, d)
        for _ in range(2):
            st = compare(ctx, orc, off, adj)
        assert st["num_components"] > 1000
    finally:
        ctx.set_tuning(**t0)


@pytest.mark.parametrize("degrees", [(0, 1, 2, 63, 64, 65), (254, 255, 256, 257, 0), (255,) * 64,
                                     (1,) * 63 + (300,), (0,) * 63 + (5,), (300, 0, 1)])
def test_first_pass_over_lists_of_every_length(ctx, orc, degrees):
    """Consecutive lists of these lengths (up to 255 entries a wave takes them
    together, 64 entries at a time), every vertex beside its component's
    smallest one: the first pass finds all labels and the second changes none."""
    r = np.random.default_rng(len(degrees))
    n, base = 64 * 9 + 13, 1400
    src, dst = [], []
    for v in range(n):  # vertex base + v: its component's smallest vertex, then others of it
        d = degrees[v % len(degrees)]
        if d == 0:
            continue
        k = v % 3
        src.append(np.full(d, base + v))
        others = base + n + k * 400 + r.permutation(400)[:d - 1]
        dst.append(r.permutation(np.append(others, k)))
    src, dst = np.concatenate(src), np.concatenate(dst)
    nv = base + n + 1200
    used = np.unique(dst[dst >= base + n])
    src = np.append(src, used)  # the others too
    dst = np.append(dst, (used - base - n) // 400)
    off, adj = orc.build_csr(nv, src, dst)
    ctx.upload_csr(off, adj, len(src))
    st = ctx.components()
    labels, ncomp, _ = orc.components(off, adj)
    np.testing.assert_array_equal(ctx.component_labels(), labels)
    assert st["num_components"] == ncomp and st["num_iters"] == 2


@pytest.mark.parametrize("nv,loops", [(1, 1), (63, 2), (64, 2), (65, 300), (1000, 255)])
def test_bytes_of_a_first_pass_alone(ctx, nv, loops):
    """Self-loops change no label, so the first pass is the only one: it reads
    every column id (4 bytes) and every vertex's bounds (8), and no label."""
    v = np.repeat(np.arange(nv), loops)
    off = np.arange(nv + 1, dtype=np.int64) * loops
    ctx.upload_csr(off, v.astype(np.int32), nv * loops // 2)
    st = ctx.components()
    assert st["num_iters"] == 1 and st["num_components"] == nv and st["labels_read"] == 0
    assert st["edge_bytes"] == 4 * nv * loops + 8 * nv


@pytest.mark.parametrize("fan", [0, 3, 254, 255, 2047, 2100])
@pytest.mark.parametrize("n", [2, 65, 600, 20000])
def test_passes_grow_with_the_logarithm_of_a_component(ctx, orc, n, fan):
    """Relabelled paths with hubs on either side of the list cuts, beside
    settled components, one of them with the vertex of largest degree: the
    first pass leaves a component with labels of half its vertices at most,
    every one from the tenth on with half of the labels, and the last changes
    none."""
    rng = np.random.default_rng(n + fan)
    a, b = np.triu_indices(60, 1)
    src, dst = [a, np.full(2200, 60)], [b, 61 + np.arange(2200)]
    base = 2300
    for _ in range(3):
        src.append(base + np.arange(n - 1))
        dst.append(base + np.arange(1, n))
        for at in (0, n // 2, n - 1):
            src.append(np.full(fan, base + at))
            dst.append(base + n + np.arange(fan))
        base += n + fan
    perm = rng.permutation(base + 7)
    s, d = perm[np.concatenate(src)], perm[np.concatenate(dst)]
    off, adj = orc.build_csr(base + 7, s, d)
    ctx.upload_csr(off, adj, len(s))
    for _ in range(2):
        st = compare(ctx, orc, off, adj)
        assert st["num_iters"] <= np.ceil(np.log2(max(n + fan, 2201))) + 9


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_components_of_many_shapes(ctx, orc, seed):
    """Forests, unions of paths, of power-law graphs and of sparse random ones,
    every id relabelled."""
    r = np.random.default_rng(seed)
    graphs = []
    for comps in (1, 40, 3000):
        nv = 20000
        v = np.arange(comps, nv)
        graphs.append((nv, v, (r.random(v.size) * v).astype(np.int64)))
    for k, length in ((1, 3000), (50, 300), (2000, 9)):
        v = np.arange(k * length).reshape(k, length)
        graphs.append((k * length, v[:, :-1].ravel(), v[:, 1:].ravel()))
    for m in (9000, 15000, 60000):
        graphs.append((30000, r.integers(0, 30000, m), r.integers(0, 30000, m)))
    parts = [orc.make_rmat(11, 8, seed=10 * seed + i) for i in range(12)]
    graphs.append((12 << 11, np.concatenate([s + (i << 11) for i, (_, s, _) in enumerate(parts)]),
                   np.concatenate([d + (i << 11) for i, (_, _, d) in enumerate(parts)])))
    for nv, s, d in graphs:
        p = r.permutation(nv + 5)
        s, d = p[s], p[d]
        off, adj = orc.build_csr(nv + 5, s, d)
        ctx.upload_csr(off, adj, len(s))
        compare(ctx, orc, off, adj)


@pytest.mark.parametrize("nv", [(1 << 22) - 1, 1 << 22])
def test_graphs_on_both_sides_of_the_root_rule(ctx, orc, nv):
    """The second pass lowers roots from 2^22 vertices on: sparse random graphs
    of hundreds of thousands of components."""
    ctx.generate_er(nv, nv, seed=nv & 3)
    off, adj = ctx.csr()
    st = ctx.components()
    labels, n, _ = orc.components(off, adj)
    np.testing.assert_array_equal(ctx.component_labels(), labels)
    assert st["num_components"] == n and st["num_iters"] <= 22 + 9


@pytest.mark.parametrize("scale", [14, 17])
def test_one_launch_a_pass_and_few_labels_read(ctx, scale):
    """An edge pass is one launch.  Where one component holds nearly all edges,
    the passes after the first read few labels: a vertex that carries its label
    reads none, and one that takes it no more."""
    ctx.generate_rmat(scale, 16, seed=scale)
    off, adj = ctx.csr()
    for _ in range(3):
        st = ctx.components()
        labels = ctx.component_labels()
        big = np.bincount(labels).max()
        assert big > 0.9 * np.count_nonzero(np.diff(off))
        assert st["pass_launches"] == st["num_iters"] >= 2
        assert st["labels_read"] <= 0.25 * (st["num_iters"] - 1) * len(adj)
