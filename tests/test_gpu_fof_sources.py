"""Friends-of-friends from the tree on the device and from the host's (gpu_tree off), with leaves below,
at and above the 64 particles that the link search takes at a time and with linking lengths from a
fraction of the spacing to several times it, against the oracle's restatement of the reference's
relabelling: group ids, counts and the catalog's members are whole numbers and equal bit for bit."""
import numpy as np
import pytest

import oracle_bind as ob
from tigergrav_amd import ics
from test_gpu_fof import NONE, _catalog, _groups

pytestmark = pytest.mark.gpu


def _set(n, kind):
    if kind == "uniform":
        return ics.uniform(n, 5)
    if kind == "twins":  # coincident particles are no friends of each other (d^2 = 0)
        x = ics.uniform(n, 6)
        x[n // 2:] = x[: n - n // 2]
        return x
    x = ics.plummer_spheres(n, 7)
    x[: n // 8] = (x[: n // 8].astype(np.int64) // 4096 - 2 ** 31 + 2 ** 20).astype(np.int32)  # at the box edge
    return x


@pytest.mark.parametrize("gpu_tree", [1, 0])
@pytest.mark.parametrize("n,leaf,link,kind", [
    (1, 32, 0.2, "uniform"), (2, 32, 5.0, "uniform"), (65, 64, 3.0, "uniform"), (1500, 1, 0.4, "uniform"),
    (2000, 64, 0.2, "cluster"), (3000, 200, 0.3, "cluster"), (2500, 129, 1.5, "uniform"), (1000, 33, 0.5, "twins"),
    (700, 16, 8.0, "uniform"),
])
def test_fof_from_either_tree(n, leaf, link, kind, gpu_tree):
    from tigergrav_amd.solver import Solver

    print(f"fof: N={n} leaf={leaf} link={link} {kind} gpu_tree={gpu_tree}", flush=True)
    x = _set(n, kind)
    s = Solver(ewald=False, soft_len=ics.soft_len(n), m=1.0 / n, theta=0.7, parts_per_node=leaf, device=0)
    s.tune("gpu_tree", gpu_tree)
    s.set_particles(x)
    g, ng = _groups(s, link)
    v = np.zeros((n, 3), np.float32)
    cat = _catalog(s, v, 1.0, 2)
    T = s.tree_arrays()
    got = g[T["order"]]
    want = ob.fof(T["pos"], ob.fof_link2(n, link))
    assert np.array_equal(got, want)
    ids, counts = np.unique(want[want != NONE], return_counts=True)
    assert ng == len(ids)
    assert [(c.id, c.N) for c in cat] == list(zip(ids.tolist(), counts.tolist()))
    assert np.array_equal(_groups(s, link)[0], g)  # with the tree on the host by now


@pytest.mark.parametrize("gpu_tree", [1, 0])
@pytest.mark.parametrize("n,leaf,link,move", [(2, 1, 0.3, 0.0), (3000, 16, 0.3, 0.5), (2000, 64, 0.2, 20.0), (1500, 1, 0.5, 2.0)])
def test_fof_after_update(n, leaf, link, move, gpu_tree):
    """Groups of particles moved under the kept tree (move: RMS displacement in mean spacings), out of
    their leaves' boxes and across the box edge: ids and counts equal the oracle's on the moved positions."""
    from tigergrav_amd.solver import Solver

    print(f"fof after update: N={n} leaf={leaf} move={move} gpu_tree={gpu_tree}", flush=True)
    if n == 2:  # two leaves with boxes far apart, then two particles side by side
        x = np.array([[-2 ** 30, 0, 0], [2 ** 30, 0, 0]], np.int32)
        y = np.array([[2 ** 28, 0, 0], [2 ** 30, 0, 0]], np.int32)
    else:
        x = _set(n, "cluster")
        d = np.random.default_rng(n).standard_normal((n, 3)) * (move * n ** (-1.0 / 3.0) * 2.0 ** 32)
        y = (x.astype(np.int64) + d.astype(np.int64)).astype(np.int32)  # wraps
    s = Solver(ewald=True, soft_len=ics.soft_len(n), m=1.0 / n, theta=0.7, parts_per_node=leaf, device=0)
    s.tune("gpu_tree", gpu_tree)
    s.set_particles(x)
    s.update_particles(y)
    g, ng = _groups(s, link)
    order = s.export("order")
    want = ob.fof(y[order], ob.fof_link2(n, link))
    assert np.array_equal(g[order], want)
    ids, counts = np.unique(want[want != NONE], return_counts=True)
    assert ng == len(ids) and ng > 0
    assert [(c.id, c.N) for c in _catalog(s, np.zeros((n, 3), np.float32), 1.0, 2)] == list(zip(ids.tolist(), counts.tolist()))


def test_fof_more_pairs_than_a_launch_takes():
    """A clump of 11,700 single-particle leaves within the linking length of each other, 6.8e7 candidate
    pairs and so more than 2^32 threads of 64 a pair, and a tighter one whose pairs, deepest in the tree,
    come last."""
    from tigergrav_amd.solver import Solver

    rng = np.random.default_rng(1)
    wide, tight = 11700, 60
    x = np.concatenate([rng.integers(-2 ** 24, 2 ** 24, (wide, 3)), 2 ** 30 + rng.integers(-2 ** 8, 2 ** 8, (tight, 3))]).astype(np.int32)
    n = wide + tight
    link = 2.0 ** 26 / 2.0 ** 32 * n ** (1.0 / 3.0)
    print(f"fof many pairs: N={n}", flush=True)
    s = Solver(ewald=False, soft_len=ics.soft_len(n), m=1.0 / n, theta=0.7, parts_per_node=1, device=0)
    s.set_particles(x)
    g, ng = _groups(s, link)
    assert ng == 2
    order = s.export("order")
    want = np.full(n, np.min(np.flatnonzero(order < wide)), np.uint64)
    want[order >= wide] = np.min(np.flatnonzero(order >= wide))
    assert np.array_equal(g[order], want)
