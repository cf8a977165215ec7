"""The device tree where its paths meet: sets up to 4,096 particles are split by one work group, larger
ones level by level with prefix counts in tiles of 4,096; levels up to 512 nodes of the multipole pass
share a launch.  Sizes at those lines, leaves of one particle (levels of thousands of nodes), coincident
particles down to the depth limit, and per-particle masses: every array against the host build, bit
for bit."""
import numpy as np
import pytest

from tigergrav_amd import ics
from tigergrav_amd.solver import Solver

pytestmark = pytest.mark.gpu

ARRAYS = ("pos", "order", "mass", "leaves", "node_range", "node_child", "node_parent", "node_level", "node_x", "node_m", "node_r",
          "node_boxid", "node_box", "node_n", "cc_d", "pp_d", "cc_e", "pc_e")


def _coincident(n):
    return np.concatenate([np.repeat(ics.uniform(1, 3), 70, axis=0), ics.uniform(n - 70, 4)])


@pytest.mark.parametrize("make,n,leaf,masses", [
    (ics.uniform, 1, 8, False), (ics.uniform, 2, 1, True), (ics.uniform, 1023, 1, False), (ics.plummer_spheres, 1025, 4, True),
    (ics.uniform, 4095, 8, True), (ics.uniform, 4096, 1, False), (ics.uniform, 4097, 1, True), (ics.plummer_spheres, 8191, 16, False),
    (ics.uniform, 8192, 1, False), (ics.plummer_spheres, 30000, 2, True), (_coincident, 2000, 32, False), (_coincident, 6000, 64, True)])
def test_tree_sizes(make, n, leaf, masses):
    x = make(n) if make is _coincident else make(n, n)
    m = np.random.default_rng(n).uniform(0.5, 1.5, n).astype(np.float32) / n if masses else None
    print(f"tree sizes {make.__name__} n={n} leaf={leaf}", flush=True)
    got = []
    for device in (-1, 0):
        s = Solver(ewald=True, soft_len=ics.soft_len(n), m=1.0 / n, theta=0.7, parts_per_node=leaf, device=device)
        s.set_particles(x, m)
        got.append({k: s.export(k) for k in ARRAYS})
        s.close()
    for k in ARRAYS:
        assert np.array_equal(got[0][k], got[1][k]), k
