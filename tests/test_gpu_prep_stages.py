"""The device preparation's scans, wave packing, item sort and range expansion where their tiles end:
node and leaf counts around 4,096 (one scan launch or three), chunks around a packing segment of 256,
items around a sort tile of 1,024, chunk lengths below, at and past a wave -- every work array
against the host's preparation, element for element."""
import numpy as np
import pytest

from tigergrav_amd import ics
from tigergrav_amd.solver import Solver

pytestmark = pytest.mark.gpu

NAMES = [f"work_{what}_{k}" for k in range(8) for what in ("items", "list")] + [f"work_owner_{k}" for k in (2, 3, 6, 7)] + [
    "slot_node", "slot_ptr", "solve_leaf_items", "solve_path", "solve_pleaf", "solve_order"]


@pytest.mark.parametrize("n,leaf,theta,chunk,ewald", [
    (2, 1, 0.7, 64, True), (300, 1, 0.5, 1, False), (1100, 1, 0.9, 63, True), (2047, 1, 0.8, 64, False), (4200, 2, 0.7, 65, True),
    (9000, 2, 0.9, 4096, False), (40, 64, 0.5, 64, True)])
def test_stages(n, leaf, theta, chunk, ewald):
    x = ics.plummer_spheres(n, n) if not ewald else ics.uniform(n, n)
    print(f"prep stages n={n} leaf={leaf} chunk={chunk}", flush=True)
    got = []
    for walk in (0, 1):
        s = Solver(ewald=ewald, soft_len=ics.soft_len(n), m=1.0 / n, theta=theta, parts_per_node=leaf, device=0)
        s.tune("gpu_walk", walk)
        s.tune("node_chunk", chunk)
        s.set_particles(x)
        got.append({name: s.export(name) for name in NAMES})
        got[-1]["info"] = s.info()
        s.close()
    for name in NAMES:
        assert np.array_equal(got[0][name], got[1][name]), name
    for key in ("count", "items", "list_len"):
        assert got[0]["info"][key] == got[1]["info"][key], key
