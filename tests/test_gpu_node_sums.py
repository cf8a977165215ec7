"""The node kinds' 26 sums and folded multipoles: a solver's node expansions (direct and Ewald, particles
and multipoles) with lists cut into slots of 1 to 65 entries, so that a wave holds one segment, two,
an odd number and 64 of them, and segments longer than a wave, against the whole lists.  Slots only
regroup FP64 sums of float terms: forces agree to a few float roundings (1e-6 RMS, the bound the
slots' own test takes); and the per-call CC and CP kinds, which sum all 35 components, against the
FP64 kernels."""
import numpy as np
import pytest

import oracle_bind as ob
from kernel_cases import PARAMS, cluster, make_multipoles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ewald", [True, False])
@pytest.mark.parametrize("chunk", [1, 2, 3, 31, 32, 33, 63, 64, 65, 130])
def test_slots(chunk, ewald):
    from tigergrav_amd import ics
    from tigergrav_amd.solver import Solver

    n = 3000
    x = ics.plummer_spheres(n, 17)
    f = []
    for c in (4096, chunk):
        s = Solver(ewald=ewald, soft_len=ics.soft_len(n), m=1.0 / n, theta=0.6, parts_per_node=16, device=0)
        s.tune("node_chunk", c)
        s.set_particles(x)
        s.solve()
        s.synchronize()
        f.append(s.forces())
    d = f[1][:, 1:] - f[0][:, 1:]
    assert np.sqrt(np.sum(d ** 2) / np.sum(f[0][:, 1:] ** 2)) < 1e-6


@pytest.mark.parametrize("nj", [1, 31, 32, 33, 64, 65, 200])
@pytest.mark.parametrize("kind", ["CC_direct", "CP_direct"])
def test_components(kind, nj):
    from tigergrav_amd import gravity as tg

    P = PARAMS["periodic"]
    rng = np.random.default_rng(nj)
    c0 = np.array([0.3, 0.6, 0.45])
    x = cluster(rng, 1, c0, 0.03)[0]
    y = make_multipoles(rng, nj, c0, 0.2, 0.04, P["m"], npart=(4, 8)) if kind[1] == "C" else cluster(rng, nj, c0 + 0.15, 0.1)
    L = np.zeros(35)
    tg.KERNELS[kind](L, x, y, opts=tg.Options(ewald=True, soft_len=P["soft_len"], m=P["m"], device=0))
    ref = ob.call_kernel("tgo64_", kind, P, x, y)[0]
    for lo, hi in ((0, 1), (1, 4), (4, 10), (10, 20), (20, 35)):
        assert np.abs(L[lo:hi] - ref[lo:hi]).max() < 1e-5 * np.abs(ref[lo:hi]).max()
