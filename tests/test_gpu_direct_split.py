"""The FP64 direct sum's split over the wave, the source chunks and the structure-factor chunks: sink
counts below, at and past a wave, particle counts below, at and past a staged tile and a chunk, and a
softening length past the periodic cut-off of half a box, against the oracle (1e-10 RMS in the
accelerations, as the direct sum's other tests)."""
import numpy as np
import pytest

import oracle_bind as ob
from tigergrav_amd import ics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ewald", [True, False], ids=["periodic", "open"])
@pytest.mark.parametrize("n,ns,h", [(2, 1, 1e-3), (17, 3, 1e-3), (64, 64, 0.2), (511, 65, 1e-3), (1025, 33, 0.6), (1300, 130, 1e-2)])
def test_direct_split(n, ns, h, ewald):
    from tigergrav_amd.accuracy import direct_forces

    x = ics.uniform(n, seed=n)
    sinks = np.random.default_rng(n).choice(n, ns, replace=False)
    print(f"direct split n={n} ns={ns} h={h} ewald={ewald}", flush=True)
    f = direct_forces(x, sinks, ewald, h, 1.0 / n)
    phi, g = ob.direct64(ewald, h, x[sinks], x, np.full(n, 1.0 / n))
    assert np.linalg.norm(f[:, 1:] - g) < 1e-10 * np.linalg.norm(g)
    assert np.all(np.abs(f[:, 0] - phi) <= (1e-7 / n if ewald else 0.0) + 1e-10 * np.abs(phi))


@pytest.mark.parametrize("ewald", [True, False], ids=["periodic", "open"])
def test_more_sinks_than_a_launch_has_blocks(ewald):
    """2^24 + 5 sinks: a block of 256 threads each would pass a launch's 2^32 threads.  The sinks repeat
    the few particles, and so do the forces (1e-12: the pair sums' order depends on the sink count)."""
    from tigergrav_amd.accuracy import direct_forces

    n, ns = 7, 2 ** 24 + 5
    x = ics.uniform(n, seed=n)
    print(f"direct split ns={ns} ewald={ewald}", flush=True)
    few = direct_forces(x, np.arange(n), ewald, 1e-3, 1.0 / n)
    f = direct_forces(x, np.arange(ns) % n, ewald, 1e-3, 1.0 / n)
    for i in range(n):
        assert np.abs(f[i::n] - few[i]).max() <= 1e-12 * np.abs(few[i]).max()
