"""The periodic correction's kinds at the edges of their wave-wide turns (their table rows are read 64 at
a time): 1 to 65 sinks, so one to 64 lanes share a sink, and source lists that end inside, at and just
past a turn, against the FP64 kernels.  A component's error is bounded by 1e-5 of the largest value its
derivative order takes over the cell (the table's interpolation error stays below 7.2e-6 of it), times
the sum of the weights that it enters with."""
import numpy as np
import pytest

import oracle_bind as ob
from kernel_cases import PARAMS, cluster, make_multipoles

pytestmark = pytest.mark.gpu
BIG = np.array([2.84, 4.0, 18.8, 96.0, 750.0])  # largest component of orders 0..4 over the cell


def _weights(kind, y):
    """sum over the sources of |weight| by the order that the weight adds (0: mass, 2, 3)"""
    if kind[1] == "P":  # particles of equal mass
        return np.array([len(y) * PARAMS["periodic"]["m"], 0.0, 0.0, 0.0])
    m = np.abs(np.asarray(y["m"], np.float64)).reshape(len(y), -1)
    return np.array([m[:, 0].sum(), 0.0, 3.0 * m[:, 1:7].sum(), 6.0 * m[:, 7:17].sum()])


def _bound(order, w):
    return 1e-5 * sum(w[k] * BIG[order + k] for k in range(4) if order + k <= 4)


@pytest.mark.parametrize("nj", [1, 2, 63, 64, 65, 129])
@pytest.mark.parametrize("kind,ns", [("PP_ewald", 1), ("PP_ewald", 2), ("PP_ewald", 33), ("PP_ewald", 64), ("PP_ewald", 65),
                                     ("PC_ewald", 1), ("PC_ewald", 33), ("PC_ewald", 65), ("CC_ewald", 1), ("CP_ewald", 1)])
def test_ewald_rows(kind, ns, nj):
    from tigergrav_amd import gravity as tg

    P = PARAMS["periodic"]
    rng = np.random.default_rng(100 * ns + nj)
    c0 = np.array([0.3, 0.6, 0.45])
    x = cluster(rng, ns, c0, 0.03)
    if kind in ("PP_ewald", "CP_ewald"):
        y = cluster(rng, nj, c0 + 0.2, 0.3)
    else:
        y = make_multipoles(rng, nj, c0, 0.35, 0.04, P["m"], npart=(4, 8))
    opts = tg.Options(ewald=True, soft_len=P["soft_len"], m=P["m"], device=0)
    w = _weights(kind[0] + kind[1], y)
    if kind[0] == "P":
        f = np.zeros((ns, 4))
        tg.KERNELS[kind](f, x, y, opts=opts)
        pick = sorted({0, min(63, ns - 1), ns - 1})
        ref = ob.call_kernel("tgo64_", kind, P, x[pick], y)[0]
        assert np.all(np.abs(f[pick, 1:] - ref[:, 1:]) < _bound(1, w))
    else:
        L = np.zeros(35)
        tg.KERNELS[kind](L, x[0], y, opts=opts)
        ref = ob.call_kernel("tgo64_", kind, P, x[0], y)[0]
        order = np.repeat(np.arange(5), [1, 3, 6, 10, 15])
        assert np.all(np.abs(L - ref) < [_bound(o, w) for o in order])
