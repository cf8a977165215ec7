"""The leaf kinds with several waves per item: list lengths around the tile counts at which the
number of waves changes (4, 8, 16 and 32 tiles of 64 sources) and where the waves' shares come out
uneven or empty, against the FP64 kernels at the kernel tests' 1e-5 RMS."""
import numpy as np
import pytest

import oracle_bind as ob
from kernel_cases import PARAMS, cluster, make_multipoles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nj", [255, 256, 257, 511, 513, 1024, 1025, 2049])
@pytest.mark.parametrize("ns", [1, 65])
@pytest.mark.parametrize("kind", ["PP_direct", "PC_direct", "PP_ewald", "PC_ewald"])
def test_leaf_waves(kind, ns, nj):
    from tigergrav_amd import gravity as tg

    P = PARAMS["periodic"]
    rng = np.random.default_rng(1000 * ns + nj)
    c0 = np.array([0.3, 0.6, 0.45])
    x = cluster(rng, ns, c0, 0.03)
    if kind.startswith("PP"):
        y = cluster(rng, nj, c0, 0.12)
    else:
        y = make_multipoles(rng, nj, c0, 0.35 if kind.endswith("ewald") else 0.2, 0.04, P["m"], npart=(4, 8))
    f = np.zeros((ns, 4))
    opts = tg.Options(ewald=True, soft_len=P["soft_len"], m=P["m"], device=0)
    tg.KERNELS[kind](f, x, y, opts=opts)
    if kind.endswith("ewald"):  # the FP64 sums take 30k flops and more a pair: the last sinks of each item
        pick = sorted({0, min(63, ns - 1), ns - 1})
        x, f = x[pick], f[pick]
    ref = ob.call_kernel("tgo64_", kind, P, x, y)[0]
    e = np.sqrt(np.sum((f[:, 1:] - ref[:, 1:]) ** 2) / np.sum(ref[:, 1:] ** 2))
    assert e < 1e-5, e
