"""The node kinds' segment sums and folded multipoles: a solver's node expansions (direct and Ewald,
particles and multipoles) with lists cut into slots of 1 to 65 entries, so that a wave holds one segment,
two, an odd number and 64 of them, and segments longer than a wave, against the whole lists.  Slots only
regroup FP64 sums of float terms: forces agree to a few float roundings (1e-6 RMS, the bound the
slots' own test takes); the per-call CC and CP kinds against the FP64 kernels; and the solver's node
expansions against the per-call kinds."""
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


@pytest.mark.parametrize("n,theta,leaf,ewald", [(1500, 0.5, 16, True), (1500, 0.6, 16, False), (400, 0.4, 4, True)])
def test_expansions(n, theta, leaf, ewald):
    """Every component of orders 2..4 of a node's expansion is the per-call kinds' sum of the same float
    terms (one per entry, slots of 64): they differ by the order of FP64 additions, 1e-12 for the few
    thousand terms of a node, where a component taken from others differs by float roundings, 1e-7."""
    from tigergrav_amd import gravity as tg
    from tigergrav_amd import ics
    from tigergrav_amd._lib import MULTI_DTYPE
    from tigergrav_amd.solver import Solver

    x = ics.plummer_spheres(n, n) if not ewald else ics.uniform(n, n)
    print(f"expansions n={n} theta={theta} ewald={ewald}", flush=True)
    m, h = 1.0 / n, ics.soft_len(n)
    s = Solver(ewald=ewald, soft_len=h, m=m, theta=theta, parts_per_node=leaf, device=0)
    s.tune("node_chunk", 64)
    s.set_particles(x)
    s.solve()
    s.synchronize()
    got = s.export("solve_expansions")
    T = s.tree_arrays()
    multi = np.zeros(len(T["node_x"]), MULTI_DTYPE)
    multi["m"], multi["x"] = T["node_m"], T["node_x"]
    opts = tg.Options(ewald=ewald, soft_len=h, m=m, device=0)
    entries = 0
    for a in range(len(multi)):
        L = np.zeros(35)
        for name, kind in (("cc_d", "CC_direct"), ("cp_d", "CP_direct"), ("cc_e", "CC_ewald"), ("cp_e", "CP_ewald")):
            v = T[name][T[name + "_ptr"][a]:T[name + "_ptr"][a + 1]]
            if name[1] == "p" and len(v):
                v = np.concatenate([np.arange(b, e) for b, e in v.reshape(-1, 2)])
            if len(v):
                tg.KERNELS[kind](L, T["node_x"][a], multi[v] if name[1] == "c" else T["pos"][v], opts=opts)
            entries += len(v)
        for lo, hi in ((4, 10), (10, 20), (20, 35)):
            assert np.abs(got[a, lo:hi] - L[lo:hi]).max() <= 1e-11 * np.abs(L[lo:hi]).max(), (a, lo)
    assert entries > n  # the lists are not empty


@pytest.mark.parametrize("make,n,leaf,theta,slot", [("uniform", 3000, 64, 0.5, 256), ("plummer_spheres", 40000, 32, 0.6, 512),
                                                    ("uniform", 100000, 8, 0.8, 4096), ("plummer_spheres", 150000, 64, 0.7, 512)])
def test_slot_sizes(make, n, leaf, theta, slot):
    """Without the knob the slots' size follows the number of nodes (and so of lists), not of particles: each
    node's slots are its lists cut into runs of that many entries."""
    from tigergrav_amd import ics
    from tigergrav_amd.solver import Solver

    s = Solver(ewald=True, soft_len=ics.soft_len(n), m=1.0 / n, theta=theta, parts_per_node=leaf, device=0)
    s.set_particles(getattr(ics, make)(n, 3))
    nn = s.info()["n_nodes"]
    print(f"slot sizes {make} n={n} nodes={nn}", flush=True)
    assert slot == (256 if nn <= 2048 else 512 if nn <= 32768 else 4096)
    want = np.zeros(nn, np.int64)
    for name in ("cc_d", "cp_d", "cc_e", "cp_e"):
        v, p = s.export(name), s.export(name + "_ptr")
        each = np.ones(len(v), np.int64) if name[1] == "c" else np.repeat(v[1::2] - v[::2], 2)
        each = np.concatenate([[0], np.cumsum(each)])
        entries = (each[p[1:]] - each[p[:-1]]) // (1 if name[1] == "c" else 2)
        want += (entries + slot - 1) // slot
    assert np.array_equal(np.diff(s.export("slot_ptr").view(np.int64)), want)
