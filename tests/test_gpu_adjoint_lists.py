"""The adjoint's by-source lists made on the device, from a device walk's lists and from a host walk's
copied there: the gradients agree to the order of the FP64 additions (atomics on the multipole adjoints;
1e-9 of the largest gradient, where FP32 terms would show at 1e-7), over leaves of one to 64 particles, a
single leaf, clustered sets whose leaf items take several waves, and per-particle masses.  And the
weights may lie in device memory."""
import ctypes as C

import numpy as np
import pytest

from tigergrav_amd import ics
from tigergrav_amd._lib import lib
from tigergrav_amd.solver import Solver

pytestmark = pytest.mark.gpu


def _solver(x, m, ewald, theta, leaf, device_lists):
    n = x.shape[0]
    s = Solver(ewald=ewald, soft_len=ics.soft_len(n), m=1.0 / n, theta=theta, parts_per_node=leaf, device=0)
    s.tune("gpu_walk", device_lists)
    s.tune("gpu_tree", device_lists)
    s.set_particles(x, m)
    s.solve()
    return s


@pytest.mark.parametrize("make,n,ewald,theta,leaf", [
    (ics.uniform, 63, True, 0.7, 64), (ics.uniform, 700, True, 0.5, 1), (ics.uniform, 3000, True, 0.6, 8),
    (ics.plummer_spheres, 20000, False, 0.7, 64), (ics.plummer_spheres, 9000, False, 0.5, 17)])
def test_adjoint_lists(make, n, ewald, theta, leaf):
    import torch

    x = make(n, n)
    rng = np.random.default_rng(n)
    m = rng.uniform(0.5, 1.5, n).astype(np.float32) / n
    w = rng.standard_normal((n, 3)).astype(np.float32)
    print(f"adjoint lists {make.__name__} n={n} leaf={leaf}", flush=True)
    dev, host = _solver(x, m, ewald, theta, leaf, 1), _solver(x, m, ewald, theta, leaf, 0)
    a, b = dev.adjoint(w), host.adjoint(w)
    for cols in (slice(0, 3), slice(3, 4)):
        assert np.max(np.abs(a[:, cols] - b[:, cols])) <= 1e-9 * np.max(np.abs(b[:, cols]))
    wd = torch.from_numpy(w).cuda()
    g = torch.zeros((n, 4), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    assert lib().tg_solver_adjoint(dev._h, C.c_void_p(wd.data_ptr()), C.c_void_p(g.data_ptr()), None) == 0
    assert np.max(np.abs(g.cpu().numpy() - a)) <= 1e-9 * np.max(np.abs(a))
    dev.close()
    host.close()


@pytest.mark.parametrize("device_lists", [0, 1])
def test_out_of_memory_while_the_lists_are_made(device_lists):
    """The first adjoint call of a tree that runs out of device memory, at every allocation it makes in
    turn, reports it; the next call starts again and gives the gradients (1e-9, as above)."""
    from tigergrav_amd._lib import TG_ENOMEM, ptr

    x = ics.uniform(700, 3)
    w = np.random.default_rng(3).standard_normal((700, 3)).astype(np.float32)
    print(f"adjoint out of memory, device_lists={device_lists}", flush=True)
    ref = _solver(x, None, True, 0.5, 8, device_lists)
    want = ref.adjoint(w)
    ref.close()
    failed = 0
    for k in range(200):
        s = _solver(x, None, True, 0.5, 8, device_lists)
        s.synchronize()
        g = np.zeros((700, 4))
        lib().tg_devmem_fail_after(k)
        rc = lib().tg_solver_adjoint(s._h, ptr(w), ptr(g), None)
        lib().tg_devmem_fail_after(-1)
        assert rc in (0, TG_ENOMEM)
        failed += rc == TG_ENOMEM
        g = s.adjoint(w)
        s.close()
        for cols in (slice(0, 3), slice(3, 4)):
            assert np.max(np.abs(g[:, cols] - want[:, cols])) <= 1e-9 * np.max(np.abs(want[:, cols]))
        if rc == 0:
            break
    assert rc == 0 and failed > 20
