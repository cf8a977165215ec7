"""Performance cases of the force solve, its adjoint and the paths around them.

Each case is one thing a program that uses this package has it do again and again, through the
package's public entry points and at sizes of its configurations, tests and benchmark:

  kernels    the per-call drop-in: the four kernels a tree walk calls for one leaf and one node
  solve      host particles to host forces on a kept Solver: rebuild, eager solve, copy back
  step       the device-resident time step: rebuild, solve and kick (Stepper)
  resident   replayed solves over a resident tree (a fixed particle set, the benchmark's region)
  adjoint    a solve and the gradients of sum_i w_i . g_i on a kept Solver
  autograd   forward and backward of tree_accelerations, as a training loop calls it
  fof        rebuild and friends-of-friends groups of a clustered set
  direct     FP64 direct sums for a sample of sinks (the accuracy check of a solve)

`exact` gives the forces and gradients in 64 bits without this package's code: direct sums with
open boundaries, a particle-mesh Ewald sum in the periodic box.
"""
import ctypes
import math

import numpy as np
import torch

import tigergrav_amd
from tigergrav_amd import gravity
from tigergrav_amd.accuracy import direct_forces
from tigergrav_amd.autograd import tree_accelerations
from tigergrav_amd.solver import Solver
from tigergrav_amd.step import Stepper

DEVICE = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
SOFT = 0.02  # softening length in units of the mean spacing, the package's default


# ---- the cases ------------------------------------------------------------------------------------

def listed():
    return [
        # the smallest work there is: one leaf's and one node's calls from a CPU tree walk, at the
        # leaf size and list lengths of the kernel tests
        {"name": "kernels_leaf64", "kind": "kernels", "ns": 64, "nj": 1000, "nc": 300, "ewald": True},
        # a small ragged set, as a test or an interactive session solves: launches and waits
        {"name": "solve_uniform_1001", "kind": "solve", "gen": "uniform", "n": 1001, "theta": 0.5, "leaf": 16},
        # 32^3 uniform particles, periodic, leaf 64
        {"name": "solve_uniform_32k", "kind": "solve", "gen": "uniform", "n": 32768, "theta": 0.7, "leaf": 64},
        # a clustered set with open boundaries: eight Plummer spheres and a uniform background
        {"name": "solve_plummer_256k", "kind": "solve", "gen": "plummer", "n": 262144, "theta": 0.7, "leaf": 64},
        # a time step of the 2M periodic box at the angle and leaf size whose force error is 1e-3
        {"name": "step_2m_t03", "kind": "step", "ngrid": 128, "n_s": -2.0, "rms": 0.3, "theta": 0.3, "leaf": 8},
        # a time step of the 16.7M periodic box
        {"name": "step_16m_t05", "kind": "step", "ngrid": 256, "n_s": -1.5, "rms": 0.5, "theta": 0.5, "leaf": 32},
        # the 2M periodic solve itself, replayed: the accurate setting and the fast one
        {"name": "resident_2m_t03", "kind": "resident", "ngrid": 128, "n_s": -2.0, "rms": 0.3, "theta": 0.3, "leaf": 8},
        {"name": "resident_2m_t06", "kind": "resident", "ngrid": 128, "n_s": -2.0, "rms": 0.3, "theta": 0.6, "leaf": 32},
        # the adjoint configuration: 64^3 periodic, leaf 64, at an angle whose gradients are good to 5%
        {"name": "adjoint_256k", "kind": "adjoint", "gen": "zeldovich", "n": 262144, "theta": 0.5, "leaf": 64},
        # one pass of a training loop over a clustered set
        {"name": "autograd_plummer_64k", "kind": "autograd", "gen": "plummer", "n": 65536, "theta": 0.7, "leaf": 64},
        # groups of a clustered 2M snapshot
        {"name": "fof_2m", "kind": "fof", "n": 2097152, "link": 0.2, "leaf": 32},
        # the accuracy sample of a 2M periodic solve
        {"name": "direct_2m", "kind": "direct", "gen": "zeldovich", "n": 2097152, "sinks": 256},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["kernels", "solve", "solve", "step", "step", "resident", "resident", "adjoint", "autograd", "fof", "direct"])
    theta = round(rng.uniform(0.3, 0.7), 2)
    leaf = rng.choice([8, 16, 24, 32, 48, 64])
    if kind == "kernels":
        return {"kind": kind, "ns": rng.randint(1, 64), "nj": _log_int(rng, 15, 4000), "nc": _log_int(rng, 15, 1000),
                "ewald": rng.random() < 0.5}
    if kind == "solve":
        gen = rng.choice(["uniform", "plummer"])
        return {"kind": kind, "gen": gen, "n": _log_int(rng, 1000, 262144), "theta": theta, "leaf": leaf}
    if kind in ("step", "resident"):
        # near-lattice forces nearly cancel: wider angles than 0.6 leave them 10% off
        return {"kind": kind, "ngrid": _log_int(rng, 24, 160), "n_s": rng.choice([-1.5, -2.0]),
                "rms": round(rng.uniform(0.3, 0.5), 2), "theta": round(rng.uniform(0.3, 0.6), 2), "leaf": leaf}
    if kind in ("adjoint", "autograd"):
        gen = rng.choice(["zeldovich", "plummer"])
        n = _log_int(rng, 16, 64 if kind == "adjoint" else 48) ** 3 if gen == "zeldovich" else _log_int(rng, 4096, 65536)
        if gen == "zeldovich":  # the mass gradient of near-lattice sets: 5% off at 0.5
            theta = round(rng.uniform(0.3, 0.5), 2)
        return {"kind": kind, "gen": gen, "n": n, "theta": theta, "leaf": leaf}
    if kind == "fof":
        return {"kind": kind, "n": _log_int(rng, 3000, 2097152), "link": round(rng.uniform(0.15, 0.3), 2), "leaf": leaf}
    gen = rng.choice(["zeldovich", "plummer"])
    return {"kind": kind, "gen": gen, "n": _log_int(rng, 16, 100) ** 3 if gen == "zeldovich" else _log_int(rng, 4096, 1000000),
            "sinks": _log_int(rng, 16, 1000)}


# ---- inputs ---------------------------------------------------------------------------------------

def _fixed(p):
    """Box positions in [0, 1) to the package's int32 fixed point, x = p 2^-32 + 0.5."""
    z = torch.round((p - 0.5) * 4294967296.0).to(torch.int64)
    return torch.where(z >= 2 ** 31, z - 2 ** 32, z).to(torch.int32)


def _rng(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _uniform(n, seed):
    return _fixed(torch.rand((n, 3), generator=_rng(seed), device=DEVICE, dtype=torch.float64))


def _plummer(n, seed, spheres=8, a=0.02, background=0.2):
    """Equal Plummer spheres in the unit box and a uniform background; samples outside are redrawn."""
    g = _rng(seed)

    def rand(*shape):
        return torch.rand(shape, generator=g, device=DEVICE, dtype=torch.float64)

    per = int(n * (1.0 - background)) // spheres
    centres = rand(spheres, 3) * 0.9 + 0.05
    out = []
    for c in centres:
        have = torch.empty((0, 3), device=DEVICE, dtype=torch.float64)
        while have.shape[0] < per:
            u = rand(2 * (per - have.shape[0]) + 8).clamp_min(1e-12)
            v = torch.randn((u.numel(), 3), generator=g, device=DEVICE, dtype=torch.float64)
            p = c + (a / torch.sqrt(u ** (-2.0 / 3.0) - 1.0))[:, None] * v / v.norm(dim=1, keepdim=True)
            have = torch.cat([have, p[((p >= 0) & (p < 1)).all(dim=1)]])[:per]
        out.append(have)
    out.append(rand(n - spheres * per, 3))
    return _fixed(torch.cat(out))


def _zeldovich(ngrid, seed, n_s=-2.0, rms=0.3):
    """(positions, displacements): an ngrid^3 lattice displaced by a Gaussian field, P(k) ~ k^n_s."""
    white = torch.randn((ngrid,) * 3, generator=_rng(seed), device=DEVICE, dtype=torch.float64)
    kf = 2 * math.pi * torch.fft.fftfreq(ngrid, d=1.0 / ngrid, device=DEVICE, dtype=torch.float64)
    kr = 2 * math.pi * torch.fft.rfftfreq(ngrid, d=1.0 / ngrid, device=DEVICE, dtype=torch.float64)
    k2 = (kf ** 2)[:, None, None] + (kf ** 2)[None, :, None] + (kr ** 2)[None, None, :]
    amp = torch.where(k2 > 0, k2 ** (n_s / 4.0) / k2, torch.zeros_like(k2))
    amp[(k2 > (math.pi * ngrid) ** 2) | (k2 == 0)] = 0.0
    dk = torch.fft.rfftn(white) * amp
    psi = torch.stack([torch.fft.irfftn(1j * k * dk, s=(ngrid,) * 3) for k in
                       (kf[:, None, None], kf[None, :, None], kr[None, None, :])], dim=-1).reshape(-1, 3)
    psi *= (rms / ngrid) / psi.square().sum(dim=1).mean().sqrt()
    q = (torch.arange(ngrid, device=DEVICE, dtype=torch.float64) + 0.5) / ngrid
    x = torch.stack(torch.meshgrid(q, q, q, indexing="ij"), dim=-1).reshape(-1, 3) + psi
    return _fixed(x - torch.floor(x)), psi


def _particles(case, seed):
    """int32 [n, 3] on the GPU, and whether the box is periodic."""
    gen = case.get("gen", "zeldovich" if "ngrid" in case else "plummer")
    if gen == "uniform":
        return _uniform(case["n"], seed), True
    if gen == "plummer":
        return _plummer(case["n"], seed), False
    ngrid = case.get("ngrid") or round(case["n"] ** (1.0 / 3.0))
    return _zeldovich(ngrid, seed, case.get("n_s", -2.0), case.get("rms", 0.3))[0], True


def _soft(n):
    return SOFT * float(n) ** (-1.0 / 3.0)


def _weights(n, seed):
    return torch.randn((n, 3), generator=_rng(seed + 7919), device=DEVICE, dtype=torch.float32)


def _kernel_inputs(case, seed):
    """One leaf's sinks, its near particles and the multipoles of distant clusters, on the host."""
    r = np.random.default_rng(seed)
    m, centre = 1.0 / 32768, r.uniform(0.3, 0.7, 3)

    def pos(p):
        z = np.rint((p - 0.5) * 4294967296.0).astype(np.int64)
        return np.where(z >= 2 ** 31, z - 2 ** 32, z).astype(np.int32)

    x = pos(centre + 0.03 * (r.random((case["ns"], 3)) - 0.5))
    y = pos(centre + 0.12 * (r.random((case["nj"], 3)) - 0.5))
    k = min(case["ns"], case["nj"])
    y[:k] = x[:k]  # a leaf is in its own list
    mult = []
    for far in (0.2, 0.35):
        a = np.zeros(case["nc"], tigergrav_amd.MULTI_DTYPE)
        v = r.normal(size=(case["nc"], 3))
        c = centre + far * (0.6 + 0.4 * r.random((case["nc"], 1))) * v / np.linalg.norm(v, axis=1, keepdims=True)
        p = c[:, None, :] + 0.04 * (r.random((case["nc"], 32, 3)) - 0.5)
        com = p.mean(axis=1)
        a["x"] = pos(com - np.floor(com))
        d = p - com[:, None, :]
        a["m"][:, 0] = 32 * m
        a["m"][:, 1:7] = np.stack([m * (d[..., i] * d[..., j]).sum(axis=1) for i, j in _S2], axis=1)
        a["m"][:, 7:] = np.stack([m * (d[..., i] * d[..., j] * d[..., l]).sum(axis=1) for i, j, l in _S3], axis=1)
        mult.append(a)
    return {"x": x, "centre": pos(centre), "y": y, "near": mult[0], "far": mult[1],
            "opts": gravity.Options(ewald=case["ewald"], soft_len=_soft(32768), m=m, device=0)}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "kernels":
        return dict(_kernel_inputs(case, seed), kind=kind)
    if kind == "step":
        x, psi = _zeldovich(case["ngrid"], seed, case["n_s"], case["rms"])
        st = Stepper(x.cpu().numpy(), psi.to(torch.float32).cpu().numpy(), ewald=True, theta=case["theta"], leaf=case["leaf"],
                     dt_max=2.0 ** -12)
        return {"kind": kind, "stepper": st}
    periodic = True
    if kind == "fof":  # a snapshot of a periodic run
        x = _plummer(case["n"], seed)
    else:
        x, periodic = _particles(case, seed)
    n = x.shape[0]
    h, m = _soft(n), 1.0 / n
    if kind == "autograd":
        return {"kind": kind, "pos": x.to(torch.float64) * 2.0 ** -32 + 0.5, "mass": torch.full((n,), m, device=DEVICE, dtype=torch.float64),
                "w": _weights(n, seed).to(torch.float64), "periodic": periodic, "h": h, "theta": case["theta"], "leaf": case["leaf"]}
    if kind == "direct":
        sinks = np.sort(np.random.default_rng(seed).choice(n, case["sinks"], replace=False))
        return {"kind": kind, "x": x.cpu().numpy(), "sinks": sinks, "periodic": periodic, "h": h, "m": m}
    s = Solver(ewald=periodic, soft_len=h, m=m, theta=case.get("theta", 0.7), parts_per_node=case["leaf"], device=0)
    state = {"kind": kind, "solver": s}
    if kind in ("solve", "fof"):
        state["x"] = x.cpu().numpy()
        state["link"] = case.get("link")
        return state
    s.set_particles(x.cpu().numpy())
    if kind == "resident":
        state["f"] = torch.zeros((n, 4), device=DEVICE, dtype=torch.float64)
    else:
        state["w"] = _weights(n, seed).cpu().numpy()
    return state


def run(state):
    kind = state["kind"]
    if kind == "kernels":
        x, o = state["x"], state["opts"]
        f, fc = np.zeros((x.shape[0], 4)), np.zeros((x.shape[0], 4))
        L, Le = np.zeros(35), np.zeros(35)
        gravity.gravity_CC_direct(L, state["centre"], state["near"], opts=o)
        gravity.gravity_CC_ewald(Le, state["centre"], state["far"], opts=o)
        gravity.gravity_PC_direct(fc, x, state["near"], opts=o)
        gravity.gravity_PP_direct(f, x, state["y"], True, opts=o)
        return {"cc": L, "cc_ewald": Le, "pc": fc, "pp": f}
    if kind == "step":
        st = state["stepper"]
        st.first()
        return {"f": st.f, "v": st.v, "rung": st.rung}
    if kind == "autograd":
        pos, mass = state["pos"].detach().requires_grad_(True), state["mass"].detach().requires_grad_(True)
        acc = tree_accelerations(pos, mass, ewald=state["periodic"], soft_len=state["h"], theta=state["theta"], leaf=state["leaf"])
        (state["w"] * acc).sum().backward()
        return {"acc": acc.detach(), "pos_grad": pos.grad, "mass_grad": mass.grad}
    if kind == "direct":
        return direct_forces(state["x"], state["sinks"], state["periodic"], state["h"], state["m"])
    s = state["solver"]
    if kind == "solve":
        s.set_particles(state["x"])
        s.solve()
        return s.forces()
    if kind == "fof":
        s.set_particles(state["x"])
        groups, count = s.find_groups(state["link"])
        return groups.view(np.int64), count
    if kind == "resident":
        s.solve_graph()
        f = state["f"]
        if tigergrav_amd.lib().tg_solver_get_forces_device(s._h, ctypes.c_void_p(f.data_ptr())) != 0:
            raise RuntimeError("tg_solver_get_forces_device")
        return f
    s.solve()
    return s.adjoint(state["w"])


def work(case):
    """Bytes: inputs read once, outputs written once.  Flops: for a solve, the interactions its opening
    angle and leaf size leave (fits of the census on near-uniform sets) at a cost per interaction of
    24 (a pair), 400 (multipole to expansion), twice that again for the adjoint."""
    kind = case["kind"]
    if kind == "kernels":
        ns, nj, nc = case["ns"], case["nj"], case["nc"]
        return {"bytes": 12 * (ns + nj) + 160 * nc + 64 * ns + 560, "flops": 24.0 * ns * nj + 478.0 * ns * nc + 1500.0 * nc}
    n = case.get("n") or case["ngrid"] ** 3
    if kind == "fof":
        return {"bytes": 20 * n, "flops": 10.0 * n * 32}
    if kind == "direct":
        images = 27 if case["gen"] == "zeldovich" else 1
        return {"bytes": 12 * n + 32 * case["sinks"], "flops": 40.0 * images * n * case["sinks"]}
    theta, leaf = case["theta"], 0.75 * case["leaf"]
    pairs = min(float(n), leaf * (2.57 + 0.79 / theta) ** 3)
    nodes = 2.0 * n / leaf
    flops = n * pairs * 24.0 + nodes * min(nodes, 13.0 / theta ** 3) * 400.0
    bytes_ = {"solve": 44, "step": 12 + 32 + 12 + 12 + 1, "resident": 16 + 32, "adjoint": 16 + 12 + 32, "autograd": 32 + 24 * 3 + 8}[kind] * n
    return {"bytes": bytes_, "flops": flops * (3.0 if kind in ("adjoint", "autograd") else 1.0)}


# ---- the same values in 64 bits -------------------------------------------------------------------

_S2 = [(i, j) for i in range(3) for j in range(i, 3)]
_S3 = [(i, j, k) for i in range(3) for j in range(i, 3) for k in range(j, 3)]
_S4 = [(i, j, k, l) for i in range(3) for j in range(i, 3) for k in range(j, 3) for l in range(k, 3)]


def _spline(r, h):
    """(f, p) of the softened pair: g = -m dx f, phi = -m p; Newton's beyond h."""
    q = r / h
    f1 = (32 / 3 - 192 / 5 * q ** 2 + 32 * q ** 3) / h ** 3
    p1 = (14 / 5 - 16 / 3 * q ** 2 + 48 / 5 * q ** 4 - 32 / 5 * q ** 5) / h
    rs = r.clamp_min(0.25 * h)  # the outer branches hold no point this near
    f2 = (64 / 3 * q ** 3 - 48 * q ** 4 + 192 / 5 * q ** 5 - 32 / 3 * q ** 6 - 1 / 15) / rs ** 3
    p2 = (-1 / 15 + 16 / 5 * q - 32 / 3 * q ** 3 + 16 * q ** 4 - 48 / 5 * q ** 5 + 32 / 15 * q ** 6) / rs
    far, mid = r >= h, r >= 0.5 * h
    return torch.where(far, rs ** -3, torch.where(mid, f2, f1)), torch.where(far, 1 / rs, torch.where(mid, p2, p1))


def _pair_sum(xi, xj, m, h, self_at=None):
    """(phi, g) at xi from particles xj by direct summation, open boundaries."""
    d = [xi[:, None, a] - xj[None, :, a] for a in range(3)]
    r2 = d[0] * d[0]
    r2 = r2 + d[1] * d[1]
    r2 = r2 + d[2] * d[2]
    soft = torch.nonzero(r2.detach() < h * h, as_tuple=True)
    r2s = r2[soft]
    r2 = r2.index_put(soft, torch.ones_like(r2s))  # their own terms below
    p = r2.rsqrt()
    f = p * p * p
    fs, ps = _spline((r2s + 1e-300).sqrt(), h)
    if self_at is not None:
        ps = torch.where(soft[0] + self_at == soft[1], torch.zeros_like(ps), ps)  # no self potential
    f, p = f.index_put(soft, fs), p.index_put(soft, ps)
    phi = -(p @ m)
    fm = f @ torch.cat([m[:, None], m[:, None] * xj], dim=1)
    return phi, fm[:, 1:] - xi * fm[:, :1]


def _open_forces(x, m, h, w=None):
    """phi, g of all particles; with w also the gradients of sum_i w_i . g_i."""
    n = x.shape[0]
    rows = max(1, min(n, int((2 ** 28 if w is None else 2 ** 26) // n)))
    phi, g = [], []
    if w is not None:
        x, m = x.detach().requires_grad_(True), m.detach().requires_grad_(True)
    for b in range(0, n, rows):
        p, a = _pair_sum(x[b:b + rows], x, m, h, self_at=b)
        if w is not None:
            (a * w[b:b + rows]).sum().backward()
        phi.append(p.detach())
        g.append(a.detach())
    return torch.cat(phi), torch.cat(g), (None if w is None else (x.grad, m.grad))


def _bspline6(t):
    """Weights of the sixth-order B-spline at the six mesh points around a position, t in [0, 1)."""
    w = [t, 1 - t]  # w[j] is the order-k spline at t + j
    for k in range(3, 7):
        w = [((t + j) * (w[j] if j < k - 1 else 0.0) + (k - t - j) * (w[j - 1] if j else 0.0)) / (k - 1) for j in range(k)]
    return torch.stack(w[::-1], dim=-1)


def _mesh_weights(x, M):
    """Per axis: mesh indices [n, 6] and weights [n, 6] of positions x in box units."""
    s = x * M
    base = torch.floor(s.detach())
    t = s - base
    idx, wts = [], []
    for a in range(3):
        w = _bspline6(t[:, a])
        i = base[:, a:a + 1].to(torch.int64) + torch.arange(-2, 4, device=x.device)
        idx.append(i % M)
        wts.append(w)
    return idx, wts


def _long_range(x, m, alpha, M):
    """phi and g of the Fourier part of the Ewald sum through a mesh of M^3 points."""
    dev = x.device
    idx, w = _mesh_weights(x, M)
    wz = w[2]
    mesh = torch.zeros(M * M * M, device=dev, dtype=torch.float64)
    for a in range(6):
        for b in range(6):
            at = ((idx[0][:, a] * M + idx[1][:, b]) * M)[:, None] + idx[2]
            mesh = mesh.index_add(0, at.reshape(-1), ((w[0][:, a] * w[1][:, b] * m)[:, None] * wz).reshape(-1))
    rho = torch.fft.rfftn(mesh.reshape(M, M, M))
    k = torch.fft.fftfreq(M, d=1.0 / M, device=dev, dtype=torch.float64)
    kz = torch.fft.rfftfreq(M, d=1.0 / M, device=dev, dtype=torch.float64)
    def one(v):  # Gaussian and the two B-splines' transforms, axis by axis
        return torch.exp(-(math.pi / alpha * v) ** 2) / torch.sinc(v / M) ** 12

    k2 = (k ** 2)[:, None, None] + (k ** 2)[None, :, None] + (kz ** 2)[None, None, :]
    k2[0, 0, 0] = 1.0
    green = one(k)[:, None, None] * one(k)[None, :, None] * one(kz)[None, None, :] / (-math.pi * k2)
    green[0, 0, 0] = 0.0
    del k2
    rho = rho * green * float(M) ** 3
    del green
    out = []
    for ax in range(4):
        if ax == 0:
            f = torch.fft.irfftn(rho, s=(M, M, M)).reshape(-1)
        else:
            q = (k[:, None, None], k[None, :, None], kz[None, None, :])[ax - 1]
            q = torch.where(q.abs() * 2 == M, torch.zeros_like(q), q)
            f = torch.fft.irfftn(rho * (-2j * math.pi * q), s=(M, M, M)).reshape(-1)
        v = 0.0
        for a in range(6):
            for b in range(6):
                at = ((idx[0][:, a] * M + idx[1][:, b]) * M)[:, None] + idx[2]
                v = v + w[0][:, a] * w[1][:, b] * (wz * f[at]).sum(dim=1)
        out.append(v)
    return out[0], torch.stack(out[1:], dim=1)


def _short_range(x, m, alpha, ncell, h, w=None):
    """phi and g of the real-space part, all pairs within a cell edge, by cells of 1 / ncell; with w
    also accumulates the gradients of sum_i w_i . g_i into x.grad and m.grad."""
    n, dev = x.shape[0], x.device
    cell = torch.floor(x.detach() * ncell).to(torch.int64).clamp_(0, ncell - 1)
    cid = (cell[:, 0] * ncell + cell[:, 1]) * ncell + cell[:, 2]
    order = torch.argsort(cid)
    count = torch.bincount(cid, minlength=ncell ** 3)
    K = int(count.max())
    start = torch.cumsum(count, 0) - count
    slot = torch.arange(n, device=dev) - start[cid[order]]
    table = torch.full((ncell ** 3, K), -1, device=dev, dtype=torch.int64)
    table[cid[order], slot] = order
    phi, g = torch.zeros(n, device=dev, dtype=torch.float64), torch.zeros((n, 3), device=dev, dtype=torch.float64)
    rc2 = (1.0 / ncell) ** 2
    step = max(1, (2 ** 27 if w is None else 2 ** 25) // (K * K))
    c3 = torch.arange(ncell ** 3, device=dev)
    cz, cy, cx = c3 % ncell, c3 // ncell % ncell, c3 // ncell // ncell
    for o in range(27):
        ox, oy, oz = o // 9 - 1, o // 3 % 3 - 1, o % 3 - 1
        other = ((cx + ox) % ncell * ncell + (cy + oy) % ncell) * ncell + (cz + oz) % ncell
        for b in range(0, ncell ** 3, step):
            ti, tj = table[b:b + step], table[other[b:b + step]]
            xi, xj, mj = x[ti.clamp_min(0)], x[tj.clamp_min(0)], m[tj.clamp_min(0)]
            d = [xi[:, :, None, a] - xj[:, None, :, a] for a in range(3)]
            d = [v - torch.round(v.detach()) for v in d]
            r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
            ok = (ti[:, :, None] >= 0) & (tj[:, None, :] >= 0) & (r2.detach() < rc2) & (ti[:, :, None] != tj[:, None, :])
            r2 = torch.where(ok, r2, torch.full_like(r2, rc2))
            r = r2.sqrt()
            e = torch.erfc(alpha * r)
            p = e / r
            f = (p + 2 * alpha / math.sqrt(math.pi) * torch.exp(-alpha * alpha * r2)) / r2
            soft = torch.nonzero(ok & (r2.detach() < h * h), as_tuple=True)
            if soft[0].numel():
                rs = (r2[soft] + 1e-300).sqrt()
                fs, ps = _spline(rs, h)
                f, p = f.index_put(soft, fs - rs ** -3, accumulate=True), p.index_put(soft, ps - 1 / rs, accumulate=True)
            mk = torch.where(ok, mj[:, None, :].expand_as(r2), torch.zeros_like(r2))
            f = f * mk
            gi = -torch.stack([(f * v).sum(dim=2) for v in d], dim=2)
            good = ti >= 0
            if w is not None:
                (gi[good] * w[ti[good]]).sum().backward()
            phi.index_add_(0, ti[good], -(p * mk).sum(dim=2)[good].detach())
            g.index_add_(0, ti[good], gi[good].detach())
    return phi, g


def _periodic_forces(x, m, h, w=None):
    """phi, g of all particles in the periodic box by a particle-mesh Ewald sum (attractive, with the
    uniform background; a particle's own images counted); with w also the gradients."""
    n = x.shape[0]
    ncell = max(3, int(round(n ** (1.0 / 3.0) / (4.0 if n < 3000000 else 3.0))))
    alpha = 4.6 * ncell
    M = 32
    while M < (3.5 if n < 3000000 else 2.6) * alpha:
        M *= 2
    if w is not None:
        x, m = x.detach().requires_grad_(True), m.detach().requires_grad_(True)
    phi, g = _long_range(x, m, alpha, M)
    if w is not None:
        (g * w).sum().backward()
    ps, gs = _short_range(x, m, alpha, ncell, h, w)
    with torch.no_grad():
        phi = phi + ps + m * (2 * alpha / math.sqrt(math.pi)) + m.sum() * (math.pi / alpha ** 2)
        g = g + gs
    return phi.detach(), g.detach(), (None if w is None else (x.grad, m.grad))


def _radial(x, d):
    """Full derivative tensors of orders 0..4 from the radial factors d_k = (1/r d/dr)^k f."""
    e = torch.eye(3, dtype=torch.float64)
    x2 = x[..., :, None] * x[..., None, :]
    x3 = x2[..., None] * x[..., None, None, :]
    ex = e[:, :, None] * x[..., None, None, :]
    ex = ex + ex.transpose(-1, -2) + ex.transpose(-1, -3)
    x4 = x3[..., None] * x[..., None, None, None, :]
    d = [v[..., None] for v in d]
    exx, ee = 0.0, 0.0
    for a, b, c, f in ((0, 1, 2, 3), (0, 2, 1, 3), (0, 3, 1, 2), (1, 2, 0, 3), (1, 3, 0, 2), (2, 3, 0, 1)):
        names = "abcd"
        s = "%s%s,...%s%s->...abcd" % (names[a], names[b], names[c], names[f])
        exx = exx + torch.einsum(s, e, x2)
        ee = ee + 0.5 * torch.einsum("%s%s,%s%s->abcd" % (names[a], names[b], names[c], names[f]), e, e)
    return [d[0][..., 0], x * d[1], x2 * d[2][..., None] + e * d[1][..., None],
            x3 * d[3][..., None, None] + ex * d[2][..., None, None],
            x4 * d[4][..., None, None, None] + exx * d[3][..., None, None, None] + ee * d[2][..., None, None, None]]


def _newton_tensors(x):
    r = x.norm(dim=-1)
    d = [-1 / r]
    for k in range(1, 5):
        d.append(-(2 * k - 1) * d[-1] / r ** 2)
    return _radial(x, d)


def _ewald_tensors(x, alpha=2.5):
    """Derivatives of the periodic potential of a unit mass less its nearest image."""
    near = _newton_tensors(x)
    out = [-v for v in near]
    out[0] = out[0] + math.pi / alpha ** 2
    rng = torch.arange(-4, 5, dtype=torch.float64)
    for nx in rng:
        img = torch.stack(torch.meshgrid(nx[None], rng, rng, indexing="ij"), dim=-1).reshape(-1, 3)
        y = x[:, None, :] - img
        r = y.norm(dim=-1)
        B, g = [torch.erfc(alpha * r) / r], torch.exp(-(alpha * r) ** 2) / (alpha * math.sqrt(math.pi))
        for k in range(1, 5):
            B.append(((2 * k - 1) * B[-1] + (2 * alpha ** 2) ** k * g) / r ** 2)
        t = _radial(y, [-(-1) ** k * b for k, b in enumerate(B)])
        out = [o + v.sum(dim=1) for o, v in zip(out, t)]
    hs = torch.arange(-6, 7, dtype=torch.float64)
    hv = torch.stack(torch.meshgrid(hs, hs, hs, indexing="ij"), dim=-1).reshape(-1, 3)
    hv = hv[(hv ** 2).sum(dim=1) > 0]
    h2 = (hv ** 2).sum(dim=1)
    c = torch.exp(-math.pi ** 2 * h2 / alpha ** 2) / (math.pi * h2)
    ph = 2 * math.pi * (x @ hv.T)
    k = 2 * math.pi * hv
    cos, sin = torch.cos(ph) * c, torch.sin(ph) * c
    fourier = [-cos.sum(dim=1), sin @ k, torch.einsum("nh,ha,hb->nab", cos, k, k),
               -torch.einsum("nh,ha,hb,hc->nabc", sin, k, k, k), -torch.einsum("nh,ha,hb,hc,hd->nabcd", cos, k, k, k, k)]
    return [o + v for o, v in zip(out, fourier)]


def _symmetric(m):
    """Full quadrupole [n, 3, 3] and octupole [n, 3, 3, 3] of stored multipoles [n, 17]."""
    q, o = torch.zeros((m.shape[0], 3, 3), dtype=torch.float64), torch.zeros((m.shape[0], 3, 3, 3), dtype=torch.float64)
    for s, (i, j) in enumerate(_S2):
        q[:, i, j] = q[:, j, i] = m[:, 1 + s]
    for s, t in enumerate(_S3):
        for i, j, k in ((0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0)):
            o[:, t[i], t[j], t[k]] = m[:, 7 + s]
    return q, o


def _m2l(D, m, q, o):
    """The 35 expansion coefficients from derivative tensors at the sink centre, summed over sources."""
    L0 = m * D[0] + 0.5 * torch.einsum("nab,nab->n", q, D[2]) - torch.einsum("nabc,nabc->n", o, D[3]) / 6
    L1 = m[:, None] * D[1] + 0.5 * torch.einsum("nbc,nabc->na", q, D[3]) - torch.einsum("nbcd,nabcd->na", o, D[4]) / 6
    L2 = m[:, None, None] * D[2] + 0.5 * torch.einsum("ncd,nabcd->nab", q, D[4])
    L3, L4 = m[:, None, None, None] * D[3], m[:, None, None, None, None] * D[4]
    L = [L0.sum()[None], L1.sum(dim=0)] + [torch.stack([t.sum(dim=0)[s] for s in idx]) for t, idx in ((L2, _S2), (L3, _S3), (L4, _S4))]
    return torch.cat(L)


def _kernels_exact(case, seed):
    c = _kernel_inputs(case, seed)
    unit, h, mass = 2.0 ** -32, c["opts"].soft_len, c["opts"].m

    def diff(a, b):  # separations as the boundary condition has them
        d = a.astype(np.int64) - b.astype(np.int64)
        if case["ewald"]:
            d = (d + 2 ** 31) % 2 ** 32 - 2 ** 31
        return torch.from_numpy(d * unit)

    out = {}
    for key, src, tensors in (("cc", c["near"], _newton_tensors), ("cc_ewald", c["far"], _ewald_tensors)):
        M = torch.from_numpy(src["m"].astype(np.float64))
        d = c["centre"][None, :].astype(np.int64) - src["x"].astype(np.int64)
        if case["ewald"] or key == "cc_ewald":
            d = (d + 2 ** 31) % 2 ** 32 - 2 ** 31
        out[key] = _m2l(tensors(torch.from_numpy(d * unit)), M[:, 0], *_symmetric(M))
    M = torch.from_numpy(c["near"]["m"].astype(np.float64))
    q, o = _symmetric(M)
    ns, nc = c["x"].shape[0], M.shape[0]
    D = _newton_tensors(diff(c["x"][:, None, :], c["near"]["x"][None, :, :]).reshape(-1, 3))
    D = [v.reshape((ns, nc) + v.shape[1:]) for v in D]
    phi = D[0] @ M[:, 0] + 0.5 * torch.einsum("jab,ijab->i", q, D[2])
    for s, t in enumerate(_S3):  # the potential's octupole counts each triple once per distinct index
        phi = phi - len(set(t)) * (1, 3, 6)[len(set(t)) - 1] / 6 * (D[3][(...,) + t] @ M[:, 7 + s])
    g = -(torch.einsum("j,ija->ia", M[:, 0], D[1]) + 0.5 * torch.einsum("jbc,ijabc->ia", q, D[3])
          - torch.einsum("jbcd,ijabcd->ia", o, D[4]) / 6)
    out["pc"] = torch.cat([phi[:, None], g], dim=1)
    d = diff(c["x"][:, None, :], c["y"][None, :, :])
    f, p = _spline(d.norm(dim=-1), h)
    phi = -mass * p.sum(dim=1) + 315.0 / 128.0 * mass / h
    out["pp"] = torch.cat([phi[:, None], -mass * (f[..., None] * d).sum(dim=1)], dim=1)
    return {k: out[k] for k in ("cc", "cc_ewald", "pc", "pp")}


def exact(case, seed):
    kind = case["kind"]
    if kind == "kernels":
        return _kernels_exact(case, seed)
    if kind in ("fof", "direct"):  # whole numbers; a 64-bit path that is compared with itself
        return None
    x, periodic = _particles(case, seed)
    n = x.shape[0]
    m = torch.full((n,), float(np.float32(1.0 / n)), device=x.device, dtype=torch.float64)
    x = x.to(torch.float64) * 2.0 ** -32 + 0.5
    x = x - torch.floor(x)
    w = _weights(n, seed).to(torch.float64) if kind in ("adjoint", "autograd") else None
    phi, g, grads = (_periodic_forces if periodic else _open_forces)(x, m, _soft(n), w)
    if kind == "adjoint":
        return torch.cat([grads[0], grads[1][:, None]], dim=1)
    if kind == "autograd":
        return {"acc": g, "pos_grad": grads[0], "mass_grad": grads[1]}
    # a solve's potential keeps the spline's value at r = 0 less the reference's self potential
    phi = phi - (14.0 / 5.0 - 315.0 / 128.0) * m / _soft(n)
    f = torch.cat([phi[:, None], g], dim=1)
    return {"f": f, "v": None, "rung": None} if kind == "step" else f
