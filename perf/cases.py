"""What the framework's users have it compute, as timed cases.

listed() names the cases, draw() gives more of the same ranges, prepare()
makes what a program holds before the call (inputs on the GPU or, where the
entry point takes host arrays, on the host; tubes, plans and weights), run()
is one pass through the public entry points, work() the bytes and operations
a pass cannot do without and exact() the same outputs in plain numpy and
torch, 64 bits.

Kinds of case:
  solve      one tube: new potential in, induced charge out (negf_solve)
  charge     integrated charge of one chain over an energy list (RGF plan)
  diag_g     one-shot call over an energy list with diag G^R written
  dos        DOS, transmission and LDOS of one tube at complex energies
  batch      one launch sequence for many uneven, biased tubes
  scf        self-consistent bias point of one tube
  batch_scf  self-consistent run of many equal tubes sharing one kernel
  block      dense-block chain: lead self-energies and block RGF
  block_mat  equilibrium charge of a block material
  sg_forward, sg_gradient  charge surrogate: estimate and training gradient
"""
import ctypes as C
import math

import numpy as np
import torch

from electrostatic_amd import _lib, negf
from electrostatic_amd.surrogate import Surrogate

KB = 8.617333262e-5            # eV / K
QE, EP0 = 1.602176634e-19, 8.8541878128e-12
GAMMA, RINGS = 2.5, 17         # hopping (eV) and atoms per ring of the (17,0) tube
TEMP, ETA = 298.0, 1e-5        # contacts (K), Im E of the real-axis paths (eV)
E_VALENCE, E_POLE = -10.0, 3.0
EQ_PTS = (30, 30, 64)
COULOMB = dict(eps_r=3.9, R_ring_nm=0.665, R_image_nm=10.0)
T_EVEN = 2.5 * math.cos(math.pi / 17)
SG_KW, SG_HALO, SG_C, SG_CP, SG_LAYERS = 9, 4, 64, 32, 6


def listed():
    return [
        # the smallest tube solve, as an outside SCF driver calls it each iteration: latency
        {"name": "solve 40 sites", "kind": "solve", "cells": 10, "modes": 1, "bias": 0.0, "noneq": 200},
        # a long device at drain bias, several modes
        {"name": "solve 4012 sites biased", "kind": "solve", "cells": 1003, "modes": 3, "bias": 0.3, "noneq": 200},
        # the benchmark's charge integral, plan kept
        {"name": "charge 4096 x 8192", "kind": "charge", "sites": 4096, "energies": 8192},
        # ragged one-shot call that wants diag G^R itself
        {"name": "diag G 1501 x 777", "kind": "diag_g", "sites": 1501, "energies": 777},
        # density-of-states output after a solve, with the per-site LDOS
        {"name": "dos 1000 sites", "kind": "dos", "cells": 250, "modes": 2, "energies": 401},
        # an array of tubes of all lengths at their own biases, one solve of all
        {"name": "batch 64 tubes", "kind": "batch", "tubes": 64, "lo": 500, "hi": 20000, "modes": 2, "noneq": 128},
        # one gate-sweep point of a short device
        {"name": "scf 400 sites", "kind": "scf", "cells": 100, "gate": 0.4},
        # many gate points of one geometry at once
        {"name": "batch scf 32 x 1024", "kind": "batch_scf", "tubes": 32, "cells": 256},
        # atomistic (16,0) tube in blocks of two rings
        {"name": "block 500 x 1024", "kind": "block", "ring": 16, "blocks": 500, "energies": 1024},
        # charge of a short atomistic device, blocks of 20 orbitals
        {"name": "block solve 40 x 20", "kind": "block_mat", "ring": 10, "blocks": 40},
        # surrogate estimate for a batch of tubes
        {"name": "surrogate 128 x 2048", "kind": "sg_forward", "samples": 128, "sites": 2048},
        # gradient of one training minibatch
        {"name": "surrogate grad 32 x 2048", "kind": "sg_gradient", "samples": 32, "sites": 2048},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "charge", "diag_g", "dos", "batch", "scf", "batch_scf", "block",
                       "block_mat", "sg_forward", "sg_gradient"])
    if kind == "solve":
        return {"kind": kind, "cells": _log(rng, 4, 1500), "modes": rng.randint(1, 4),
                "bias": rng.choice([0.0, round(rng.uniform(0.05, 0.5), 3)]), "noneq": rng.randint(100, 300)}
    if kind == "charge":
        return {"kind": kind, "sites": _log(rng, 300, 4096), "energies": _log(rng, 200, 8192)}
    if kind == "diag_g":
        return {"kind": kind, "sites": _log(rng, 200, 3000), "energies": _log(rng, 100, 1500)}
    if kind == "dos":
        return {"kind": kind, "cells": _log(rng, 10, 400), "modes": rng.randint(1, 3),
                "energies": _log(rng, 50, 500)}
    if kind == "batch":
        return {"kind": kind, "tubes": _log(rng, 8, 64), "lo": rng.randint(100, 1000),
                "hi": rng.randint(2000, 20000), "modes": rng.randint(1, 2), "noneq": rng.randint(64, 128)}
    if kind == "scf":
        return {"kind": kind, "cells": _log(rng, 20, 150), "gate": round(rng.uniform(0.0, 1.0), 3)}
    if kind == "batch_scf":
        return {"kind": kind, "tubes": _log(rng, 4, 32), "cells": _log(rng, 30, 256)}
    if kind == "block":
        return {"kind": kind, "ring": rng.randint(5, 16), "blocks": _log(rng, 10, 500),
                "energies": _log(rng, 30, 1024)}
    if kind == "block_mat":
        return {"kind": kind, "ring": rng.randint(5, 16), "blocks": _log(rng, 5, 80)}
    return {"kind": kind, "samples": _log(rng, 4, 128 if kind == "sg_forward" else 32),
            "sites": _log(rng, 100, 2048)}


# ---------------------------------------------------------------- inputs
def _smooth(rng, N, lo, hi):
    """Sum of eight random Fourier modes rescaled to [lo, hi] eV."""
    x = np.arange(N) / N
    U = np.zeros(N)
    for k in range(1, 9):
        U += rng.normal() * np.cos(2 * np.pi * k * x + rng.uniform(0, 2 * np.pi))
    return lo + (hi - lo) * (U - U.min()) / (U.max() - U.min())


def _bumps(rng, N, amp):
    n = np.arange(N)
    U = np.zeros(N)
    for _ in range(4):
        c, w, a = rng.uniform(0, N), rng.uniform(N / 20, N / 5), rng.uniform(-amp, amp)
        U += a * np.exp(-0.5 * ((n - c) / w) ** 2)
    return U


def _gl(n):
    """Gauss-Legendre nodes and weights by the reference's Newton iteration
    (stop 3e-11, weight from the last derivative taken)."""
    x, w = np.zeros(n), np.zeros(n)
    for i in range(1, (n + 1) // 2 + 1):
        z = math.cos(math.pi * (i - 0.25) / (n + 0.5))
        while True:
            p1, p2 = 1.0, 0.0
            for j in range(1, n + 1):
                p1, p2 = ((2.0 * j - 1.0) * z * p1 - (j - 1.0) * p2) / j, p1
            pp = n * (z * p1 - p2) / (z * z - 1.0)
            z1, z = z, z - p1 / pp
            if not abs(z - z1) > 3.0e-11:
                break
        x[i - 1], x[n - i] = -z, z
        w[i - 1] = w[n - i] = 2.0 / ((1.0 - z * z) * pp * pp)
    return x, w


def _line(a, b, n):
    x, w = _gl(n)
    return (b - a) * 0.5 * x + (b + a) * 0.5, w * (b - a) * 0.5


def _arc(a, b, n):
    """Circular arc from a to b (centre on Im = Im b): energies, w dE."""
    x, w = _gl(n)
    c = (b.real ** 2 - a.real ** 2 - a.imag ** 2) / (2 * (b.real - a.real))
    R = c - b.real
    t1 = math.asin(abs(a.imag) / R)
    if c > a.real:
        t1 = math.pi - t1
    th = (math.pi - t1) * 0.5 * x + (math.pi + t1) * 0.5
    return c + R * np.cos(th) + 1j * (b.imag + R * np.sin(th)), w * (math.pi - t1) * 0.5 * R * np.exp(1j * th) * 1j


def _chain_inputs(case, seed):
    """Chain potential, and energies (half on the equilibrium contour arc for
    mu = 0, half on the real axis) with the charge coefficients."""
    N, nE = case["sites"], case["energies"]
    U = _smooth(np.random.default_rng([seed, 1]), N, -0.5, 0.5)
    kT = KB * TEMP
    poles = int((E_POLE - math.pi * kT) / (2 * math.pi * kT) + 1)
    # the few per cent of shift in the real-axis window is the seed's
    s = np.random.default_rng([seed, 2]).uniform(-0.05, 0.05)
    na = nE // 2
    Ea, da = _arc(complex(-14 * kT, 2 * poles * math.pi * kT), complex(E_VALENCE, ETA), na)
    Er, dr = _line(complex(-3.0 + s, ETA), complex(3.0 + s, ETA), nE - na)
    E = np.concatenate([Ea, Er])
    f = 1.0 / (np.exp(E / kT) + 1.0)
    return U, E, 2j / math.pi * np.concatenate([da, dr]) * f


def _tube_keys(cells, modes, bias, noneq, eq=EQ_PTS):
    return dict(num_unitcells=cells, num_modes=modes, contact_mu=(-1.0, -1.0 - bias), eq_integration_pts=eq,
                noneq_integration_pts=(noneq,), E_zPlus_imag=ETA, E_valence_min=E_VALENCE, E_pole_max=E_POLE)


def _batch_shape(case, seed):
    """Lengths (log-uniform, the case's own) and biases of a batch."""
    r = np.random.default_rng(3)
    cells = np.maximum(1, np.round(np.exp(r.uniform(math.log(case["lo"]), math.log(case["hi"]), case["tubes"])) / 4))
    bias = np.random.default_rng([seed, 4]).uniform(0.02, 0.5, case["tubes"])
    return cells.astype(int), bias


def _batch_potential(seed, i, N):
    return _smooth(np.random.default_rng([seed, 5, i]), N, -0.3, 0.3)


def _scf_inputs(case, seed):
    T, N = case.get("tubes", 1), 4 * case["cells"]
    U = np.stack([_bumps(np.random.default_rng([seed, 6, t]), N, 0.3) for t in range(T)])
    V = np.linspace(0.0, 1.0, T) if case["kind"] == "batch_scf" else np.array([case["gate"]])
    return U, V


def _ring_blocks(m):
    """Nearest-neighbour (m,0) tube in blocks of two rings: (H0, T)."""
    zig = np.eye(m) + np.roll(np.eye(m), -1, axis=1)
    H0 = np.zeros((2 * m, 2 * m))
    H0[:m, m:], H0[m:, :m] = -GAMMA * zig, -GAMMA * zig.T
    T = np.zeros((2 * m, 2 * m))
    j = np.arange(m)
    T[m + j, (-j) % m] = -GAMMA
    return H0, T


def _block_inputs(case, seed):
    nb, m = case["blocks"], 2 * case["ring"]
    r = np.random.default_rng([seed, 7])
    v = r.normal(0.0, 0.05, (nb, m)) + 0.2 * np.sin(np.linspace(0, np.pi, nb))[:, None]
    if case["kind"] == "block_mat":
        return v
    nE = case["energies"]
    E = np.concatenate([np.linspace(-3, 3, nE // 2) + 1j * ETA,
                        -1.0 + 1.5 * np.exp(1j * np.linspace(0.01, np.pi - 0.01, nE - nE // 2))])
    return v, E, np.exp(1j * r.uniform(0, 2 * np.pi, nE)) / nE


def _sg_layout():
    """Per layer: channels in and out (stored, real) and the offset of W."""
    out, off = [], 0
    for l in range(SG_LAYERS):
        ci, co = SG_CP if l == 0 else SG_C, SG_CP if l == SG_LAYERS - 1 else SG_C
        out.append((ci, co, 3 if l == 0 else SG_C, 1 if l == SG_LAYERS - 1 else SG_C, off))
        off += co * SG_KW * ci + co
    return out, off


def _sg_inputs(case, seed):
    """Weights of variance 1 / fan-in, potentials an SCF visits and, for the
    gradient, target charges."""
    B, N = case["samples"], case["sites"]
    r = np.random.default_rng([seed, 8])
    lay, n = _sg_layout()
    w = np.zeros(n, np.float32)
    for ci, co, cir, cor, off in lay:
        lim = math.sqrt(3.0 / (cir * SG_KW))
        W = np.zeros((co, SG_KW, ci), np.float32)
        W[:cor, :, :cir] = r.uniform(-lim, lim, (cor, SG_KW, cir))
        b = np.zeros(co, np.float32)
        b[:cor] = r.uniform(-0.1, 0.1, cor)
        w[off:off + W.size] = W.ravel()
        w[off + W.size:off + W.size + co] = b
    U = np.stack([_smooth(r, N, -0.4, 0.4) - r.uniform(-0.2, 1.2) for _ in range(B)])
    Q = 0.3 * np.tanh(2.0 * U) + 0.02 * np.stack([_smooth(r, N, -1.0, 1.0) for _ in range(B)])
    return w, U, Q


# ---------------------------------------------------------------- prepare, run
def _dev(a):
    a = np.ascontiguousarray(a)
    return torch.from_numpy(a.view(np.float64) if a.dtype == np.complex128 else a).cuda()


def _ptr(t):
    return None if t is None else C.c_void_p(t.data_ptr())


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


class _Plan:
    """RGF plan handle of the C ABI, destroyed with the state."""

    def __init__(self, p, dU, nE, dE, dc):
        self.h = C.c_void_p()
        _lib.check(_lib.load().negf_rgf_plan_create(C.byref(p), _ptr(dU), nE, _ptr(dE), _ptr(dc), 0, C.byref(self.h)))

    def __del__(self):
        _lib.load().negf_rgf_plan_destroy(self.h)


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "solve":
        s["tube"] = negf.Tube(**_tube_keys(case["cells"], case["modes"], case["bias"], case["noneq"]))
        s["U"] = _smooth(np.random.default_rng([seed, 1]), 4 * case["cells"], -0.3, 0.3)
    elif kind in ("charge", "diag_g"):
        U, E, coef = _chain_inputs(case, seed)
        p = _lib.negf_chain_params()
        p.N, p.t_even, p.t_odd = U.size, T_EVEN, 2.5
        p.Uc[0], p.Uc[1] = U[0], U[-1]
        s.update(p=p, nE=E.size, dU=_dev(U), dE=_dev(E), dc=_dev(coef))
        s["acc"] = torch.empty(U.size, dtype=torch.float64, device="cuda")
        if kind == "charge":
            s["plan"] = _Plan(p, s["dU"], E.size, s["dE"], s["dc"])
        else:
            s["dG"] = torch.empty((E.size, U.size, 2), dtype=torch.float64, device="cuda")
    elif kind == "dos":
        s["tube"] = negf.Tube(**_tube_keys(case["cells"], case["modes"], 0.0, 200))
        s["tube"].set_potential(_smooth(np.random.default_rng([seed, 1]), 4 * case["cells"], -0.3, 0.3))
        s["E"] = np.linspace(-2.0, 1.0, case["energies"]) + 1j * ETA
    elif kind == "batch":
        tubes = []
        for i, (cells, bias) in enumerate(zip(*_batch_shape(case, seed))):
            t = negf.Tube(**_tube_keys(int(cells), case["modes"], float(bias), case["noneq"], (32, 32, 64)))
            t.set_potential(_batch_potential(seed, i, t.N))
            tubes.append(t)
        s["batch"] = negf.Batch(tubes)
        s["batch"].use_graph(True)
        s["Q"] = torch.empty(int(s["batch"].offsets[-1]), dtype=torch.float64, device="cuda")
    elif kind in ("scf", "batch_scf"):
        U_ext, V = _scf_inputs(case, seed)
        tubes = [negf.Tube(**_tube_keys(case["cells"], 1, 0.0, 200)) for _ in range(len(V))]
        keys = dict(Broyden_fraction=0.1, Broyden_max_norm=1e-6, Broyden_threshold_maxstep=200,
                    reset_with_previous_charge_distribution=0, **COULOMB)
        if kind == "scf":
            s["scf"] = negf.Scf(tubes[0], **keys)
            s["scf"].set_external_potential(U_ext[0])
            s["V"] = float(V[0])
        else:
            s["batch"] = negf.Batch(tubes)
            s["scf"] = negf.BatchScf(s["batch"], **keys)
            s["scf"].set_external_potential(U_ext)
            s["V"], s["n0"] = V, np.zeros(U_ext.shape)
    elif kind == "block":
        v, E, coef = _block_inputs(case, seed)
        s["chain"] = negf.BlockChain(case["blocks"], *_ring_blocks(case["ring"]))
        s["chain"].set_potential(v, (0.0, 0.0))
        s.update(E=E, coef=coef)
    elif kind == "block_mat":
        s["chain"] = negf.BlockChain(case["blocks"], *_ring_blocks(case["ring"]))
        s["mat"] = negf.BlockMaterial(s["chain"], contact_mu=(-1.0, -1.0), eq_integration_pts=EQ_PTS,
                                      E_zPlus_imag=ETA, E_valence_min=E_VALENCE, E_pole_max=E_POLE)
        s["v"] = _block_inputs(case, seed)
    else:
        w, U, Q = _sg_inputs(case, seed)
        s["net"] = Surrogate(case["sites"], seed=1)
        s["net"].set_params(w, np.array([0.01, 0.3]))
        s["U"], s["Q"] = _dev(U), _dev(Q)
    return s


def run(s):
    kind = s["kind"]
    if kind == "solve":
        s["tube"].set_potential(s["U"])
        return s["tube"].solve(1)[0]
    if kind == "charge":
        _lib.check(_lib.load().negf_rgf_plan_execute(s["plan"].h, _ptr(s["acc"]), None, _stream()))
        return s["acc"]
    if kind == "diag_g":
        _lib.check(_lib.load().negf_rgf_diag_accumulate(C.byref(s["p"]), _ptr(s["dU"]), s["nE"], _ptr(s["dE"]),
                                                        _ptr(s["dc"]), _ptr(s["acc"]), _ptr(s["dG"]), _stream()))
        return s["acc"], s["dG"]
    if kind == "dos":
        return s["tube"].dos_complex(s["E"], want_ldos=True)
    if kind == "batch":
        s["batch"].solve_device(1, s["Q"].data_ptr(), torch.cuda.current_stream().cuda_stream)
        return s["Q"]
    if kind == "scf":
        return s["scf"].bias_point(s["V"])[:3]
    if kind == "batch_scf":
        s["scf"].set_input_charge(s["n0"])
        return s["scf"].run(s["V"])[:3]
    if kind == "block":
        return s["chain"].rgf(s["E"], s["coef"])[0]
    if kind == "block_mat":
        s["mat"].set_potential(s["v"])
        return s["mat"].solve()[0]
    if kind == "sg_forward":
        return s["net"].forward(s["U"])
    return s["net"].gradient(s["U"], s["Q"])


# ---------------------------------------------------------------- work
EQ_FLOP, NEQ_FLOP = 31.0, 63.0     # per energy and site, FMA = 2


def _eq_energies(bias):
    return sum(EQ_PTS) + (0 if bias else int((E_POLE - math.pi * KB * TEMP) / (2 * math.pi * KB * TEMP) + 1))


def work(case):
    kind = case["kind"]
    if kind == "solve":
        N, m = 4 * case["cells"], case["modes"]
        f = m * N * (_eq_energies(case["bias"]) * EQ_FLOP + (case["noneq"] * NEQ_FLOP if case["bias"] else 0.0))
        return {"bytes": 16.0 * N, "flops": f}
    if kind in ("charge", "diag_g"):
        N, nE = case["sites"], case["energies"]
        return {"bytes": 16.0 * N + 32.0 * nE + (16.0 * N * nE if kind == "diag_g" else 0.0),
                "flops": EQ_FLOP * N * nE}
    if kind == "dos":
        N, nE = 4 * case["cells"], case["energies"]
        return {"bytes": 8.0 * N + 32.0 * nE + 8.0 * N * nE, "flops": NEQ_FLOP * N * nE * case["modes"]}
    if kind == "batch":
        sites = 4.0 * float(_batch_shape(case, 0)[0].sum())
        return {"bytes": 16.0 * sites,
                "flops": sites * case["modes"] * (128 * EQ_FLOP + case["noneq"] * NEQ_FLOP)}
    if kind in ("scf", "batch_scf"):
        # about 25 iterations: the charge, the kernel product and the Broyden sums
        T, N = case.get("tubes", 1), 4 * case["cells"]
        return {"bytes": 25.0 * 8 * N * N + 25.0 * 16 * T * N, "flops":
                25.0 * T * (N * _eq_energies(0.0) * EQ_FLOP + 2.0 * N * N + 100.0 * N)}
    if kind in ("block", "block_mat"):
        m, nb = 2 * case["ring"], case["blocks"]
        nE = case["energies"] if kind == "block" else _eq_energies(0.0)
        return {"bytes": 16.0 * nb * m + 32.0 * nE, "flops": nE * m ** 3 * (36.0 * nb + 2 * 15 * 56.0)}
    B, N = case["samples"], case["sites"]
    f = 2.0 * SG_KW * B * N * (3 * SG_C + 4 * SG_C * SG_C + SG_C)
    n = 4.0 * _sg_layout()[1]
    return {"bytes": 16.0 * B * N + n / 2, "flops": f} if kind == "sg_forward" else \
        {"bytes": 16.0 * B * N + 1.5 * n, "flops": 3 * f}


# ---------------------------------------------------------------- exact
def _surface(E, U, te, to):
    """Lead self-energy: root with Im g < 0 of the alternating chain's end."""
    e2 = (E - U) ** 2
    fac = e2 + to * to - te * te
    root = torch.sqrt(fac * fac - 4.0 * e2 * to * to)
    den = 2.0 * to * to * (E - U)
    a, b = (fac + root) / den, (fac - root) / den
    zero = torch.zeros_like(a)
    return to * to * torch.where(a.imag < 0, a, torch.where(b.imag < 0, b, zero))


def _green(E, U, te, to, Uc0, Uc1, last, columns=False):
    """Chains in columns: diag G [N][C] of the tridiagonal matrices with
    energies E [C], potentials U [N][C] or [N][1], links te (even) and to
    (odd) and ends at site last [C]; with columns, also Gamma_L |G_n0|^2 and
    Gamma_R |G_n,last|^2."""
    N, nc = U.shape[0], E.numel()
    SL, SR = _surface(E, Uc0, te, to), _surface(E, Uc1, te, to)
    t2 = (te * te, torch.full_like(te, to * to))
    ragged = int(last.min()) < N - 1
    sL = torch.empty((N, nc), dtype=E.dtype, device=E.device)
    sL[0] = SL
    for n in range(N - 1):
        sL[n + 1] = t2[n & 1] / (E - U[n] - sL[n])
    G = sL
    sR = torch.empty_like(sL) if columns else None
    aR = torch.empty((N, nc), dtype=torch.float64, device=E.device) if columns else None
    cur, g2 = SR, None
    for n in range(N - 1, -1, -1):
        if n < N - 1:
            cur = t2[n & 1] / (E - U[n + 1] - cur)
            if ragged:
                cur = torch.where(last <= n, SR, cur)
        left = E - U[n] - sL[n]
        g = 1.0 / (left - cur)
        if columns:
            sR[n] = cur
            here = g.real ** 2 + g.imag ** 2
            if g2 is None:
                g2 = here
            else:
                g2 = g2 * t2[n & 1] / (left.real ** 2 + left.imag ** 2)
                if ragged:
                    g2 = torch.where(last <= n, here, g2)
            aR[n] = -2.0 * SR.imag * g2
        G[n] = g
    if not columns:
        return G
    aL = torch.empty_like(aR)
    g2 = G[0].real ** 2 + G[0].imag ** 2
    aL[0] = -2.0 * SL.imag * g2
    for n in range(1, N):
        right = E - U[n] - sR[n]
        g2 = g2 * t2[(n - 1) & 1] / (right.real ** 2 + right.imag ** 2)
        aL[n] = -2.0 * SL.imag * g2
    return G, aL, aR


def _where(size):
    return "cuda" if size > 1e6 and torch.cuda.is_available() else "cpu"


def _modes(nm):
    """Lowest modes of the (17,0) tube by gap: hopping and degeneracy."""
    gap = {}
    for p in range(1, RINGS + 1):
        gap.setdefault(min(abs(3 * p - 2 * RINGS), abs(3 * p - RINGS)), []).append(p)
    best = [gap[k] for k in sorted(gap)][:nm]
    return [(abs(2 * GAMMA * math.cos(math.pi * js[0] / RINGS)), len(js)) for js in best]


def _limits(mu):
    kT = KB * TEMP
    lo, hi = min(mu), max(mu)
    np_ = int((E_POLE - math.pi * kT) / (2 * math.pi * kT) + 1)
    top = 2 * np_ * math.pi * kT
    right = complex(hi + 14 * kT, ETA)
    if hi - lo > 1e-8:
        r = lo - 14 * kT
        return complex(r, ETA), complex(r, top), complex(r - 14 * kT, top), right, []
    return right, complex(right.real, top), complex(lo - 14 * kT, top), right, \
        [complex(lo, math.pi * kT * (2 * q + 1)) for q in range(np_)]


def _fermi(x):
    return 1.0 / (np.exp(x / (KB * TEMP)) + 1.0)


def _paths(mu, eq, noneq):
    """Energies and weights per unit degeneracy: the equilibrium charge is
    Re(c G_nn) summed, the non-equilibrium one cL Gamma_L |G_n0|^2 + cR ...
    """
    a, zeta, eta, right, poles = _limits(mu)
    p = [_line(a, zeta, eq[0]), _line(zeta, eta, eq[1]), _arc(eta, complex(E_VALENCE, ETA), eq[2])]
    E, d = np.concatenate([x for x, _ in p]), np.concatenate([x for _, x in p])
    c = -1j * (-2.0 / math.pi) * d * _fermi(E - min(mu))
    if poles:
        return np.concatenate([E, poles]), np.concatenate([c, np.full(len(poles), -4.0 * KB * TEMP)]), None
    En, dn = _line(a, right, noneq)
    w = -1.0 / math.pi
    return E, c, (En, w * (_fermi(En - mu[0]) * dn).real, w * (_fermi(En - mu[1]) * dn).real)


def _rho0_path():
    _, zeta, eta, _, _ = _limits((0.0, 0.0))
    p = [_line(complex(0.0, ETA), zeta, 30), _line(zeta, eta, 30), _arc(eta, complex(E_VALENCE, ETA), 30)]
    return np.concatenate([x for x, _ in p]), 2j / math.pi * np.concatenate([x for _, x in p])


def _tubes_charge(U, modes, sets, dev, rho0=None):
    """Charge of tubes of potentials U [t][N_t] with energy sets [t] =
    (E, c, noneq or None), all of one size; returns [t][N_t]."""
    Ns = [len(u) for u in U]
    N, T, md = max(Ns), len(U), _modes(modes)
    P = torch.zeros((N, T), dtype=torch.float64)
    for t, u in enumerate(U):
        P[:len(u), t] = torch.as_tensor(u)
    P = P.to(dev)
    ends = torch.tensor([[u[0], u[-1]] for u in U], dtype=torch.float64, device=dev)
    out = torch.zeros((N, T), dtype=torch.float64, device=dev)

    def each(E, *cs):
        # chains ordered (tube, mode, energy)
        e = torch.as_tensor(np.concatenate([np.tile(x, modes) for x in E])).to(dev)
        n = len(E[0])
        te = torch.tensor(np.tile(np.repeat([b for b, _ in md], n), T), device=dev)
        g = np.repeat([float(d) for _, d in md], n)
        w = [torch.as_tensor(np.concatenate([np.tile(x, modes) * g for x in c])).to(dev) for c in cs]
        k = modes * n
        last = torch.tensor(np.repeat(np.array(Ns) - 1, k), device=dev)
        return e, te, k, last, w, ends.repeat_interleave(k, 0)

    def total(x):
        return x.reshape(N, T, -1).sum(2)

    e, te, k, last, (c,), uc = each([s[0] for s in sets], [s[1] for s in sets])
    G = _green(e, P.repeat_interleave(k, 1), te, GAMMA, uc[:, 0], uc[:, 1], last)
    out += total((c * G).real)
    del G
    if sets[0][2] is not None:
        e, te, k, last, (cl, cr), uc = each(*[[s[2][q] for s in sets] for q in range(3)])
        _, aL, aR = _green(e, P.repeat_interleave(k, 1), te, GAMMA, uc[:, 0], uc[:, 1], last, True)
        out += total(cl * aL + cr * aR)
        del aL, aR
    if rho0 is None:
        rho0 = _rho0(Ns, modes, dev)
    out = out.cpu().numpy()
    return [out[:n, t] - rho0[n] for t, n in enumerate(Ns)]


def _rho0(Ns, modes, dev):
    """Rho0 by chain length; all lengths as the columns of one sweep."""
    E, c = _rho0_path()
    Ls, md = sorted(set(Ns)), _modes(modes)
    n, N = len(E), max(Ns)
    e = torch.as_tensor(np.tile(E, modes * len(Ls))).to(dev)
    te = torch.tensor(np.tile(np.repeat([b for b, _ in md], n), len(Ls)), device=dev)
    w = torch.as_tensor(np.tile(c, modes) * np.repeat([float(d) for _, d in md], n)).to(dev)
    last = torch.tensor(np.repeat(np.array(Ls) - 1, modes * n), device=dev)
    zero = torch.zeros((N, 1), dtype=torch.float64, device=dev)
    G = _green(e, zero, te, GAMMA, 0.0, 0.0, last)
    r = (w * G.reshape(N, len(Ls), -1)).real.sum(2).cpu().numpy()
    return {L: r[:L, i] for i, L in enumerate(Ls)}


def _coulomb(cells):
    acc = 1.42e-10
    r = np.arange(4 * cells)
    y = np.array([1.0, 1.5, 2.5, 3.0])[r % 4] * acc + 3 * acc * (r // 4)
    d2 = ((y[:, None] - y[None, :]) / 1e-9) ** 2
    ke = QE / (4.0 * math.pi * EP0) * 1e9
    return ke / COULOMB["eps_r"] * (1 / np.sqrt(d2 + COULOMB["R_ring_nm"] ** 2) -
                                    1 / np.sqrt(d2 + COULOMB["R_image_nm"] ** 2))


class _Mixer:
    """Broyden's second method, modified (fraction 0.1, absolute norm)."""

    def __init__(self, n):
        self.n, self.prev, self.F, self.V, self.W, self.step = n, np.zeros_like(n), np.zeros_like(n), [], [], 0

    def update(self, n_out):
        Fn = self.n - n_out
        dF, self.F = Fn - self.F, Fn
        s = np.zeros_like(Fn)
        if self.step > 0:
            W = -0.1 * dF + (self.n - self.prev) - sum((w * (v @ dF) for v, w in zip(self.V, self.W)),
                                                       np.zeros_like(Fn))
            self.V.append(dF / (dF @ dF))
            self.W.append(W)
            s = sum(w * (v @ Fn) for v, w in zip(self.V, self.W))
        self.prev, self.n = self.n, self.n - 0.1 * Fn - s
        self.step += 1
        return np.abs(Fn).max()


def _scf(case, seed):
    U_ext, V = _scf_inputs(case, seed)
    T, N = U_ext.shape
    K = _coulomb(case["cells"])
    E = _paths((-1.0, -1.0), EQ_PTS, 200)
    dev = _where(T * N * len(E[0]))
    rho0 = _rho0([N], 1, dev)
    mix = [_Mixer(np.zeros(N)) for _ in range(T)]
    out, active = {}, list(range(T))
    it = 0
    while active and it < 200:
        it += 1
        U = [U_ext[t] - V[t] - K @ mix[t].n for t in active]
        Q = _tubes_charge(U, 1, [E] * len(active), dev, rho0)
        for t, u, q in zip(list(active), U, Q):
            if mix[t].update(q) <= 1e-6:
                out[t] = (u, q, it)
                active.remove(t)
    return tuple(np.stack([np.asarray(out[t][k]) for t in range(T)]) for k in range(3))


def _block_diag(v, H0, T, E):
    """diag G [E][nb][m] of the block chain, leads by decimation."""
    nb, m = v.shape
    dev = _where(len(E) * nb * m * m)
    E = torch.as_tensor(E).to(dev)[:, None, None]
    I = torch.eye(m, dtype=torch.complex128, device=dev)
    H0, T = (torch.as_tensor(x + 0j).to(dev) for x in (H0, T))
    Tt = T.T.contiguous()

    def surface(a, b):
        es = e = H0.expand(len(E), m, m)
        a, b = a.expand(len(E), m, m), b.expand(len(E), m, m)
        for _ in range(200):
            g = torch.linalg.inv(E * I - e)
            ga, gb = g @ a, g @ b
            es, e = es + a @ gb, e + a @ gb + b @ ga
            a, b = a @ ga, b @ gb
            if max(float(a.abs().max()), float(b.abs().max())) < 1e-12:
                break
        return torch.linalg.inv(E * I - es)

    SL, SR = Tt @ surface(Tt, T) @ T, T @ surface(T, Tt) @ Tt
    vd = torch.as_tensor(v).to(dev)
    gs = []
    for b in range(nb):
        A = E * I - H0 - torch.diag(vd[b]) - (SL if b == 0 else Tt @ gs[-1] @ T)
        gs.append(torch.linalg.inv(A - SR if b == nb - 1 else A))
    G, out = gs[-1], [None] * nb
    for b in range(nb - 1, -1, -1):
        if b < nb - 1:
            X = gs[b] @ T
            G = gs[b] + X @ G @ X.transpose(1, 2).contiguous()
        out[b] = torch.diagonal(G, dim1=1, dim2=2)
    return torch.stack(out, 1).cpu().numpy()


def _sg_net(w, U, dev):
    """The network in 64 bits: leaves (W, b per layer) and the output q."""
    B, N = U.shape
    lay, _ = _sg_layout()
    par, n = [], torch.arange(N, device=dev)
    x = torch.stack([2.0 * U, torch.exp(-torch.minimum(n, N - 1 - n) / 16.0).expand(B, N), torch.zeros_like(U)], 2)
    for l, (ci, co, cir, cor, off) in enumerate(lay):
        W = w[off:off + co * SG_KW * ci].reshape(co, SG_KW, ci)[:cor, :, :cir]
        W = torch.as_tensor(W.astype(np.float64)).to(dev).requires_grad_()
        b = w[off + co * SG_KW * ci:off + co * SG_KW * ci + cor]
        b = torch.as_tensor(b.astype(np.float64)).to(dev).requires_grad_()
        par.append((W, b))
        xp = torch.nn.functional.pad(x, (0, 0, SG_HALO, SG_HALO))
        y = sum((xp[:, t:t + N] .reshape(B * N, cir) @ W[:, t].T for t in range(SG_KW)), b).reshape(B, N, cor)
        x = torch.tanh(y) if l < SG_LAYERS - 1 else y
    return par, x[:, :, 0]


def exact(case, seed):
    kind = case["kind"]
    if kind == "solve":
        N = 4 * case["cells"]
        U = _smooth(np.random.default_rng([seed, 1]), N, -0.3, 0.3)
        E = _paths((-1.0, -1.0 - case["bias"]), EQ_PTS, case["noneq"])
        return _tubes_charge([U], case["modes"], [E], _where(N * case["modes"] * 500))[0]
    if kind in ("charge", "diag_g"):
        U, E, coef = _chain_inputs(case, seed)
        dev = _where(U.size * E.size)
        e, c = torch.as_tensor(E).to(dev), torch.as_tensor(coef).to(dev)
        te = torch.full((E.size,), T_EVEN, dtype=torch.float64, device=dev)
        last = torch.full((E.size,), U.size - 1, device=dev)
        G = _green(e, torch.as_tensor(U).to(dev)[:, None], te, 2.5, U[0], U[-1], last)
        acc = (c * G).real.sum(1)
        return acc if kind == "charge" else (acc, torch.view_as_real(G.T.contiguous()))
    if kind == "dos":
        N, nm, E = 4 * case["cells"], case["modes"], np.linspace(-2.0, 1.0, case["energies"]) + 1j * ETA
        U = _smooth(np.random.default_rng([seed, 1]), N, -0.3, 0.3)
        dev, nE, md = _where(N * nm * case["energies"]), case["energies"], _modes(nm)
        e = torch.as_tensor(np.tile(E, nm)).to(dev)
        te = torch.tensor(np.repeat([b for b, _ in md], nE), device=dev)
        g = torch.tensor(np.repeat([float(d) for _, d in md], nE), device=dev)
        last = torch.full((nm * nE,), N - 1, device=dev)
        _, aL, aR = _green(e, torch.as_tensor(U).to(dev)[:, None], te, GAMMA, U[0], U[-1], last, True)
        ld = ((aL + aR) * g / (2.0 * math.pi)).reshape(N, nm, nE).sum(1).T
        tr = (aL[N - 1] * g * -2.0 * _surface(e, U[-1], te, GAMMA).imag).reshape(nm, nE).sum(0)
        return 2.0 * ld.sum(1) / (4 * RINGS), tr, ld.contiguous()
    if kind == "batch":
        cells, bias = _batch_shape(case, seed)
        U = [_batch_potential(seed, i, 4 * int(c)) for i, c in enumerate(cells)]
        sets = [_paths((-1.0, -1.0 - b), (32, 32, 64), case["noneq"]) for b in bias]
        return np.concatenate(_tubes_charge(U, case["modes"], sets, _where(1e9)))
    if kind == "scf":
        U, Q, it = _scf(case, seed)
        return U[0], Q[0], None
    if kind == "batch_scf":
        U, Q, it = _scf(case, seed)
        return U, Q, None
    if kind == "block":
        v, E, coef = _block_inputs(case, seed)
        return (coef[:, None, None] * _block_diag(v, *_ring_blocks(case["ring"]), E)).imag.sum(0)
    if kind == "block_mat":
        v, HT = _block_inputs(case, seed), _ring_blocks(case["ring"])
        E, c, _ = _paths((-1.0, -1.0), EQ_PTS, 0)
        E0, c0 = _rho0_path()
        # Re(c G) of the tube's weights per spin pair, one orbital each
        return (c[:, None, None] * _block_diag(v, *HT, E)).real.sum(0) - \
            (c0[:, None, None] * _block_diag(0.0 * v, *HT, E0)).real.sum(0)
    w, U, Q = _sg_inputs(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    U, Q = torch.as_tensor(U).to(dev), torch.as_tensor(Q).to(dev)
    if kind == "sg_forward":
        with torch.no_grad():
            return 0.01 + 0.3 * _sg_net(w, U, dev)[1]
    par, q = _sg_net(w, U, dev)
    loss = ((q - (Q - 0.01) / 0.3) ** 2).mean()
    loss.backward()
    lay, n = _sg_layout()
    g = np.zeros(n)
    for (ci, co, cir, cor, off), (W, b) in zip(lay, par):
        full = np.zeros((co, SG_KW, ci))
        full[:cor, :, :cir] = W.grad.cpu().numpy()
        g[off:off + full.size] = full.ravel()
        g[off + full.size:off + full.size + cor] = b.grad.cpu().numpy()
    return float(loss.detach()), g
