"""What the speed of this framework is measured on: pressure solves, time steps,
operators and the learned preconditioner, each called as a user's program calls it.

listed() holds the measured cases, draw() makes more of the same ranges,
prepare() builds what a program has in hand before the call, run() is one pass
through the public entry points, work() counts what a pass cannot do without,
and exact() is the same result in 64 bits by plain NumPy and torch, for the
cases that have one (the direct solution of the discrete system behind an
iterative solve, the network in float64).
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import moons_amd as M
from moons_amd import _lib
from moons_amd.duct import Duct
from moons_amd.ensemble import LDC_U, PSEUDO_VACUUM, Ensemble

PRESET = (5, 1e-6, 1e-13, 1)        # the solver settings of U and B
PPE = (20000, 1e-8, 1e-300, 1)      # the pressure solve
PHI = (20000, 1e-12, 1e-300, 1)     # the phi cleaning, which sets div B


def listed():
    return [
        # the induction source curl(U x B) of one small ragged block: a few launches, latency
        {"name": "ct_source_50x39x45", "kind": "ct", "nx": 50, "ny": 39, "nz": 45},
        # the pressure solve of the 32^3 lid-driven cavity by the plain Jacobi-PCG: launches count
        {"name": "ppe_jacobi_cavity_32", "kind": "ppe", "prec": "Lap_SF", "bc": "cavity", "nx": 32, "ny": 32, "nz": 32,
         "stretched": False, "learned": False},
        # the plain FP64 pressure solve at the size of the headline benchmark: the rectangular duct
        {"name": "ppe_jacobi_duct_128", "kind": "ppe", "prec": "Lap_SF", "bc": "duct", "nx": 128, "ny": 128, "nz": 128,
         "stretched": True, "learned": False},
        # the headline benchmark's own solve: mixed precision with the network on the 32^3 level
        {"name": "ppe_learned_duct_128", "kind": "ppe", "prec": "MG_FP32", "bc": "duct", "nx": 128, "ny": 128,
         "nz": 128, "stretched": True, "learned": True},
        # a large pressure solve, inflow and outflow along x: the largest grid of the list
        {"name": "ppe_mixed_channel_256", "kind": "ppe", "prec": "MG_FP32", "bc": "channel", "nx": 256, "ny": 256,
         "nz": 256, "stretched": True, "learned": False},
        # a whole time step of the 64^3 MHD cavity, every solve by the reference's own preconditioner
        {"name": "mhd_cavity_64_step", "kind": "mhd", "n": 64, "Re": 400.0, "Ha": 10.0, "alpha": 1.0, "prec": "Lap_SF"},
        # a whole time step of the 128^3 duct (Ha 100, thin conducting walls) with the mixed solvers
        {"name": "duct_128_step", "kind": "duct", "nx": 128, "ny": 128, "nz": 128},
        # one step of a batch of independent cavities, each a captured graph, over four streams
        {"name": "ensemble_8_step", "kind": "ensemble", "sizes": "32 48 64 96 32 48 64 32"},
        # the energy equation with every source and the three-stage march, on a large ragged block
        {"name": "energy_120x100x110_step", "kind": "energy", "nx": 120, "ny": 100, "nz": 110, "method": 5, "stages": 3,
         "sources": True},
        # the cosine-transform pressure solve
        {"name": "fft_128", "kind": "fft", "nx": 128, "ny": 128, "nz": 128, "dir": 3},
        # one application of the network as a preconditioner
        {"name": "unet_prec_64", "kind": "unet_prec", "nx": 64, "ny": 64, "nz": 64},
        # one training sample: loss and gradient of every weight, forward and backward, from host arrays
        {"name": "unet_grad_32", "kind": "unet_grad", "nx": 32, "ny": 32, "nz": 32},
    ]


def _log(rng, lo, hi, step=1):
    """A whole number of [lo, hi], a multiple of step, even over its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["ct", "ppe", "ppe", "mixed", "mixed", "mhd", "duct", "ensemble", "energy", "fft", "unet_prec",
                       "unet_grad"])
    if kind == "ct":
        return {"kind": "ct", "nx": _log(rng, 8, 160), "ny": _log(rng, 8, 160), "nz": _log(rng, 8, 160)}
    if kind == "ppe":
        return {"kind": "ppe", "prec": "Lap_SF", "bc": rng.choice(["cavity", "duct", "channel", "phi"]),
                "nx": _log(rng, 8, 112), "ny": _log(rng, 8, 112), "nz": _log(rng, 8, 112),
                "stretched": rng.random() < 0.5, "learned": False}
    if kind == "mixed":
        # periodic directions need even counts in the multigrid; an odd count ends its coarsening,
        # so odd ones are met on small grids
        bc = rng.choice(["cavity", "channel", "phi", "duct"])
        learned = rng.random() < 0.25
        if learned:  # the network's level, a quarter of the grid, has counts that are multiples of 4
            lo, hi, step = 96, 192, 16
        else:
            lo, hi, step = rng.choice([(16, 64, 2 if bc == "duct" else 1), (16, 192, 8), (16, 192, 8)])
        return {"kind": "ppe", "prec": "MG_FP32", "bc": bc, "nx": _log(rng, lo, hi, step), "ny": _log(rng, lo, hi, step),
                "nz": _log(rng, lo, hi, step), "stretched": rng.random() < 0.5, "learned": learned}
    if kind == "mhd":
        Ha = rng.choice([0.0, round(rng.uniform(1.0, 100.0), 3)])
        return {"kind": "mhd", "n": _log(rng, 16, 72), "Re": round(rng.uniform(100.0, 1000.0), 3), "Ha": Ha,
                "alpha": rng.choice([0.0, 1.0]), "prec": "Lap_SF"}
    if kind == "duct":
        return {"kind": "duct", "nx": _log(rng, 16, 128, 8), "ny": _log(rng, 16, 128, 8), "nz": _log(rng, 16, 128, 8)}
    if kind == "ensemble":
        return {"kind": "ensemble", "sizes": " ".join(str(rng.choice([16, 24, 32, 48, 64])) for _ in range(rng.randint(2, 8)))}
    if kind == "energy":
        return {"kind": "energy", "nx": _log(rng, 12, 144), "ny": _log(rng, 12, 144), "nz": _log(rng, 12, 144),
                "method": rng.choice([2, 3, 4, 5]), "stages": rng.choice([1, 3]), "sources": rng.random() < 0.5}
    if kind == "fft":
        return {"kind": "fft", "nx": _log(rng, 12, 160), "ny": _log(rng, 12, 160), "nz": _log(rng, 12, 160),
                "dir": rng.choice([2, 3])}
    hi = 80 if kind == "unet_prec" else 48
    return {"kind": kind, "nx": _log(rng, 8, hi, 4), "ny": _log(rng, 8, hi, 4), "nz": _log(rng, 8, hi, 4)}


# ------------------------------------------------------------------ pieces
def _with_ghosts(x):
    """Node coordinates with a ghost node at each end, the wall spacing repeated."""
    return np.concatenate([[2 * x[0] - x[1]], x, [2 * x[-1] - x[-2]]])


def _nodes(n, stretched):
    """n cells on [0, 1]; stretched: clustered at both walls as the duct's are."""
    s = np.linspace(-1.0, 1.0, n + 1)
    if not stretched:
        return _with_ghosts(0.5 * (s + 1.0))
    a = 0.5 * math.log(2.05 / 0.05)
    return _with_ghosts(0.5 * (1.0 + np.tanh(a * s) / math.tanh(a)))


def _ppe_nodes(c):
    # the duct's and the channel's flow direction x is uniform
    along_x = c["stretched"] and c["bc"] in ("cavity", "phi")
    return [_nodes(c["nx"], along_x), _nodes(c["ny"], c["stretched"]), _nodes(c["nz"], c["stretched"])]


BCS = {"cavity": ["Neumann"] * 6, "duct": ["Periodic"] * 2 + ["Neumann"] * 4,
       "channel": ["Neumann", "Dirichlet"] + ["Neumann"] * 4, "phi": ["Dirichlet"] * 6}


def _singular(c):
    return c["bc"] in ("cavity", "duct")


def _rhs(c, seed):
    """A pressure right-hand side (z, y, x): smooth modes and the divergence of noise."""
    rng = np.random.default_rng(seed)
    n = (c["nz"], c["ny"], c["nx"])
    ax = [(np.arange(m) + 0.5) / m for m in n]
    f = 0.3 * rng.standard_normal(n)
    for _ in range(3):
        k = rng.integers(1, 5, size=3)
        ph = rng.random(3) * 2 * np.pi
        m = [np.cos(2 * np.pi * k[d] * ax[d] + ph[d]) for d in range(3)]
        f += rng.standard_normal() * m[0][:, None, None] * m[1][None, :, None] * m[2][None, None, :]
    return f


def _padded(f):
    return np.pad(f, 1).transpose(2, 1, 0)  # a field's (x, y, z) with ghosts, x fastest in memory


class _Span:
    """A field's memory for torch, which holds this object, and with it the field and its owner, as long as a tensor of it lives."""

    def __init__(self, f, owner):
        p = ctypes.c_void_p()
        _lib.check(_lib.load().moons_field_device_ptr(f.handle, ctypes.byref(p)))
        self.kept = (f, f.m, owner)
        self.__cuda_array_interface__ = {"shape": f.shape[::-1], "typestr": "<f8", "data": (p.value, False), "version": 2}


def _view(f, owner=None):
    """A field's device memory as a torch tensor (z, y, x), ghosts included, without a copy."""
    return torch.as_tensor(_Span(f, owner), device="cuda")


def _field(m, dl, rng, amp, mean=0.0):
    f = M.SF(m, dl)
    return f.upload((mean + amp * (2.0 * rng.random(f.shape[::-1]) - 1.0)).transpose(2, 1, 0))


LAYERS = [(4, 16), (16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (96, 32), (32, 32), (48, 16), (16, 16), (16, 1)]
LEVELS = [0, 0, 1, 1, 2, 2, 1, 1, 0, 0, 0]


def _weights(seed):
    """He-scaled weights W[tap][in][out] and small biases, layer by layer."""
    rng = np.random.default_rng(seed)
    w = []
    for ci, co in LAYERS:
        w += [math.sqrt(2.0 / (27 * ci)) * rng.standard_normal(27 * ci * co), 0.02 * rng.standard_normal(co)]
    return np.concatenate(w).astype(np.float32)


class _Checkpoint:
    """The start of a run kept on the device: run() advances from it each time."""

    def __init__(self, fields, zeroed):
        self.pairs = [(f, M.SF(f.m, f.dl).assign(f)) for f in fields]
        self.zeroed = zeroed

    def restore(self):
        for f, kept in self.pairs:
            f.assign(kept)
        for f in self.zeroed:
            f.fill(0.0)


# ----------------------------------------------------------------- prepare
def prepare(case, seed):
    c, kind = case, case["kind"]
    rng = np.random.default_rng(seed)
    s = {"case": c}
    if kind == "ct":
        m = M.mesh(_nodes(c["nx"], False), _nodes(c["ny"], True), _nodes(c["nz"], True))
        edge = (6, 5, 3)
        s["U_E"] = [_field(m, edge[d], rng, 1.0) for d in (0, 0, 1, 1, 2, 2)]
        s["B"] = [_field(m, 1 << d, rng, 0.5, 0.3) for d in range(3)]
        s["adv"] = [M.SF(m, 1 << d).fill(0.0) for d in range(3)]
        # face2Edge's six off-diagonal components: Bx@y, Bx@z, By@x, By@z, Bz@x, Bz@y
        s["tf"] = [M.SF(m, edge[d]) for d in (1, 2, 0, 2, 0, 1)]
        s["te"] = [M.SF(m, edge[d]) for d in range(3)]
        s["out"] = [_view(f) for f in s["adv"]]
    elif kind == "ppe":
        m = M.mesh(*_ppe_nodes(c))
        s["b"] = M.SF(m, "CC").upload(_padded(_rhs(c, seed)))
        s["x"] = M.SF(m, "CC").fill(0.0).set_BCs(BCS[c["bc"]], None, all_Neumann=_singular(c))
        s["P"] = M.PCG_solver_SF(m, s["x"], M.iter_solver_params(*PPE), prec=c["prec"])
        if c["learned"]:
            # the network of the 1/4 level; a program has trained it, its cost is that of any weights
            s["net"] = M.UNet(seed=0)
            s["net"].set_weights(_weights(1000))
            s["P"].set_MG_UNet(s["net"], 2, cycles=1)
        s["view"] = _view(s["x"])[1:-1, 1:-1, 1:-1]
    elif kind == "mhd":
        m = M.mesh.cube_uniform(c["n"])
        U = [_field(m, 1 << d, rng, 1e-3).set_BCs(*LDC_U[d]) for d in range(3)]
        for u in U:
            M.apply_BCs(u)
        p = M.SF(m, "CC").fill(0.0).set_BCs(["Neumann"] * 6, None, all_Neumann=True)
        kw = {}
        fields = U + [p]
        if c["Ha"] > 0:
            B = [M.SF(m, 1 << d).fill(0.0).set_BCs(*PSEUDO_VACUUM[d]) for d in range(3)]
            phi = M.SF(m, "CC").fill(0.0).set_BCs(["Dirichlet"] * 6)
            kw = dict(B=B, phi=phi, Ha=c["Ha"], Rem=1.0, B0=(0.0, 1.0, 0.0), isp_B=PRESET, isp_phi=PHI)
            fields = fields + B + [phi]
        s["st"] = M.MHD_step(m, U, p, Re=c["Re"], dt=5e-4, alpha_U=c["alpha"], isp_U=PRESET, isp_p=PPE,
                             prec_p=c["prec"], **kw)
        history = ("F", "FB", "J", "jCrossB") if c["Ha"] > 0 else ("F",)
        s["start"] = _Checkpoint(fields, [f for h in history for f in s["st"].field(h)])
        s["fields"], s["out"] = fields, [_view(f) for f in fields]
    elif kind == "duct":
        # wall conductance 1: the walls of the set-up that stays bounded
        s["D"] = Duct(n=(c["nx"], c["ny"], c["nz"]), c_w=1.0, prec_p="MG_FP32", prec_phi="MG_FP32", seed=seed)
        fields = s["D"].U + [s["D"].p] + s["D"].B + [s["D"].phi]
        s["start"] = _Checkpoint(fields, [f for h in ("F", "FB", "J", "jCrossB") for f in s["D"].st.field(h)])
        s["out"] = [_view(f) for f in fields]
    elif kind == "ensemble":
        s["E"] = Ensemble(member_sizes=[int(n) for n in c["sizes"].split()], seed=seed)
        s["out"] = [_view(f) for mb in s["E"].members for f in mb.U + [mb.p] + mb.B]
    elif kind == "energy":
        m = M.mesh(_nodes(c["nx"], False), _nodes(c["ny"], True), _nodes(c["nz"], True))
        U = [_field(m, 1 << d, rng, 0.5) for d in range(3)]
        T = _field(m, "CC", rng, 0.1, 0.5).set_BCs(["Dirichlet", "Dirichlet"] + ["Neumann"] * 4, [1.0, 0, 0, 0, 0, 0])
        M.apply_BCs(T)
        k = [_field(m, 1 << d, rng, 0.2, 1.0) for d in range(3)]
        kw = {}
        if c["sources"]:
            on = (True, 0.01)
            kw = dict(diffusion=on, KE_diffusion=on, viscous_dissipation=on, joule_heating=on, volumetric_heating=on,
                      J=[_field(m, dl, rng, 0.1) for dl in (6, 5, 3)], sigma_inv=M.SF(m, "CC").fill(1.0))
        s["st"] = M.Energy_step(m, T, U, k, dt=5e-5, method=c["method"], Pe=100.0, rk_stages=c["stages"],
                                isp_T=(1000, 1e-8, 1e-300, 1), **kw)
        s["start"] = _Checkpoint([T], [s["st"].field("F")])
        s["start"].pairs.append((s["st"].field("Tnm1"), s["start"].pairs[0][1]))
        s["keep"], s["out"] = (U, k), [_view(T), _view(s["st"].field("F"), s["st"])]
    elif kind == "fft":
        # planes normal to the direction have equal spacings, as the transform wants
        h = 1.0 / 64
        m = M.mesh(*[_with_ghosts(np.arange(n + 1) * h) for n in (c["nx"], c["ny"], c["nz"])])
        s["f"] = M.SF(m, "CC").upload(_padded(_rhs(c, seed)))
        s["u"] = M.SF(m, "CC").fill(0.0).set_BCs(["Neumann"] * 6, None, all_Neumann=True)
        s["F"] = M.FFT_solver_SF(m, c["dir"])
        s["out"] = _view(s["u"])[1:-1, 1:-1, 1:-1]
    elif kind == "unet_prec":
        m = M.mesh(*_unet_nodes(c))
        s["r"] = M.SF(m, "CC").upload(_padded(_residual(c, seed)))
        s["z"] = M.SF(m, "CC").fill(0.0).set_BCs(["Neumann"] * 6, None, all_Neumann=True)
        s["net"] = M.UNet(seed=0)
        s["net"].set_weights(_weights(seed))
        s["P"] = M.PCG_solver_SF(m, s["z"], M.iter_solver_params(*PPE), prec="UNet")
        s["P"].set_UNet(s["net"])
        s["out"] = _view(s["z"])[1:-1, 1:-1, 1:-1]
    elif kind == "unet_grad":
        M.init(0)
        s["net"] = M.UNet(seed=0)
        s["net"].set_weights(_weights(seed))
        s["in"], s["target"] = _sample(c, seed)
    return s


def _unet_nodes(c):
    return [_nodes(c["nx"], False), _nodes(c["ny"], True), _nodes(c["nz"], True)]


def _residual(c, seed):
    """A residual as the solver holds it: a right-hand side times the cell volumes (z, y, x)."""
    dh = [np.diff(h)[1:-1] for h in _unet_nodes(c)]
    return _rhs(c, seed) * (dh[2][:, None, None] * dh[1][None, :, None] * dh[0][None, None, :])


def _channels(c, f):
    """The network's four channels (float64, (4, z, y, x)) and the scale of f: f vol^(2/3) / rms and log aspect ratios."""
    dh = [np.diff(h)[1:-1] for h in _unet_nodes(c)]
    w = [dh[0][None, None, :], dh[1][None, :, None], dh[2][:, None, None]]
    vol = w[0] * w[1] * w[2]
    g = f * np.cbrt(vol) ** 2
    rms = math.sqrt(float(np.mean(g * g)))
    return np.stack([g / rms] + [np.broadcast_to(np.log(w[d] / np.cbrt(vol)), vol.shape) for d in range(3)]), rms


def _sample(c, seed):
    x, _ = _channels(c, _rhs(c, seed))
    t = _rhs(c, seed + 7777)
    t = t / math.sqrt(float(np.mean(t * t)))
    pad = [np.pad(a, 1).transpose(2, 1, 0).astype(np.float32) for a in list(x) + [t]]
    return np.stack(pad[:4]), pad[4]


# --------------------------------------------------------------------- run
def run(state):
    s, kind = state, state["case"]["kind"]
    if kind == "ct":
        M.advect_B(s["adv"], s["U_E"], s["B"], s["tf"], s["te"])
        return s["out"]
    if kind == "ppe":
        s["x"].fill(0.0)
        s["P"].solve(s["x"], s["b"])
        # with walls all round the pressure is known up to a constant: its mean is taken out
        return s["view"] - s["view"].mean() if _singular(s["case"]) else s["view"]
    if kind in ("mhd", "energy"):
        s["start"].restore()
        s["st"].step(1)
        return s["out"]
    if kind == "duct":
        s["start"].restore()
        s["D"].step(1)
        return s["out"]
    if kind == "ensemble":
        s["E"].step(1)
        return s["out"]
    if kind == "fft":
        s["F"].solve(s["u"], s["f"])
        return s["out"]
    if kind == "unet_prec":
        s["P"].apply_prec(s["r"], s["z"])
        return s["out"]
    loss, grad = s["net"].grad(s["in"], s["target"])
    return {"loss": loss, "grad": grad}


# -------------------------------------------------------------------- work
def work(case):
    """Fields read and written once; the network's multiplications and additions."""
    c, kind = case, case["kind"]
    if kind == "mhd":
        fields = (14 if c["Ha"] > 0 else 7)  # U, p, F (B, phi, F_B) in and out
        return {"bytes": 16.0 * fields * c["n"] ** 3, "flops": 0.0}
    if kind == "ensemble":
        return {"bytes": 16.0 * 14 * sum(int(n) ** 3 for n in c["sizes"].split()), "flops": 0.0}
    cells = float(c["nx"]) * c["ny"] * c["nz"]
    if kind == "ct":
        return {"bytes": 8.0 * (6 + 3 + 3) * cells, "flops": 27.0 * cells}
    if kind == "duct":
        return {"bytes": 16.0 * 14 * cells, "flops": 0.0}
    if kind == "energy":
        # T and F in and out, U, k (an implicit march) and the Joule heating's J and 1/sigma in
        reads = 3 + (3 if c["method"] >= 3 else 0) + (4 if c["sources"] else 0)
        return {"bytes": (32.0 + 8.0 * reads) * cells, "flops": 0.0}
    if kind in ("ppe", "fft"):
        return {"bytes": 16.0 * cells, "flops": 0.0}
    flops = sum(2.0 * 27 * ci * co * cells / 8 ** lev for (ci, co), lev in zip(LAYERS, LEVELS))
    if kind == "unet_prec":
        return {"bytes": 16.0 * cells, "flops": flops}
    return {"bytes": 20.0 * cells + 8.0 * sum(27 * a * b + b for a, b in LAYERS), "flops": 3.0 * flops}


# ------------------------------------------------------------------- exact
def _laplacian_modes(h, lo, hi):
    """Eigenvectors and values of the 1D cell-centred second difference of nodes h with its
    boundary conditions, symmetric in the cell widths' inner product."""
    dh, hc = np.diff(h), 0.5 * (h[1:] + h[:-1])
    n = len(dh) - 2
    up = 1.0 / np.diff(hc)  # between padded cells i and i + 1
    A = np.zeros((n, n))
    for i in range(n):
        for j, g in ((i - 1, up[i]), (i + 1, up[i + 1])):
            A[i, i] -= g
            if 0 <= j < n:
                A[i, j] += g
            else:
                bc = lo if j < 0 else hi
                if bc == "Periodic":
                    A[i, j % n] += g
                else:
                    A[i, i] += g if bc == "Neumann" else -g
    w = np.sqrt(dh[1:-1])
    lam, V = np.linalg.eigh(A / w[:, None] / w[None, :])
    return w, lam, V


def _along(mats, f):
    """f(z, y, x) with a matrix applied along each direction (x, y, z)."""
    f = f @ mats[0].T
    f = np.matmul(mats[1], f)
    return np.tensordot(mats[2], f, axes=(1, 0))


def _exact_ppe(c, seed):
    f = _rhs(c, seed)
    hs, bc = _ppe_nodes(c), BCS[c["bc"]]
    md = [_laplacian_modes(hs[d], bc[2 * d], bc[2 * d + 1]) for d in range(3)]
    lam = md[2][1][:, None, None] + md[1][1][None, :, None] + md[0][1][None, None, :]
    g = _along([V.T * w for w, _, V in md], f)
    if _singular(c):
        # the constant mode: the solver takes the right-hand side's mean out
        at = tuple(int(np.argmax(md[d][1])) for d in (2, 1, 0))
        lam[at], g[at] = 1.0, 0.0
    x = _along([V / w[:, None] for w, _, V in md], g / lam)
    return x - x.mean() if _singular(c) else x


def _exact_fft(c, seed):
    f = _rhs(c, seed)
    keep = c["dir"] - 1
    lam, T = 0.0, []
    for d, n in enumerate((c["nx"], c["ny"], c["nz"])):
        if d == keep:
            T.append(np.eye(n))
            continue
        k = np.arange(n)
        C = np.cos(np.pi * k[:, None] * (k[None, :] + 0.5) / n) * np.sqrt(np.where(k == 0, 1.0, 2.0) / n)[:, None]
        T.append(C)
        lam = lam + ((2.0 * np.cos(np.pi * k / n) - 2.0) * 64.0 ** 2).reshape([-1 if 2 - e == d else 1 for e in range(3)])
    lam = np.broadcast_to(lam, f.shape).copy()
    g = _along(T, f)
    zero = lam == 0.0
    lam[zero], g[zero] = 1.0, 0.0
    return _along([C.T for C in T], g / lam)


def _net(P, x):
    """The network in float64: x (1, 4, z, y, x)."""
    F = torch.nn.functional

    def conv(a, l, relu=True):
        a = F.conv3d(a, P[2 * l], P[2 * l + 1], padding=1)
        return F.relu(a) if relu else a

    def up(a):
        return F.interpolate(a, scale_factor=2, mode="nearest")

    e1 = conv(conv(x, 0), 1)
    e2 = conv(conv(F.avg_pool3d(e1, 2), 2), 3)
    b = conv(conv(F.avg_pool3d(e2, 2), 4), 5)
    d2 = conv(conv(torch.cat([up(b), e2], 1), 6), 7)
    return conv(conv(conv(torch.cat([up(d2), e1], 1), 8), 9), 10, relu=False)


def _parameters(seed):
    w, P, at = _weights(seed).astype(np.float64), [], 0
    for ci, co in LAYERS:
        W = w[at:at + 27 * ci * co].reshape(3, 3, 3, ci, co).transpose(4, 3, 0, 1, 2)
        at += 27 * ci * co
        P += [torch.tensor(np.ascontiguousarray(W)), torch.tensor(w[at:at + co])]
        at += co
    return P


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "ppe":
        return _exact_ppe(c, seed)
    if kind == "fft":
        return _exact_fft(c, seed)
    if kind == "unet_prec":
        dh = [np.diff(h)[1:-1] for h in _unet_nodes(c)]
        x, rms = _channels(c, _residual(c, seed) / (dh[2][:, None, None] * dh[1][None, :, None] * dh[0][None, None, :]))
        with torch.no_grad():
            return rms * _net(_parameters(seed), torch.tensor(x[None]))[0, 0]
    if kind == "unet_grad":
        x, t = (torch.tensor(a.astype(np.float64)) for a in _sample(c, seed))
        inner = (slice(1, -1),) * 3
        P = [p.requires_grad_() for p in _parameters(seed)]
        out = _net(P, x[(slice(None),) + inner].permute(0, 3, 2, 1)[None].contiguous())[0, 0]
        loss = ((out - t[inner].permute(2, 1, 0)) ** 2).mean()
        loss.backward()
        flat = [P[q].grad.permute(2, 3, 4, 1, 0).reshape(-1) if q % 2 == 0 else P[q].grad for q in range(len(P))]
        return {"loss": float(loss.detach()), "grad": torch.cat(flat)}
    return None
