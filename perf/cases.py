"""Timing cases of the framework's public entry points.

Each case is one call that a SFEMaNS run makes, on the inputs it has in hand
at that moment, device resident unless the case says otherwise:

* the azimuthal products at the nodes (``FFT_PAR_CROSS_PROD_DCL``), from a few
  hundred points to a full mesh, on device arrays and on the host arrays of a
  Fortran caller;
* the nonlinear term at the Gauss points, fused to its right-hand side, its
  tangent and its adjoint;
* the right-hand sides of the momentum and temperature equations;
* the products on the reference's own odd grid of a multiphase step (velocity
  from momentum, entropy viscosity).

Sizes are those of the bench workloads and tests (40x80, 158x316 and 224x448
squares, m_max from 8 to 128) with ragged ones between them.  Mode lists are
0..M-1.  Fields have N(0,1) coefficients with the spectral decay exp(-m/4).
"""
from __future__ import annotations

import math

import numpy as np
import torch

from sfemans_amd import fft_parallele as FP
from sfemans_amd import nonlinear as NL
from sfemans_amd.mesh import rectangle_p2
from sfemans_amd.synth import level_set_density

F64 = torch.float64


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # u x B at the nodes of a toy problem: launch and call cost
        {"name": "cross_small", "kind": "cross", "points": 500, "M": 8},
        # the same call from a host program with its arrays in host memory
        {"name": "cross_host", "kind": "cross_host", "points": 13041, "M": 16},
        # u x B at the nodes of a production mesh (Maxwell update)
        {"name": "cross_nodes", "kind": "cross", "points": 402753, "M": 64},
        # the nonlinear term of a small run: 6,400 triangles, 8 modes
        {"name": "nl_small", "kind": "nl", "nx": 40, "ny": 80, "M": 8},
        # the nonlinear term of a production run: 200,704 triangles, 64 modes
        {"name": "nl", "kind": "nl", "nx": 224, "ny": 448, "M": 64},
        # the nonlinear term fused to rhs_3x3, a mode count between two grids
        {"name": "nl_rhs", "kind": "nl_rhs", "nx": 150, "ny": 301, "M": 100},
        # adjoint of the linearised term (stability analysis), production size
        {"name": "adjoint", "kind": "adjoint", "nx": 224, "ny": 448, "M": 64},
        # tangent of the linearised term, the stability workload's size
        {"name": "tangent", "kind": "tangent", "nx": 158, "ny": 316, "M": 32},
        # full explicit momentum right-hand side with the LES stress
        {"name": "rhs_ns", "kind": "rhs_ns", "nx": 160, "ny": 321, "M": 48},
        # temperature right-hand side of a small run, ragged
        {"name": "temperature", "kind": "temperature", "nx": 113, "ny": 225, "M": 24},
        # velocity from momentum and level-set density at the nodes (division)
        {"name": "velocity", "kind": "velocity", "points": 402753, "M": 64},
        # entropy viscosity of the momentum equation at the Gauss points
        {"name": "entropy", "kind": "entropy", "points": 351232, "M": 32},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# points*M (or triangles*M) of the largest drawn case of a kind
_MOST = {"cross": 402753 * 64, "cross_host": 402753 * 8, "nl": 200704 * 64, "nl_rhs": 90300 * 100,
         "adjoint": 200704 * 40, "tangent": 99856 * 64, "rhs_ns": 102720 * 48, "temperature": 100000 * 48,
         "velocity": 402753 * 64, "entropy": 351232 * 32}
_HIGH = {"cross": 128, "cross_host": 64, "nl": 128, "nl_rhs": 128, "adjoint": 128, "tangent": 128, "rhs_ns": 96,
         "temperature": 128, "velocity": 96, "entropy": 64}


def draw(rng):
    kind = rng.choice(sorted(_MOST))
    M = _log_int(rng, 6, _HIGH[kind])
    # the products cost the same per mode up to a padded grid, the direct sums
    # of the odd grid grow with M
    room = _MOST[kind] / M if kind not in ("velocity", "entropy") else _MOST[kind] / M * min(1.0, 48.0 / M)
    if M & (M - 1) and kind not in ("velocity", "entropy", "rhs_ns"):
        room *= M / float(1 << M.bit_length())
    if kind in ("cross", "cross_host", "velocity"):
        return {"kind": kind, "points": _log_int(rng, 500, max(600, min(402753, room))), "M": M}
    if kind == "entropy":
        return {"kind": kind, "points": 7 * _log_int(rng, 100, max(120, min(200704, room / 7))), "M": M}
    me = _log_int(rng, 400, max(500, min(200704, room)))
    nx = max(5, int(math.sqrt(me / 4.0) * rng.uniform(0.8, 1.25)))
    return {"kind": kind, "nx": nx, "ny": max(5, me // (2 * nx)), "M": M}


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _field(gen, npts, nc, M, decay=4.0, mean=None, scale=1.0):
    """(M, nc, npts): N(0,1) exp(-m/decay), no sine of mode 0."""
    t = torch.randn((M, nc, npts), generator=gen, device="cuda", dtype=F64)
    t *= (scale * torch.exp(-torch.arange(M, device="cuda", dtype=F64) / decay))[:, None, None]
    t[0, 1::2] = 0.0
    if mean is not None:
        t[0, 0] = mean
    return t


def _f(t):
    """The Fortran view (points, columns, modes) of a base array."""
    return t.permute(*reversed(range(t.dim())))


def _density(gen, npts, M):
    """Coefficients of the density of a level set (a sphere) at random meridian points."""
    x = torch.rand((2, npts), generator=gen, device="cuda", dtype=F64)
    rr = np.stack([x[0].cpu().numpy(), 2.0 * x[1].cpu().numpy() - 1.0])
    c = torch.rand(2, generator=gen, device="cuda", dtype=F64).cpu()
    return level_set_density(torch, rr, M, x0=0.2 + 0.2 * float(c[0]), radius=0.2 + 0.1 * float(c[1]))


def _inputs(case, seed):
    """The arrays of a case, (modes, columns, points) contiguous, on the GPU."""
    g, k, M = _gen(seed), case["kind"], case["M"]
    if k in ("cross", "cross_host"):
        n = case["points"]
        return {"a": _field(g, n, 6, M), "b": _field(g, n, 6, M)}
    if k == "velocity":
        n = case["points"]
        return {"m": _field(g, n, 6, M), "rho": _density(g, n, M).permute(2, 1, 0)}
    if k == "entropy":
        n = case["points"]
        d = {n_: _field(g, n, 6, M) for n_ in ("u", "res", "g1", "g2", "g3")}
        d["h"] = 0.005 + 0.01 * torch.rand(n // 7, generator=g, device="cuda", dtype=F64).repeat_interleave(7)
        return d
    me = 2 * case["nx"] * case["ny"]
    n, G = (2 * case["nx"] + 1) * (2 * case["ny"] + 1), 7 * me
    d = {"u": _field(g, n, 6, M)}
    if k == "adjoint":
        d["y"] = _field(g, G, 6, M)
    elif k == "tangent":
        d["u"][5:] = 0.0
        d["u"][1:5] *= 0.1
        d["d"] = _field(g, n, 6, M, 2.0)
    elif k == "temperature":
        d["T"], d["ff"] = _field(g, n, 2, M), _field(g, n, 2, M)
        d["hc"] = 0.5 + torch.rand(me, generator=g, device="cuda", dtype=F64)
    elif k == "rhs_ns":
        d["rotv"], d["ff"] = _field(g, G, 6, M), _field(g, n, 6, M)
        d["p"], d["pinc"] = _field(g, n, 2, M), _field(g, n, 2, M, scale=0.1)
        t = torch.randn((M, 6, G, 3), generator=g, device="cuda", dtype=F64)
        t *= (0.01 * torch.exp(-torch.arange(M, device="cuda", dtype=F64) / 4.0))[:, None, None, None]
        d["tensor"] = t
    return d


def _p2(case):
    return rectangle_p2(case["nx"], case["ny"])


def prepare(case, seed):
    k, M = case["kind"], case["M"]
    s = {"kind": k, "modes": list(range(M))}
    d = _inputs(case, seed)
    if k == "cross_host":
        s |= {n: np.asfortranarray(_f(t).cpu().numpy()) for n, t in d.items()}
        s["out"] = np.zeros((case["points"], 6, M), order="F")
        return s
    s |= {n: _f(t) for n, t in d.items()}
    if k == "cross" or k == "velocity":
        s["out"] = FP.fortran_empty((case["points"], 6, M))
        return s
    if k == "entropy":
        s["outs"] = [FP.fortran_empty((case["points"], 6, M)) for _ in range(3)]
        return s
    p2 = _p2(case)
    s["mesh"] = mesh = NL.Mesh.from_p2(p2)
    n, G, me = p2.np, p2.n_gauss, p2.me
    if k == "nl" or k == "tangent":
        s["out"] = FP.fortran_empty((G, 6, M))
    elif k == "nl_rhs" or k == "rhs_ns":
        s["v145"], s["v236"] = FP.fortran_empty((n, 3, M)), FP.fortran_empty((n, 3, M))
        s["work"] = torch.empty(36 * me * M, dtype=F64, device="cuda")
    elif k == "adjoint":
        s["out"] = FP.fortran_empty((n, 6, M))
        s["work"] = torch.empty(36 * me * M, dtype=F64, device="cuda")
    elif k == "temperature":
        s["out"] = FP.fortran_empty((n, 2, M))
        s["work"] = torch.empty(12 * me * M, dtype=F64, device="cuda")
    mesh.list_mode_device(s["modes"])
    return s


# the entropy viscosity's parameters: residual normalisation, LES_coeff1, 2, 4
_RES, _C1, _C2, _C4 = 1.0, 0.3, 0.9, 0.8


def run(s):
    k = s["kind"]
    if k in ("cross", "cross_host"):
        return FP.FFT_PAR_CROSS_PROD_DCL(None, s["a"], s["b"], s["out"])
    if k == "velocity":
        return FP.FFT_SCALAR_VECT_DCL(None, s["m"], s["rho"], s["out"], 2)
    if k == "entropy":
        return list(FP.FFT_COMPUTE_ENTROPY_VISC(None, None, s["u"], s["res"], s["g1"], s["g2"], s["g3"], s["h"],
                                                *s["outs"], _RES, 7, _C1, _C2, _C4))
    mesh, modes = s["mesh"], s["modes"]
    if k == "nl":
        return NL.smb_cross_prod_gauss_sft_par(None, mesh, modes, s["u"], s["out"])
    if k == "nl_rhs":
        return list(NL.nl_rhs_3x3(mesh, modes, s["u"], s["v145"], s["v236"], -1.0, s["work"]))
    if k == "adjoint":
        return NL.nl_adjoint(mesh, modes, s["u"], s["y"], s["out"], s["work"])
    if k == "tangent":
        return NL.nl_tangent(mesh, modes, s["u"], s["d"], s["out"])
    if k == "temperature":
        return NL.nl_qs_00(mesh, modes, s["hc"], s["u"], s["T"], s["out"], s["ff"], -1.0, s["work"])
    return list(NL.rhs_ns_3x3(mesh, modes, s["rotv"], s["u"], s["ff"], s["p"], s["pinc"], s["v145"], s["v236"],
                              s["work"], opt_tensor=s["tensor"]))


# ---------------------------------------------------------------- work

def _fft(M, nf, ops):
    """Flops per point of nf real transforms and ops flops per angle on the 3/2 grid."""
    N = 3 * M
    return nf * 2.5 * N * math.log2(N) + ops * N


def work(case):
    """Inputs read once, outputs written once; real transforms at 2.5 N log2 N
    on the 3/2 grid, or 4 M m_max_pad (sums folded over the angle pairs) on the
    reference's odd, often prime grid."""
    k, M = case["kind"], case["M"]
    if k in ("cross", "cross_host"):
        return {"bytes": 18.0 * 8 * case["points"] * M, "flops": case["points"] * _fft(M, 9, 9)}
    if k == "velocity":
        return {"bytes": 14.0 * 8 * case["points"] * M, "flops": case["points"] * 7.0 * 4 * M * (3 * M // 2)}
    if k == "entropy":
        return {"bytes": 8.0 * case["points"] * (48 * M + 1), "flops": case["points"] * 24.0 * 4 * M * (3 * M // 2)}
    me = 2 * case["nx"] * case["ny"]
    n, G = (2 * case["nx"] + 1) * (2 * case["ny"] + 1), 7 * me
    mesh = 24.0 * me + 16.0 * n
    nod, gau = 48.0 * n * M, 48.0 * G * M
    b2 = G * (_fft(M, 9, 9) + 168.0 * M)
    if k == "nl":
        return {"bytes": nod + gau + mesh, "flops": b2}
    if k == "nl_rhs":
        return {"bytes": 2 * nod + mesh, "flops": b2 + 72.0 * G * M}
    if k == "adjoint":
        return {"bytes": 2 * nod + gau + mesh, "flops": 2 * b2}
    if k == "tangent":
        return {"bytes": 2 * nod + gau + mesh, "flops": G * (_fft(M, 15, 18) + 336.0 * M)}
    if k == "temperature":
        return {"bytes": 2 * nod + mesh, "flops": G * (_fft(M, 9, 8) + 160.0 * M)}
    return {"bytes": 3 * nod + 2 * nod / 3 + 4 * gau + mesh, "flops": G * M * 500.0}


# ------------------------------------------- the same results in plain torch

def _tables(M, N):
    """cos and sin (2 pi m j / N), (M, N), from exact residues of m j mod N."""
    mj = (np.arange(M, dtype=np.int64)[:, None] * np.arange(N, dtype=np.int64)[None, :]) % N
    t = 2 * np.longdouble("3.141592653589793238462643383279502884197") * mj.astype(np.longdouble) / N
    dev = lambda x: torch.tensor(x.astype(np.float64), device="cuda")
    return dev(np.cos(t)), dev(np.sin(t))


class _Dft:
    def __init__(self, M, N=None):
        self.M, self.N = M, 2 * (3 * M // 2) - 1 if N is None else N
        self.c, self.s = _tables(M, self.N)
        self.w = torch.full((M, 1), 2.0 / self.N, device="cuda", dtype=F64)
        self.w[0] = 1.0 / self.N

    def grid(self, c):
        """(M, 2, n) coefficients -> (N, n) values."""
        return self.c.t() @ c[:, 0] + self.s[1:].t() @ c[1:, 1]

    def fields(self, v):
        """(M, 2 k, n) -> k arrays of values."""
        return [self.grid(v[:, 2 * i:2 * i + 2]) for i in range(v.shape[1] // 2)]

    def back(self, ws):
        """k arrays (N, n) -> (M, 2 k, n); the sine of mode 0 is zero."""
        return torch.stack([x for w in ws for x in (self.w * (self.c @ w), self.w * (self.s @ w))], dim=1)


def _cross(a, b):
    return [a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]]


def _element():
    """Quadratic shape functions w(6,7), their derivatives d(2,6,7) and the weights of the 7-point rule."""
    sq = math.sqrt(15.0)
    s1, t1, s2, t2 = (6 - sq) / 21, (9 + 2 * sq) / 21, (6 + sq) / 21, (9 - 2 * sq) / 21
    x = np.array([1 / 3, s1, s1, t1, s2, s2, t2])
    y = np.array([1 / 3, s1, t1, s1, s2, t2, s2])
    p = 0.5 * np.array([9 / 40] + 3 * [(155 - sq) / 1200] + 3 * [(155 + sq) / 1200])
    z = 1 - x - y
    w = np.stack([z * (2 * z - 1), x * (2 * x - 1), y * (2 * y - 1), 4 * x * y, 4 * y * z, 4 * x * z])
    o = np.zeros(7)
    dx = np.stack([1 - 4 * z, 4 * x - 1, o, 4 * y, -4 * y, 4 * (z - x)])
    dy = np.stack([1 - 4 * z, o, 4 * y - 1, 4 * x, 4 * (z - y), -4 * x])
    return tuple(torch.tensor(v, device="cuda") for v in (w, np.stack([dx, dy]), p))


class _Fem:
    """Gauss values of nodal fields on the elements e0..e1 of a mesh."""

    def __init__(self, p2, e0, e1):
        self.jj = torch.tensor(p2.jj[:, e0:e1].astype(np.int64) - 1, device="cuda")      # (6, e)
        rr = torch.tensor(p2.rr, device="cuda")[:, self.jj]                              # (2, 6, e)
        self.w, dd, p = _element()
        J = torch.einsum("knm,jnl->kjml", rr, dd)                                        # (2, 2, e, 7)
        det = J[0, 0] * J[1, 1] - J[0, 1] * J[1, 0]
        self.dr = (dd[0][:, None, :] * J[1, 1] - dd[1][:, None, :] * J[1, 0]) / det      # (6, e, 7)
        self.dz = (dd[1][:, None, :] * J[0, 0] - dd[0][:, None, :] * J[0, 1]) / det
        self.r = torch.einsum("nm,nl->ml", rr[0], self.w)
        self.wgt = det.abs() * p * self.r                                                # (e, 7)

    def at(self, v):
        """v (M, c, np) -> values, d/dr, d/dz, each (M, c, e, 7)."""
        x = v[:, :, self.jj]                                                             # (M, c, 6, e)
        out = [0.0, 0.0, 0.0]
        for n in range(6):
            xn = x[:, :, n, :, None]
            out = [out[0] + xn * self.w[n], out[1] + xn * self.dr[n], out[2] + xn * self.dz[n]]
        return out

    def value_curl(self, v, m):
        W, R, Z = self.at(v)
        q = m[:, None, None] / self.r
        c = [q * W[:, 5] - Z[:, 2], -q * W[:, 4] - Z[:, 3], Z[:, 0] - R[:, 4], Z[:, 1] - R[:, 5],
             W[:, 2] / self.r + R[:, 2] - q * W[:, 1], W[:, 3] / self.r + R[:, 3] + q * W[:, 0]]
        return W, torch.stack(c, dim=1)

    def scatter(self, out, g, grad_r=None, grad_z=None):
        """out (M, c, np) += sum over the Gauss points of wgt (w g + dw/dr grad_r + dw/dz grad_z)."""
        for n in range(6):
            t = (g * (self.w[n] * self.wgt)).sum(-1)
            if grad_r is not None:
                t = t + (grad_r * (self.dr[n] * self.wgt) + grad_z * (self.dz[n] * self.wgt)).sum(-1)
            out.index_add_(2, self.jj[n], t)


def _pt(x):
    return x.reshape(x.shape[0], x.shape[1], -1)


def exact(case, seed):
    k, M = case["kind"], case["M"]
    d, D = _inputs(case, seed), _Dft(M)
    m = torch.arange(M, device="cuda", dtype=F64)
    if k in ("cross", "cross_host", "velocity"):
        n = case["points"]
        out = torch.empty((M, 6, n), device="cuda", dtype=F64)
        for i in range(0, n, 65536):
            c = slice(i, min(n, i + 65536))
            if k == "velocity":
                rho = D.grid(d["rho"][..., c])
                w = [x / rho for x in D.fields(d["m"][..., c])]
            else:
                w = _cross(D.fields(d["a"][..., c]), D.fields(d["b"][..., c]))
            out[..., c] = D.back(w)
        return _f(out).cpu() if k == "cross_host" else _f(out)
    if k == "entropy":
        n = case["points"]
        outs = [torch.empty((M, 6, n), device="cuda", dtype=F64) for _ in range(3)]
        for i in range(0, n, 7 * 8192):
            c = slice(i, min(n, i + 7 * 8192))
            u, r = D.fields(d["u"][..., c]), D.fields(d["res"][..., c])
            a = (u[0] ** 2 + u[1] ** 2 + u[2] ** 2).sqrt().reshape(D.N, -1, 7).amax(-1)
            a = torch.maximum(a, torch.maximum(a.roll(1, 0), a.roll(-1, 0))).repeat_interleave(7, dim=1)
            dot = (u[0] * r[0] + u[1] * r[1] + u[2] * r[2]).abs()
            v = -_C1 + torch.minimum(_C4 * a, _C2 * d["h"][c] * dot / (_RES + 1.0e-14))
            for o, name in zip(outs, ("g1", "g2", "g3")):
                o[..., c] = D.back([v * x for x in D.fields(d[name][..., c])])
        return [_f(o) for o in outs]
    p2 = _p2(case)
    me, n = p2.me, p2.np
    step = max(512, int(40_000_000 / (42 * M)))
    blocks = [(e, min(me, e + step)) for e in range(0, me, step)]

    def term(fem, a, b):
        """P[(curl a) x b] at the Gauss points of a block, (M, 6, points)."""
        Wa, Ra = fem.value_curl(a, m)
        Wb = Wa if a is b else fem.at(b)[0]
        return D.back(_cross(D.fields(_pt(Ra)), D.fields(_pt(Wb))))

    if k in ("nl", "tangent"):
        out = torch.empty((M, 6, 7 * me), device="cuda", dtype=F64)
        for e0, e1 in blocks:
            fem = _Fem(p2, e0, e1)
            if k == "nl":
                out[..., 7 * e0:7 * e1] = term(fem, d["u"], d["u"])
            else:
                out[..., 7 * e0:7 * e1] = term(fem, d["u"], d["d"]) + term(fem, d["d"], d["u"])
        return _f(out)
    if k == "adjoint":
        # F is quadratic: its tangent's transpose is the gradient of <F(u), y>
        out = torch.zeros((M, 6, n), device="cuda", dtype=F64)
        for e0, e1 in blocks:
            fem = _Fem(p2, e0, e1)
            nodes = torch.unique(fem.jj)
            local = torch.empty(n, dtype=torch.int64, device="cuda")
            local[nodes] = torch.arange(len(nodes), device="cuda")
            fem.jj = local[fem.jj]
            u = d["u"][..., nodes].clone().requires_grad_(True)
            term(fem, u, u).backward(d["y"][..., 7 * e0:7 * e1])
            out.index_add_(2, nodes, u.grad)
        return _f(out)
    if k == "nl_rhs":
        v = torch.zeros((M, 6, n), device="cuda", dtype=F64)
        for e0, e1 in blocks:
            fem = _Fem(p2, e0, e1)
            fem.scatter(v, -term(fem, d["u"], d["u"]).reshape(M, 6, -1, 7))
        return [_f(v[:, [0, 3, 4]]), _f(v[:, [1, 2, 5]])]
    if k == "temperature":
        v = torch.zeros((M, 2, n), device="cuda", dtype=F64)
        for e0, e1 in blocks:
            fem = _Fem(p2, e0, e1)
            W, R, Z = fem.at(d["u"])
            C, Cr, Cz = fem.at(d["T"])
            hc = d["hc"][e0:e1, None]
            q = m[:, None, None] / fem.r
            div = torch.stack([R[:, 0] + W[:, 0] / fem.r + q * W[:, 3] + Z[:, 4],
                               R[:, 1] + W[:, 1] / fem.r - q * W[:, 2] + Z[:, 5]], dim=1)
            g = hc * torch.stack([Cr[:, 0], Cr[:, 1], q * C[:, 1], -q * C[:, 0], Cz[:, 0], Cz[:, 1]], dim=1)
            gf, uf = D.fields(_pt(g)), D.fields(_pt(W))
            t = sum(x * y for x, y in zip(gf, uf)) + D.grid(_pt(div)) * D.grid(_pt(hc * C))
            t = D.back([t]).reshape(M, 2, -1, 7)
            fem.scatter(v, -(hc * fem.at(d["ff"])[0] + t))
        return _f(v)
    v = torch.zeros((M, 6, n), device="cuda", dtype=F64)
    for e0, e1 in blocks:
        fem = _Fem(p2, e0, e1)
        q = m[:, None, None] / fem.r
        g = fem.at(d["u"])[0] + fem.at(d["ff"])[0] - d["rotv"][..., 7 * e0:7 * e1].reshape(M, 6, -1, 7)
        for name in ("p", "pinc"):
            P, Pr, Pz = fem.at(d[name])
            g = g + torch.stack([-Pr[:, 0], -Pr[:, 1], -q * P[:, 1], q * P[:, 0], -Pz[:, 0], -Pz[:, 1]], dim=1)
        T = d["tensor"][:, :, 7 * e0:7 * e1].reshape(M, 6, -1, 7, 3)
        mm, r = m[:, None, None], fem.r
        g = g + torch.stack([-mm * T[:, 3, ..., 0] + T[:, 2, ..., 1], mm * T[:, 2, ..., 0] + T[:, 3, ..., 1],
                             -T[:, 2, ..., 0] - mm * T[:, 3, ..., 1], -T[:, 3, ..., 0] + mm * T[:, 2, ..., 1],
                             -mm * T[:, 3, ..., 2], mm * T[:, 2, ..., 2]], dim=1) / r
        gr = torch.stack([T[:, c % 2, ..., c // 2] for c in range(6)], dim=1)
        gz = torch.stack([T[:, 4 + c % 2, ..., c // 2] for c in range(6)], dim=1)
        fem.scatter(v, g, gr, gz)
    return [_f(v[:, [0, 3, 4]]), _f(v[:, [1, 2, 5]])]
