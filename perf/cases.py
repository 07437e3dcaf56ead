"""Workloads of the even-odd domain-wall path, through its public entry points.

A case is a dict of plain values.  `kind` names the call:

  hermop   Mpc^+ Mpc of a half field in device memory (FP64), what a caller's
           own eigensolver, smoother or CG applies
  mhost    multiply_m / multiply_mdag of a full 5D field in host memory
  solve5d  one 5D source, device memory, with one of the three solvers
  prop     a 12-column point-source propagator, device memory
  batch    several 5D sources times several masses in one call
  force    the fermion force and link gradient of one pseudofermion
  qed      one 4D source with the U(1) domain-wall operator, host memory

Links are exp(i 0.3 H) with Gaussian H and antiperiodic time, M5 = 1.8, the
synthetic configuration of the repository's benchmark and tests.  The solvers
run to tight residuals (1e-11, 1e-12), as for a force or a low-noise
correlator: solutions then agree to 1e-9 whatever their rounding.
"""

import math

import numpy as np
import torch

import qlattice_amd as q

M5 = 1.8
SIGMA = 0.3
KINDS = ("hermop", "mhost", "solve5d", "prop", "batch", "force", "qed")


def listed():
    return [
        # the smallest lattice of the test suite: launches and latency only
        {"name": "hermop_4c8_ls8", "kind": "hermop", "site": "4.4.4.8", "ls": 8, "scale": 2.0, "mass": 0.1, "eo": 1},
        # a thermalisation-size lattice that fits the last-level cache
        {"name": "hermop_16c32_ls8", "kind": "hermop", "site": "16.16.16.32", "ls": 8, "scale": 2.0, "mass": 0.03,
         "eo": 1},
        # the benchmark's lattice: fields far beyond any cache
        {"name": "hermop_24c64_ls12", "kind": "hermop", "site": "24.24.24.64", "ls": 12, "scale": 2.0, "mass": 0.01,
         "eo": 1},
        # unequal extents, a half volume that is no multiple of a block, an Ls
        # between the kernels' sizes, complex fifth-dimension coefficients
        {"name": "hermop_ragged_zmobius_ls10", "kind": "hermop", "site": "6.10.14.22", "ls": 10, "scale": 0.0,
         "mass": 0.05, "eo": 2},
        # the full operator on numpy fields, as a script checking a solution calls it
        {"name": "mdag_host_12c24_ls12", "kind": "mhost", "site": "12.12.12.24", "ls": 12, "scale": 2.0, "mass": 0.01,
         "dag": True},
        # the default (FP64) solver on the smallest lattice of the benchmark
        {"name": "solve_fp64_8c16_ls8", "kind": "solve5d", "site": "8.8.8.16", "ls": 8, "scale": 2.0, "mass": 0.1,
         "solver": "fp64", "stop": 1e-11},
        # one column at the benchmark's size with the FP32 solver
        {"name": "solve_mixed_24c64_ls12", "kind": "solve5d", "site": "24.24.24.64", "ls": 12, "scale": 2.0,
         "mass": 0.1, "solver": "mixed", "stop": 1e-11},
        # a propagator on a small lattice with the fifth dimension of production actions
        {"name": "prop_mixed16_8c16_ls24", "kind": "prop", "site": "8.8.8.16", "ls": 24, "scale": 4.0, "mass": 0.1,
         "solver": "mixed16", "stop": 1e-11},
        # a propagator on the lattice of the batch and force workloads
        {"name": "prop_mixed16_16c32_ls12", "kind": "prop", "site": "16.16.16.32", "ls": 12, "scale": 2.0,
         "mass": 0.05, "solver": "mixed16", "stop": 1e-11},
        # noise sources times four masses in one call, columns retiring at different times
        {"name": "batch_mixed16_16c32_ls8", "kind": "batch", "site": "16.16.16.32", "ls": 8, "scale": 2.0,
         "masses": "0.02/0.05/0.1/0.3", "sources": 3, "solver": "mixed16", "stop": 1e-11},
        # one force evaluation of a molecular-dynamics step
        {"name": "force_16c32_ls8", "kind": "force", "site": "16.16.16.32", "ls": 8, "scale": 2.0, "mass": 0.1,
         "stop": 1e-11},
        # a QED column on numpy fields
        {"name": "qed_8c16_ls8", "kind": "qed", "site": "8.8.8.16", "ls": 8, "scale": 1.0, "mass": 0.1,
         "stop": 1e-12},
    ]


# A draw keeps to the listed sizes' span: lattices from 4^3 x 8 up, with
# unequal extents, every Ls the kinds meet, and at most this many
# 5D-site-columns (the listed maximum of the kind).
_CAP = {"hermop": 24**3 * 64 * 12, "mhost": 12**3 * 24 * 12, "solve5d": 24**3 * 64 * 6, "prop": 16**3 * 32 * 12 * 8,
        "batch": 16**3 * 32 * 8 * 8, "force": 16**3 * 32 * 8, "qed": 8**3 * 16 * 8}


def draw(rng):
    kind = rng.choice(("hermop", "hermop", "mhost", "solve5d", "prop", "batch", "force", "qed"))
    ls = rng.choice((8,) if kind == "qed" else (6, 8, 8, 10, 12, 12, 14, 16, 20, 24))
    ncol = {"prop": 12, "batch": 6}.get(kind, 1)
    lo, hi = 4**3 * 8, _CAP[kind] // (ls * ncol)
    vol = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    side = max(2.0, (vol / 2.0) ** 0.25)
    while True:
        site = [2 * max(2, round(0.5 * side * f * rng.uniform(0.75, 1.3))) for f in (1.0, 1.0, 1.0, 1.8)]
        if math.prod(site) <= hi:
            break
        side *= 0.95
    case = {"kind": kind, "site": ".".join(map(str, site)), "ls": ls, "scale": rng.choice((1.0, 2.0, 2.0, 4.0)),
            "mass": round(rng.uniform(0.03, 0.3), 3)}
    if kind == "hermop":
        case["eo"] = rng.choice((1, 2))
        if rng.random() < 0.3:
            case["scale"] = 0.0
    elif kind == "mhost":
        case["dag"] = rng.random() < 0.5
    elif kind in ("solve5d", "prop"):
        case["solver"] = rng.choice(("fp64", "mixed", "mixed16")) if kind == "solve5d" else rng.choice(("mixed", "mixed16"))
        case["stop"] = 1e-11
    elif kind == "batch":
        case["masses"] = rng.choice(("0.03/0.1", "0.02/0.05/0.2"))
        case["sources"] = 6 // len(case["masses"].split("/"))
        case["solver"], case["stop"] = rng.choice(("mixed", "mixed16")), 1e-11
        del case["mass"]
    elif kind == "force":
        case["stop"] = 1e-11
    else:
        case["scale"], case["stop"] = 1.0, 1e-12
    return case


# ------------------------------------------------------------------ inputs


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _site(case):
    return tuple(int(v) for v in case["site"].split("."))


def _masses(case):
    return [float(m) for m in case["masses"].split("/")] if "masses" in case else [case["mass"]]


def _generator(seed):
    return torch.Generator(device=_device()).manual_seed(seed)


def _noise(gen, *shape):
    re_im = torch.randn(*shape, 2, generator=gen, device=_device(), dtype=torch.float64)
    return torch.view_as_complex(re_im)


def _links(site, gen):
    """(V, 4, 3, 3) SU(3) links exp(i SIGMA H), antiperiodic in time."""
    n = math.prod(site) * 4
    h = torch.randn(n, 8, generator=gen, device=_device(), dtype=torch.float64)
    a = torch.zeros(n, 3, 3, device=_device(), dtype=torch.complex128)
    for k, (r, c) in enumerate(((0, 1), (0, 2), (1, 2))):
        a[:, r, c] = 0.5 * (h[:, 2 * k] - 1j * h[:, 2 * k + 1])
        a[:, c, r] = 0.5 * (h[:, 2 * k] + 1j * h[:, 2 * k + 1])
    d8 = 0.5 * h[:, 7] / math.sqrt(3.0)
    a[:, 0, 0], a[:, 1, 1], a[:, 2, 2] = 0.5 * h[:, 6] + d8, d8 - 0.5 * h[:, 6], -2.0 * d8
    a *= 1j * SIGMA / 16.0
    out = torch.eye(3, device=a.device, dtype=a.dtype).expand_as(a).clone()
    term = out.clone()
    for k in range(1, 13):  # exp by its series at 1/16 of the argument, then four squarings
        term = _mul3(term, a) / k
        out += term
    for _ in range(4):
        out = _mul3(out, out)
    u = out.view(site[3], -1, 4, 3, 3)
    u[site[3] - 1, :, 3] *= -1.0
    return out.view(-1, 4, 3, 3)


def _mul3(a, b):
    return (a[:, :, 0, None] * b[:, None, 0] + a[:, :, 1, None] * b[:, None, 1]) + a[:, :, 2, None] * b[:, None, 2]


def _coefficients(case):
    """(b_s, c_s): Moebius from the scale, zMoebius (scale 0) from complex omega."""
    ls = case["ls"]
    if case["scale"] > 0:
        return np.full(ls, 0.5 * case["scale"] + 0.5 + 0j), np.full(ls, 0.5 * case["scale"] - 0.5 + 0j)
    b = 0.5 * (1.0 / np.asarray(_omega(ls)) + 1.0)
    return b, b - 1.0


def _omega(ls):
    om = [complex(1.1 - 0.8 * s / (ls - 1)) for s in range(ls)]
    om[-2], om[-1] = complex(0.35, -0.05), complex(0.35, 0.05)
    return om


def _fields(case, seed):
    """Links and the field or fields that the call works on."""
    gen, site, ls = _generator(seed), _site(case), case["ls"]
    vol = math.prod(site)
    if case["kind"] == "qed":
        phase = 0.3 * torch.randn(vol, 4, generator=gen, device=_device(), dtype=torch.float64)
        return torch.polar(torch.ones_like(phase), phase), _noise(gen, vol, 4)
    u = _links(site, gen)
    if case["kind"] in ("hermop", "force"):
        return u, _noise(gen, vol // 2, ls, 12)
    if case["kind"] == "prop":
        src = torch.zeros(vol, 12, 12, device=_device(), dtype=torch.complex128)
        x = int(torch.randint(vol, (1,), generator=gen, device=_device()))
        src[x] = torch.eye(12, device=_device(), dtype=src.dtype)
        return u, src
    if case["kind"] == "batch":
        return u, [_noise(gen, vol, ls, 12) for _ in range(case["sources"])]
    return u, _noise(gen, vol, ls, 12)


# ------------------------------------------------------------------- calls


def _inverter(case, gf, mass):
    omega = None if case["scale"] > 0 else _omega(case["ls"])
    fa = q.FermionAction(mass=mass, ls=case["ls"], m5=M5, mobius_scale=case["scale"], omega=omega)
    inv = q.InverterDomainWall(gf=gf, fa=fa, solver=case.get("solver", "fp64"))
    inv.set_stop_rsd(case.get("stop", 1e-8))
    inv.set_max_num_iter(2000)
    return inv


def prepare(case, seed):
    u, f = _fields(case, seed)
    site = _site(case)
    if case["kind"] == "qed":
        return {"case": case, "gf1": u.cpu().numpy(), "src": f.cpu().numpy(), "site": site}
    geo = q.Geometry(site)
    gf = q.GaugeField(geo)
    gf.data = u.cpu().numpy()
    invs = [_inverter(case, gf, m) for m in _masses(case)]
    state = {"case": case, "inv": invs[0], "invs": invs, "lib": q.load_library()}
    if case["kind"] == "mhost":
        state["src"] = q.FermionField5d(geo, case["ls"], 0)
        state["src"].data = f.cpu().numpy()
    elif case["kind"] == "batch":
        state["src"] = f * len(invs)
        state["cdata"] = [inv.cdata for inv in invs for _ in f]
        state["out"] = [torch.empty_like(s) for s in state["src"]]
    else:
        state["src"] = f
        state["out"] = torch.empty_like(f)
        if case["kind"] == "force":
            del state["out"]
            state["force"], state["grad"] = torch.empty_like(u), torch.empty_like(u)
    if torch.cuda.is_available():
        torch.cuda.synchronize()
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "qed":
        out, _ = q.invert_dwf_qed(state["src"], state["gf1"], case["mass"], M5, case["ls"], state["site"],
                                  stop_rsd=case["stop"])
        return out
    inv, lib = state["inv"], state["lib"]
    if kind == "hermop":
        lib.multiply_hermop_sym2_device(inv.cdata, state["out"].data_ptr(), state["src"].data_ptr(), case["eo"])
    elif kind == "mhost":
        return (q.multiply_mdag if case["dag"] else q.multiply_m)(None, state["src"], inv).data
    elif kind == "solve5d":
        lib.invert_5d(inv.cdata, state["out"].data_ptr(), state["src"].data_ptr(), True)
    elif kind == "prop":
        lib.invert_prop(inv.cdata, state["out"].data_ptr(), state["src"].data_ptr(), True)
    elif kind == "batch":
        lib.invert_5d_batch(state["cdata"], [t.data_ptr() for t in state["out"]],
                            [t.data_ptr() for t in state["src"]], True)
    else:
        action, _, _ = lib.fermion_force(inv.cdata, state["src"].data_ptr(), case["stop"], state["force"].data_ptr(),
                                         state["grad"].data_ptr(), True)
        return {"action": action, "force": state["force"], "grad": state["grad"]}
    return state["out"]


# -------------------------------------------------------------------- work


def work(case):
    """Inputs and outputs once; the arithmetic of a solve for a nominal 16
    iterations per decade of the residual."""
    vol, ls, kind = math.prod(_site(case)), case["ls"], case["kind"]
    nc = 1 if kind == "qed" else 3
    n5 = vol // 2 * ls  # 5D sites of one parity
    hop = 128 * nc * nc + 56 * nc  # 1320 for colour
    smat = 2 * 24 * ls if case["scale"] > 0 else 4 * 24 * ls
    links = vol * 4 * nc * nc * 16
    field = 16 * 4 * nc  # one FP64 spinor
    hermop = n5 * (4 * hop + 4 * smat)
    if kind == "hermop":
        return {"bytes": 2 * n5 * field + links, "flops": hermop}
    if kind == "mhost":
        return {"bytes": 4 * n5 * field + links, "flops": 2 * n5 * (hop + 2 * smat)}
    iters = -16.0 * math.log10(case["stop"])
    ncol = {"prop": 12, "batch": len(_masses(case)) * case.get("sources", 1)}.get(kind, 1)
    ends = {"prop": 2 * vol * 144 * 16, "force": n5 * field + 2 * links, "qed": 2 * vol * field}.get(
        kind, 4 * n5 * field * ncol)
    return {"bytes": ends + links, "flops": iters * ncol * hermop * (2 if kind == "qed" else 1)}


# --------------------------------------------------- the same in plain torch


class _Dwf:
    """The domain-wall operator on full-lattice fields [T, Z, Y, X, colour,
    column, spin, s] in complex128; a half field is one with zeros on the
    other parity."""

    def __init__(self, case, mass, links):
        site, ls = _site(case), case["ls"]
        self.site, self.ls = site, ls
        self.nc = 1 if case["kind"] == "qed" else 3
        self.u = links.reshape(*reversed(site), 4, self.nc, self.nc)
        b, c = _coefficients(case)
        eye = np.eye(ls)
        down, up = np.eye(ls, k=-1), np.eye(ls, k=1)
        down[0, ls - 1] = up[ls - 1, 0] = -mass
        d = np.diag
        pre = [d(b) + d(c) @ s for s in (down, up)]
        mee = [d(1 + b * (4 - M5)) - d(1 - c * (4 - M5)) @ s for s in (down, up)]
        inv = [np.linalg.inv(m) for m in mee]
        sets = {"P": pre, "M": mee, "I": inv, "K": [p @ i for p, i in zip(pre, inv)], "C": [d(1 - c * (4 - M5))] * 2,
                "N": [-d(c)] * 2}
        self.mat = {}
        for k, ms in sets.items():
            self.mat[k] = [torch.tensor(m + 0j * eye, device=links.device) for m in ms]
            self.mat[k + "+"] = [m.conj().T.contiguous() for m in self.mat[k]]
        x = torch.meshgrid(*[torch.arange(n, device=links.device) for n in reversed(site)], indexing="ij")
        odd = (x[0] + x[1] + x[2] + x[3]) % 2
        self.odd = odd.reshape(-1).bool()
        self.mask = {1: odd[..., None, None, None, None].double(), 2: (1 - odd)[..., None, None, None, None].double()}

    def s(self, name, f):
        m = self.mat[name]
        return torch.cat([(f[..., 2 * i:2 * i + 2, :].reshape(-1, self.ls) @ m[i].T).view(*f.shape[:-2], 2, self.ls)
                          for i in (0, 1)], dim=-2)

    def hop(self, f, dag=False):
        out = torch.zeros_like(f)
        for mu in range(4):
            for fwd in (True, False):
                sg = 1.0 if fwd == dag else -1.0
                p = torch.roll(f, -1 if fwd else 1, dims=3 - mu)
                w = p[..., :2, :] + sg * self._b(mu, p[..., 2:, :], False)
                del p
                u = self.u[..., mu, :, :]
                if not fwd:
                    u = torch.roll(u, 1, dims=3 - mu).transpose(-1, -2).conj()
                y = torch.empty_like(w)
                for i in range(self.nc):
                    t = u[..., i, 0, None, None, None] * w[..., 0, :, :, :]
                    for j in range(1, self.nc):
                        t = t + u[..., i, j, None, None, None] * w[..., j, :, :, :]
                    y[..., i, :, :, :] = t
                out[..., :2, :] += y
                out[..., 2:, :] += sg * self._b(mu, y, True)
        return -0.5 * out

    @staticmethod
    def _b(mu, v, adjoint):
        """B (or B^+) of gamma_mu = [[0, B], [B^+, 0]] on two spins."""
        a, b = v[..., 0, :], v[..., 1, :]
        if mu == 0:
            r = (1j * b, 1j * a)
        elif mu == 1:
            r = (-b, a)
        elif mu == 2:
            r = (1j * a, -1j * b)
        else:
            r = (a, b)
        sign = -1.0 if adjoint and mu != 3 else 1.0
        return sign * torch.stack(r, dim=-2)

    def mpc(self, f):
        return f - self.hop(self.s("K", self.hop(self.s("K", f))))

    def mpcdag(self, f):
        return f - self.s("K+", self.hop(self.s("K+", self.hop(f, True)), True))

    def hermop(self, f):
        return self.mpcdag(self.mpc(f))

    def m(self, f):
        return self.s("M", f) + self.hop(self.s("P", f))

    def mdag(self, f):
        return self.s("M+", f) + self.s("P+", self.hop(f, True))

    def solve(self, src):
        """M x = D_- src by the odd-site Schur complement."""
        d = self.s("C", src) + self.hop(self.s("N", src))
        even, odd = self.mask[2], self.mask[1]
        rhs = odd * (d - self.hop(self.s("P", self.s("I", even * d))))
        y = self.cg(self.hermop, self.mpcdag(rhs))
        xo = self.s("I", y)
        return xo + self.s("I", even * (d - self.hop(self.s("P", xo))))

    @staticmethod
    def cg(op, b, tol=1e-13):
        def dot(x, y):  # per column
            return (x.conj() * y).real.sum(dim=(0, 1, 2, 3, 4, 6, 7), keepdim=True)

        x, r, p = torch.zeros_like(b), b.clone(), b.clone()
        rr = dot(r, r)
        stop = tol * tol * rr
        for _ in range(2000):
            ap = op(p)
            alpha = torch.where(rr > 0, rr / dot(p, ap).clamp_min(1e-300), rr)
            x += alpha * p
            r -= alpha * ap
            new = dot(r, r)
            if bool((new <= stop).all()):
                break
            p = r + torch.where(rr > 0, new / rr.clamp_min(1e-300), rr) * p
            rr = new
        return x

    # library layouts: [site][s][spin * nc + colour], a column index last
    def load(self, a, eo=0):
        t = a.reshape(a.shape[0], self.ls, 4, self.nc, -1)
        if eo:
            full = torch.zeros(2 * a.shape[0], *t.shape[1:], device=a.device, dtype=a.dtype)
            full[self.odd if eo == 1 else ~self.odd] = t
            t = full
        return t.permute(0, 3, 4, 2, 1).contiguous().view(*reversed(self.site), self.nc, -1, 4, self.ls)

    def store(self, f, eo=0):
        t = f.reshape(-1, *f.shape[4:]).permute(0, 4, 3, 1, 2)
        if eo:
            t = t[self.odd if eo == 1 else ~self.odd]
        return t.reshape(t.shape[0], self.ls, -1, f.shape[5]).contiguous()


def _embed(src, ls):
    """4D -> 5D: spins 0, 1 at s = 0 and spins 2, 3 at s = Ls - 1."""
    out = torch.zeros(src.shape[0], ls, *src.shape[1:], device=src.device, dtype=src.dtype)
    half = src.shape[1] // 2
    out[:, 0, :half], out[:, ls - 1, half:] = src[:, :half], src[:, half:]
    return out


def _project(sol):
    """5D -> 4D: spins 0, 1 from s = Ls - 1 and spins 2, 3 from s = 0."""
    half = sol.shape[2] // 2
    return torch.cat([sol[:, -1, :half], sol[:, 0, half:]], dim=1)


def exact(case, seed):
    kind, ls = case["kind"], case["ls"]
    # the solves' reference CG takes too long beyond this many 5D-site-columns
    columns = {"prop": 12, "batch": len(_masses(case)) * case.get("sources", 1)}.get(kind, 1)
    if kind in ("solve5d", "prop", "batch", "force") and math.prod(_site(case)) * ls * columns > 5 * 2**19:
        return None
    u, f = _fields(case, seed)
    if kind == "batch":
        src = torch.stack(f, dim=-1)
        out = []
        for mass in _masses(case):
            op = _Dwf(case, mass, u)
            sol = op.store(op.solve(op.load(src)))
            out += [sol[..., j].contiguous() for j in range(len(f))]
        return out
    op = _Dwf(case, case["mass"], u)
    if kind == "hermop":
        return op.store(op.hermop(op.load(f, case["eo"])), case["eo"])[..., 0]
    if kind == "mhost":
        return op.store((op.mdag if case["dag"] else op.m)(op.load(f)))[..., 0].cpu().numpy()
    if kind == "solve5d":
        return op.store(op.solve(op.load(f)))[..., 0]
    if kind == "prop":
        return _project(op.store(op.solve(op.load(_embed(f, ls)))))
    if kind == "qed":
        rhs = op.load(_embed(f, ls))
        return _project(op.store(op.cg(lambda v: op.mdag(op.m(v)), op.mdag(rhs)))[..., 0]).cpu().numpy()
    phi = op.load(f, 1)
    x = op.cg(op.hermop, phi)
    with torch.enable_grad():
        op.u = op.u.clone().requires_grad_(True)
        y = op.mpc(x)
        norm = torch.view_as_real(y).square().sum()
        (grad,) = torch.autograd.grad(-norm, op.u)
    grad = grad.reshape(-1, 4, 3, 3)
    mat = torch.einsum("nmij,nmkj->nmik", u, grad.conj())
    anti = 0.5 * (mat - mat.transpose(-1, -2).conj())
    trace = torch.diagonal(anti, dim1=-2, dim2=-1).sum(-1)[..., None, None]
    force = anti - trace / 3.0 * torch.eye(3, device=u.device, dtype=u.dtype)
    return {"action": float((phi.conj() * x).real.sum()), "force": force, "grad": grad}
