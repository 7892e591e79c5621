"""The measured workloads of the domain-wall framework.

Each case is one call, or the few calls that belong together, which a user's
program makes through dwf_amd: an operator application, a solve, a shifted
solve, the fermion force on fresh links, a gauge step of the molecular dynamics,
an application or a training step of the network preconditioner.  Fields live in
device memory, as in the HMC driver; the tensors returned are views of them.

listed(), draw(rng), prepare(case, seed), run(state), work(case) and
exact(case, seed), the last in plain torch in 64 bits.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "lqcd-dwf-hmc_amd"))

EPS, RHO = 0.3, 0.1                     # link disorder exp(i EPS H), stout parameter
ELEM = {"double": 8, "float": 4, "half": 2, "bfloat16": 2}
TORCH = {"double": torch.float64, "float": torch.float32, "half": torch.float16,
         "bfloat16": torch.bfloat16}
TYPESTR = {"double": "<f8", "float": "<f4", "half": "<f2", "bfloat16": "<i2"}
# Iwasaki-type improved gauge action of the 2+1-flavour benchmark
BETA, C_PLAQ, C_RECT = 4.17, 1.66666666666666666666, -0.08333333333333333333
NPATH = 11                              # transports of one network layer


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    shamir = dict(M0=1.6, b=1.0, c=0.0)
    moebius = dict(M0=1.0, b=1.5, c=0.5)
    return [
        # the even-odd hop in FP64 on the benchmark lattice: the framework's headline kernel
        dict(name="hop f64 16x16x16x32", kind="operator", lattice="16x16x16x32", Ls=16,
             precision="double", mode="Deo", mq=0.01, **shamir),
        # one D of the smallest lattice of the tests: the latency of a call
        dict(name="D f64 4x4x4x8", kind="operator", lattice="4x4x4x8", Ls=8, precision="double",
             mode="D", mq=0.02, **moebius),
        # the operator of the mixed solve's inner CG, 16-bit storage
        dict(name="DdagD f16 16x16x16x32", kind="operator", lattice="16x16x16x32", Ls=16,
             precision="half", mode="DdagD", mq=0.01, **shamir),
        # the reference scheme's inner operator on the largest lattice of the workloads
        dict(name="DdagD f32 24x24x24x48", kind="operator", lattice="24x24x24x48", Ls=16,
             precision="float", mode="DdagD", mq=0.01, **shamir),
        # extents and Ls away from the usual ones: partial blocks, Ls without a compiled kernel
        dict(name="Ddag f32 6x10x14x18 Ls10", kind="operator", lattice="6x10x14x18", Ls=10,
             precision="float", mode="Ddag", mq=0.05, **moebius),
        # a small lattice solved in FP64: many short launches in a dependent chain
        dict(name="CG f64 8x8x8x8", kind="cg", lattice="8x8x8x8", Ls=8, stop=1e-24, mq=0.02,
             **shamir),
        # the time-to-solution workload: FP64 Richardson around a 16-bit CG
        dict(name="mixed CG 16x16x16x32", kind="mixed", lattice="16x16x16x32", Ls=16,
             precision="half", inner=2e-4, stop=1e-24, mq=0.01, **shamir),
        # the rational force's shifted solves, 16 poles
        dict(name="multishift 16x16x16x16 Ls12", kind="multishift", lattice="16x16x16x16", Ls=12,
             shifts=16, stop=1e-24, mq=0.02, **moebius),
        # molecular dynamics: the fermion force right after the links have moved
        dict(name="force 32x16x16x24 Ls12", kind="force", lattice="32x16x16x24", Ls=12, nsmear=3,
             mq=0.002, **moebius),
        # molecular dynamics: one innermost step, the gauge force and the link update
        dict(name="gauge step 32x16x16x24", kind="gauge", lattice="32x16x16x24"),
        # the network preconditioner inside a solve: forward only, on the benchmark lattice
        dict(name="network 16x16x16x32", kind="network", lattice="16x16x16x32", Ls=16,
             channels="1,8,8,8,1", **shamir),
        # one training step of the network: forward, adjoint and weight gradient
        dict(name="network grad 8x8x8x16", kind="network_grad", lattice="8x8x8x16", Ls=16,
             channels="1,8,8,8,1", batch=4, **shamir),
    ]


def _extents(rng, vmin, vmax):
    """A lattice of even extents with a volume of about exp(uniform)."""
    while True:
        d = [rng.choice((4, 6, 8, 10, 12, 14, 16, 18, 20, 24, 32)) for _ in range(4)]
        want = math.exp(rng.uniform(math.log(vmin), math.log(vmax)))
        V = d[0] * d[1] * d[2] * d[3]
        if 0.7 < V / want < 1.4 and vmin <= V <= vmax:
            return "%dx%dx%dx%d" % tuple(d)


def draw(rng):
    kind = rng.choice(("operator", "operator", "operator", "operator", "cg", "mixed",
                       "multishift", "force", "gauge", "network", "network_grad"))
    act = rng.choice((dict(M0=1.6, b=1.0, c=0.0), dict(M0=1.0, b=1.5, c=0.5),
                      dict(M0=1.8, b=1.25, c=0.25)))
    mq = round(math.exp(rng.uniform(math.log(0.01), math.log(0.1))), 4)
    Ls = rng.choice((8, 10, 12, 12, 16, 16))
    if kind == "operator":
        return dict(kind=kind, lattice=_extents(rng, 512, 400000),
                    Ls=rng.choice((4, 6, 8, 10, 12, 12, 16, 16)),
                    precision=rng.choice(("double", "double", "float", "float", "half", "bfloat16")),
                    mode=rng.choice(("Deo", "Doe", "D", "Ddag", "DdagD", "DdagD", "Dee_inv", "H")),
                    mq=mq, **act)
    if kind == "cg":
        return dict(kind=kind, lattice=_extents(rng, 512, 20000), Ls=Ls, stop=1e-24, mq=mq, **act)
    if kind == "mixed":
        prec = rng.choice(("half", "float"))
        return dict(kind=kind, lattice=_extents(rng, 4096, 100000), Ls=Ls, precision=prec,
                    inner=2e-4 if prec == "half" else 1e-8, stop=1e-24, mq=mq, **act)
    if kind == "multishift":
        return dict(kind=kind, lattice=_extents(rng, 2048, 50000), Ls=Ls,
                    shifts=rng.choice((4, 12, 15, 16)), stop=1e-24, mq=mq, **act)
    if kind == "force":
        return dict(kind=kind, lattice=_extents(rng, 2048, 150000), Ls=Ls,
                    nsmear=rng.choice((1, 2, 3)), mq=mq, **act)
    if kind == "gauge":
        return dict(kind=kind, lattice=_extents(rng, 512, 300000))
    channels = rng.choice(("1,8,8,8,1", "1,8,1", "1,4,4,1", "1,6,6,1", "1,3,1", "1,8,8,1"))
    if kind == "network":
        return dict(kind=kind, lattice=_extents(rng, 512, 100000), Ls=Ls, channels=channels, **act)
    return dict(kind=kind, lattice=_extents(rng, 512, 8192), Ls=Ls, channels=channels,
                batch=rng.choice((1, 2, 4)), **act)


def _dims(case):
    return tuple(int(v) for v in case["lattice"].split("x"))


def _volume(case):
    return math.prod(_dims(case))


def _hops(mode):
    return {"Deo": 1, "Doe": 1, "D": 2, "Ddag": 2, "H": 2, "DdagD": 4, "Dee_inv": 0}[mode]


def work(case):
    """Bytes: every input read once, every output written once.  Flops: 1320 per 4D hop
    and site, 4 Ls per component and chiral matrix; a solve takes about ten D^+D per
    decade of its criterion, each reading and writing one field and the links."""
    V = _volume(case)
    kind = case["kind"]
    if kind == "gauge":
        # U and iP in; U, iP and the force out; 6 + 18 staples of 2 products per link
        return dict(bytes=4 * V * 18 * 8 * 5, flops=4 * V * (3 * 8 * 2 * 198 + 8 * 198))
    Ls = case["Ls"]
    spinor, links = V // 2 * Ls * 24, 4 * V * 18
    hop = V // 2 * Ls * (1320 + 24 * 4 * Ls)
    if kind == "operator":
        e, n = ELEM[case["precision"]], _hops(case["mode"])
        return dict(bytes=e * (2 * spinor + (links if n else 0)),
                    flops=n * hop + (0 if n else spinor * 4 * Ls))
    if kind in ("cg", "mixed", "multishift"):
        e = ELEM[case.get("precision", "double")]
        n = 10 * -math.log10(case["stop"])
        return dict(bytes=n * e * (2 * spinor + links) + 8 * spinor * (1 + case.get("shifts", 1)),
                    flops=n * (4 * hop + 10 * spinor))
    if kind == "force":
        # eta and the links in, the force and the smeared levels out
        n = case["nsmear"]
        return dict(bytes=8 * (spinor + links * (2 + n)),
                    flops=6 * hop + 2 * V * Ls * 4 * 3 * 3 * 3 * 8 + n * 4 * V * 60 * 198)
    ch = [int(v) for v in case["channels"].split(",")]
    pairs = sum(a * b for a, b in zip(ch, ch[1:]))
    fwd = V * Ls * (pairs * NPATH * 384 + sum(ch[:-1]) * 8 * 288)
    if kind == "network":
        return dict(bytes=4 * (2 * spinor + links), flops=fwd)
    n = case["batch"]
    return dict(bytes=4 * (2 * n * spinor + links) + 8 * pairs * NPATH * 32, flops=3 * n * fwd)


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------

DEVICE = "cuda" if torch.cuda.is_available() else "cpu"


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEVICE, dtype=torch.float64)


def _mm(a, b):
    """a b of 3x3 matrices (..., 3, 3), without a batched library product."""
    r = a[..., :, 0, None] * b[..., None, 0, :]
    r = r + a[..., :, 1, None] * b[..., None, 1, :]
    return r + a[..., :, 2, None] * b[..., None, 2, :]


def _dag(a):
    return a.conj().transpose(-1, -2)


def _at(m):
    """Traceless anti-hermitian part."""
    a = 0.5 * (m - _dag(m))
    tr = a.diagonal(dim1=-2, dim2=-1).sum(-1) / 3.0
    return a - tr[..., None, None] * torch.eye(3, dtype=a.dtype, device=a.device)


def _exp(m, terms=14, halvings=3):
    """exp of small 3x3 matrices: Taylor on m / 2^halvings, then squarings."""
    one = torch.eye(3, dtype=m.dtype, device=m.device)
    m = m * 0.5 ** halvings
    r = one.expand_as(m)
    for k in range(terms, 0, -1):
        r = one + _mm(m, r) / k
    for _ in range(halvings):
        r = _mm(r, r)
    return r


def _links(dims, g):
    """exp(i EPS H), H Gaussian traceless Hermitian: complex (4, Nt, Nz, Ny, Nx, 3, 3)."""
    shape = (4,) + tuple(dims[::-1]) + (3, 3)
    out = torch.empty(shape, dtype=torch.complex128, device=DEVICE)
    for mu in range(4):
        a = torch.complex(_randn(g, *shape[1:]), _randn(g, *shape[1:]))
        out[mu] = _exp(EPS * _at(1j * (a + _dag(a)) / 2))
    return out


def _field_g(M):
    """Field_G (4, V, 18) doubles of complex (4, Nt, Nz, Ny, Nx, 3, 3) matrices."""
    return torch.view_as_real(M.contiguous()).reshape(4, -1, 18)


def _spinor(g, dims, Ls, dtype=torch.float64):
    """Gaussian field of one parity in the device layout (V/2, 24, Ls)."""
    return _randn(g, math.prod(dims) // 2, 24, Ls).to(dtype)


def _momenta(g, dims):
    """Gaussian momenta in su(3)."""
    shape = (4,) + tuple(dims[::-1]) + (3, 3)
    return _at(torch.complex(_randn(g, *shape), _randn(g, *shape)))


def _weights(g, channels, noise=0.05, scale=0.5):
    """Channel 0 carried by the identity path, plus noise: a network early in training."""
    parts = []
    for l, (cin, cout) in enumerate(zip(channels, channels[1:])):
        w = noise * _randn(g, NPATH, cout, cin, 4, 4, 2)
        w[0, 0, 0, :, :, 0] += (scale if l == len(channels) - 2 else 1.0) * torch.eye(
            4, dtype=torch.float64, device=w.device)
        parts.append(w.reshape(-1))
    return torch.cat(parts).float()


def _channels(case):
    return tuple(int(v) for v in case["channels"].split(","))


def _inputs(case, seed):
    """Everything random of a case."""
    g = _generator(seed)
    dims = _dims(case)
    d = dict(U=_links(dims, g))
    kind = case["kind"]
    if kind == "operator":
        d["w"] = _spinor(g, dims, case["Ls"], TORCH[case["precision"]])
    elif kind in ("cg", "mixed", "multishift", "force"):
        d["w"] = _spinor(g, dims, case["Ls"])
    elif kind == "gauge":
        d["iP"] = _momenta(g, dims)
    else:
        d["weights"] = _weights(g, _channels(case))
        if kind == "network":
            d["w"] = _spinor(g, dims, case["Ls"], torch.float32)
        else:   # (source, solution) pairs of the operator, sources of norm 1
            op = _Operator(case, _smear(d["U"], 2), mq=0.01)
            d["pairs"] = []
            for _ in range(case["batch"]):
                x = _to_complex(_spinor(g, dims, case["Ls"]))
                b = op.mult("DdagD", x)
                s = 1.0 / b.abs().square().sum().sqrt()
                d["pairs"].append((_to_real(b * s).float(), _to_real(x * s).float()))
    return d


# ---------------------------------------------------------------------------
# the calls
# ---------------------------------------------------------------------------

class _Buffer:
    """Device memory of the library as an array that torch can wrap; keeps its owner alive."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner, self.ptr, self.n = owner, ptr, math.prod(shape)
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=typestr,
                                             data=(ptr, False), version=2, strides=None)


def _view(owner, ptr, shape, precision="double"):
    t = torch.as_tensor(_Buffer(owner, ptr, shape, TYPESTR[precision]), device="cuda")
    return t.view(torch.bfloat16) if precision == "bfloat16" else t


def _new_field(op, precision, value=None):
    f = op.new_field()
    v = _view(f, f.ptr, (op.Vh, 24, op.Ls), precision)
    if value is not None:
        v.copy_(value)
    return f, v


def _gauge(dims, value):
    """A device Field_G of the HMC driver holding value, and its tensor view."""
    from dwf_amd import hmc
    f = hmc.GaugeField(dims)
    v = _view(f, f.ptr, f.shape)
    v.copy_(_field_g(value))
    return f, v


def _fopr(director, case, precision, mq=None):
    from dwf_amd import hmc
    return hmc.SmearedFopr(director, _dims(case), case["Ls"], case["mq"] if mq is None else mq,
                           case["M0"], case["b"], case["c"], (1, 1, 1, -1), precision)


def prepare(case, seed):
    import dwf_amd
    from dwf_amd import hmc
    from dwf_amd.ptc import ParallelTransportNet
    dims, kind = _dims(case), case["kind"]
    d = _inputs(case, seed)
    s = dict(kind=kind)
    s["U"], s["U_view"] = _gauge(dims, d["U"])
    if kind == "gauge":
        s["iP"], s["iP_view"] = _gauge(dims, d["iP"])
        s["F"] = hmc.GaugeField(dims)
        s["F_view"] = _view(s["F"], s["F"].ptr, s["F"].shape)
        s["action"] = hmc.Action_G_Rectangle(dims, BETA, C_PLAQ, C_RECT)
        s["action"].set_config(s["U"])
        s["update"] = hmc.Integrator_UpdateU([])
        torch.cuda.synchronize()
        return s
    s["director"] = hmc.Director(dims, RHO, case.get("nsmear", 2))
    s["director"].set_config(s["U"])
    torch.cuda.synchronize()
    if kind == "operator":
        s["op"] = _fopr(s["director"], case, case["precision"]).refresh()
        s["op"].set_mode(case["mode"])
        s["w"], _ = _new_field(s["op"], case["precision"], d["w"])
        s["v"], s["out"] = _new_field(s["op"], case["precision"])
    elif kind in ("cg", "mixed", "multishift"):
        op = s["op"] = _fopr(s["director"], case, "double").refresh()
        op.set_mode("DdagD")
        s["b"], _ = _new_field(op, "double", d["w"])
        if kind == "multishift":
            n = case["shifts"]
            s["sigma"] = [math.exp(math.log(1e-4) + i * math.log(1e5) / (n - 1)) for i in range(n)]
            s["x"], s["out"] = zip(*[_new_field(op, "double") for _ in range(n)])
            s["solver"] = dwf_amd.AShiftsolver_CG(op, 10000, case["stop"])
        else:
            s["x"], s["out"] = _new_field(op, "double")
            if kind == "cg":
                s["solver"] = dwf_amd.ASolver_CG(op, 10000, case["stop"])
            else:
                s["op_f"] = _fopr(s["director"], case, case["precision"]).refresh()
                s["op_f"].set_mode("DdagD")
                s["solver"] = dwf_amd.ASolver_Richardson(op, s["op_f"], 100, case["stop"], 10000,
                                                         case["inner"])
    elif kind == "force":
        s["fopr"] = _fopr(s["director"], case, "double")
        op = s["fopr"].op
        s["eta"], _ = _new_field(op, "double", d["w"])
        s["force"] = dwf_amd.AForce_F_Smeared_alt(dwf_amd.AForce_F_Domainwall_5din_eo(op),
                                                  s["director"].sm)
        s["F"] = s["force"].new_force()
        s["F_view"] = _view(s["F"], s["F"].ptr, s["F"].shape)
    else:
        op = s["op"] = _fopr(s["director"], case, "float", mq=0.01).refresh()
        s["net"] = ParallelTransportNet(op, _channels(case))
        s["net"].set_weights(d["weights"].cpu().numpy())
        if kind == "network":
            s["w"], _ = _new_field(op, "float", d["w"])
            s["v"], s["out"] = _new_field(op, "float")
        else:
            s["b"] = [_new_field(op, "float", b)[0] for b, _ in d["pairs"]]
            s["x"] = [_new_field(op, "float", x)[0] for _, x in d["pairs"]]
    torch.cuda.synchronize()
    dwf_amd.synchronize()
    return s


def run(s):
    kind = s["kind"]
    if kind == "operator":
        s["op"].mult(s["v"], s["w"])
        return s["out"]
    if kind in ("cg", "mixed"):
        s["solver"].solve(s["x"], s["b"])
        return s["out"]
    if kind == "multishift":
        s["solver"].solve(s["x"], s["sigma"], s["b"])
        return list(s["out"])
    if kind == "force":
        s["director"].notify_linkv()         # the links have moved: smear them again
        s["fopr"].refresh()
        s["force"].force_core(s["F"], s["eta"])
        return s["F_view"]
    if kind == "gauge":
        s["action"].force(s["F"])
        s["iP"].axpy(0.02, s["F"])
        s["update"].evolve(0.02, s["iP"], s["U"])
        return dict(F=s["F_view"], iP=s["iP_view"], U=s["U_view"])
    if kind == "network":
        s["net"].apply(s["v"], s["w"])
        return s["out"]
    loss, grad = s["net"].loss_grad(s["b"], s["x"])
    return dict(loss=loss, grad=grad)


# ---------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ---------------------------------------------------------------------------

def _roll(a, mu, step):
    """v(x) = a(x + step mu) for fields (Nt, Nz, Ny, Nx, ...)."""
    return torch.roll(a, -step, dims=3 - mu)


def _staples(U, mu, nu):
    """U_nu(x) U_mu(x+nu) U_nu(x+mu)^+ and U_nu(x-nu)^+ U_mu(x-nu) U_nu(x-nu+mu)."""
    up = _mm(_mm(U[nu], _roll(U[mu], nu, 1)), _dag(_roll(U[nu], mu, 1)))
    lo = _roll(_mm(_mm(_dag(U[nu]), U[mu]), _roll(U[nu], mu, 1)), nu, -1)
    return up, lo


def _smear(U, levels):
    for _ in range(levels):
        new = []
        for mu in range(4):
            C = 0
            for nu in range(4):
                if nu != mu:
                    up, lo = _staples(U, mu, nu)
                    C = C + RHO * (up + lo)
            new.append(_mm(_exp(_at(_mm(C, _dag(U[mu])))), U[mu]))
        U = torch.stack(new)
    return U


def _to_complex(w):
    """(V/2, 24, Ls) reals -> complex (V/2, 4, 3, Ls)."""
    w = w.double().reshape(w.shape[0], 4, 3, 2, -1)
    return torch.complex(w[..., 0, :].contiguous(), w[..., 1, :].contiguous())


def _to_real(v):
    return torch.stack((v.real, v.imag), dim=3).reshape(v.shape[0], 24, v.shape[-1])


def _half_sites(dims, parity):
    """Coordinates (x, y, z, t) of the half sites of one parity, x/2 fastest."""
    Nx, Ny, Nz, Nt = dims
    i = torch.arange(Nx * Ny * Nz * Nt // 2, device=DEVICE)
    x2, r = i % (Nx // 2), i // (Nx // 2)
    y, r = r % Ny, r // Ny
    z, t = r % Nz, r // Nz
    return [2 * x2 + (y + z + t + parity) % 2, y, z, t]


# (spin partner of 0, factor), (spin partner of 1, factor): (1 - gamma_mu) psi has the upper
# components psi_0 + f0 psi_p0 and psi_1 + f1 psi_p1, the lower ones follow from them
_PROJ = [((3, 1j), (2, 1j)), ((3, 1.0), (2, -1.0)), ((2, 1j), (3, -1j))]


class _Operator:
    """The even-odd Moebius operator on complex (V/2, 4, 3, Ls) fields, Dirac basis."""

    def __init__(self, case, U, mq=None):
        self.dims, self.Ls = _dims(case), case["Ls"]
        mq = case["mq"] if mq is None else mq
        self.geometry(U)
        Ls, M0, b, c = self.Ls, case["M0"], case["b"], case["c"]
        one = torch.eye(Ls, dtype=torch.float64, device=DEVICE)
        up = torch.roll(one, 1, dims=1)          # (up psi)_s = psi_{s+1}, -mq at the wall
        up[Ls - 1, 0] = -mq
        shift = (up.T.contiguous(), up)          # P+ takes s - 1, P- takes s + 1
        # per chirality: the 5D factor of the hop, D_ee and its inverse
        self.Mp = [-0.5 * (b * one + c * m) for m in shift]
        dee = [(b * (4 - M0) + 1) * one + (c * (4 - M0) - 1) * m for m in shift]
        self.Di = [torch.linalg.inv(m.cpu()).to(DEVICE) for m in dee]
        r = one.flip(0)
        self.R = [r, -r]

    def geometry(self, U):
        Nx, Ny, Nz, Nt = N = self.dims
        self.nb, self.link = [], []
        for p in range(2):
            x = _half_sites(self.dims, p)
            nb, link = [], []
            for mu in range(4):
                for step in (1, -1):
                    y = list(x)
                    y[mu] = (x[mu] + step) % N[mu]
                    at = y if step < 0 else x
                    u = U[mu][at[3], at[2], at[1], at[0]]
                    u = u if step > 0 else _dag(u)
                    if mu == 3:                  # antiperiodic in t
                        wrap = x[3] == (N[3] - 1 if step > 0 else 0)
                        u = u * torch.where(wrap, -1.0, 1.0)[:, None, None]
                    nb.append(y[0] // 2 + (Nx // 2) * (y[1] + Ny * (y[2] + Nz * y[3])))
                    link.append(u)
            self.nb.append(nb)
            self.link.append(link)

    def transport(self, h, p, d):
        """U(x, d) h(x + d) for fields (V/2, spins, 3, Ls) of parity 1 - p."""
        g, u = h[self.nb[p][d]], self.link[p][d]
        return sum(u[:, None, :, b, None] * g[:, :, b, None, :] for b in range(3))

    def hop(self, psi, p):
        """Wilson hop onto the sites of parity p."""
        out = [0, 0, 0, 0]
        for d in range(8):
            mu, sign = d // 2, 1.0 if d % 2 == 0 else -1.0      # 1 - sign gamma_mu
            if mu == 3:
                k = 2 if d == 6 else 0
                h = self.transport(2.0 * psi[:, k:k + 2], p, d)
                out[k], out[k + 1] = out[k] + h[:, 0], out[k + 1] + h[:, 1]
                continue
            (p0, f0), (p1, f1) = _PROJ[mu]
            f0, f1 = sign * f0, sign * f1
            h = self.transport(torch.stack((psi[:, 0] + f0 * psi[:, p0],
                                            psi[:, 1] + f1 * psi[:, p1]), dim=1), p, d)
            out[0], out[1] = out[0] + h[:, 0], out[1] + h[:, 1]
            out[p0] = out[p0] + complex(f0).conjugate() * h[:, 0]
            out[p1] = out[p1] + complex(f1).conjugate() * h[:, 1]
        return torch.stack(out, dim=1)

    @staticmethod
    def gm5(psi):
        return torch.cat((psi[:, 2:], psi[:, :2]), dim=1)

    def chiral(self, M, psi, transpose=False):
        """M[0] on P+ psi plus M[1] on P- psi, along s."""
        g = self.gm5(psi)
        m = [a.T if transpose else a for a in M]
        a = torch.matmul(0.5 * (psi + g), m[0].T.to(psi.dtype))
        return a + torch.matmul(0.5 * (psi - g), m[1].T.to(psi.dtype))

    def mult(self, mode, w):
        if mode in ("Deo", "Doe"):
            return self.hop(self.chiral(self.Mp, w), 0 if mode == "Deo" else 1)
        if mode == "Dee_inv":
            return self.chiral(self.Di, w)
        if mode == "D":
            t = self.chiral(self.Di, self.mult("Doe", w))
            return w - self.chiral(self.Di, self.mult("Deo", t))
        if mode == "Ddag":
            t = self.chiral(self.Di, w, True)
            t = self.chiral(self.Mp, self.gm5(self.hop(self.gm5(t), 1)), True)
            t = self.chiral(self.Di, t, True)
            return w - self.chiral(self.Mp, self.gm5(self.hop(self.gm5(t), 0)), True)
        if mode == "H":                          # gamma_5 R D
            return self.chiral(self.R, self.mult("D", w))
        return self.mult("Ddag", self.mult("D", w))


def _solve(op, b, sigma, stop):
    """(D^+D + sigma_j) x_j = b by multishift CG."""
    n = len(sigma)
    x = [torch.zeros_like(b) for _ in sigma]
    r, p = b, [b.clone() for _ in sigma]
    rr = float(b.abs().square().sum())
    limit, zeta, zold, beta_old, alpha = stop * rr, [1.0] * n, [1.0] * n, 1.0, 0.0
    live = [True] * n
    while rr > limit:
        q = op.mult("DdagD", p[0]) + sigma[0] * p[0]
        beta = rr / float((p[0].conj() * q).sum().real)
        r = r - beta * q
        new = float(r.abs().square().sum())
        nalpha = new / rr
        for j in range(n):
            if not live[j]:
                continue
            z = zeta[j] * zold[j] * beta_old / (
                beta * alpha * (zold[j] - zeta[j])
                + zold[j] * beta_old * (1 + (sigma[j] - sigma[0]) * beta))
            x[j] = x[j] + (beta * z / zeta[j]) * p[j]
            p[j] = (nalpha * (z / zeta[j]) ** 2) * p[j] + z * r
            zold[j], zeta[j] = zeta[j], z
            live[j] = j == 0 or z * z * new > limit
        rr, beta_old, alpha = new, beta, nalpha
    return x


def _gauge_step(U, iP, e):
    F = []
    for mu in range(4):
        S = 0
        for nu in range(4):
            if nu == mu:
                continue
            Um, Un = U[mu], U[nu]
            up, lo = _staples(U, mu, nu)
            side, back = _staples(U, nu, mu)
            Um_n, Un_m = _roll(Um, nu, 1), _roll(Un, mu, 1)
            S = S + C_PLAQ * (up + lo)
            R = _mm(Un, _mm(Um_n, _dag(_roll(side, mu, 1))))
            R = R + _mm(Un, _mm(_roll(up, nu, 1), _dag(Un_m)))
            R = R + _mm(back, _mm(Um_n, _dag(Un_m)))
            L = _mm(_dag(Un), _mm(Um, _roll(side, mu, 1)))
            L = L + _mm(_dag(Un), _mm(lo, Un_m))
            L = L + _mm(_dag(back), _mm(Um, Un_m))
            S = S + C_RECT * (R + _roll(L, nu, -1))
        F.append(-(BETA / 3.0) * _at(_mm(U[mu], _dag(S))))
    F = torch.stack(F)
    P = iP + e * F
    V = _mm(_exp(e * P, terms=16, halvings=2), U)
    r0 = V[..., 0, :] / V[..., 0, :].abs().square().sum(-1, keepdim=True).sqrt()
    r1 = V[..., 1, :] - (r0.conj() * V[..., 1, :]).sum(-1, keepdim=True) * r0
    r1 = r1 / r1.abs().square().sum(-1, keepdim=True).sqrt()
    r2 = torch.linalg.cross(r0, r1).conj()
    return dict(F=_field_g(F), iP=_field_g(P), U=_field_g(torch.stack((r0, r1, r2), dim=-2)))


def _network(op, W, channels, w):
    """The parallel-transport network on an even field; pairs (even, odd) per channel."""
    act, off = [(w, torch.zeros_like(w))], 0
    for cin, cout in zip(channels, channels[1:]):
        n = NPATH * cin * cout * 32
        m = torch.view_as_complex(W[off:off + n].reshape(NPATH, cout, cin, 4, 4, 2))
        off += n
        new = [[0, 0] for _ in range(cout)]
        for b in range(cin):
            for q in range(NPATH):
                for p in range(2):
                    f = act[b][p]
                    if q == 0:
                        t = f
                    elif q <= 8:
                        t = op.transport(act[b][1 - p], p, q - 1)
                    else:
                        z = torch.zeros_like(f[..., :1])
                        t = torch.cat((f[..., 1:], z) if q == 9 else (z, f[..., :-1]), dim=-1)
                    u = [t[:, j, None] for j in range(4)]
                    for a in range(cout):
                        k = m[q, a, b]
                        new[a][p] = new[a][p] + sum(k[:, j, None, None] * u[j] for j in range(4))
        act = new
    return act[0][0]


def exact(case, seed):
    kind, V = case["kind"], _volume(case)
    size = V * case.get("Ls", 1)
    if (kind in ("cg", "mixed", "multishift") and size * case.get("shifts", 1) > 400000
            or kind == "network" and size > 2200000 or kind == "network_grad" and size > 140000):
        return None                              # too long in plain torch
    d = _inputs(case, seed)
    if kind == "gauge":
        return _gauge_step(d["U"], d["iP"], 0.02)
    if kind == "force":
        # S = |D eta|^2 of the thin links U: dS = Re tr(X U G^+) for U -> exp(X) U
        U = d["U"].clone().requires_grad_(True)
        op = _Operator(case, _smear(U, case["nsmear"]))
        S = op.mult("D", _to_complex(d["w"])).abs().square().sum()
        G, = torch.autograd.grad(S, U)
        return _field_g(-_at(_mm(d["U"], _dag(G))))
    U = _smear(d["U"], 2)
    if kind in ("network", "network_grad"):
        op = _Operator(case, U, mq=0.01)
        W = d["weights"].to(torch.bfloat16).double()
        if kind == "network":
            return _to_real(_network(op, W, _channels(case), _to_complex(d["w"])))
        loss, grad = 0.0, torch.zeros_like(W)
        for b, x in d["pairs"]:
            w = W.clone().requires_grad_(True)
            y = _network(op, w, _channels(case), _to_complex(b))
            L = (y - _to_complex(x)).abs().square().sum()
            grad += torch.autograd.grad(L, w)[0]
            loss += float(L.detach())
        return dict(loss=loss, grad=grad.cpu().numpy())
    op = _Operator(case, U)
    w = _to_complex(d["w"])
    if kind == "operator":
        return _to_real(op.mult(case["mode"], w))
    if kind == "multishift":
        n = case["shifts"]
        sigma = [math.exp(math.log(1e-4) + i * math.log(1e5) / (n - 1)) for i in range(n)]
        return [_to_real(x) for x in _solve(op, w, sigma, 1e-28)]
    return _to_real(_solve(op, w, [0.0], 1e-29)[0])
