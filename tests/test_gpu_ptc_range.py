"""The network's matrix-core kernels at the ends of the FP32 range, where the three-part split
of the transports is not exact: tiny inputs, infinities, NaN.

Bars: those of the network's other tests (2e-5 forward, 1e-4 gradient, against the FP64 oracle
of the stored input).  The smallest scale, 1e-37, has a tenth of its normal components in FP32's
denormals, spaced 1.4e-45, 1e-8 of it.  What infinities and NaN become is what the VALU
kernels make of them: the same elements are NaN, +inf and -inf.
"""
import numpy as np
import pytest

import ptc_oracle as po
import dwf_amd
from dwf_amd import lattice
from dwf_amd.ptc import ParallelTransportNet

pytestmark = pytest.mark.gpu


def rel(a, b):
    m = np.abs(b).max()
    return np.linalg.norm(a / m - b / m) / np.linalg.norm(b / m)


def make(dims, Ls, ch):
    U = lattice.random_gauge(dims, 0.4, 51)
    op = dwf_amd.AFopr_Domainwall_5din_eo(dims, Ls, 0.05, 1.6, 1.0, 0.0, (1, 1, 1, -1), "float")
    op.set_config(U)
    net = ParallelTransportNet(op, ch)
    net.set_weights((0.2 * np.random.default_rng(52).standard_normal(net.nw)).astype(np.float32))
    return U, op, net


def field(op, x):
    f = op.new_field()
    op.convert(f, x)
    return f


SHAPES = [((2, 2, 2, 6), 16, (1, 8, 8, 1)), ((2, 4, 2, 2), 12, (1, 7, 5, 1)),
          ((2, 2, 2, 4), 4, (1, 13, 11, 1))]


@pytest.mark.parametrize("dims,Ls,ch", SHAPES + [((2, 2, 2, 6), 5, (1, 3, 1))])
@pytest.mark.parametrize("scale", [1e-37, 1e-34, 1e36])
def test_forward(dims, Ls, ch, scale):
    print("case ptc range forward", dims, Ls, ch, scale, flush=True)
    U, op, net = make(dims, Ls, ch)
    fi, fo = field(op, scale * lattice.random_spinor5(dims, Ls, 53)), op.new_field()
    net.apply(fo, fi)
    want = po.apply(po.Lattice(dims, U, Ls), net.get_weights().astype(np.float64), ch,
                    op.reverse(fi))
    assert rel(op.reverse(fo), want) < 2e-5


@pytest.mark.parametrize("dims,Ls,ch", SHAPES)
@pytest.mark.parametrize("scale", [1e-37, 1e-34])
def test_gradient(dims, Ls, ch, scale):
    print("case ptc range gradient", dims, Ls, ch, scale, flush=True)
    U, op, net = make(dims, Ls, ch)
    b = field(op, scale * lattice.random_spinor5(dims, Ls, 54))
    x = field(op, lattice.random_spinor5(dims, Ls, 55))
    loss, grad = net.loss_grad([b], [x])
    lo, go = po.loss_grad(po.Lattice(dims, U, Ls), net.get_weights().astype(np.float64), ch,
                          [(op.reverse(b), op.reverse(x))])
    assert abs(loss - lo) / lo < 1e-5
    assert rel(grad, go) < 1e-4


def same(a, b):
    return (np.array_equal(np.isnan(a), np.isnan(b))
            and np.array_equal(np.isposinf(a), np.isposinf(b))
            and np.array_equal(np.isneginf(a), np.isneginf(b)))


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("dims,Ls,ch", [((4, 2, 2, 4), 16, (1, 1)), ((4, 2, 2, 4), 5, (1, 1)),
                                        ((4, 4, 4, 4), 8, (1, 7, 6, 1))])
def test_not_finite(dims, Ls, ch, value, monkeypatch):
    print("case ptc range", dims, Ls, ch, value, flush=True)
    _, op, net = make(dims, Ls, ch)
    h = lattice.random_spinor5(dims, Ls, 56)
    h.reshape(-1)[1234] = value
    fi, fx, fo = field(op, h), field(op, lattice.random_spinor5(dims, Ls, 57)), op.new_field()
    out, grad = {}, {}
    for kernel in ("", "valu", "valu-wgrad"):
        monkeypatch.setenv("DWF_PTC_KERNEL", kernel)
        net.apply(fo, fi)
        out[kernel] = op.reverse(fo)
        grad[kernel] = net.loss_grad([fi], [fx])[1]
    assert not np.isfinite(out["valu"]).all() and np.isfinite(out["valu"]).any()
    assert same(out[""], out["valu"])
    assert same(grad[""], grad["valu-wgrad"])
