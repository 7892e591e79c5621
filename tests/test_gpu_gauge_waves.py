"""The wave-gathered gauge kernels (rectangle force, stout smearing and its force)
at the sizes where their 64-site chunks can go wrong: volumes below, at and just
past a multiple of 64, extents 1 and 2 (both neighbours the same site, two-step
neighbours wrapping), and fields that are not 16-byte aligned, which take the
per-lane loads.

Bar: 1e-13 relative in the 2-norm.  A force or smeared link is a sum of at most
about 50 products of up to six unitary matrices, a few hundred roundings of
1.1e-16 each, mostly independent; the stout force adds the exp(iQ) derivatives,
hence 1e-12 there (the bar of its parity test).
"""
import numpy as np
import pytest

import gauge_oracle as go
import dwf_amd
from dwf_amd import _lib, lattice
from oracle import stout_force_udiv, stout_smear

pytestmark = pytest.mark.gpu

DIMS = [(2, 2, 2, 2), (2, 2, 2, 6), (4, 2, 2, 4), (4, 4, 2, 6), (6, 2, 2, 10), (3, 5, 1, 7)]


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


class Shifted:
    """A device field that starts `skip` bytes into an allocation."""

    def __init__(self, a, skip):
        self.shape, self.skip = a.shape, skip // 8
        self.buf = dwf_amd.DeviceArray((a.size + self.skip,))
        self.buf.from_host(np.concatenate([np.zeros(self.skip), a.ravel()]))
        self.ptr = self.buf.ptr + skip

    def host(self):
        return self.buf.to_host()[self.skip:].reshape(self.shape)


@pytest.mark.parametrize("skip", [0, 8])
@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("c_rect", [-0.0833, 0.0])
def test_rect_force(dims, c_rect, skip):
    print("case rect force", dims, c_rect, skip, flush=True)
    U = lattice.random_gauge(dims, 0.5, 3)
    u, f = Shifted(U, skip), Shifted(np.zeros_like(U), skip)
    d = (_lib.C.c_int * 4)(*dims)
    _lib.check("rect", _lib.load().dwf_hmc_rect_force(d, f.ptr, u.ptr, 4.17, 1.6667, c_rect))
    dwf_amd.synchronize()
    assert rel(f.host(), go.rect_force(U, dims, 4.17, 1.6667, c_rect)) < 1e-13


@pytest.mark.parametrize("skip", [0, 8])
@pytest.mark.parametrize("dims", DIMS)
def test_stout_and_its_force(dims, skip):
    print("case stout", dims, skip, flush=True)
    U = lattice.random_gauge(dims, 0.5, 5)
    sm = dwf_amd.Director_alt_Smear(dims, 0.1, 2)
    sm.set_config(U)
    want = stout_smear(dims, 0.1, U)
    assert rel(sm.get_config(1), want) < 1e-13
    assert rel(sm.get_config(2), stout_smear(dims, 0.1, want)) < 1e-13
    S = np.random.default_rng(6).standard_normal(U.shape)
    a, b = Shifted(S, skip), Shifted(np.zeros_like(S), skip)
    L = _lib.load()
    _lib.check("udiv", L.dwf_smear_force_udiv(sm._h, 1, b.ptr, a.ptr))
    _lib.check("udiv", L.dwf_smear_force_udiv(sm._h, 1, a.ptr, a.ptr))   # in place
    dwf_amd.synchronize()
    ref = stout_force_udiv(dims, 0.1, S, want)
    assert rel(b.host(), ref) < 1e-12
    assert np.array_equal(a.host(), b.host())
