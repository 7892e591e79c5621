"""k_dwf on the lattices of the other tests.

Those are small, and by the rule between the two operator kernels their launches go to
k_dwf_small.  Here every operator is made with DWF_HOP_KERNEL=full, so the same checks
against the oracle, with the same bars, run on k_dwf: partial last blocks, 16-bit storage at
Ls = 8, runtime Ls, the fused CG updates, several right-hand sides of one lattice, the force
and the learned polynomial.  The last test runs k_dwf_small where the rule would not take it.
"""
import pytest

import test_gpu_batch as batch
import test_gpu_force as force
import test_gpu_lpc as lpc
import test_gpu_parity as parity
import test_gpu_small_kernel as small

pytestmark = pytest.mark.gpu


@pytest.fixture
def full(monkeypatch):
    monkeypatch.setenv("DWF_HOP_KERNEL", "full")


@pytest.mark.parametrize("precision", ["double", "float", "half", "bfloat16"])
@pytest.mark.parametrize("dims,Ls", [c for c in small.CASES if c[1] != 23])
def test_modes(full, dims, Ls, precision):
    small.test_modes(dims, Ls, precision)


@pytest.mark.parametrize("prm", parity.PARAMS + parity.LS16[1:] + parity.LS12
                         + parity.LS12_PARTIAL)
def test_modes_fp64(full, prm):
    parity.test_modes_fp64(prm)


@pytest.mark.parametrize("prm", parity.PARAMS + parity.LS16 + parity.LS12 + parity.LS12_PARTIAL)
@pytest.mark.parametrize("precision,tol", [("float", 2e-6), ("half", 4e-3), ("bfloat16", 3e-2)])
def test_modes_reduced_precision(full, prm, precision, tol):
    parity.test_modes_reduced_precision(prm, precision, tol)


@pytest.mark.parametrize("inner", ["half", "float", "bfloat16", "double"])
@pytest.mark.parametrize("prm", parity.LS16 + parity.LS12 + parity.LS12_PARTIAL)
def test_fused_cg(full, prm, inner):
    parity.test_richardson_low_precision_inner_matrix_core(prm, inner)


def test_multishift(full):
    parity.test_multishift_matches_oracle()
    parity.test_multishift_ddagger_mode_matches_oracle()


@pytest.mark.parametrize("prm,nrhs", [
    (((4, 4, 4, 4), 6, 0.05, 1.6, 1.0, 0.0), 3),
    (((4, 4, 4, 8), 16, 0.05, 1.6, 1.5, 0.5), 4),
    (((4, 4, 4, 8), 12, 0.05, 1.6, 1.0, 0.0), 2),
    (((6, 6, 2, 6), 12, 0.05, 1.6, 1.5, 0.5), 3),      # a partial last block
    (((6, 2, 2, 6), 8, 0.05, 1.6, 1.0, 0.0), 2),
], ids=["ls6-3rhs", "ls16-4rhs", "ls12-2rhs", "ls12-partial-3rhs", "ls8-partial-2rhs"])
def test_multi_rhs(full, prm, nrhs):
    batch.test_batch_multi_rhs_matches_oracle(prm, nrhs)


def test_multi_rhs_graph(full):
    batch.test_batch_graph_replay_matches_direct()


@pytest.mark.parametrize("prm", force.PARAMS)
def test_force_modes(full, prm):
    force.test_force_modes_match_oracle(prm)


@pytest.mark.parametrize("case", lpc.CASES)
@pytest.mark.parametrize("prec,tol", [("double", 1e-12), ("float", 1e-5), ("half", 5e-3)])
def test_polynomial(full, case, prec, tol):
    lpc.test_apply_matches_oracle(case, prec, tol)


@pytest.mark.parametrize("precision", ["double", "float", "half", "bfloat16"])
@pytest.mark.parametrize("dims,Ls", [((6, 6, 6, 26), 16), ((6, 6, 10, 18), 12),
                                     ((6, 10, 14, 26), 8)])
def test_small_kernel_beyond_its_lines(monkeypatch, dims, Ls, precision):
    monkeypatch.setenv("DWF_HOP_KERNEL", "small")
    small.test_modes(dims, Ls, precision)
