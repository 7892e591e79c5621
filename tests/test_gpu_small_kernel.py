"""The small-lattice operator kernel and k_dwf on both sides of the rule between them.

The rule counts blocks of 64 / Ls sites; the lattices below sit just under and just
over its lines for FP64 and FP32 hops (640 blocks at Ls = 12 and 16, 1300 at Ls = 8, 1200
or 1500 above Ls = 10; test_gpu_hop_kernel.py has both kernels in every type), with a ragged last block on each side, idle lanes (Ls = 5, 7, 10, 11, 12, 14, 18),
one and two matrix elements per thread (Ls = 16, 18), the largest Ls of the small kernel
(22) and the first beyond it (23).  Bars as in the parity tests: FP64 1e-13, FP32 2e-6,
FP16 4e-3, BF16 3e-2.
"""
import numpy as np
import pytest

from oracle import OracleDWF
import dwf_amd
from dwf_amd import lattice

pytestmark = pytest.mark.gpu

TOL = {"double": 1e-13, "float": 2e-6, "half": 4e-3, "bfloat16": 3e-2}
CASES = [((2, 2, 2, 2), 5), ((4, 2, 6, 2), 7), ((6, 2, 2, 10), 10), ((4, 6, 2, 4), 11),
         ((4, 2, 2, 6), 14), ((4, 4, 2, 2), 18), ((2, 4, 2, 6), 22), ((2, 4, 2, 6), 23),
         ((6, 6, 6, 22), 16), ((6, 6, 6, 26), 16),        # 594 and 702 blocks
         ((6, 6, 10, 16), 12), ((6, 6, 10, 18), 12),      # 576 and 648
         ((6, 10, 14, 24), 8), ((6, 10, 14, 26), 8),      # 1260 and 1365
         ((6, 10, 14, 14), 11), ((6, 10, 14, 18), 11)]    # 1176 and 1512


@pytest.mark.parametrize("dims,Ls", CASES)
@pytest.mark.parametrize("precision", ["double", "float", "half", "bfloat16"])
def test_modes(dims, Ls, precision):
    print("case", dims, Ls, precision, flush=True)
    U = np.tile(lattice.random_gauge((2, 2, 2, 2), 0.5, 11), (1, lattice.volume(dims) // 16, 1))
    prm = (dims, Ls, 0.05, 1.1, 1.5, 0.5)
    orc = OracleDWF(*prm)
    orc.set_config(U)
    gpu = dwf_amd.AFopr_Domainwall_5din_eo(*prm, (1, 1, 1, -1), precision)
    gpu.set_config(U)
    x = lattice.random_spinor5(dims, Ls, 12)
    for mode, dag in (("D", False), ("DdagD", False), ("Hdag", False), ("Doe", False),
                      ("Deo", True), ("Dee_inv", True)):
        want = orc.mult_dag(mode, x) if dag else orc.mult(mode, x)
        got = gpu.apply(mode, x, dagger=dag)
        err = np.linalg.norm(got - want) / np.linalg.norm(want)
        assert err < TOL[precision], (mode, dag, err)
