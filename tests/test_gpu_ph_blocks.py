"""The fused commutator with 222_ph by block quadruples (k_comm222ph_blk)
against the oracle, on bases whose (l, j, tz) blocks hold 3 to 7 orbits:
whole quadruples and ones cut in J or in their members, pairs inside one
block, channels of opposite Tz with different holes.  All four hermiticity
pairs; the two instances of a batch."""
import numpy as np
import pytest
import torch

from conftest import assert_rel
from test_gpu_122_tiles import HERMS, _basis, _op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("emax,lmax,nucleus", [(5, 5, "O16"), (6, 6, "O22"), (7, 7, "Ca40"), (8, 4, "C14"),
                                               (12, 2, "He4")])
def test_commutator_vs_oracle(gpu, emax, lmax, nucleus):
    from eom_imsrg import Batch
    b, o = _basis(emax, lmax, nucleus)
    for hL, hR in HERMS:
        print(f"[ph blocks] eMax {emax} lMax {lmax} {nucleus} herm ({hL},{hR})", flush=True)
        Ls, Rs = [_op(b, hL, s) for s in (5, 6)], [_op(b, hR, s) for s in (7, 8)]
        bt = Batch(b, 2, graphs=False)
        RES = bt.zeros()
        bt.commutator(torch.from_numpy(np.stack(Ls)).cuda(), hL, torch.from_numpy(np.stack(Rs)).cuda(), hR, RES)
        torch.cuda.synchronize()
        for k in range(2):
            assert_rel(RES[k].cpu().numpy(), o.commutator(Ls[k], hL, Rs[k], hR, -hL * hR), what=f"instance {k}")
