"""121 and 221 with one or two lanes a thread (by the results of a launch and the
terms of one): the instances of a batch large enough for two lanes have the bits
of single commutators, and the oracle's values."""
import numpy as np
import pytest
import torch

from conftest import assert_rel
from test_gpu_122_tiles import _basis, _op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("emax,lmax,nucleus,ninst", [(2, 2, "He4", 2), (4, 4, "O22", 40), (6, 6, "Ca40", 16), (8, 4, "C14", 12)])
def test_batch_has_the_bits_of_single_commutators(gpu, emax, lmax, nucleus, ninst):
    from eom_imsrg import Batch
    b, o = _basis(emax, lmax, nucleus)
    print(f"[onebody] eMax {emax} lMax {lmax} {nucleus} x {ninst}", flush=True)
    L, R = _op(b, -1, 41), _op(b, 1, 42)
    scale = np.linspace(0.5, 1.5, ninst)[:, None]
    Ls, Rs = torch.from_numpy(scale * L).cuda(), torch.from_numpy(scale[::-1] * R).cuda()
    bt, one = Batch(b, ninst, graphs=False), Batch(b, 1, graphs=False)
    RES, X = bt.zeros(), one.zeros()
    bt.commutator(Ls, -1, Rs, 1, RES)
    for k in (0, ninst // 2, ninst - 1):
        one.commutator(Ls[k: k + 1].contiguous(), -1, Rs[k: k + 1].contiguous(), 1, X)
        assert torch.equal(RES[k], X[0]), k
        assert_rel(X[0].cpu().numpy(), o.commutator(scale[k] * L, -1, scale[ninst - 1 - k] * R, 1, 1), what=f"instance {k}")
