"""The GEMM tile shapes of the fused commutator's families against the oracle
on channels around the register-direct blocks (64 x 32 and 32 x 32 a wave):
matrices smaller than a block, cut by its edge, odd leading dimensions (operands
at 8-byte alignment), K below one chunk of 8 and with each remainder."""
import numpy as np
import pytest
import torch

from conftest import assert_rel
from test_gpu_122_tiles import _basis, _op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [5, 6, 7])
@pytest.mark.parametrize("emax,lmax,nucleus", [(2, 2, "He4"), (4, 4, "O16"), (5, 3, "C14"), (6, 6, "O22"), (9, 2, "He4")])
def test_shapes_vs_oracle(gpu, emax, lmax, nucleus, shape):
    from eom_imsrg import Batch, _lib
    b, o = _basis(emax, lmax, nucleus)
    print(f"[gemm edges] eMax {emax} lMax {lmax} {nucleus} shape {shape}", flush=True)
    for fam in ("PPPP", "PPX", "XX", "PH"):
        _lib.check(_lib.lib.imsrg_set_gemm_tile(b.handle, _lib.GEMM[fam], shape))
    for hL, hR in ((-1, 1), (1, 1)):
        L, R = _op(b, hL, 11), _op(b, hR, 12)
        bt = Batch(b, 1, graphs=False)
        RES = bt.zeros()
        bt.commutator(torch.from_numpy(L[None]).cuda(), hL, torch.from_numpy(R[None]).cuda(), hR, RES)
        torch.cuda.synchronize()
        assert_rel(RES[0].cpu().numpy(), o.commutator(L, hL, R, hR, -hL * hR), what=f"shape {shape} herm ({hL},{hR})")


@pytest.mark.parametrize("shape", [6, 7])
def test_matrix_edges_do_not_leak(gpu, shape):
    """An infinite element reaches only the outputs whose sums hold it: rows,
    columns and k that a block reads at a clamped place stay out."""
    from eom_imsrg import Batch, _lib
    b, o = _basis(4, 4, "O16")
    L, R = _op(b, -1, 21), _op(b, 1, 22)
    n = b.oplen
    at = n - 1                      # the last stored element: a clamped read's neighbour
    R2 = R.copy()
    R2[at] = np.inf
    out = []
    for s in (5, shape):
        for fam in ("PPPP", "PPX", "XX", "PH"):
            _lib.check(_lib.lib.imsrg_set_gemm_tile(b.handle, _lib.GEMM[fam], s))
        bt = Batch(b, 1, graphs=False)
        RES = bt.zeros()
        bt.commutator(torch.from_numpy(L[None]).cuda(), -1, torch.from_numpy(R2[None]).cuda(), 1, RES)
        torch.cuda.synchronize()
        out.append(np.isfinite(RES[0].cpu().numpy()))
    assert np.array_equal(out[0], out[1])
    assert out[0].any() and not out[0].all()
