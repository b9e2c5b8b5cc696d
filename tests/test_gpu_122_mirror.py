"""commutator_122's result is exactly (anti)hermitian: the lower triangles of the
square blocks are the upper ones times RES.herm to the last bit, whichever
kernel and path forms them."""
import pytest
import torch

from test_gpu_122_tiles import HERMS, _basis, _op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("emax,lmax,nucleus", [(4, 4, "O16"), (6, 6, "O16"), (8, 4, "C14"), (10, 3, "Ca40"), (12, 3, "He4")])
def test_lower_triangles_mirror_the_upper(gpu, emax, lmax, nucleus):
    from eom_imsrg import SqOp, commutators as cm
    b, _ = _basis(emax, lmax, nucleus)
    for hL, hR in HERMS:
        L, R = SqOp.from_numpy(b, _op(b, hL, 3), hL), SqOp.from_numpy(b, _op(b, hR, 4), hR)
        for path in (0, 1):
            b.set_path(path)
            for h in (-hL * hR, hL * hR):   # RES.herm drives the fill, whatever the operands are
                print(f"[122 mirror] eMax {emax} lMax {lmax} {nucleus} herm ({hL},{hR}) RES {h} path {path}", flush=True)
                RES = SqOp.zeros(b, h)
                cm.commutator_122(L, R, RES)
                for q in range(b.nblocks):
                    for g in (0, 3, 4):
                        n, _ = b.block_shape(q, g)
                        o = int(b.goff[q, g])
                        X = RES.data[o: o + n * n].view(n, n).T   # column-major
                        assert torch.equal(torch.tril(X, -1), h * torch.triu(X, 1).T + 0.0), (q, g)
        b.set_path(0)
