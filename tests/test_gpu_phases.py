"""The commutator of a small basis in three launches (k_phase1, 2, 3) against
the launch per term, which a 64 x 64 tile shape of one family selects: the same
bodies, and tile shapes that sum in the same order, so the same bits.  Bases
without particle-hole channels beside hh, of one shell, ragged; batches; BCH
(with E0) and Magnus (without)."""
import numpy as np
import pytest
import torch

from test_gpu_122_tiles import _basis, _op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("emax,lmax,nucleus", [(1, 1, "He4"), (2, 2, "O16"), (3, 1, "He4"), (3, 3, "O16"), (4, 2, "C14"),
                                               (4, 4, "O22"), (4, 4, "O16")])
def test_same_bits_as_the_term_launches(gpu, emax, lmax, nucleus):
    from eom_imsrg import Batch, Flow, SqOp, _lib
    b, _ = _basis(emax, lmax, nucleus)
    L, R = [_op(b, -1, s) for s in (31, 32)], [_op(b, 1, s) for s in (33, 34)]
    res = []
    for shape in (5 | 8, 0):
        print(f"[phases] eMax {emax} lMax {lmax} {nucleus} shape {shape}", flush=True)
        _lib.check(_lib.lib.imsrg_set_gemm_tile(b.handle, _lib.GEMM["PPPP"], shape))
        bt = Batch(b, 2, graphs=False)
        RES = bt.zeros()
        bt.commutator(torch.from_numpy(np.stack(L)).cuda(), -1, torch.from_numpy(np.stack(R)).cuda(), 1, RES)
        f = Flow(b)
        HS, DG = SqOp.zeros(b), SqOp.from_numpy(b, 0.1 * L[1], -1)
        G = SqOp.from_numpy(b, 0.02 * L[0], -1)
        for _ in range(2):   # captured, then replayed
            f.BCH_EXPAND(HS, G, SqOp.from_numpy(b, R[0], 1))
        f.MAGNUS_EXPAND(DG, G)
        torch.cuda.synchronize()
        res.append((RES.clone(), HS.data.clone(), DG.data.clone()))
    for x, y, what in zip(res[0], res[1], ("commutator", "BCH", "Magnus")):
        assert torch.equal(x, y), what
