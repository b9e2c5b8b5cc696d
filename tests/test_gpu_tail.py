"""The last pass of a nested commutator (k_comm_tail: lower triangles, append
and norm at once) against the plain path, which appends and takes the norm in
a pass of its own, over a BCH and a Magnus expansion: square blocks below one
tile, of exactly one and of several, rectangular blocks
and the one-body part beside them."""
import numpy as np
import pytest
import torch

from conftest import assert_rel
from test_gpu_122_tiles import _basis, _op

pytestmark = pytest.mark.gpu

@pytest.mark.parametrize("emax,lmax,nucleus", [(1, 1, "He4"), (2, 2, "He4"), (3, 3, "O16"), (4, 2, "C14"),
                                               (4, 4, "O16"), (5, 5, "O22"), (9, 1, "He4")])
def test_expansions_vs_plain_path(gpu, emax, lmax, nucleus):
    from eom_imsrg import Flow, SqOp
    b, _ = _basis(emax, lmax, nucleus)
    res = []
    for path in (0, 1):
        print(f"[tail] eMax {emax} lMax {lmax} {nucleus} path {path}", flush=True)
        b.set_path(path)
        try:
            f = Flow(b, graphs=path == 0)
            HS, DG = SqOp.zeros(b), SqOp.from_numpy(b, 0.1 * _op(b, -1, 5), -1)
            G = SqOp.from_numpy(b, 0.02 * _op(b, -1, 3), -1)
            nt, adv = f.BCH_EXPAND(HS, G, SqOp.from_numpy(b, _op(b, 1, 4), 1))
            nc = f.MAGNUS_EXPAND(DG, G)
            torch.cuda.synchronize()
            res.append((HS.numpy(), DG.numpy(), nt, nc, np.array(adv)))
        finally:
            b.set_path(0)
    (h0, d0, n0, c0, a0), (h1, d1, n1, c1, a1) = res
    assert (n0, c0) == (n1, c1)
    assert_rel(h0, h1, what="BCH")
    assert_rel(d0, d1, what="Magnus")
    assert_rel(a0, a1, what="norms")
