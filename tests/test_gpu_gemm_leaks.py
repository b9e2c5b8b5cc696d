"""Infinite elements at the edges of the GEMM families' matrices reach only the
outputs whose sums hold them, with the register-direct shapes (6, 7: clamped rows,
pairs of rows moved back, zeroed K tails) as with the 32x32 tiles through LDS, which
select zeros.  The matrices have more than one row and column, are cut by the
blocks' edges, and their K is not a multiple of 8."""
import numpy as np
import pytest
import torch

from test_gpu_122_tiles import _basis, _op

pytestmark = pytest.mark.gpu

FORWARD = ("PPPP", "PPX", "XX", "PH")
BASES = [(4, 4, "O16"), (6, 4, "O22")]


def _set(b, families, shape):
    from eom_imsrg import _lib
    for fam in families:
        _lib.check(_lib.lib.imsrg_set_gemm_tile(b.handle, _lib.GEMM[fam], shape))


def _channels(b):
    """channels whose pp x pp and pp x (ph|hh) products have ragged edges in m, n and k"""
    d = np.asarray(b.dims).reshape(-1, 3)
    return [q for q, (np_, nb, nh) in enumerate(d) if np_ > 32 and np_ % 2 == 1 and np_ % 8 and nb > 1 and nb + nh > 1]


def _corners(b, q):
    """(operand index list) of the last row, the last column and the last element of every block of channel q"""
    out = []
    for g in range(6):
        n1, n2 = b.block_shape(q, g)
        if n1 < 2 or n2 < 2:
            continue
        for i, j in ((n1 - 1, n2 - 1), (n1 - 1, 0), (0, n2 - 1)):
            at = [int(b.goff[q, g]) + i + j * n1]
            if g in (0, 3, 4):
                at.append(int(b.goff[q, g]) + j + i * n1)   # the mirrored element of a square block
            out.append((g, (i, j), at))
    return out


@pytest.mark.parametrize("shape", [6, 7])
@pytest.mark.parametrize("emax,lmax,nucleus", BASES)
def test_forward_products(gpu, emax, lmax, nucleus, shape):
    from eom_imsrg import Batch
    b, _ = _basis(emax, lmax, nucleus)
    L, R = _op(b, -1, 21), _op(b, 1, 22)
    qs = _channels(b)
    assert qs
    for q in (qs[0], qs[-1]):
        for g, ij, at in _corners(b, q):
            for which in (0, 1):
                ops = [torch.from_numpy(X[None].copy()).cuda() for X in (L, R)]
                ops[which][0, at] = float("inf")
                masks = []
                for s in (5, shape):
                    _set(b, FORWARD, s)
                    bt = Batch(b, 1, graphs=False)
                    RES = bt.zeros()
                    bt.commutator(ops[0], -1, ops[1], 1, RES)
                    masks.append(torch.isfinite(RES[0]))
                print(f"[gemm leaks] {emax} {lmax} {nucleus} shape {shape} channel {q} block {g} {ij} operand {which}: "
                      f"{int((~masks[0]).sum())} of {b.oplen}", flush=True)
                assert masks[0].any() and not masks[0].all()
                assert torch.equal(masks[0], masks[1])


@pytest.mark.parametrize("shape", [6, 7])
def test_cross_coupled_product(gpu, shape):
    from eom_imsrg import CCMat, CCWork, SqOp, commutators as cm
    b, _ = _basis(6, 4, "O22")
    LCC, RCC = CCMat(b, -1), CCMat(b, 1)
    cm.calculate_cross_coupled(SqOp.from_numpy(b, _op(b, -1, 23), -1), LCC)
    cm.calculate_cross_coupled(SqOp.from_numpy(b, _op(b, 1, 24), 1), RCC)
    blocks = [q for q in range(b.ncc) if b.rlen[q] > 32 and b.rlen[q] % 64 and b.ncol[q] > 1 and b.ncol[q] % 8]
    assert blocks
    for q in (blocks[0], blocks[-1]):
        r, n = int(b.rlen[q]), int(b.ncol[q])
        for i, k in ((r - 1, n - 1), (r - 1, 0), (0, n - 1)):
            for X in (LCC, RCC):
                at = int(b.ccoff[q]) + i + k * r
                keep = X.data[at].clone()
                X.data[at] = float("inf")
                masks = []
                for s in (5, shape):
                    _set(b, ("PH",), s)
                    RES, WCC = SqOp.zeros(b, 1), CCWork(b)
                    cm.commutator_222_ph(LCC, RCC, RES, WCC)
                    o = int(b.wcoff[q])
                    W = torch.triu(WCC.data[o: o + r * r].view(r, r).T)   # the documented part
                    masks.append((torch.isfinite(W), torch.isfinite(RES.data)))
                X.data[at] = keep
                print(f"[gemm leaks] W' shape {shape} block {q} ({r} x {n}) at {(i, k)}", flush=True)
                assert not masks[0][0].all() and masks[0][0].any()
                assert all(torch.equal(x, y) for x, y in zip(*masks))


@pytest.mark.parametrize("shape", [6, 7])
def test_reverse_products(gpu, shape):
    """the transposed 222_pp_hh products (their operands in every orientation)"""
    from eom_imsrg import SqOp, adjoint
    b, _ = _basis(4, 4, "O16")
    L, R, C = SqOp.from_numpy(b, _op(b, -1, 25), -1), SqOp.from_numpy(b, _op(b, 1, 26), 1), _op(b, 1, 27)
    for q in _channels(b)[:1]:
        for g, ij, at in _corners(b, q):
            Cb = torch.from_numpy(C.copy()).cuda()
            Cb[at] = float("inf")
            masks = []
            for s in (5, shape):
                _set(b, ("ADJ", "ADJ_PP"), s)
                Lb, Rb = torch.zeros_like(L.data), torch.zeros_like(R.data)
                adjoint.commutator_vjp(L, R, Cb, 1, Lb, Rb)
                masks.append((torch.isfinite(Lb), torch.isfinite(Rb)))
            print(f"[gemm leaks] reverse shape {shape} channel {q} block {g} {ij}: {int((~masks[0][0]).sum())}", flush=True)
            assert not masks[0][0].all() and masks[0][0].any()
            assert all(torch.equal(x, y) for x, y in zip(*masks))
