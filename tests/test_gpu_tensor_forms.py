"""The two forms of the tensor terms 212 and 222_ph, one thread per output and
one wave per pack of alike orbit quadruples: which one a tensor's size
selects, and each against the oracle."""
import numpy as np
import pytest
import torch

from test_gpu_tensor import Basis, CCMat, SqOp, _case, _close, cm, tensor

pytestmark = pytest.mark.gpu


def _packs(emax, rank, dpar):
    b = Basis.oxygen16(emax)
    tl = tensor.TensorLayout(b, rank, dpar)
    print(f"[tensor forms] eMax {emax} rank {rank} dpar {dpar}", flush=True)
    assert tl.packs == 0   # nothing on the device yet
    RES = tensor.TensorOp.zeros(tl, 1)
    tensor.TS_commutator_212(SqOp.zeros(b, -1), tensor.TensorOp.zeros(tl, 1), RES)
    torch.cuda.synchronize()
    return tl.packs


# eMax 5 rank 8: 888 k outputs of 128 k quadruples; eMax 6 rank 0: 958 k of 376 k
@pytest.mark.parametrize("emax,rank,dpar,by_packs", [(2, 2, 2, False), (4, 8, 0, False), (5, 4, 0, False),
                                                     (5, 8, 0, False), (6, 0, 0, True), (6, 2, 2, True)])
def test_packs_only_where_they_run(emax, rank, dpar, by_packs):
    """a tensor whose terms run one thread per output holds no pack lists"""
    assert (_packs(emax, rank, dpar) > 0) == by_packs


HERMS = [(-1, 1), (-1, -1), (1, 1), (1, -1)]


@pytest.mark.parametrize("form", ["outputs", "packs"])
@pytest.mark.parametrize("emax,rank,dpar", [(1, 2, 0), (2, 2, 2), (3, 8, 0), (3, 6, 2), (4, 4, 0)])
def test_forms_vs_oracle(emax, rank, dpar, form):
    """both forms of 212 and 222_ph against the oracle at every pair of
    hermiticities: one shell, packs of one quadruple and of 64, more outputs than
    a lane accumulates at a time, equal orbits in a pair, odd parity change"""
    for hL, hR in HERMS:
        b, o, ot, tl, L, R, P = _case(emax, rank, dpar, hL, hR, seed=7)
        tl.set_form(form)
        hC = -hL * hR
        print(f"[tensor forms] eMax {emax} rank {rank} dpar {dpar} herm ({hL},{hR}) {form}", flush=True)
        Ld, Rd = SqOp.from_numpy(b, L, hL), tensor.TensorOp.from_numpy(tl, R, hR)
        LCC, RCC = CCMat(b, hL), tensor.TensorCC(tl)
        cm.calculate_cross_coupled(Ld, LCC)
        X = tensor.TensorOp.from_numpy(tl, P, hC)
        tensor.TS_commutator_212(Ld, Rd, X)
        _close(X.numpy(), ot.ts212(L, hL, R, hR, P.copy(), hC), f"212 {form} ({hL},{hR})")
        X = tensor.TensorOp.from_numpy(tl, P, hC)
        tensor.TS_commutator_222_ph(LCC, RCC, Rd, X)
        _close(X.numpy(), ot.ts222ph(L, hL, R, hR, P.copy(), hC), f"222_ph {form} ({hL},{hR})")
        assert (tl.packs > 0) == (form == "packs")


def test_form_is_set_before_the_first_use():
    from eom_imsrg import _lib
    b = Basis.oxygen16(2)
    tl = tensor.TensorLayout(b, 2, 0)
    tl.set_form("packs")
    tl.set_form("size")
    with pytest.raises(_lib.ImsrgError):
        _lib.check(_lib.lib.imsrg_tensor_set_form(tl.handle, 3))
    tensor.TS_commutator_212(SqOp.zeros(b, -1), tensor.TensorOp.zeros(tl, 1), tensor.TensorOp.zeros(tl, 1))
    with pytest.raises(_lib.ImsrgError):
        tl.set_form("outputs")


@pytest.mark.parametrize("emax,rank,dpar", [(2, 2, 2), (4, 4, 0), (3, 8, 0)])
def test_nonfinite_elements_reach_the_same_outputs(emax, rank, dpar):
    """an infinite element of L, R or a cross-coupled set reaches the outputs whose
    sums hold it and no other, in both forms"""
    b, _, _, tl, L, R, _ = _case(emax, rank, dpar, -1, 1, seed=9)
    two = b.off_fpp + b.npart ** 2
    rng = np.random.default_rng(emax)
    spread = [0, 0]
    for at in [two + int(x) for x in rng.integers(0, b.oplen - two, 6)] + [b.off_fph, b.off_fpp + 1]:
        out = []
        for form in ("outputs", "packs"):
            t = tensor.TensorLayout(b, rank, dpar)
            t.set_form(form)
            L2, R2 = L.copy(), R.copy()
            (L2 if at >= two else R2)[at] = np.inf
            X = tensor.TensorOp.zeros(t, 1)
            tensor.TS_commutator_212(SqOp.from_numpy(b, L2, -1), tensor.TensorOp.from_numpy(t, R2, 1), X)
            LCC, RCC, Y = CCMat(b, -1), tensor.TensorCC(t), tensor.TensorOp.zeros(t, 1)
            cm.calculate_cross_coupled(SqOp.from_numpy(b, L, -1), LCC)
            LCC.data[at * 7919 % b.cclen] = float("inf")
            tensor.TS_commutator_222_ph(LCC, RCC, tensor.TensorOp.from_numpy(t, R, 1), Y)
            out.append([np.isfinite(Z.numpy()) for Z in (X, Y)])
        print(f"[tensor forms] eMax {emax} rank {rank} inf at {at}", [int((~m).sum()) for o in out for m in o], flush=True)
        for k, what in enumerate(("212", "222_ph")):
            assert np.array_equal(out[0][k], out[1][k]), f"{what}, element {at}"
            spread[k] += int((~out[0][k]).sum())
    assert spread[0] > 0 and spread[1] > 0


@pytest.mark.parametrize("emax,rank,dpar", [(2, 2, 2), (4, 4, 0), (3, 8, 0)])
def test_forbidden_elements_stay_zero(emax, rank, dpar):
    """two equal orbits do not couple to odd J: where one thread per output leaves
    such an element exactly zero, so do the packs"""
    b, _, _, tl, L, R, _ = _case(emax, rank, dpar, -1, 1, seed=13)
    zero = []
    for form in ("outputs", "packs"):
        t = tensor.TensorLayout(b, rank, dpar)
        t.set_form(form)
        Ld, Rd = SqOp.from_numpy(b, L, -1), tensor.TensorOp.from_numpy(t, R, 1)
        X, Y = tensor.TensorOp.zeros(t, 1), tensor.TensorOp.zeros(t, 1)
        tensor.TS_commutator_212(Ld, Rd, X)
        LCC, RCC = CCMat(b, -1), tensor.TensorCC(t)
        cm.calculate_cross_coupled(Ld, LCC)
        tensor.TS_commutator_222_ph(LCC, RCC, Rd, Y)
        zero.append([Z.numpy() == 0.0 for Z in (X, Y)])
    odd = np.zeros(tl.oplen, bool)
    for q, g, ix, jx, (a, c), (d, e), J1, J2, at in tl.elements():
        odd[at] = (a == c and J1 // 2 % 2 == 1) or (d == e and J2 // 2 % 2 == 1)
    print(f"[tensor forms] eMax {emax} rank {rank}: {int(odd.sum())} forbidden, zero by form",
          [[int(z[odd].sum()) for z in f] for f in zero], flush=True)
    for k, what in enumerate(("212", "222_ph")):
        assert odd.any() and zero[0][k][odd].any()
        assert not (zero[0][k] & odd & ~zero[1][k]).any(), what
