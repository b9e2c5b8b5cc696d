"""Which form the fused commutator of a small basis takes: three launches where
every GEMM family is on 32x32 tiles and the instances do not fill the chip, a
launch per term otherwise; and the same bits from both."""
import numpy as np
import pytest
import torch

from test_gpu_122_tiles import _basis, _op

pytestmark = pytest.mark.gpu

FAMILIES = ("PPPP", "PPX", "XX", "PH")


def _set(b, shapes):
    from eom_imsrg import _lib
    for fam, s in zip(FAMILIES, shapes):
        _lib.check(_lib.lib.imsrg_set_gemm_tile(b.handle, _lib.GEMM[fam], s))


def _phases(b):
    from eom_imsrg import _lib
    return int(_lib.lib.imsrg_basis_size(b.handle, _lib.SIZE["PHASES"]))


@pytest.mark.parametrize("emax,lmax,nucleus", [(1, 1, "He4"), (2, 2, "O16"), (3, 1, "He4"), (3, 3, "O16"), (4, 2, "C14"),
                                               (4, 4, "O22"), (4, 4, "O16")])
def test_both_forms_run_and_agree(gpu, emax, lmax, nucleus):
    from eom_imsrg import Batch
    b, _ = _basis(emax, lmax, nucleus)
    L, R = (torch.from_numpy(np.stack([_op(b, h, s) for s in (61, 62)])).cuda() for h in (-1, 1))
    out = []
    for shapes, three in (((13, 13, 13, 13), True), ((8, 13, 13, 13), False)):
        _set(b, shapes)
        bt = Batch(b, 2, graphs=False)
        RES = bt.zeros()
        bt.commutator(L, -1, R, 1, RES)
        print(f"[phases] eMax {emax} lMax {lmax} {nucleus} shapes {shapes}: up to {_phases(b)} instances", flush=True)
        assert (_phases(b) >= 2) == three
        out.append(RES)
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("emax,lmax,nucleus", [(2, 2, "He4"), (4, 4, "O16"), (6, 3, "O16")])
def test_large_batches_take_the_term_launches(gpu, emax, lmax, nucleus):
    """untuned shapes; batches just below and above the limit have the same bits"""
    from eom_imsrg import Batch
    b, _ = _basis(emax, lmax, nucleus)
    assert _phases(b) == 0   # no device plan yet
    one = Batch(b, 1, graphs=False)
    L, R, X = (torch.from_numpy(_op(b, h, 63)[None]).cuda() for h in (-1, 1, 1))
    one.commutator(L, -1, R, 1, X)
    n = _phases(b)
    print(f"[phases] eMax {emax} lMax {lmax} {nucleus}: up to {n} instances", flush=True)
    assert 1 <= n < 64
    for k in (n, n + 1):
        bt = Batch(b, k, graphs=False)
        RES = bt.zeros()
        bt.commutator(L.expand(k, -1).contiguous(), -1, R.expand(k, -1).contiguous(), 1, RES)
        assert torch.equal(RES, X.expand(k, -1))
