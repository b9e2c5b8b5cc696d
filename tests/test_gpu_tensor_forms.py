"""The two forms of the tensor terms 212 and 222_ph, one thread per output and
one wave per pack of alike orbit quadruples: which one a tensor's size
selects."""
import pytest
import torch

from test_gpu_tensor import Basis, SqOp, tensor

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
