"""The tensor terms 212 and 222_ph in both forms (one thread per output below
800,000 outputs, packs of orbit quadruples from there) against the oracle
where they have their edges: one shell, rank 8 with more outputs than a lane of
a pack accumulates at a time, odd parity change, quadruples with equal orbits
in a pair; the last case runs by packs."""
import pytest

from test_gpu_tensor import test_full_commutator_and_norm_vs_oracle as full

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("emax,rank,dpar", [(1, 2, 0), (2, 2, 2), (3, 8, 0), (4, 6, 2), (4, 8, 0), (5, 8, 0)])
def test_both_forms(emax, rank, dpar):
    print(f"[tensor packs] eMax {emax} rank {rank} dpar {dpar}", flush=True)
    full(emax, rank, dpar, -1, 1)
