"""The tensor terms that run by packs of orbit quadruples (212, 222_ph) against
the oracle where the packs have their edges: one shell (packs of one
quadruple), more outputs than a lane accumulates at a time (j up to 9/2, rank
8), odd parity change, quadruples with equal orbits in a pair."""
import pytest

from test_gpu_tensor import test_full_commutator_and_norm_vs_oracle as full

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("emax,rank,dpar", [(1, 2, 0), (2, 2, 2), (3, 8, 0), (4, 6, 2), (4, 8, 0)])
def test_packs(emax, rank, dpar):
    print(f"[tensor packs] eMax {emax} rank {rank} dpar {dpar}", flush=True)
    full(emax, rank, dpar, -1, 1)
