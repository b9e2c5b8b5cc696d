"""commutator_122 by closed tiles (k_comm122t) against the oracle, on bases
whose (l, j, tz) blocks select each variant of the kernel (up to 4, 5, 6 and
7 orbits a block), with partly filled channels and slabs, and on one basis
with a block too large for a tile and one too small to fill the chip (the
list kernel).  All four hermiticity pairs; RES starts from an unsymmetric
prior (the term assigns).  The form that stores upper triangles only runs in
the fused commutator (test_gpu_ph_blocks)."""
import numpy as np
import pytest
import torch

from conftest import assert_rel
from test_gpu_nuclei import _holes

pytestmark = pytest.mark.gpu

HERMS = [(-1, 1), (-1, -1), (1, 1), (1, -1)]
SHAPES = [(6, 6, "O16"), (7, 4, "O22"), (8, 4, "C14"), (10, 3, "Ca40"), (12, 3, "He4"), (14, 1, "He4"), (5, 5, "O16")]


def _basis(emax, lmax, nucleus):
    from eom_imsrg import Basis, hk_orbits, oxygen16_holes
    from oracle.oracle import OracleBasis
    o = hk_orbits(emax, lmax)
    hole = oxygen16_holes(o) if nucleus == "O16" else _holes(o, nucleus)
    b = Basis(o["n"], o["l"], o["jj"], o["tz"], hole, o["e"])
    return b, OracleBasis(b.n, b.l, b.jj, b.tz, b.hole)


def _op(b, herm, seed):
    from eom_imsrg import synth
    return synth.hermitian_random(b, seed, 1.0) if herm == 1 else synth.antihermitian(b, seed, 1.0)


@pytest.mark.parametrize("emax,lmax,nucleus", SHAPES)
def test_122_vs_oracle(gpu, emax, lmax, nucleus):
    from eom_imsrg import SqOp, commutators as cm
    b, o = _basis(emax, lmax, nucleus)
    rng = np.random.default_rng(emax)
    two = slice(b.off_fpp + b.npart ** 2, b.oplen)
    for hL, hR in HERMS:
        print(f"[122 tiles] eMax {emax} lMax {lmax} {nucleus} herm ({hL},{hR})", flush=True)
        L, R, h = _op(b, hL, 3), _op(b, hR, 4), -hL * hR
        prior = rng.normal(0, 1, b.oplen)
        ref = prior.copy()
        o.comm122(L, hL, R, hR, ref, h)
        for path in (0, 1):
            b.set_path(path)
            RES = SqOp.from_numpy(b, prior, h)
            cm.commutator_122(SqOp.from_numpy(b, L, hL), SqOp.from_numpy(b, R, hR), RES)
            torch.cuda.synchronize()
            got = RES.numpy()
            assert_rel(got[two], ref[two], what=f"122 path {path}")
            assert np.array_equal(got[: two.start], ref[: two.start])
        b.set_path(0)
