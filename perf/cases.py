"""The calls that a user of this framework makes, as measurable cases.

A run of the reference's ``magnus_decouple`` spends its time in nested
commutators of scalar operators (BCH_EXPAND, MAGNUS_EXPAND); around them stand
the single terms of the commutator, many-instance batches, reverse-mode
derivatives and the commutator with a tensor observable.  Each case is one
call of those (or, for ``steps``, the first steps of a flow).

A case is a dict with

  kind     commutator | c122 | pphh | ph | bch | steps | decouple | batch |
           vjp | grad | tensor
  emax     HO orbits with 2n + l <= emax (0-based shells)
  lmax     and l <= lmax (lmax < emax gives ragged channel lists)
  nucleus  the holes of the reference state
  ...      the options of the kind

Inputs are random operators of the shapes a nuclear Hamiltonian and a Magnus
operator have: matrix elements that fall off with the HO energy of their
orbits, zero where the Pauli principle or the (l, j, tz) selection rules say
so.  They are drawn on the GPU from the seed alone.
"""
from __future__ import annotations

import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "eom-imsrg_amd"))

from eom_imsrg import Basis, Batch, CCMat, CCWork, Flow, SqOp, adjoint, hk_orbits, tensor, tune, workload  # noqa: E402
from eom_imsrg import commutators as cm  # noqa: E402

ROWS, COLS, SQUARE = (0, 0, 0, 1, 2, 1), (0, 1, 2, 1, 2, 2), (0, 3, 4)


def listed():
    return [
        # one commutator through the public term routines, at the size of a
        # quick test run: a dozen small launches, latency only
        {"name": "commutator_e4", "kind": "commutator", "emax": 4, "lmax": 4, "nucleus": "O16"},
        # a whole flow at the size of a tutorial: launches and the host's loop
        {"name": "decouple_e4", "kind": "decouple", "emax": 4, "lmax": 4, "nucleus": "O16", "generator": "white"},
        # e^Omega H e^-Omega for an open-shell reference at an ordinary small size
        {"name": "bch_e6_O22", "kind": "bch", "emax": 6, "lmax": 6, "nucleus": "O22", "sigma": 0.1},
        # production size: the first two steps of a flow (the benchmark's work)
        {"name": "steps_e8", "kind": "steps", "emax": 8, "lmax": 8, "nucleus": "O16", "steps": 2},
        # the largest basis that the repository runs
        {"name": "bch_e10", "kind": "bch", "emax": 10, "lmax": 10, "nucleus": "O16", "sigma": 0.1},
        # single terms, as a caller that composes its own commutator uses them
        {"name": "c122_e8_Ca40", "kind": "c122", "emax": 8, "lmax": 8, "nucleus": "Ca40", "hL": -1, "hR": 1},
        {"name": "pphh_e8", "kind": "pphh", "emax": 8, "lmax": 8, "nucleus": "O16", "hL": -1, "hR": 1},
        # the particle-hole term on an odd shell and a cut in l
        {"name": "ph_e7_l5_C14", "kind": "ph", "emax": 7, "lmax": 5, "nucleus": "C14", "hL": -1, "hR": 1},
        # an ensemble of Hamiltonians (uncertainty quantification) in one batch
        {"name": "batch64_e6", "kind": "batch", "emax": 6, "lmax": 6, "nucleus": "O16", "ninst": 64, "sigma": 0.1},
        # reverse mode: one commutator's transpose, and the gradient of a whole flow
        {"name": "vjp_e8", "kind": "vjp", "emax": 8, "lmax": 8, "nucleus": "O16", "hL": -1, "hR": 1},
        {"name": "grad_e6", "kind": "grad", "emax": 6, "lmax": 6, "nucleus": "O16", "ckpt": 0},
        # a rank-2 observable's nested commutator (transform_sq_op_BCH)
        {"name": "tensor_e8_r4", "kind": "tensor", "emax": 8, "lmax": 8, "nucleus": "O16", "rank": 4, "dpar": 0},
    ]


def draw(rng):
    """one more case of the same ranges; none costs more than the largest listed one"""
    kind = rng.choice(["commutator", "c122", "pphh", "ph", "bch", "bch", "steps", "steps", "decouple", "batch", "vjp",
                       "grad", "tensor"])
    nucleus = rng.choice(["He4", "O16", "O16", "C14", "O22", "Ca40"])
    top = {"commutator": 9, "c122": 9, "pphh": 9, "ph": 9, "bch": 9, "steps": 9, "decouple": 5, "batch": 6, "vjp": 8,
           "grad": 5, "tensor": 7}[kind]
    emax = rng.randint(3, top)
    lmax = emax if rng.random() < 0.6 else rng.randint(2, emax)
    c = {"kind": kind, "emax": emax, "lmax": lmax, "nucleus": nucleus}
    if kind in ("c122", "pphh", "ph", "vjp"):
        c["hL"] = rng.choice([-1, -1, 1])
        c["hR"] = rng.choice([1, 1, -1])
    if kind in ("steps", "decouple", "grad"):
        # flows converge from a closed shell
        c["nucleus"] = "O16"
    if kind in ("bch", "batch"):
        c["sigma"] = round(rng.uniform(0.05, 0.12), 3)
    if kind == "steps":
        c["steps"] = rng.randint(1, 3)
    if kind == "decouple":
        c["generator"] = rng.choice(["white", "atan", "w2"])
    if kind == "batch":
        # the product of instances and their size stays below the listed batch
        c["ninst"] = max(2, min(96, int(2 ** rng.uniform(1, 5.5) * 4 ** (6 - emax) / (1 if emax == 6 else 2))))
    if kind == "grad":
        c["ckpt"] = rng.choice([0, 4])
    if kind == "tensor":
        c["rank"] = rng.choice([0, 2, 4])
        c["dpar"] = rng.choice([0, 2]) if c["rank"] else 0
        c["nucleus"] = rng.choice(["He4", "O16"])
    return c


# ------------------------------------------------------------------ bases
def _holes(o, nucleus):
    n, l, jj, tz = (np.asarray(o[k]) for k in ("n", "l", "jj", "tz"))
    s = (n == 0) & (l == 0)
    sp = (n == 0) & (l <= 1)
    return {
        "He4": s,
        "O16": sp,
        "C14": sp & ~((l == 1) & (jj == 1) & (tz == -1)),
        "O22": sp | ((n == 0) & (l == 2) & (jj == 5) & (tz == 1)),
        "Ca40": 2 * n + l <= 2,
    }[nucleus].astype(np.int32)


@functools.lru_cache(maxsize=None)
def _basis(emax, lmax, nucleus):
    """the basis handle: built once by a program and used for every operator,
    with the shipped GEMM tile choice where there is one"""
    o = hk_orbits(emax, lmax)
    b = Basis(o["n"], o["l"], o["jj"], o["tz"], _holes(o, nucleus), o["e"])
    choice = tune.lookup(b)
    if choice is not None:
        tune.apply(b, choice)
    return b


@functools.lru_cache(maxsize=None)
def _layout(emax, lmax, nucleus, rank, dpar):
    return tensor.TensorLayout(_basis(emax, lmax, nucleus), rank, dpar)


def _of(case):
    return _basis(case["emax"], case["lmax"], case["nucleus"])


# ------------------------------------------------------------------ inputs
def _pair_weights(b, q, cls, damp):
    pr = b.pairs[q][cls]
    w = np.exp(-(b.e[pr[:, 0]] + b.e[pr[:, 1]]) / 8.0) if damp else np.ones(len(pr))
    if (int(b.jtp[q, 0]) // 2) % 2 == 1:
        w = np.where(pr[:, 0] == pr[:, 1], 0.0, w)
    return torch.from_numpy(w).cuda()


def _operators(b, gen, ninst, herm, two, one, diag=None):
    """(ninst, oplen): one-body elements N(0, one) inside the (l, j, tz)
    blocks (plus `diag` on the diagonal), two-body elements
    N(0, two) exp(-(e_a + e_b + e_c + e_d) / 8)"""
    x = torch.zeros(ninst, b.oplen, dtype=torch.float64, device="cuda")
    key = [(int(b.l[a]), int(b.jj[a]), int(b.tz[a])) for a in range(b.norb)]
    same = torch.tensor([[u == v for v in key] for u in key], dtype=torch.float64, device="cuda")
    f = torch.randn(ninst, b.norb, b.norb, dtype=torch.float64, device="cuda", generator=gen) * one
    f = torch.triu(f, 1)
    f = (f + herm * f.transpose(1, 2)) * same
    if diag is not None:
        f = f + torch.diag(diag)
    h, p = torch.from_numpy(b.holes).cuda(), torch.from_numpy(b.parts).cuda()
    A, P = b.nhole, b.npart
    x[:, b.off_fhh: b.off_fhh + A * A] = f[:, h][:, :, h].transpose(1, 2).reshape(ninst, -1)
    x[:, b.off_fph: b.off_fph + P * A] = f[:, p][:, :, h].transpose(1, 2).reshape(ninst, -1)
    x[:, b.off_fpp: b.off_fpp + P * P] = f[:, p][:, :, p].transpose(1, 2).reshape(ninst, -1)
    o2 = b.off_fpp + P * P
    x[:, o2:] = torch.randn(ninst, b.oplen - o2, dtype=torch.float64, device="cuda", generator=gen) * two
    for q in range(b.nblocks):
        w = [_pair_weights(b, q, c, True) for c in range(3)]
        for g in range(6):
            n1, n2 = b.block_shape(q, g)
            if n1 * n2 == 0:
                continue
            o = int(b.goff[q, g])
            v = x[:, o: o + n1 * n2].view(ninst, n2, n1)   # column-major blocks
            v *= w[COLS[g]][:, None] * w[ROWS[g]][None, :]
            if g in SQUARE:
                u = torch.tril(v, -1)                      # the block's upper triangle
                d = torch.diag_embed(torch.diagonal(v, dim1=1, dim2=2)) if herm == 1 else 0.0
                v.copy_(u + herm * u.transpose(1, 2) + d)
    return x


def _hamiltonian(b, gen, ninst=1):
    """vacuum t + V, hbar omega = 20 MeV"""
    d = torch.from_numpy(20.0 * (b.e + 1.5)).cuda()
    return _operators(b, gen, ninst, 1, 1.0, 0.5, d)


def _any(b, gen, herm, sigma=0.1):
    """a Hamiltonian-like (herm 1) or Omega-like (herm -1) operator"""
    if herm == 1:
        return SqOp(b, _hamiltonian(b, gen)[0], 1)
    return SqOp(b, _operators(b, gen, 1, -1, sigma, sigma)[0], -1)


def _tensor_operator(tl, gen):
    """a random tensor observable of the layout's selection rules"""
    b = tl.basis
    x = torch.zeros(tl.oplen, dtype=torch.float64, device="cuda")
    l, jj, tz = (np.asarray(v) for v in (b.l, b.jj, b.tz))

    def ok1(r, c):
        r, c = r[:, None], c[None, :]
        return torch.from_numpy((tz[r] == tz[c]) & ((l[r] + l[c] + tl.dpar // 2) % 2 == 0)
                                & (np.abs(jj[r] - jj[c]) <= tl.rank) & (tl.rank <= jj[r] + jj[c])).cuda()

    def randn(n1, n2):
        return torch.randn(n1, n2, dtype=torch.float64, device="cuda", generator=gen)

    H, P = b.holes, b.parts
    for r, off in ((H, b.off_fhh), (P, b.off_fpp)):
        ph = torch.from_numpy(1.0 - 2.0 * ((np.abs(jj[r][:, None] - jj[r][None, :]) // 2) % 2)).cuda()
        u = torch.triu(randn(len(r), len(r)), 1)
        m = (u + (ph * u).T) * ok1(r, r) + torch.diag(torch.diagonal(ok1(r, r)) * randn(1, len(r))[0])
        x[off: off + len(r) ** 2] = m.T.reshape(-1)
    m = randn(len(P), len(H)) * ok1(P, H)
    x[b.off_fph: b.off_fph + len(P) * len(H)] = m.T.reshape(-1)
    mirror = (0, 7, 6, 3, 4, 8, 2, 1, 5)   # the sub-block that holds the transposed element at J1 = J2
    look = {tuple(int(v) for v in tl.info[q, :4]): q for q in range(tl.nblocks)}
    weights = {}

    def weight(q, cls):
        if (q, cls) not in weights:
            weights[q, cls] = _pair_weights(b, q, cls, True)
        return weights[q, cls]

    for q in range(tl.nblocks):
        J1, J2, t, P1, P2, q1, q2 = (int(v) for v in tl.info[q])
        if q2 < 0:
            continue
        for g in range(9):
            n1, n2 = tl.shape(q, g)
            if n1 * n2 == 0:
                continue
            v = randn(n2, n1) * weight(q2, tl.SEA2[g])[:, None] * weight(q1, tl.SEA1[g])[None, :]
            o = int(tl.goff[q, g])
            if J1 == J2:
                qm, gm = look[(J1, J1, t, P2)], mirror[g]
                if (qm, gm) < (q, g):
                    om = int(tl.goff[qm, gm])
                    v = x[om: om + n1 * n2].view(n1, n2).T
                elif (qm, gm) == (q, g):
                    v = torch.tril(v) + torch.tril(v, -1).T
            x[o: o + n1 * n2] = v.reshape(-1)
    return tensor.TensorOp(tl, x, 1)


def prepare(case, seed):
    b, kind = _of(case), case["kind"]
    gen = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)
    s = {"kind": kind, "basis": b, "case": case}
    if kind in ("commutator", "c122", "pphh", "ph", "vjp"):
        hL, hR = case.get("hL", -1), case.get("hR", 1)
        s["L"], s["R"] = _any(b, gen, hL), _any(b, gen, hR)
        s["RES"] = SqOp.zeros(b, -hL * hR)
        if kind in ("commutator", "pphh"):
            s["w1"], s["w2"] = SqOp.zeros(b), SqOp.zeros(b)
        if kind == "ph":
            s["LCC"], s["RCC"] = CCMat(b, hL), CCMat(b, hR)
            s["WCC"] = CCWork(b)
        if kind == "vjp":
            s["RESb"] = _operators(b, gen, 1, -hL * hR, 1.0, 0.5)[0]
            s["Lb"], s["Rb"] = torch.zeros_like(s["L"].data), torch.zeros_like(s["R"].data)
    elif kind == "bch":
        s["G"], s["H"] = _any(b, gen, -1, case["sigma"]), _any(b, gen, 1)
        s["HS"] = SqOp.zeros(b, 1)
        s["flow"] = Flow(b, graphs=True)
    elif kind in ("steps", "decouple"):
        s["H"] = _any(b, gen, 1)
        cm.normal_order(s["H"])
        s["HS"], s["G"] = SqOp.zeros(b, 1), SqOp.zeros(b, -1)
        s["DG"] = SqOp.zeros(b, -1)
        s["flow"] = Flow(b, graphs=True, generator=case.get("generator", "white"))
    elif kind == "batch":
        n = case["ninst"]
        s["G"] = _operators(b, gen, n, -1, case["sigma"], case["sigma"])
        s["H"] = _hamiltonian(b, gen, n)
        s["batch"] = Batch(b, n, graphs=True)
        s["HS"] = s["batch"].zeros()
    elif kind == "grad":
        s["T"] = _hamiltonian(b, gen)[0]
        s["flow"] = Flow(b, graphs=True)
    else:
        tl = _layout(case["emax"], case["lmax"], case["nucleus"], case["rank"], case["dpar"])
        s["G"], s["O"] = _any(b, gen, -1), _tensor_operator(tl, gen)
        s["RES"] = tensor.TensorOp.zeros(tl, 1)
    return s


def _padded(rows, n):
    """the rows of a call's log, to a length that does not depend on the data"""
    out = np.zeros((n,) + rows.shape[1:])
    out[: len(rows)] = rows
    return out


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "commutator":
        cm.commutator(s["L"], s["R"], s["RES"], s["w1"], s["w2"])
        return s["RES"].data
    if kind == "c122":
        cm.commutator_122(s["L"], s["R"], s["RES"])
        return s["RES"].data
    if kind == "pphh":
        cm.clear_sq_op(s["RES"])   # the term adds to RES
        cm.commutator_222_pp_hh(s["L"], s["R"], s["RES"], s["w1"], s["w2"])
        return {"RES": s["RES"].data, "w1": s["w1"].data, "w2": s["w2"].data}
    if kind == "ph":
        cm.clear_sq_op(s["RES"])
        cm.calculate_cross_coupled(s["L"], s["LCC"])
        cm.calculate_cross_coupled(s["R"], s["RCC"])
        cm.commutator_222_ph(s["LCC"], s["RCC"], s["RES"], s["WCC"])
        return {"RES": s["RES"].data, "LCC": s["LCC"].data, "RCC": s["RCC"].data}
    if kind == "bch":
        index, norms = s["flow"].BCH_EXPAND(s["HS"], s["G"], s["H"])
        return {"HS": s["HS"].data, "index": index, "norms": _padded(norms, 40)}
    if kind == "steps":
        s["HS"].data.copy_(s["H"].data)
        s["G"].data.zero_()
        cm.build_gs_white(s["HS"], s["DG"])
        log = [s["flow"].magnus_step(s["HS"], s["G"], s["DG"], s["H"]) for _ in range(case["steps"])]
        return {"HS": s["HS"].data, "G": s["G"].data, "DG": s["DG"].data, "log": np.array(log, np.float64)}
    if kind == "decouple":
        s["HS"].data.copy_(s["H"].data)
        s["G"].data.zero_()
        log = s["flow"].magnus_decouple(s["HS"], s["G"])
        return {"HS": s["HS"].data, "G": s["G"].data, "log": _padded(log, 200)}
    if kind == "batch":
        index = s["batch"].BCH_EXPAND(s["HS"], s["G"], s["H"])
        return {"HS": s["HS"], "index": index}
    if kind == "vjp":
        s["Lb"].zero_()
        s["Rb"].zero_()
        adjoint.commutator_vjp(s["L"], s["R"], s["RESb"], s["RES"].herm, s["Lb"], s["Rb"])
        return {"Lb": s["Lb"], "Rb": s["Rb"]}
    if kind == "grad":
        e0, g, steps = adjoint.flow_grad(s["flow"], s["T"], ckpt=case["ckpt"])
        return {"E0": e0, "g": g, "steps": steps}
    tensor.TS_commutator(s["G"], s["O"], s["RES"])
    return s["RES"].data


# ------------------------------------------------------------------ work
def work(case):
    """Matrix-product flops of the terms (each product that the path cannot do
    without) and every input read and output written once.  The number of
    nested commutators depends on the data: the typical one of these inputs."""
    b, kind = _of(case), case["kind"]
    op, F = 8.0 * b.oplen, workload.commutator_flops(b)
    if kind == "commutator":
        return {"bytes": 3 * op, "flops": F}
    if kind == "c122":
        # two one-body partners of both pairs, L and R: about 8 products of
        # (l, j, tz) block size for each stored element
        n = b.norb / (4.0 * case["lmax"] + 2)
        return {"bytes": 3 * op, "flops": 16.0 * n * b.e2_count()}
    if kind == "pphh":
        return {"bytes": 5 * op, "flops": workload.pphh_flops(b)}
    if kind == "ph":
        return {"bytes": 3 * op + 16.0 * b.cclen, "flops": workload.ph_gemm_flops(b)}
    if kind == "bch":
        return {"bytes": 3 * op, "flops": 19 * F}
    if kind == "steps":
        return {"bytes": 6 * op, "flops": (8, 21, 35)[case["steps"] - 1] * F}
    if kind == "decouple":
        return {"bytes": 3 * op, "flops": 170 * F}
    if kind == "batch":
        return {"bytes": 3 * op * case["ninst"], "flops": 18 * F * case["ninst"]}
    if kind == "vjp":
        return {"bytes": 5 * op, "flops": 2 * F}
    if kind == "grad":
        return {"bytes": 2 * op, "flops": 3 * 160 * F}
    tl = _layout(case["emax"], case["lmax"], case["nucleus"], case["rank"], case["dpar"])
    return {"bytes": 16.0 * tl.oplen + op, "flops": _tensor_flops(b, tl)}


def _tensor_flops(b, tl):
    """the products of the pp / hh intermediates and of the cross-coupled blocks"""
    f = 0.0
    for q in range(tl.nblocks):
        d1, d2 = tl.dims[q, :3].astype(float), tl.dims[q, 3:].astype(float)
        for r in range(3):
            for c in range(3):
                f += 2.0 * d1[r] * d2[c] * (d1[0] + d2[0] + d1[2] + d2[2])
    per = b.jtotal_max + 1
    for k3 in range(per):
        for k4 in range(k3, min(per, k3 + tl.rank // 2 + 1)):
            if k3 + k4 < tl.rank // 2:
                continue
            for x in range(4):
                s1, s2 = k3 + per * x, k4 + per * (x ^ (2 if tl.dpar else 0))
                f += 2.0 * b.rlen[s1] * b.rlen[s2] * (int(b.ncol[s1]) + (int(b.ncol[s2]) if k3 != k4 else 0))
    return f


# ------------------------------------------------- the same in dense form
# exact(): the commutator from its orbit-space formulas on dense arrays
# V[J][a, b, c, d] over all ordered orbits (unnormalised, antisymmetric), with
# none of the channel, class or cross-coupled bookkeeping of the framework.
class _Dense:
    def __init__(self, b):
        self.b, N = b, b.norb
        dev = "cuda"
        self.N = N
        self.jj = torch.from_numpy(b.jj.astype(np.int64)).to(dev)
        self.n = torch.from_numpy(b.hole.astype(np.float64)).to(dev)
        self.nJ = int(b.jj.max()) + 1
        jv = np.unique(b.jj)
        self.jc = torch.from_numpy(np.searchsorted(jv, b.jj)).to(dev)
        self.jv, self._six = jv, {}
        key = torch.from_numpy(b.l.astype(np.int64) * 1000 + b.jj * 10 + b.tz).to(dev)
        self.same = (key[:, None] == key[None, :]).double()
        at, J, orb, fac, herm = [], [], [], [], []
        for q in range(b.nblocks):
            for g in range(6):
                n1, n2 = b.block_shape(q, g)
                if n1 * n2 == 0:
                    continue
                r, c = b.pairs[q][ROWS[g]], b.pairs[q][COLS[g]]
                jx, ix = np.divmod(np.arange(n1 * n2), n1)
                at.append(int(b.goff[q, g]) + np.arange(n1 * n2))
                J.append(np.full(n1 * n2, int(b.jtp[q, 0]) // 2))
                orb.append(np.stack([r[ix, 0], r[ix, 1], c[jx, 0], c[jx, 1]], 1))
                fac.append(np.sqrt((1.0 + (r[ix, 0] == r[ix, 1])) * (1.0 + (c[jx, 0] == c[jx, 1]))))
                herm.append(np.full(n1 * n2, g not in SQUARE))
        cat = lambda v: torch.from_numpy(np.concatenate(v)).to(dev)  # noqa: E731
        self.at, self.J, self.orb, self.fac, self.rect = cat(at), cat(J), cat(orb).long(), cat(fac), cat(herm)

    def flat_index(self, a, b, c, d, J):
        return (((J * self.N + a) * self.N + b) * self.N + c) * self.N + d

    def of(self, x, herm):
        """(E0, f, V) of a flat operator"""
        b, N = self.b, self.N
        h, p = torch.from_numpy(b.holes).cuda(), torch.from_numpy(b.parts).cuda()
        A, P = b.nhole, b.npart
        f = torch.zeros(N, N, dtype=torch.float64, device="cuda")
        ph = x[b.off_fph: b.off_fph + P * A].view(A, P).T
        f[h[:, None], h[None, :]] = x[b.off_fhh: b.off_fhh + A * A].view(A, A).T
        f[p[:, None], h[None, :]] = ph
        f[h[:, None], p[None, :]] = herm * ph.T
        f[p[:, None], p[None, :]] = x[b.off_fpp: b.off_fpp + P * P].view(P, P).T
        V = torch.zeros(self.nJ * N ** 4, dtype=torch.float64, device="cuda")
        v = x[self.at] * self.fac
        a, bb, c, d = self.orb.unbind(1)
        J = self.J
        s1 = 1.0 - 2.0 * ((1 + (self.jj[a] + self.jj[bb]) // 2 - J) % 2)
        s2 = 1.0 - 2.0 * ((1 + (self.jj[c] + self.jj[d]) // 2 - J) % 2)
        for (i, j, si) in ((a, bb, 1.0), (bb, a, s1)):
            same = i is bb
            for (k, l, sk) in ((c, d, 1.0), (d, c, s2)):
                w = v * si * sk
                keep = torch.ones_like(w, dtype=torch.bool)
                if same:
                    keep &= a != bb
                if k is d:
                    keep &= c != d
                V[self.flat_index(i, j, k, l, J)[keep]] = w[keep]
                keep &= self.rect
                V[self.flat_index(k, l, i, j, J)[keep]] = herm * w[keep]
        return 0.0, f, V.view(self.nJ, N, N, N, N)

    def flat(self, E0, f, V):
        b = self.b
        h, p = torch.from_numpy(b.holes).cuda(), torch.from_numpy(b.parts).cuda()
        x = torch.zeros(b.oplen, dtype=torch.float64, device="cuda")
        x[0] = E0
        if f is not None:
            for r, c, o in ((h, h, b.off_fhh), (p, h, b.off_fph), (p, p, b.off_fpp)):
                x[o: o + len(r) * len(c)] = f[r][:, c].T.reshape(-1)
        a, bb, c, d = self.orb.unbind(1)
        x[self.at] = V.reshape(-1)[self.flat_index(a, bb, c, d, self.J)] / self.fac
        return x

    def six(self, J, K):
        """{ja jb J; jc jd K} over the distinct j, by the Racah sum"""
        if (J, K) not in self._six:
            m = len(self.jv)
            t = np.zeros((m, m, m, m))
            for ia, a in enumerate(self.jv):
                for ib, b in enumerate(self.jv):
                    for ic, c in enumerate(self.jv):
                        for id_, d in enumerate(self.jv):
                            t[ia, ib, ic, id_] = _racah(int(a), int(b), 2 * J, int(c), int(d), 2 * K)
            self._six[J, K] = torch.from_numpy(t).cuda()
        return self._six[J, K]

    def recouple(self, X):
        """Y[J](a, d, c, b) = - sum_K (2K+1) {ja jd J; jc jb K} X[K](a, b, c, d)
        (its own inverse: the second call brings (a, d, c, b) back)"""
        Y = torch.zeros_like(X)
        j = self.jc
        for J in range(self.nJ):
            for K in range(self.nJ):
                t = self.six(J, K)
                if not bool(t.any()):
                    continue
                w = t[j[:, None, None, None], j[None, :, None, None], j[None, None, :, None], j[None, None, None, :]]
                Y[J] -= (2 * K + 1) * w * X[K].permute(0, 3, 2, 1)
        return Y

    def c122(self, L, R):
        V = torch.zeros_like(L[2])
        for (f, W, s) in ((L[1], R[2], 1.0), (R[1], L[2], -1.0)):
            N = self.N
            n3 = (self.nJ, N, N, N, N)
            V += s * torch.matmul(f, W.reshape(self.nJ, N, N ** 3)).view(n3)
            V += s * torch.matmul(f, W.reshape(self.nJ * N, N, N * N)).view(n3)
            V -= s * torch.matmul(f.T, W.reshape(self.nJ * N * N, N, N)).view(n3)
            V -= s * torch.matmul(W.reshape(-1, N), f).view(n3)
        return V

    def ladder(self, L, R):
        """(L D R) with D = pp and D = hh separately (half: ordered pairs count twice)"""
        N, n = self.N, self.n
        pp = 0.5 * torch.outer(1 - n, 1 - n).reshape(-1)
        hh = 0.5 * torch.outer(n, n).reshape(-1)
        l, r = L[2].view(self.nJ, N * N, N * N), R[2].view(self.nJ, N * N, N * N)
        return torch.bmm((l * pp).contiguous(), r.contiguous()), torch.bmm((l * hh).contiguous(), r.contiguous())

    def ph(self, L, R):
        N, n = self.N, self.n
        x, y = self.recouple(L[2]).view(self.nJ, N * N, N * N), self.recouple(R[2]).view(self.nJ, N * N, N * N)
        occ = (n[:, None] - n[None, :]).reshape(-1)
        z = self.recouple(torch.bmm((x * occ).contiguous(), y.contiguous()).view(self.nJ, N, N, N, N))
        del x, y
        out = torch.zeros_like(z)
        for J in range(self.nJ):
            s = 1.0 - 2.0 * (((self.jj[:, None] + self.jj[None, :]) // 2 - J) % 2)
            t = s[:, :, None, None] * z[J].permute(1, 0, 2, 3) - z[J]
            out[J] = t - s[None, None] * t.permute(0, 1, 3, 2)
        return out

    def commutator(self, L, R):
        n, N, jj = self.n, self.N, self.jj.double()
        fl, fr = L[1], R[1]
        occ = n[:, None] * (1 - n[None, :])
        E = float(((jj[:, None] + 1) * occ * (fl * fr.T - fr * fl.T)).sum())
        hh = torch.outer(n, n).reshape(-1)
        pp = torch.outer(1 - n, 1 - n).reshape(-1)
        f = fl @ fr - fr @ fl
        g = torch.zeros_like(f)
        d = n[:, None] - n[None, :]
        lad = self.ladder(L, R)
        rad = self.ladder(R, L)
        for J in range(self.nJ):
            l, r = L[2][J].view(N * N, N * N), R[2][J].view(N * N, N * N)
            E += 0.25 * (2 * J + 1) * float((hh[:, None] * pp[None, :] * (l * r.T - r * l.T)).sum())
            w = (2 * J + 1) / (jj + 1)
            g += w[:, None] * (torch.einsum("ab,biaj->ij", fl * d, R[2][J]) - torch.einsum("ab,biaj->ij", fr * d, L[2][J]))
            mp = (lad[0][J] - rad[0][J]).view(N, N, N, N)
            mh = (lad[1][J] - rad[1][J]).view(N, N, N, N)
            g += w[:, None] * (torch.einsum("c,cicj->ij", n, mp) + torch.einsum("c,cicj->ij", 1 - n, mh))
        f += g * self.same   # the traces are scalars: they keep (l, j, tz)
        V = self.c122(L, R) + (lad[0] - lad[1] - rad[0] + rad[1]).view_as(L[2])
        del lad, rad
        V += self.ph(L, R)
        return E, f, V


@functools.lru_cache(maxsize=None)
def _racah(a, b, c, d, e, f):
    """{a b c; d e f}, twice the angular momenta"""
    def delta(x, y, z):
        if z < abs(x - y) or z > x + y or (x + y + z) % 2:
            return None
        F = math.factorial
        return F((x + y - z) // 2) * F((x - y + z) // 2) * F((-x + y + z) // 2) / F((x + y + z) // 2 + 1)

    ds = [delta(a, b, c), delta(a, e, f), delta(d, b, f), delta(d, e, c)]
    if any(x is None for x in ds):
        return 0.0
    F = math.factorial
    lo = max(a + b + c, a + e + f, d + b + f, d + e + c) // 2
    hi = min(a + b + d + e, b + c + e + f, a + c + d + f) // 2
    s = 0
    for t in range(lo, hi + 1):
        den = (F(t - (a + b + c) // 2) * F(t - (a + e + f) // 2) * F(t - (d + b + f) // 2) * F(t - (d + e + c) // 2)
               * F((a + b + d + e) // 2 - t) * F((b + c + e + f) // 2 - t) * F((a + c + d + f) // 2 - t))
        s += (-1) ** t * F(t + 1) / den
    return math.sqrt(math.prod(ds)) * s


@functools.lru_cache(maxsize=2)
def _dense(emax, lmax, nucleus):
    return _Dense(_basis(emax, lmax, nucleus))


def exact(case, seed):
    """The outputs in dense 64-bit torch.  None for the whole flows, the
    gradients and the tensor commutator, and for bases whose dense arrays
    (orbits^4 for every J) do not fit the time."""
    kind, b = case["kind"], _of(case)
    if kind not in ("commutator", "c122", "pphh", "ph", "bch") or b.norb > (56 if kind == "bch" else 90):
        return None
    s = prepare(case, seed)
    D = _dense(case["emax"], case["lmax"], case["nucleus"])
    L, R = (s["G"], s["H"]) if kind == "bch" else (s["L"], s["R"])
    l, r = D.of(L.data, L.herm), D.of(R.data, R.herm)
    if kind == "commutator":
        return D.flat(*D.commutator(l, r))
    if kind == "c122":
        x = D.flat(0.0, None, D.c122(l, r))
        return x
    if kind == "ph":
        return {"RES": D.flat(0.0, None, D.ph(l, r)), "LCC": None, "RCC": None}
    if kind == "pphh":
        lad, rad = D.ladder(l, r), D.ladder(r, l)
        # w1, w2: the pp and hh intermediates; square blocks hold one order of the product
        w = []
        for p, m in zip(lad, rad):
            one, both = D.flat(0.0, None, p), D.flat(0.0, None, p - m)
            w.append(one.index_copy(0, D.at[D.rect], both[D.at[D.rect]]))
        return {"RES": D.flat(0.0, None, lad[0] - lad[1] - rad[0] + rad[1]), "w1": w[0], "w2": w[1]}
    # BCH_EXPAND: sum of ad^n / n! until a term's Frobenius norm is below 1e-6
    weight = torch.zeros(b.oplen, dtype=torch.float64, device="cuda")
    weight[D.at] = 1.0 + D.rect.double()
    weight[b.off_fhh: b.off_fpp + b.npart ** 2] = 1.0
    weight[b.off_fph: b.off_fpp] = 2.0
    total, term, coef, norms = s["H"].data.clone(), r, 1.0, []
    conv = float(np.float32(1e-6))
    for i in range(2, 41):
        coef /= i - 1.0
        term = D.commutator(l, term)
        flat = D.flat(*term)
        total += coef * flat
        norms.append(float((weight * flat * flat).sum().sqrt()) * coef)
        if norms[-1] < conv:
            break
    return {"HS": total, "index": i, "norms": _padded(np.array(norms), 40)}
