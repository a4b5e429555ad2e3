"""Pins the oracle's digit conversions Q_j -> T and PQ -> T (CPU only) where the float
overflow estimate rounds up to the next integer: the top residues of a block.  A block of
one prime is the residue itself, always; a block of several may come out one multiple of its
product lower, the same integer modulo every T prime."""
import numpy as np
import pytest

import oracle_lib as orc
import params as Pm


def ends(mods, n):
    """[len(mods)][n]: the last and first n/2 values of [0, product) of all moduli"""
    M = 1
    for m in mods:
        M *= m
    vals = [M - 1 - i for i in range(n // 2)] + list(range(n // 2))
    return vals, np.array([[v % m for v in vals] for m in mods], dtype=np.uint64), M


def short_k2():
    """digits of two 28-bit primes, whose product is below every T prime"""
    p = orc.primes_descending(1 << 28, 8192, 6)
    return dict(log_n=12, q=p[2:], p=p[:2], t=orc.primes_descending(1 << 60, 1 << 17, 4), gamma=2, plain=65537)


CHAINS = {"k1_gamma1": lambda: Pm.chain60(12, 4, 1, 3, 1), "k1_gamma2": lambda: Pm.chain60(12, 4, 1, 4, 2),
          "short_k2": short_k2}


@pytest.mark.parametrize("chain", list(CHAINS))
@pytest.mark.parametrize("which", ["qj", "pq"])
def test_top_residues(chain, which):
    d = CHAINS[chain]()
    oc = orc.Ctx(d["log_n"], d["q"], d["p"], d["t"], d["gamma"], d["plain"])
    T = [int(v) for v in oc.mod[oc.oT:oc.oT + oc.tn]]
    src, width = (d["q"], len(d["p"])) if which == "qj" else (list(d["p"]) + list(d["q"]), d["gamma"])
    blocks = [src[i:i + width] for i in range(0, len(src), width)]
    parts = [ends(b, oc.n) for b in blocks]
    x = np.concatenate([p[1] for p in parts])
    out = (oc.modup_qj_to_t if which == "qj" else oc.modup_pq_to_t)(x)
    for b, (vals, _, M) in enumerate(parts):
        for k in list(range(0, 64)) + [oc.n // 2 - 1, oc.n // 2, oc.n - 1]:
            got = [int(v) for v in out[b, :, k]]
            if got == [vals[k] % t for t in T]:
                continue
            assert len(blocks[b]) > 1 and got == [(vals[k] - M) % t for t in T], (b, k)
