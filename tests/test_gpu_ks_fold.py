"""GPU: the key-switch tail where its sums are folded at bit 60 (primes near 2^60) and where
they are Barrett-reduced (others), in one chain, one and two special primes: the fused
kernel, with the addend, against the separate modUp and modDown kernels; residues at the
ends of their range; bit-exact."""
import numpy as np
import pytest

import oracle_lib as orc
import params as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("special,mixed", [(1, False), (1, True), (2, True)])
def test_tail_against_separate_kernels(special, mixed):
    import kunpbfv_amd as kb
    m = 1 << 17
    d = P.chain60(12, 4, 1, 4, 2)
    q, p = list(d["q"]), d["p"]
    if special == 1 and mixed:  # below the line of the folded form, and far below
        q[1] = orc.primes_descending((1 << 60) - (1 << 28), m, 1)[0]
        q[3] = orc.primes_descending(1 << 59, m, 1)[0]
    if special == 2:  # digits of two primes fit the basis T if one of them is short
        p = orc.primes_descending(1 << 50, m, 2)
        q[1], q[2] = orc.primes_descending(1 << 36, m, 2)
    ctx = kb.Context(12, q, p, d["t"], d["gamma"], d["plain"])
    n, batch, rng = ctx.n, 3, np.random.default_rng(special)

    def rand(lead, mods):
        out = np.empty((*lead, len(mods), n), dtype=np.uint64)
        for i, v in enumerate(mods):
            out[..., i, :] = rng.integers(0, int(v), size=(*lead, n), dtype=np.uint64)
            out[..., i, :8] = int(v) - 1
            out[..., i, 8:16] = 0
        return kb.to_device(out)

    x = rand((batch, 2, ctx.ri_blocks), ctx.mod[ctx.oT:ctx.oT + ctx.tn])  # coefficient form, over T
    d01 = rand((batch, 2), ctx.mod[ctx.oQ:ctx.oQ + ctx.qn])
    pq, want = ctx.empty(batch, 2, ctx.pn + ctx.qn, n), ctx.empty(batch, 2, ctx.qn, n)
    ctx.modup_t_to_pq(x, pq, batch=batch)
    ctx.moddown(pq, want, add=d01, add_stride=2 * ctx.qn * n, batch=batch)
    ctx.ntt(want, want, +1, ctx.oQ, ctx.qn, polys=2 * batch)
    ctx.ntt(x, x, +1, ctx.oT, ctx.tn, polys=2 * ctx.ri_blocks * batch)
    got = ctx.mult_after_ip(x, d01)
    assert np.array_equal(kb.to_host(got), kb.to_host(want))
