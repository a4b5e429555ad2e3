"""GPU: the key-switch tail (transform over T, modUp to PQ, modDown, addend, transform)
with the blocks of a coefficient split over two to eight threads or none: every fused shape
of (auxiliary primes, gamma, special primes), block counts that the split does not divide,
near-2^60 and other primes in one chain, residues at the ends of their range; against
the oracle."""
import numpy as np
import pytest

import oracle_lib as orc
import params as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tn,gamma,special,qn,bits,batch", [
    (4, 2, 1, 4, 60, 1), (4, 2, 1, 12, 60, 1), (4, 2, 1, 28, 60, 1), (4, 2, 1, 13, 60, 20), (4, 2, 1, 13, 60, 33),
    (4, 2, 1, 6, 0, 2), (4, 2, 2, 4, 50, 1), (4, 2, 2, 13, 50, 2), (3, 1, 1, 10, 60, 2), (2, 1, 1, 1, 36, 1),
    (2, 1, 1, 2, 36, 3), (2, 1, 1, 16, 36, 1)])
def test_tail(tn, gamma, special, qn, bits, batch):
    import kunpbfv_amd as kb
    d = P.chain60(12, qn, 1, tn, gamma)
    q, p = list(d["q"]), list(d["p"])
    if bits == 0:  # both kinds of primes
        q[1::2] = orc.primes_descending(1 << 50, 1 << 17, len(q[1::2]))
    elif bits != 60:
        short = orc.primes_descending(1 << bits, 8192, qn + special)
        q, p = short[special:], short[:special]
    args = (12, q, p, d["t"], gamma, d["plain"])
    ctx, oc = kb.Context(*args), orc.Ctx(*args)
    rng = np.random.default_rng(qn + batch)

    def rand(lead, mods):
        out = np.empty((*lead, len(mods), ctx.n), dtype=np.uint64)
        for i, v in enumerate(mods):
            out[..., i, :] = rng.integers(0, int(v), size=(*lead, ctx.n), dtype=np.uint64)
            out[..., i, :8] = int(v) - 1
            out[..., i, 8:16] = 0
        return out

    x = rand((batch, 2, ctx.ri_blocks), ctx.mod[ctx.oT:ctx.oT + ctx.tn])  # coefficient form, over T
    add = rand((batch, 2), q)
    xn = kb.to_device(x)
    ctx.ntt(xn, xn, +1, ctx.oT, ctx.tn, polys=2 * ctx.ri_blocks * batch)
    got = kb.to_host(ctx.mult_after_ip(xn, kb.to_device(add)))
    mods = np.array(q, dtype=np.uint64)[:, None]
    for b in {0, batch - 1}:
        want = (oc.moddown(oc.modup_t_to_pq(x[b])) + add[b]) % mods
        assert np.array_equal(got[b], oc.ntt_fwd(want, ctx.oQ, qn, 2)), b
