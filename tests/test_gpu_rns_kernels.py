"""GPU parity of base conversion and scale-and-round at the edges of the two
kernels that compute them: the matrix kernel's shortest chain and its chunk
boundaries (60-bit primes), and the register kernel's groups of 15 rows up to
its longest chain (55-bit primes, which the matrix kernel does not take)."""
import numpy as np
import pytest

import oracle_lib as orc
import params as P
from test_gpu_rns_sizes import rand_mod

pytestmark = pytest.mark.gpu

CHAINS = [(60, 10), (60, 11), (60, 12), (60, 13), (60, 14), (60, 22), (60, 23), (55, 10), (55, 14), (55, 15), (55, 16), (55, 29),
          (55, 30), (36, 4)]


@pytest.mark.parametrize("bits,qn", CHAINS)
def test_conversions(bits, qn):
    import kunpbfv_amd as kb
    if bits == 60:
        d = P.chain60(12, qn, 1, 4, 2)
    else:
        primes = orc.primes_descending(1 << bits, 8192, qn + 1)
        d = dict(log_n=12, q=primes[1:], p=primes[:1], t=orc.primes_descending(1 << 60, 1 << 17, 4), gamma=2,
                 plain=65537)
    ctx = kb.Context(d["log_n"], d["q"], d["p"], d["t"], d["gamma"], d["plain"])
    oc = orc.Ctx(d["log_n"], d["q"], d["p"], d["t"], d["gamma"], d["plain"])
    rng = np.random.default_rng(1000 * bits + qn)
    q, r = ctx.mod[ctx.oQ:ctx.oQ + ctx.qn], ctx.mod[ctx.oR:ctx.oR + ctx.rn]
    for extreme in (False, True):
        for mods, q_to_r, ref, outs in ((q, True, oc.bconv_q_to_r, ctx.rn), (r, False, oc.bconv_r_to_q, ctx.qn)):
            x = rand_mod(rng, mods, ctx.n, 2, extreme)
            y = ctx.empty(2, outs, ctx.n)
            ctx.bconv(kb.to_device(x), y, q_to_r, polys=2)
            got = kb.to_host(y)
            for p in range(2):
                assert np.array_equal(got[p], ref(x[p])), (q_to_r, extreme, p)
        x = rand_mod(rng, ctx.mod[ctx.oQ:ctx.oQ + ctx.qn + ctx.rn], ctx.n, 2, extreme)
        y = ctx.empty(2, ctx.rn, ctx.n)
        ctx.scale_round(kb.to_device(x), y, polys=2)
        got = kb.to_host(y)
        for p in range(2):
            assert np.array_equal(got[p], oc.scale_round(x[p])), (extreme, p)
