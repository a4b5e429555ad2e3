"""GPU parity of base conversion and scale-and-round at the lines between their
launches: outputs of a coefficient split over eight, four, two threads or none, and the
register kernel against the matrix kernel; both ends of every line, first and last
polynomial against the oracle."""
import numpy as np
import pytest

import oracle_lib as orc
import params as P
from test_gpu_rns_sizes import rand_mod

pytestmark = pytest.mark.gpu


# (prime bits, primes, polynomials of 2^12 coefficients)
@pytest.mark.parametrize("bits,qn,polys", [(60, 9, 5), (60, 12, 16), (60, 12, 17), (60, 12, 33), (60, 13, 16),
                                           (60, 13, 17), (60, 14, 16), (60, 15, 8), (60, 15, 9), (60, 28, 1),
                                           (55, 17, 32), (55, 30, 17), (55, 30, 33)])
def test_conversions(bits, qn, polys):
    import kunpbfv_amd as kb
    if bits == 60:
        d = P.chain60(12, qn, 1, 4, 2)
    else:
        primes = orc.primes_descending(1 << bits, 8192, qn + 1)
        d = dict(log_n=12, q=primes[1:], p=primes[:1], t=orc.primes_descending(1 << 60, 1 << 17, 4), gamma=2,
                 plain=65537)
    args = (12, d["q"], d["p"], d["t"], d["gamma"], d["plain"])
    ctx, oc = kb.Context(*args), orc.Ctx(*args)
    rng = np.random.default_rng(1000 * polys + qn)
    q, r = ctx.mod[ctx.oQ:ctx.oQ + ctx.qn], ctx.mod[ctx.oR:ctx.oR + ctx.rn]
    for mods, q_to_r, ref, outs in ((q, True, oc.bconv_q_to_r, ctx.rn), (r, False, oc.bconv_r_to_q, ctx.qn)):
        x = rand_mod(rng, mods, ctx.n, polys, polys % 2 == 0)
        y = ctx.empty(polys, outs, ctx.n)
        ctx.bconv(kb.to_device(x), y, q_to_r, polys=polys)
        got = kb.to_host(y)
        for p in {0, polys - 1}:
            assert np.array_equal(got[p], ref(x[p])), (q_to_r, p)
    x = rand_mod(rng, ctx.mod[ctx.oQ:ctx.oQ + ctx.qn + ctx.rn], ctx.n, polys, polys % 2 == 0)
    y = ctx.empty(polys, ctx.rn, ctx.n)
    ctx.scale_round(kb.to_device(x), y, polys=polys)
    got = kb.to_host(y)
    for p in {0, polys - 1}:
        assert np.array_equal(got[p], oc.scale_round(x[p])), p
