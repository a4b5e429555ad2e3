"""GPU: transforms modulo primes 2^60 - c run on signed values for c up to 2^28 and on
Shoup products past it: primes on both sides of that line and a large one in one
launch, every ring degree, residues at the ends of their range, against the oracle;
the unscaled inverse and long sums inside HomMult are covered by its own tests."""
import numpy as np
import pytest

import oracle_lib as orc
import params as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log_n", [12, 13, 14, 15, 16])
def test_both_sides_of_the_line(log_n):
    import kunpbfv_amd as kb
    m, line = 1 << 17, (1 << 60) - (1 << 28)
    below = orc.primes_descending(line, m, 2)  # c just above 2^28
    above = orc.primes_descending(line + 512 * m, m, 64)  # c just below 2^28
    above = sorted(v for v in above if v > line)[:2]
    assert len(above) == 2
    q = [above[0], below[0], orc.primes_descending(1 << 60, m, 8)[7], above[1], below[1]]
    d = P.chain60(log_n, 2, 1, 4, 2)
    args = (log_n, q, d["p"], d["t"], d["gamma"], d["plain"])
    ctx, oc = kb.Context(*args), orc.Ctx(*args)
    rng = np.random.default_rng(log_n)
    for polys in (1, max(2, (1 << 20 >> log_n) // len(q))):  # small tiles, large tiles
        x = np.empty((polys, len(q), ctx.n), dtype=np.uint64)
        for i, v in enumerate(q):
            x[:, i] = rng.integers(0, v, size=(polys, ctx.n), dtype=np.uint64)
            x[0, i, ::3] = v - 1
        x[-1, :, :] = np.where(np.arange(ctx.n) % 2, np.array(q, dtype=np.uint64)[:, None] - np.uint64(1), np.uint64(0))
        y = kb.to_device(x)
        ctx.ntt(y, y, +1, ctx.oQ, len(q), polys=polys)
        got = kb.to_host(y)
        for k in (0, polys - 1):
            assert np.array_equal(got[k:k + 1], oc.ntt_fwd(np.ascontiguousarray(x[k:k + 1]), ctx.oQ, len(q), 1)), k
        ctx.ntt(y, y, -1, ctx.oQ, len(q), polys=polys)
        assert np.array_equal(kb.to_host(y), x), polys
