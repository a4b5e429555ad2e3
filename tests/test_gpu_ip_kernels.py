"""GPU parity of the key-switch inner product at the edges of its kernels: the
streaming kernel (1 to 4 ciphertexts), the key-holding one (odd batches, digit
counts around its register sizes and its carries after 8 and 16 terms), the
matrix-core one (long keys, large batches) and keys past 32 digits; 60-bit and
50-bit auxiliary primes; bit-exact with the oracle."""
import numpy as np
import pytest

import oracle_lib as orc
import params as P

pytestmark = pytest.mark.gpu

# (digits, auxiliary prime bits, batches)
CASES = [(1, 60, (1, 3)), (2, 60, (1, 2, 5)), (8, 60, (2, 3)), (9, 60, (1, 4)), (12, 50, (1, 2, 7)), (13, 60, (3,)),
         (16, 60, (1, 4, 17)), (17, 60, (1, 2, 4, 5)), (24, 60, (6, 45)), (25, 60, (3, 7)), (32, 60, (1, 9, 44)),
         (33, 60, (1, 2, 5))]


@pytest.mark.parametrize("digits,bits,batches", CASES)
def test_inner_product(digits, bits, batches):
    import kunpbfv_amd as kb
    if bits == 60:
        d = P.chain60(12, digits, 1, 4, 2)
    else:
        primes = orc.primes_descending(1 << 36, 8192, digits + 1)
        d = dict(log_n=12, q=primes[1:], p=primes[:1], t=orc.primes_descending(1 << bits, 1 << 17, 4), gamma=2,
                 plain=65537)
    ctx = kb.Context(d["log_n"], d["q"], d["p"], d["t"], d["gamma"], d["plain"])
    oc = orc.Ctx(d["log_n"], d["q"], d["p"], d["t"], d["gamma"], d["plain"])
    N, D, B, tn = ctx.n, ctx.dnum, ctx.ri_blocks, ctx.tn
    assert D == digits
    rng = np.random.default_rng(digits * 100 + bits)
    tm = [int(v) for v in ctx.mod[ctx.oT:ctx.oT + tn]]
    key = np.empty((2, D, B, tn, N), dtype=np.uint64)
    cin = np.empty((max(batches), D, tn, N), dtype=np.uint64)
    for k, q in enumerate(tm):
        key[:, :, :, k, :] = rng.integers(0, q, size=(2, D, B, N), dtype=np.uint64)
        cin[:, :, k, :] = rng.integers(0, q, size=(len(cin), D, N), dtype=np.uint64)
        cin[:, :, k, :16] = q - 1  # the largest sums
        key[:, :, :, k, :8] = q - 1
    dkey = kb.to_device(key)
    for batch in batches:
        out = ctx.empty(batch, 2, B, tn, N)
        ctx.inner_product(kb.to_device(cin[:batch]), dkey, out, batch=batch)
        got = kb.to_host(out)
        for ct in {0, batch // 2, batch - 1}:
            assert np.array_equal(got[ct], oc.inner_product(cin[ct], key)), (batch, ct)
