"""GPU: ciphertext chains that mix primes near 2^60 (signed butterflies, their own
twiddle form and order) with others: the external product's digit transforms against
the oracle, the near prime first, in the middle and last, through the general path and
the auxiliary basis; and the tuner's pass timings, which run the same launches."""
import numpy as np
import pytest

import oracle_lib as orc
import params as P

pytestmark = pytest.mark.gpu

# near = a prime of the 60-bit chain, else one of 50 bits
MIXES = [(True, False), (False, True), (True, False, True), (False, True, False), (True, True, False, False, True)]


def make(mix, log_n=12):
    import kunpbfv_amd as kb
    d = P.chain60(log_n, len(mix), 1, 4, 2)
    short = orc.primes_descending(1 << 50, 1 << 17, len(mix))
    q = [a if near else b for near, a, b in zip(mix, d["q"], short)]
    args = (log_n, q, d["p"], d["t"], d["gamma"], d["plain"])
    return kb, kb.Context(*args), args


# base 2^30 is past the auxiliary basis and still splits its digits in the transform
@pytest.mark.parametrize("mix", MIXES)
@pytest.mark.parametrize("bits,batch", [(20, 1), (20, 3), (20, 50), (30, 50), (30, 3)])
def test_external_product(mix, bits, batch):
    kb, ctx, args = make(mix)
    oc = orc.Ctx(*args)
    rng = np.random.default_rng(batch + bits)
    rows = ctx.rgsw_rows(bits)
    rgsw = np.empty((rows, 2, ctx.qn, ctx.n), dtype=np.uint64)
    ct = np.empty((batch, 2, ctx.qn, ctx.n), dtype=np.uint64)
    for l in range(ctx.qn):
        q = int(ctx.mod[ctx.oQ + l])
        rgsw[:, :, l] = rng.integers(0, q, size=(rows, 2, ctx.n), dtype=np.uint64)
        ct[:, :, l] = rng.integers(0, q, size=(batch, 2, ctx.n), dtype=np.uint64)
    out = kb.to_host(ctx.external_product(kb.to_device(rgsw), kb.to_device(ct), bits))
    for b in {0, batch - 1}:
        assert np.array_equal(out[b], oc.external_product(rgsw, ct[b], bits)), b


@pytest.mark.parametrize("mix", [(True, False), (False, True, True)])
@pytest.mark.parametrize("log_n", [12, 15])
def test_autotune_times_the_range_it_is_given(mix, log_n):
    import torch
    kb, ctx, _ = make(mix, log_n)
    polys = 5
    scratch = torch.full((polys, ctx.qn, ctx.n), 7, dtype=torch.int64, device="cuda")
    for direction in (+1, -1):
        ctx.autotune_ntt(direction, ctx.oQ, ctx.qn, polys, reps=1, scratch=scratch)
        # it transforms residues of 0: every launch of the right kind leaves residues of 0
        assert int(torch.count_nonzero(scratch)) == 0, direction
