"""GPU parity of the external product through the auxiliary basis (large
batches): bit-exact with the oracle over ring sizes, gadget bases, three and
four auxiliary primes, row chunks that do not divide the rows, and the largest
sums (every residue q - 1); and, where the oracle is slow, with the same
ciphertexts one at a time, which take the other path."""
import numpy as np
import pytest

import oracle_lib as orc
import params as P

pytestmark = pytest.mark.gpu


def make(chain, log_n, qn):
    import kunpbfv_amd as kb
    d = P.c1_params() if chain == "36bit" else P.chain60(log_n, qn, 1, 4, 2)
    d = dict(d, log_n=log_n)
    args = (d["log_n"], d["q"], d["p"], d["t"], d["gamma"], d["plain"])
    return kb.Context(*args), args


def operands(ctx, rows, batch, seed):
    rng = np.random.default_rng(seed)
    rgsw = np.empty((rows, 2, ctx.qn, ctx.n), dtype=np.uint64)
    ct = np.empty((batch, 2, ctx.qn, ctx.n), dtype=np.uint64)
    for l in range(ctx.qn):
        q = int(ctx.mod[ctx.oQ + l])
        rgsw[:, :, l] = rng.integers(0, q, size=(rows, 2, ctx.n), dtype=np.uint64)
        ct[:, :, l] = rng.integers(0, q, size=(batch, 2, ctx.n), dtype=np.uint64)
        rgsw[:, :, l, 0] = ct[:, :, l, 0] = q - 1
        # the second entry's transform is q - 1 everywhere: its digits are the largest
        ct[1, :, l] = q - 1
    return rgsw, ct


@pytest.mark.parametrize("chain,log_n,qn,bits,batch", [
    ("36bit", 12, 2, 20, 50), ("36bit", 12, 2, 5, 51), ("60bit", 12, 8, 20, 13), ("60bit", 13, 9, 20, 12),
    ("60bit", 13, 7, 27, 15), ("60bit", 14, 8, 16, 13)])
def test_matches_oracle(chain, log_n, qn, bits, batch):
    import kunpbfv_amd as kb
    ctx, args = make(chain, log_n, qn)
    oc = orc.Ctx(*args)
    rows = ctx.rgsw_rows(bits)
    rgsw, ct = operands(ctx, rows, batch, 31 * qn + bits)
    out = kb.to_host(ctx.external_product(kb.to_device(rgsw), kb.to_device(ct), bits))
    for b in (0, 1, batch - 1):
        assert np.array_equal(out[b], oc.external_product(rgsw, ct[b], bits)), b


@pytest.mark.parametrize("log_n,qn,bits,batch", [(15, 8, 20, 13), (16, 9, 20, 12), (16, 12, 24, 17)])
def test_matches_single_ciphertexts(log_n, qn, bits, batch):
    import torch
    import kunpbfv_amd as kb
    ctx, _ = make("60bit", log_n, qn)
    rows = ctx.rgsw_rows(bits)
    rgsw, ct = operands(ctx, rows, batch, 7 * log_n + qn)
    rgsw, ct = kb.to_device(rgsw), kb.to_device(ct)
    want = torch.cat([ctx.external_product(rgsw, ct[b:b + 1], bits) for b in range(batch)])
    assert torch.equal(ctx.external_product(rgsw, ct, bits), want)
    assert torch.equal(ctx.external_product(rgsw, ct, bits, out=ct), want)  # in place
