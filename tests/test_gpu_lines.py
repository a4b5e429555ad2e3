"""GPU parity at the lines where a call changes its kernels: the key-switch inner product
of more than 16 digits between the holding and the matrix kernel, and the external
product between the general path and the auxiliary basis; both sides of every line,
first and last ciphertext against the oracle."""
import numpy as np
import pytest

import oracle_lib as orc
import params as P

pytestmark = pytest.mark.gpu


def make(log_n, qn):
    import kunpbfv_amd as kb
    d = P.chain60(log_n, qn, 1, 4, 2)
    args = (d["log_n"], d["q"], d["p"], d["t"], d["gamma"], d["plain"])
    return kb, kb.Context(*args), orc.Ctx(*args)


def rand(rng, lead, mods, n):
    out = np.empty((*lead, len(mods), n), dtype=np.uint64)
    for i, q in enumerate(mods):
        out[..., i, :] = rng.integers(0, int(q), size=(*lead, n), dtype=np.uint64)
        out[..., i, :4] = int(q) - 1
    return out


@pytest.mark.parametrize("digits,batches", [(17, (14, 15, 16, 17, 23, 24, 33)), (21, (16, 25, 26, 34, 35, 48, 49))])
def test_inner_product(digits, batches):
    kb, ctx, oc = make(12, digits)
    n, B, tn = ctx.n, ctx.ri_blocks, ctx.tn
    rng = np.random.default_rng(digits)
    T = ctx.mod[ctx.oT:ctx.oT + tn]
    key, cin = rand(rng, (2, digits, B), T, n), rand(rng, (max(batches), digits), T, n)
    dkey, dcin = kb.to_device(key), kb.to_device(cin)
    want = {}
    for batch in batches:
        out = ctx.empty(batch, 2, B, tn, n)
        ctx.inner_product(dcin[:batch], dkey, out, batch=batch)
        got = kb.to_host(out)
        for ct in (0, batch - 1):
            if ct not in want:
                want[ct] = oc.inner_product(cin[ct], key)
            assert np.array_equal(got[ct], want[ct]), (batch, ct)


@pytest.mark.parametrize("log_n,qn,batches", [(12, 6, (17, 18)), (14, 10, (16, 17)), (15, 8, (14, 15)), (15, 12, (12, 13)),
                                              (16, 12, (11, 12)), (15, 2, (50,)), (15, 3, (33, 34))])
def test_external_product(log_n, qn, batches):
    import torch
    kb, ctx, oc = make(log_n, qn)
    rows = ctx.rgsw_rows(20)
    m = torch.tensor([int(v) for v in ctx.mod[ctx.oQ:ctx.oQ + qn]], device="cuda")
    torch.manual_seed(qn)

    def rnd(*lead):
        return torch.randint(1 << 62, (*lead, qn, ctx.n), dtype=torch.int64, device="cuda") % m[:, None]

    rgsw, ct = rnd(rows, 2), rnd(max(batches), 2)
    single = {}
    for batch in batches:
        out = ctx.external_product(rgsw, ct[:batch], 20)
        for b in (0, batch - 1):
            if b not in single:
                single[b] = ctx.external_product(rgsw, ct[b:b + 1], 20)[0]
            assert torch.equal(out[b], single[b]), (batch, b)
    if log_n == 12:
        want = oc.external_product(kb.to_host(rgsw), kb.to_host(ct[0]), 20)
        assert np.array_equal(kb.to_host(single[0]), want)
