"""GPU: buffers aligned to their 8-byte words only (the second word of an allocation) give
the same bits as allocations do, in the calls whose kernels move 16 bytes per lane: the
key-switch inner product of one ciphertext to many, the external product through both
paths, encryption."""
import pytest

import params as P

pytestmark = pytest.mark.gpu


def make(log_n, qn):
    import torch
    import kunpbfv_amd as kb
    d = P.chain60(log_n, qn, 1, 4, 2)
    ctx = kb.Context(log_n, d["q"], d["p"], d["t"], d["gamma"], d["plain"])
    torch.manual_seed(qn)

    def rnd(lead, mods):
        m = torch.tensor([int(v) for v in mods], device="cuda")
        return torch.randint(1 << 62, (*lead, len(m), ctx.n), dtype=torch.int64, device="cuda") % m[:, None]

    return ctx, rnd


def shifted(x):
    """the same tensor one word past an allocation's start"""
    import torch
    y = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)[1:].view(x.shape)
    y.copy_(x)
    assert y.data_ptr() % 16 == 8
    return y


@pytest.mark.parametrize("digits", [2, 17])
def test_inner_product(digits):
    import torch
    ctx, rnd = make(12, digits)
    T = ctx.mod[ctx.oT:ctx.oT + ctx.tn]
    key, cin = rnd((2, ctx.dnum, ctx.ri_blocks), T), rnd((16, ctx.dnum), T)
    for batch in (1, 2, 3, 5, 16):
        want = ctx.empty(batch, 2, ctx.ri_blocks, ctx.tn, ctx.n)
        ctx.inner_product(cin, key, want, batch=batch)
        got = shifted(torch.zeros_like(want))
        ctx.inner_product(shifted(cin), shifted(key), got, batch=batch)
        assert torch.equal(got, want), batch


@pytest.mark.parametrize("qn,batch", [(2, 3), (6, 20)])
def test_external_product(qn, batch):
    import torch
    import kunpbfv_amd as kb
    ctx, rnd = make(12, qn)
    Q = ctx.mod[ctx.oQ:ctx.oQ + qn]
    rgsw, ct = rnd((ctx.rgsw_rows(20), 2), Q), rnd((batch, 2), Q)
    want = ctx.external_product(rgsw, ct, 20)
    need = kb.lib.kbfv_external_product_workspace_bytes(ctx.h, batch, 20)
    ctx._ws = torch.empty(need + 8, dtype=torch.uint8, device="cuda")[8:]
    got = ctx.external_product(shifted(rgsw), shifted(ct), 20, out=shifted(torch.zeros_like(ct)))
    assert torch.equal(got, want)


def test_encrypt():
    import torch
    import kunpbfv_amd as kb
    ctx, rnd = make(13, 3)
    sk = ctx.keygen_sk(bytes([1]) * 32)
    pk = ctx.keygen_pk(bytes([2]) * 32, sk)
    m = torch.randint(ctx.plain, (3, ctx.n), dtype=torch.int64, device="cuda")
    want = ctx.encrypt(bytes([3]) * 32, pk, m)
    need = kb.lib.kbfv_encrypt_workspace_bytes(ctx.h, 3)
    ctx._ws = torch.empty(need + 8, dtype=torch.uint8, device="cuda")[8:]
    assert torch.equal(ctx.encrypt(bytes([3]) * 32, shifted(pk), shifted(m)), want)
