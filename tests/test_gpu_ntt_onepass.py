"""GPU: the one-pass transforms that the built-in plan takes for launches of many
limbs (a limb, or half of one of 2^16, held by one workgroup) agree bit for bit with
the tiled passes and, on some limbs, with the oracle: every ring degree, row counts
around the rule's lines and past one round of workgroups, both directions, in place
and out of place with gaps, the unscaled two-source inverse inside HomMult, residues
at the ends of their range, a launch with a modulus that the kernel does not take."""
import numpy as np
import pytest

import oracle_lib as orc
import params as P

pytestmark = pytest.mark.gpu

# polynomials of 5 limbs at each ring degree
POLYS = {12: (26, 103, 420), 13: (13, 52, 210), 14: (22, 23, 110), 15: (29, 30, 51, 53), 16: (40, 41, 51, 102)}


def contexts(log_n, q=None):
    import kunpbfv_amd as kb
    d = P.chain60(log_n, 5, 1, 4, 2)
    args = (d["log_n"], q or d["q"], d["p"], d["t"], d["gamma"], d["plain"])
    tiled = kb.Context(*args)
    plan = [p for p in kb.ntt_plan_candidates(log_n) if p & 15 != log_n and p >> 12 == 0][0]
    for b in range(kb.lib.kbfv_ntt_plan_bucket(1 << 40) + 1):
        tiled.set_ntt_plan(+1, b, plan)
        tiled.set_ntt_plan(-1, b, plan)
    return kb, kb.Context(*args), tiled, orc.Ctx(*args)


def check(kb, ctx, tiled, oc, polys, limbs=5):
    import torch
    n, mod0 = ctx.n, ctx.oQ
    mods = torch.tensor([int(v) for v in ctx.mod[mod0:mod0 + limbs]], device="cuda")
    torch.manual_seed(polys)
    x = torch.randint(1 << 62, (polys, limbs + 1, n), dtype=torch.int64, device="cuda")
    x[:, :limbs] %= mods[:, None]
    x[0, :limbs, ::3] = mods[:, None] - 1
    x[-1, :limbs] = torch.where(torch.arange(n, device="cuda") % 2 == 0, mods[:, None] - 1, 0)
    before = x.clone()
    s, d = (0, (limbs + 1) * n, n), (0, limbs * n, n)
    for dirn in (+1, -1):
        got, want = ctx.empty(polys, limbs, n), ctx.empty(polys, limbs, n)
        ctx.ntt(x, got, dirn, mod0, limbs, polys=polys, s=s, d=d)
        tiled.ntt(x, want, dirn, mod0, limbs, polys=polys, s=s, d=d)
        assert torch.equal(got, want) and torch.equal(x, before), (polys, dirn)
        if dirn > 0:
            for k in (0, polys - 1):
                host = np.ascontiguousarray(kb.to_host(x[k:k + 1, :limbs].contiguous()))
                assert np.array_equal(kb.to_host(got[k:k + 1].contiguous()), oc.ntt_fwd(host, mod0, limbs, 1)), k
        ctx.ntt(got, got, -dirn, mod0, limbs, polys=polys)  # in place
        assert torch.equal(got, x[:, :limbs].contiguous()), (polys, dirn)


@pytest.mark.parametrize("log_n", [12, 13, 14, 15, 16])
def test_rows(log_n):
    kb, ctx, tiled, oc = contexts(log_n)
    for polys in POLYS[log_n]:
        check(kb, ctx, tiled, oc, polys)


def test_mixed_moduli():
    d = P.chain60(13, 5, 1, 4, 2)
    kb, ctx, tiled, oc = contexts(13, d["q"][:2] + orc.primes_descending(1 << 50, 1 << 17, 1) + d["q"][3:])
    check(kb, ctx, tiled, oc, 100)


@pytest.mark.parametrize("log_n,batch", [(12, 20), (13, 14), (14, 12), (15, 13), (16, 13)])
def test_hommult(log_n, batch):
    import torch
    kb, ctx, tiled, _ = contexts(log_n)
    torch.manual_seed(log_n)

    def rand(lead, mods):
        m = torch.tensor([int(v) for v in mods], device="cuda")
        return torch.randint(1 << 62, (*lead, len(m), ctx.n), dtype=torch.int64, device="cuda") % m[:, None]

    q = ctx.mod[ctx.oQ:ctx.oQ + ctx.qn]
    rlk = rand((2, ctx.dnum, ctx.ri_blocks), ctx.mod[ctx.oT:ctx.oT + ctx.tn])
    c1, c2 = rand((batch, 2), q), rand((batch, 2), q)
    assert torch.equal(ctx.mult_relin(rlk, c1, c2), tiled.mult_relin(rlk, c1, c2))
