"""GPU: the small-tile transforms that built-in plans take up to 2^19 words agree,
bit for bit, with the oracle and with the tiled passes (an explicit plan), at sizes
around the limit, at every ring degree, both directions, out of place with gaps
between limbs, polynomials and batch entries, in place, and for the two-source
unscaled inverse inside HomMult."""
import numpy as np
import pytest

import oracle_lib as orc
import params as P

pytestmark = pytest.mark.gpu

LIMIT = 1 << 19


def make(log_n, qn=5):
    import kunpbfv_amd as kb
    d = P.chain60(log_n, qn, 1, 4, 2)
    args = (d["log_n"], d["q"], d["p"], d["t"], d["gamma"], d["plain"])
    tiled = kb.Context(*args)
    # tiled passes: two passes, not the built-in plan's word
    plan = [p for p in kb.ntt_plan_candidates(log_n) if p & 15 != log_n and p >> 12 == 0][0]
    for b in range(kb.lib.kbfv_ntt_plan_bucket(1 << 40) + 1):
        tiled.set_ntt_plan(+1, b, plan)
        tiled.set_ntt_plan(-1, b, plan)
    return kb, kb.Context(*args), tiled, orc.Ctx(*args)


@pytest.mark.parametrize("log_n", [12, 13, 14, 15, 16])
def test_sizes(log_n):
    kb, ctx, tiled, oc = make(log_n)
    n, mod0, limbs = ctx.n, ctx.oQ, 4
    mods = [int(v) for v in ctx.mod[mod0:mod0 + limbs]]
    rng = np.random.default_rng(log_n)
    rows = LIMIT >> log_n
    for polys, batch in ((1, 1), (3, 1), (1, 2), (rows // limbs, 1), (rows // limbs + 1, 1)):
        if polys == 0:
            continue
        x = np.empty((batch, polys, limbs + 1, n), dtype=np.uint64)  # one spare row
        for i in range(limbs):
            x[:, :, i] = rng.integers(0, mods[i], size=(batch, polys, n), dtype=np.uint64)
            x[:, :, i, :3] = mods[i] - 1
        x[:, :, limbs] = 12345
        xd = kb.to_device(x)
        src = (polys * (limbs + 1) * n, (limbs + 1) * n, n)
        for d in (+1, -1):
            got, want = ctx.empty(batch, polys, limbs, n), ctx.empty(batch, polys, limbs, n)
            dst = (polys * limbs * n, limbs * n, n)
            ctx.ntt(xd, got, d, mod0, limbs, polys=polys, batch=batch, s=src, d=dst)
            tiled.ntt(xd, want, d, mod0, limbs, polys=polys, batch=batch, s=src, d=dst)
            assert np.array_equal(kb.to_host(got), kb.to_host(want)), (polys, batch, d)
            if d > 0:
                first = np.ascontiguousarray(x[0, :1, :limbs])
                assert np.array_equal(kb.to_host(got)[0, :1], oc.ntt_fwd(first, mod0, limbs, 1))
                ctx.ntt(got, got, -1, mod0, limbs, polys=polys, batch=batch, s=dst, d=dst)  # in place
                assert np.array_equal(kb.to_host(got), x[:, :, :limbs]), (polys, batch)
            assert np.array_equal(kb.to_host(xd), x)  # the source and its spare rows


@pytest.mark.parametrize("log_n,qn,batch", [(12, 1, 1), (12, 2, 3), (13, 3, 1), (14, 2, 2), (15, 2, 1), (16, 1, 2)])
def test_hommult(log_n, qn, batch):
    kb, ctx, tiled, _ = make(log_n, qn)
    rng = np.random.default_rng(log_n * 10 + qn)

    def rand(lead, mods):
        out = np.empty((*lead, len(mods), ctx.n), dtype=np.uint64)
        for i, q in enumerate(mods):
            out[..., i, :] = rng.integers(0, int(q), size=(*lead, ctx.n), dtype=np.uint64)
        return kb.to_device(out)

    q = ctx.mod[ctx.oQ:ctx.oQ + qn]
    rlk = rand((2, ctx.dnum, ctx.ri_blocks), ctx.mod[ctx.oT:ctx.oT + ctx.tn])
    c1, c2 = rand((batch, 2), q), rand((batch, 2), q)
    assert np.array_equal(kb.to_host(ctx.mult_relin(rlk, c1, c2)), kb.to_host(tiled.mult_relin(rlk, c1, c2)))
