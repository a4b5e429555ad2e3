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


# one launch for both kinds (small tiles, large tiles), and run by run
@pytest.mark.parametrize("mix,polys", [((True, False, True), 7), ((True, False) * 4, 40), ((True,) * 7 + (False,), 100),
                                       ((False,) + (True,) * 7, 100)])
@pytest.mark.parametrize("log_n", [13, 15])
def test_transforms(mix, polys, log_n):
    import torch
    kb, ctx, args = make(mix, log_n)
    oc, q = orc.Ctx(*args), ctx.mod[ctx.oQ:ctx.oQ + ctx.qn]
    polys = max(2, polys >> (log_n - 13))
    x = torch.empty(polys, ctx.qn, ctx.n, dtype=torch.int64, device="cuda")
    torch.manual_seed(polys)
    for l, v in enumerate(q):
        x[:, l] = torch.randint(int(v), (polys, ctx.n), dtype=torch.int64, device="cuda")
        x[0, l, ::3] = int(v) - 1
    for tiles in (False, True):
        if tiles:  # explicit plans: another split, chunks
            plan = (ctx.log_n + 1) // 2 - 1 | 12 << 4 | 12 << 8 | 2 << 14
            assert kb.lib.kbfv_ntt_plan_valid(log_n, plan) == 0
            for b in range(4):
                ctx.set_ntt_plan(+1, b, plan)
                ctx.set_ntt_plan(-1, b, plan)
        y = ctx.ntt(x, torch.empty_like(x), +1, ctx.oQ, ctx.qn, polys=polys)
        for k in (0, polys - 1):
            assert np.array_equal(kb.to_host(y[k:k + 1]), oc.ntt_fwd(kb.to_host(x[k:k + 1]), ctx.oQ, ctx.qn, 1)), k
        ctx.ntt(y, y, -1, ctx.oQ, ctx.qn, polys=polys)
        assert torch.equal(y, x)


@pytest.mark.parametrize("mix,batch", [((True, False), 1), ((False, True, True), 3), ((True, False, False, True), 35)])
def test_product_and_rotation(mix, batch):
    kb, ctx, args = make(mix)
    oc = orc.Ctx(*args)
    sk = ctx.keygen_sk(bytes([1]) * 32)
    pk = ctx.keygen_pk(bytes([2]) * 32, sk)
    rlk, g = ctx.keygen_rlk(bytes([3]) * 32, sk), ctx.galois_elt(3)
    gkey = ctx.keygen_galois(bytes([4]) * 32, sk, g)
    m = np.random.default_rng(batch).integers(0, ctx.plain, size=(batch, ctx.n), dtype=np.uint64)
    ct = ctx.encrypt(bytes([5]) * 32, pk, kb.to_device(m))
    host, prod, rot = kb.to_host(ct), kb.to_host(ctx.mult_relin(rlk, ct, ct.flip(0).contiguous())), \
        kb.to_host(ctx.rotate(gkey, g, ct))
    for b in {0, batch - 1}:
        assert np.array_equal(host[b], oc.encrypt(bytes([5]) * 32, kb.to_host(pk), m[b], entry=b)), b
        assert np.array_equal(prod[b], oc.mult_relin(kb.to_host(rlk), host[b], host[batch - 1 - b])), b
        assert np.array_equal(rot[b], oc.rotate(kb.to_host(gkey), g, host[b])), b
