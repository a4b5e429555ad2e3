"""GPU: encryption's one-launch sampler at its edges (the fewest and the most 512-word
runs, one and many limbs, odd batches, a message at the ends of its range) against the
oracle's ciphertexts; bit-exact."""
import numpy as np
import pytest

import oracle_lib as orc
import params as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log_n,qn,batch,plain", [(12, 1, 1, 65537), (12, 3, 5, 257), (14, 2, 3, 786433), (16, 4, 2, 65537)])
def test_encrypt(log_n, qn, batch, plain):
    import kunpbfv_amd as kb
    d = P.chain60(log_n, qn, 1, 4, 2, plain=plain)
    args = (d["log_n"], d["q"], d["p"], d["t"], d["gamma"], d["plain"])
    ctx, oc = kb.Context(*args), orc.Ctx(*args)
    seed = bytes([log_n + qn]) * 32
    sk = ctx.keygen_sk(bytes([1]) * 32)
    pk = ctx.keygen_pk(bytes([2]) * 32, sk)
    m = np.random.default_rng(qn).integers(0, plain, size=(batch, ctx.n), dtype=np.uint64)
    m[0, :4] = (0, plain - 1, plain // 2, plain // 2 + 1)
    got = kb.to_host(ctx.encrypt(seed, pk, kb.to_device(m)))
    for b in range(batch):
        assert np.array_equal(got[b], oc.encrypt(seed, kb.to_host(pk), m[b], entry=b)), b
