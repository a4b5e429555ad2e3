"""GPU: key-switch digits at the top residues of their blocks, where the float overflow
estimate rounds up to the next integer: both conversions against the oracle, bit for bit
(test_oracle_ks_ends.py pins the oracle there), and a product that meets such a residue (the
third ciphertext, squared) against the oracle and by decryption."""
import numpy as np
import pytest

import oracle_lib as orc
import params as P
from test_oracle_ks_ends import CHAINS, ends

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chain", list(CHAINS))
def test_top_residues(chain):
    import kunpbfv_amd as kb
    d = CHAINS[chain]()
    args = (d["log_n"], d["q"], d["p"], d["t"], d["gamma"], d["plain"])
    ctx, oc = kb.Context(*args), orc.Ctx(*args)

    def tops(src, width):
        return np.concatenate([ends(src[i:i + width], ctx.n)[1] for i in range(0, len(src), width)])

    x = tops(d["q"], len(d["p"]))
    out = ctx.empty(1, ctx.dnum, ctx.tn, ctx.n)
    ctx.modup_qj_to_t(kb.to_device(x), out)
    assert np.array_equal(kb.to_host(out)[0], oc.modup_qj_to_t(x))
    x = tops(list(d["p"]) + list(d["q"]), d["gamma"])
    out = ctx.empty(1, ctx.ri_blocks, ctx.tn, ctx.n)
    ctx.modup_pq_to_t(kb.to_device(x), out)
    assert np.array_equal(kb.to_host(out)[0], oc.modup_pq_to_t(x))


def test_product_with_a_top_residue_among_its_digits():
    import kunpbfv_amd as kb
    d = P.chain60(12, 4, 1, 4, 2)
    args = (12, d["q"], d["p"], d["t"], d["gamma"], d["plain"])
    ctx, oc = kb.Context(*args), orc.Ctx(*args)
    sk = ctx.keygen_sk(bytes([1]) * 32)
    pk = ctx.keygen_pk(bytes([2]) * 32, sk)
    rlk = ctx.keygen_rlk(bytes([3]) * 32, sk)
    m = np.random.default_rng(1).integers(0, ctx.plain, size=(3, ctx.n), dtype=np.uint64)
    ct = ctx.encrypt(bytes([4]) * 32, pk, kb.to_device(m))[2:].contiguous()
    host = kb.to_host(ct)[0]
    digits = oc.mult_tensor(host, host)[0]
    q = np.array(d["q"], dtype=np.uint64)[:, None]
    assert ((q - digits).astype(np.float64) < q.astype(np.float64) * 2.0 ** -25).any()  # the case is what it says
    prod = ctx.mult_relin(rlk, ct, ct)
    assert np.array_equal(kb.to_host(prod)[0], oc.mult_relin(kb.to_host(rlk), host, host))
    full = np.convolve(m[2].astype(object), m[2].astype(object))
    want = full[:ctx.n].copy()
    want[:ctx.n - 1] -= full[ctx.n:]
    assert np.array_equal(kb.to_host(ctx.decrypt(sk, prod))[0].astype(object), want % ctx.plain)
