"""GPU: an external product of more ciphertexts than a grid dimension holds (65535), through
the auxiliary basis: the ones around that line and the last equal the same ciphertexts
taken one at a time, by the general path."""
import pytest

import params as P

pytestmark = pytest.mark.gpu


def test_more_ciphertexts_than_a_grid_dimension():
    import torch
    import kunpbfv_amd as kb
    d = P.chain60(12, 1, 1, 4, 2)
    ctx = kb.Context(12, d["q"], d["p"], d["t"], d["gamma"], d["plain"])
    batch, kinds, q = 65537, 29, int(ctx.mod[ctx.oQ])
    torch.manual_seed(3)
    rgsw = torch.randint(q, (ctx.rgsw_rows(20), 2, 1, ctx.n), dtype=torch.int64, device="cuda")
    some = torch.randint(q, (kinds, 2, 1, ctx.n), dtype=torch.int64, device="cuda")
    ct = some.repeat(-(-batch // kinds), 1, 1, 1)[:batch]
    out = ctx.external_product(rgsw, ct, 20)
    for b in (0, 65534, 65535, 65536):
        want = ctx.external_product(rgsw, some[b % kinds:b % kinds + 1], 20)
        assert torch.equal(out[b:b + 1], want), b
