"""The MTP head's input from embedding rows (lollm_mtp_rows) against the two norms and the
concatenation it fuses: the same bits; and the vectors of a block over an empty cache."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L,H", [(1, 1, 8), (3, 2, 264), (16, 1, 4096), (600, 1, 512), (2, 5, 8192)])
@pytest.mark.parametrize("rope", [True, False])
def test_mtp_rows_equals_norms_cat(B, L, H, rope):
    from lollm_amd import ops
    print(f"case mtp rows B={B} L={L} H={H} rope={rope}", flush=True)
    g = torch.Generator().manual_seed(B + H)
    emb, hidden = ((torch.randn(B, L, H, generator=g) * s).bfloat16().cuda() for s in (0.02, 3.0))
    w_e, w_h = ((torch.randn(H, generator=g) * 0.1).bfloat16().cuda() for _ in range(2))
    out, lengths, kv_len, first = ops.mtp_rows(emb, hidden, w_e, w_h, 1e-6, rope=rope)
    want = torch.cat([ops.rmsnorm(emb, w_e, 1e-6), ops.rmsnorm(hidden, w_h, 1e-6)], -1)
    assert torch.equal(out, want)
    assert lengths.tolist() == [0] * B and kv_len.tolist() == [L] * B
    assert first.tolist() == [1] * B if rope else first is None


def test_mtp_rows_rejects_other_shapes():
    from lollm_amd import ops
    x = torch.zeros(2, 3, 64, dtype=torch.bfloat16, device="cuda")
    w = torch.zeros(64, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(ValueError):
        ops.mtp_rows(x[:, :2].contiguous(), x, w, w, 1e-6)
