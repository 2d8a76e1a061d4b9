"""The chunks of a long GDN call spread over the chip (lollm_gdn_layer_split) against the kernel
that walks them (lollm_gdn_layer_chunked, held to the oracle in test_gdn_layer_gpu.py; calls
with few heads there take the spread form): the same arithmetic per chunk, so outputs differ by
isolated bf16 roundings and states by summation order."""

import pytest
import torch

pytestmark = pytest.mark.gpu
D, K = 128, 4


def call(ops, m, spread, fresh, monkeypatch):
    """One long call in the spread or the walked form (also where the rule would take the other),
    held to that kernel's entry."""
    from lollm_amd import _lib
    monkeypatch.setattr(ops, "GDN_SPLIT_MAX_HEADS", 1 << 30 if spread else 0)
    monkeypatch.setattr(ops, "GDN_CHUNK", 0)
    ran = []
    for name in ("lollm_gdn_layer_split", "lollm_gdn_layer_chunked"):
        fn = getattr(_lib.lib(), name)
        monkeypatch.setattr(_lib.lib(), name, lambda *a, fn=fn, name=name: ran.append(name) or fn(*a))
    win, rec = m["win"].clone(), m["rec"].clone()
    out = ops.gdn_layer(m["proj"], m["conv_w"], m["A_log"], m["dt_bias"], m["norm_w"], win, m["off"], rec,
                        m["half"], m["rep"], m["replay"], fresh, m["B"], m["T"], m["Hk"], m["Hv"], D, K, 1e-6,
                        chunked=True)
    torch.cuda.synchronize()
    monkeypatch.undo()
    assert ran == ["lollm_gdn_layer_split" if spread else "lollm_gdn_layer_chunked"]
    return out.float().cpu(), rec.cpu(), win.cpu()


def make(B, T, Hk, Hv, seed, S=4):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rn(*shape, scale=1.0):
        return scale * torch.randn(*shape, device="cuda", generator=g)

    C, W = 2 * Hk * D + Hv * D, K - 1 + S
    P = -(-(C + Hv * D + 2 * Hv) // 8) * 8
    half = torch.randint(0, 2, (B,), device="cuda", generator=g, dtype=torch.int32)
    return dict(B=B, T=T, Hk=Hk, Hv=Hv, proj=rn(B, T, P).bfloat16(), conv_w=rn(C, K, scale=0.5).bfloat16(),
                A_log=rn(Hv, scale=0.5), dt_bias=rn(Hv, scale=0.5), norm_w=(1 + rn(D, scale=0.1)).bfloat16(),
                win=rn(B, 2 * W, C).bfloat16(), rec=rn(B, 2, Hv, D, D, scale=0.02), half=half, off=half * W + 2,
                rep=torch.zeros(B, 2, Hv, S, 4 * D + 16, dtype=torch.uint8, device="cuda"),
                replay=torch.zeros(B, dtype=torch.int32, device="cuda"))


CASES = [
    # B, T, Hk, Hv
    (1, 65, 16, 32),      # one token in the second chunk
    (1, 128, 1, 2),       # whole chunks; heads not a multiple of 8
    (2, 191, 2, 4),       # one token short of a chunk
    (3, 66, 1, 3),        # three v-heads per qk-head, 9 heads
    (1, 64, 8, 16),       # a single chunk
    (1, 8257, 16, 32),    # more chunks than a segment holds
]


@pytest.mark.parametrize("B,T,Hk,Hv", CASES)
@pytest.mark.parametrize("fresh", [True, False])
def test_spread_chunks_equal_walked_chunks(B, T, Hk, Hv, fresh, monkeypatch):
    from lollm_amd import ops
    print(f"case gdn spread B={B} T={T} Hk={Hk} Hv={Hv} fresh={fresh}", flush=True)
    m = make(B, T, Hk, Hv, seed=T + Hv)
    out, rec, win = call(ops, m, True, fresh, monkeypatch)
    ref, rec0, win0 = call(ops, m, False, fresh, monkeypatch)
    assert torch.equal(win, win0)
    # hi + lo products carry 2^-17 relative error and the sums run in another order: states
    # agree to a few 1e-6 of their scale, outputs but for a rounding flip where the sum lies
    # near a bf16 midpoint (2^-9 of the elements would already be 2^-17 / 2^-8 apart)
    for b in range(B):
        h = 1 - int(m["half"][b])
        assert torch.equal(rec[b, 1 - h], rec0[b, 1 - h])
        assert (rec[b, h] - rec0[b, h]).abs().max() <= 5e-5 * rec0[b, h].abs().max()
    assert (out != ref).float().mean() <= 1e-2
    torch.testing.assert_close(out, ref, rtol=2e-2, atol=1e-2)


def test_spread_workspace_is_validated():
    """A short or missing workspace is refused before any launch; bad sizes give -1."""
    from lollm_amd import _lib, ops
    L = _lib.lib()
    assert L.lollm_gdn_split_workspace_bytes(1, 0, 16, 32) == -1
    assert L.lollm_gdn_split_workspace_bytes(1, 100, 3, 32) == -1
    need = L.lollm_gdn_split_workspace_bytes(1, 70, 1, 2)
    m = make(1, 70, 1, 2, seed=3)
    buf = torch.empty(need, dtype=torch.uint8, device="cuda")
    out = torch.empty(1, 70, 2 * D, dtype=torch.bfloat16, device="cuda")
    p = ops._ptr
    for ws, n in ((None, need), (p(buf), need - 1)):
        rc = L.lollm_gdn_layer_split(
            p(m["proj"]), m["proj"].shape[-1], p(m["conv_w"]), p(m["A_log"]), p(m["dt_bias"]), p(m["norm_w"]),
            p(m["win"]), p(m["off"]), 7, p(m["rec"]), p(m["half"]), p(m["rep"]), p(m["replay"]), 4, 0, p(out), ws,
            n, 1, 70, 1, 2, D, D, K, 1e-6, None)
        assert rc == 1
