"""The long-call attention kernel (many new positions per sequence) and the many-token
attention prologue, against the oracle and against the kernels of the short calls.

An explicit `grid` always takes the split-K kernels, so the same operands reach both; without
one, a call that leaves its workspace as it was has taken the long-call kernel."""

import pytest
import torch

from test_attn_gpu import D, TOL, make_case, oracle

pytestmark = pytest.mark.gpu


def long_call(q, kc, vc, kl, gate):
    """ops.attn_verify without a grid, held to the long-call kernel."""
    from lollm_amd import ops
    B, T, Hq, _ = q.shape
    n = ops.attn_workspace_bytes(B, T, Hq, kc.shape[1], D, kc.shape[2])
    ws = torch.full((n,), 0x5A, dtype=torch.uint8, device="cuda")
    out = ops.attn_verify(q.cuda(), kc.cuda(), vc.cuda(), kl.cuda(), None if gate is None else gate.cuda(), workspace=ws)
    assert bool((ws == 0x5A).all()), "the call took the split-K kernels"
    return out


CASES = [   # 80 tiles of 128 rows or more: the long-call kernel's line on 256 CUs
    # B, T, Hq, Hkv, lens
    (40, 16, 8, 2, [16 + 3 * b for b in range(40)]),          # the shortest long call; 64 rows of a 128-row tile
    (10, 17, 32, 4, [17 + 40 * b for b in range(10)]),        # one row past a tile (16 positions x 8 heads)
    (20, 33, 4, 4, [33] + [500] * 19),                        # n_rep 1: 33 rows
    (40, 43, 6, 2, [75] * 40),                                # n_rep 3: 42 positions per tile, 2 rows of it unused
    (7, 50, 32, 1, [64 + b for b in range(7)]),               # n_rep 32: 4 positions per tile
    (10, 100, 10, 2, [100 + 3 * b for b in range(10)]),       # n_rep 5; key blocks cut at many residues
    (40, 31, 8, 2, [511] * 40),                               # one position short of a block end
    (20, 64, 8, 2, [64, 20] * 10),                            # kv_len < T: the first rows see no key
    (40, 16, 8, 2, [16, 0] * 20),                             # empty sequences
    (1, 2053, 8, 2, [2053]),                                  # many tiles, odd sizes
    (4, 200, 32, 4, [200, 900, 333, 1200]),
]


@pytest.mark.parametrize("B,T,Hq,Hkv,lens", CASES)
@pytest.mark.parametrize("gated", [True, False])
def test_long_call_matches_oracle_and_split(B, T, Hq, Hkv, lens, gated):
    from lollm_amd import ops
    print(f"case long attention B={B} T={T} Hq={Hq} Hkv={Hkv} lens={lens} gated={gated}", flush=True)
    q, kc, vc, kl, gate = make_case(B, T, Hq, Hkv, lens, seed=sum(lens) + T, max_len=max(lens) + 3)
    gate = gate if gated else None
    out = long_call(q, kc, vc, kl, gate)
    split = ops.attn_verify(q.cuda(), kc.cuda(), vc.cuda(), kl.cuda(), gate.cuda() if gated else None, grid=64)
    torch.cuda.synchronize()
    assert torch.isfinite(out.float()).all()
    # the split kernels round P to bf16 (relative 2^-9) and both the output
    torch.testing.assert_close(out.float(), split.float(), rtol=1.6e-2, atol=1e-2)
    pick = [b for b in range(B) if lens[b] >= T]
    pick = sorted({pick[0], pick[len(pick) // 2], pick[-1]})
    ref = oracle(q[pick], kc[pick], vc[pick], kl[pick], gate[pick] if gated else None)
    torch.testing.assert_close(out[pick].cpu().float(), ref, **TOL)


def test_two_row_groups_match_oracle():
    """Enough 256-row tiles for the 64-rows-per-wave form (512, its line is 384 on 256 CUs), odd
    lengths; two of the sequences against the oracle, all against the split kernels."""
    from lollm_amd import ops
    B, T, Hq, Hkv = 16, 231, 32, 4
    lens = [T + 37 * b for b in range(B)]
    print("case two row groups", flush=True)
    q, kc, vc, kl, gate = make_case(B, T, Hq, Hkv, lens, seed=5, max_len=max(lens) + 1)
    out = long_call(q, kc, vc, kl, gate)
    split = ops.attn_verify(q.cuda(), kc.cuda(), vc.cuda(), kl.cuda(), gate.cuda(), grid=256)
    torch.testing.assert_close(out.float(), split.float(), rtol=1.6e-2, atol=1e-2)
    pick = [0, 15]
    torch.testing.assert_close(out[pick].cpu().float(),
                               oracle(q[pick], kc[pick], vc[pick], kl[pick], gate[pick]), **TOL)


@pytest.mark.parametrize("B,T,Hq,Hkv,L", [(4, 100, 32, 4, 100), (1, 600, 32, 4, 700), (2, 1600, 32, 4, 1600)])
@pytest.mark.parametrize("scale", [1.0, 2.0])
def test_long_call_error_is_the_output_rounding(B, T, Hq, Hkv, L, scale):
    """Against 64 bits: the weights carry 16 bits and their sum 24, so the error is that of
    rounding the exact result to bf16 (2^-16 of the weights beside it: under 1% of it); the
    split kernels, whose weights carry 8 bits, are further away."""
    from lollm_amd import ops
    print(f"case long attention error B={B} T={T} L={L} scale={scale}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T)
    q = (scale * torch.randn(B, T, Hq, D, device="cuda", generator=g)).bfloat16()
    kc, vc = (torch.randn(B, Hkv, L, D, device="cuda", generator=g).bfloat16() for _ in range(2))
    kl = torch.full((B,), L, dtype=torch.int32, device="cuda")
    out = long_call(q, kc, vc, kl, None).double().view(B, T, Hq, D)
    split = ops.attn_verify(q, kc, vc, kl, grid=256).double().view(B, T, Hq, D)
    seen = torch.arange(L, device="cuda") <= (L - T + torch.arange(T, device="cuda"))[:, None]
    err, err_split, rounding = 0.0, 0.0, 0.0
    for b in range(B):
        for h in range(Hq):
            s = (q[b, :, h].double() @ kc[b, h * Hkv // Hq].double().t()) * D ** -0.5
            o = s.masked_fill(~seen, float("-inf")).softmax(-1) @ vc[b, h * Hkv // Hq].double()
            err += (out[b, :, h] - o).square().sum().item()
            err_split += (split[b, :, h] - o).square().sum().item()
            rounding += (o.bfloat16().double() - o).square().sum().item()
    assert err <= 1.02 * rounding and err <= err_split


@pytest.mark.parametrize("B,T,Hq,Hkv", [(10, 100, 32, 4), (16, 231, 32, 4)])
def test_infinite_values_stay_infinite(B, T, Hq, Hkv):
    """Infinite and NaN V entries reach the rows that see them as they are (key 0: every row, the
    first with a weight of exactly 1), as from the split kernels, and no other column."""
    from lollm_amd import ops
    print(f"case infinite values B={B} T={T}", flush=True)
    q, kc, vc, kl, gate = make_case(B, T, Hq, Hkv, [T] * B, seed=B + T)
    clean = long_call(q, kc, vc, kl, gate)
    inf, nan, late = float("inf"), float("nan"), 37
    vc[:, :, 0, 3], vc[:, :, 0, 200], vc[:, :, 0, 64] = inf, -inf, nan
    vc[:, :, late, 5], vc[:, :, late, 130] = -inf, inf
    out = long_call(q, kc, vc, kl, gate)
    split = ops.attn_verify(q.cuda(), kc.cuda(), vc.cuda(), kl.cuda(), gate.cuda(), grid=256)
    out, split, clean = (t.cpu().float().view(B, T, Hq, D) for t in (out, split, clean))
    for o in (out, split):
        assert (o[..., 3] == inf).all() and (o[..., 200] == -inf).all() and o[..., 64].isnan().all()
        assert (o[:, late:, :, 5] == -inf).all() and (o[:, late:, :, 130] == inf).all()
    rest = [c for c in range(D) if c not in (3, 200, 64, 5, 130)]
    assert torch.equal(out[..., rest], clean[..., rest])


def test_large_scores_move_the_reference_maximum():
    """Keys whose scores grow along the context: the running maximum moves often, by far more
    than the rescale threshold, and differently per row."""
    B, T, Hq, Hkv = 4, 300, 8, 2
    q, kc, vc, kl, gate = make_case(B, T, Hq, Hkv, [300] * B, seed=9)
    kc = (kc.float() * torch.linspace(0.2, 12, 300)[None, None, :, None]).bfloat16()
    print("case growing scores", flush=True)
    out = long_call(q, kc, vc, kl, gate)
    torch.testing.assert_close(out.cpu().float(), oracle(q, kc, vc, kl, gate), **TOL)


@pytest.mark.parametrize("B,T,Hq,Hkv", [(10, 100, 10, 2), (16, 231, 32, 4)])
def test_cache_strides_beyond_packed(B, T, Hq, Hkv):
    """Heads and sequences of the caches further apart than packed (the library's strides; NaN in
    the gaps), in both tile heights: the bits of the packed caches."""
    from lollm_amd import _lib, ops
    print(f"case long attention strides B={B} T={T}", flush=True)
    q, kc, vc, kl, gate = make_case(B, T, Hq, Hkv, [T + 2 * b for b in range(B)], seed=T)
    packed = long_call(q, kc, vc, kl, gate)
    n = kc.shape[2]
    head, seq = (n + 3) * D, Hkv * (n + 3) * D + 5 * D
    wide = []
    for c in (kc, vc):
        buf = torch.full((B * seq,), float("nan"), dtype=torch.bfloat16, device="cuda")
        buf.as_strided((B, Hkv, n, D), (seq, head, D, 1)).copy_(c)
        wide.append(buf)
    qd, gd, kld, out = q.cuda(), gate.cuda(), kl.cuda(), torch.zeros_like(packed)
    need = ops.attn_workspace_bytes(B, T, Hq, Hkv, D, n)
    ws = torch.full((need,), 0x5A, dtype=torch.uint8, device="cuda")
    p = ops._ptr
    rc = _lib.lib().lollm_attn_verify(p(qd), p(wide[0]), p(wide[1]), p(kld), p(gd), p(out), p(ws), need, B, T, Hq,
                                      Hkv, D, n, seq, head, 0, D ** -0.5, ops._stream())
    assert rc == 0
    assert torch.equal(out, packed) and bool((ws == 0x5A).all())


@pytest.mark.parametrize("B,T,Hq,Hkv,rd,rope", [(2, 150, 8, 2, 64, None), (4, 64, 5, 2, 256, "start"),
                                               (3, 100, 4, 1, 16, "token"), (2, 128, 3, 3, 0, None),
                                               (2, 130, 4, 2, 128, "token")])
def test_many_token_prologue_equals_few_token_prologue(B, T, Hq, Hkv, rd, rope):
    """256 tokens or more take the token-per-workgroup kernel; the same tokens in calls of
    fewer take the head-per-workgroup kernel.  Same bits, also at the cache's end."""
    from lollm_amd import ops
    print(f"case prologue B={B} T={T} Hq={Hq} Hkv={Hkv} rd={rd} rope={rope}", flush=True)
    g = torch.Generator().manual_seed(B * T)
    max_len = T + 20
    qkv = torch.randn(B, T, Hq * 2 * D + 2 * Hkv * D, generator=g).bfloat16().cuda()
    qn, kn = ((0.1 * torch.randn(D, generator=g)).bfloat16().cuda() for _ in range(2))
    freq = (1.0 / (1e7 ** (torch.arange(0, max(rd, 2), 2).float() / max(rd, 2)))).cuda()
    lengths = torch.randint(0, 30, (B,), generator=g, dtype=torch.int32).cuda()   # some rows past max_len
    pos = {None: None, "start": torch.randint(0, 40000, (B,), generator=g, dtype=torch.int32),
           "token": torch.randint(0, 40000, (B, T), generator=g, dtype=torch.int32)}[rope]
    kc, vc = (torch.zeros(B, Hkv, max_len, D, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    kc2, vc2 = torch.zeros_like(kc), torch.zeros_like(vc)
    q, gate = ops.attn_prologue(qkv, qn, kn, freq, lengths, B, T, Hq, Hkv, D, rd, 1e-6, kc, vc,
                                rope_pos=None if pos is None else pos.cuda())
    for b in range(B):
        q1, g1 = ops.attn_prologue(qkv[b:b + 1].contiguous(), qn, kn, freq, lengths[b:b + 1].clone(), 1, T, Hq,
                                   Hkv, D, rd, 1e-6, kc2[b:b + 1], vc2[b:b + 1],
                                   rope_pos=None if pos is None else pos[b:b + 1].cuda())
        assert torch.equal(q1[0].cpu(), q[b].cpu()) and torch.equal(g1[0].cpu(), gate[b].cpu())
    assert torch.equal(kc.cpu(), kc2.cpu()) and torch.equal(vc.cpu(), vc2.cpu())
