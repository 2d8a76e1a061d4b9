"""The one-launch repetition penalty of sample_next against the bitmap path, bit for bit."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V,n", [(8, 3), (2048, 100), (2056, 896), (32768, 896), (151936, 517), (151936, 1)])
@pytest.mark.parametrize("pen", [1.1, 0.7])
def test_penalised_row_equals_bitmap_path(V, n, pen):
    from array import array
    from lollm_amd import ops
    print(f"case penalised row V={V} n={n} pen={pen}", flush=True)
    g = torch.Generator().manual_seed(V + n)
    x = (4 * torch.randn(1, V, generator=g)).bfloat16().cuda()
    tok = torch.randint(-2, V + 3, (n,), generator=g, dtype=torch.int32)   # some outside, some twice
    tok[:: 7] = tok[0]
    tok[-1] = V - 1
    got = ops.penalised_row(x, array("i", tok.tolist()), pen)
    ref = x.clone()
    ops.repetition_penalty(ref, ops.seen_mark(ops.new_seen(1, V, "cuda"), tok.cuda(), V), pen)
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("n", [0, 5, 896, 897, 3000])
def test_sample_next_same_token_for_every_context_form(n):
    """Contexts a launch carries and longer ones, as a list, a tuple and an iterator, from an
    aligned row and a view; the row itself is not changed."""
    from lollm_amd.generate import sample_next
    print(f"case sample_next context {n}", flush=True)
    g = torch.Generator().manual_seed(n)
    V = 4096
    buf = (3 * torch.randn(V + 8, generator=g)).bfloat16().cuda()
    ids = torch.randint(0, V, (n,), generator=g).tolist()
    row, keep = buf[8:], buf.clone()
    want = None
    for form in (ids, tuple(ids), iter(list(ids)) if n else []):
        for x in (row, row.float(), torch.stack([row, row], 1)[:, 0], torch.cat([row[:1], row])[1:]):
            if not isinstance(form, (list, tuple)):
                form = iter(list(ids)) if n else []
            t = sample_next(x, 0.8, 20, 0.9, 1.3, form, seed=5, offset=3)
            want = t if want is None else want
            assert t == want and isinstance(t, int)
    assert torch.equal(buf.view(torch.int16), keep.view(torch.int16))
