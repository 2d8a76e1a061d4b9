"""lollm_sample_rows with a row's counts spread over workgroups (few rows) against the one
workgroup per row that a workspace without room for the counts takes: the same token."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def rows_of(V, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(9, V, generator=g) * 3
    x[1] = -x[1].abs() - 0.25                # all negative
    x[2, V // 2] = float("inf")
    x[3, V - 1] = float("nan")
    x[4, 0] = 80.0                           # far above the rest: most slices weigh nothing
    x[5] = -1e-6                             # every key flushed to 0
    x[6, : V // 3] = -1.0e30                 # whole slices beyond the counted distances
    x[7] = torch.randint(-2, 3, (V,), generator=g).float()   # many ties
    x[8] = float("-inf")
    x[8, V - 3 :] = 1.0
    return x.bfloat16().cuda()


# the shortest rows the slices take (with a small top-k, without) and slices of unequal length;
# chunks past the registers of a slice's threads (4 x 1024 x 16 slices); the longest rows, and
# one past them
@pytest.mark.parametrize("V", [49144, 49152, 50304, 147456, 151936, 524288 + 8 * 17, 16 * 65528,
                               16 * 65528 + 8])
@pytest.mark.parametrize("temp,top_k,top_p", [(0.7, 0, 1.0), (0.7, 20, 0.8), (1.7, 0, 0.5), (1.0, 3000, 1.0),
                                              (400.0, 1, 0.9)])
def test_few_rows_draw_the_same_tokens(V, temp, top_k, top_p):
    from lollm_amd import ops
    print(f"case sample slices V={V} T={temp} top_k={top_k} top_p={top_p}", flush=True)
    rows = rows_of(V, seed=V % 1000)
    small = torch.empty(9 * 152, dtype=torch.uint8, device="cuda")   # the row statistics alone
    assert ops.sample_workspace_bytes(9) > small.numel()
    for off in range(4):
        want = ops.sample_rows(rows, temp, top_k, top_p, 31, off, row_base=3, slot=1, workspace=small)
        got = ops.sample_rows(rows, temp, top_k, top_p, 31, off, row_base=3, slot=1)
        assert torch.equal(got, want)
