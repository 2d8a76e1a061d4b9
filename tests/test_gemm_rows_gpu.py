"""The many-row GEMM (lollm_gemm_rows) against fp32, at the edges of its tiles, and, with K
whole, its row independence of M and tile; the rule that picks its tile is checked on the CPU."""

import pytest
import torch

TILES = (44, 34, 43, 24)


def case(M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(M, K, generator=g).bfloat16(), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16()


def close(got, ref):
    # fp32 sums of exact bf16 products, one rounding to bf16 (2^-9 of the value)
    torch.testing.assert_close(got.float().cpu(), ref, rtol=2 ** -8, atol=1e-3)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K", [(1, 64, 128), (65, 64, 128), (129, 320, 256), (255, 256, 384), (257, 192, 128),
                                   (300, 832, 512), (193, 1088, 128)])
def test_gemm_rows_matches_fp32(M, N, K, tile):
    from lollm_amd import ops
    print(f"case gemm rows M={M} N={N} K={K} tile={tile}", flush=True)
    x, W = case(M, N, K, seed=M + N + K)
    t = ops.gemm_tile_weights(W.cuda())
    out = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device="cuda")
    from lollm_amd import _lib
    xd = x.cuda()
    rc = _lib.lib().lollm_gemm_rows(xd.data_ptr(), K, t.data_ptr(), out.data_ptr(), N, M, N, K, 0, tile, 1, None, 0,
                                    torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    close(out[:M], x.float() @ W.float().t())
    assert (out[M] == 7.0).all()          # nothing written past the last row


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K", [(130, 448, 256), (517, 1600, 128), (70, 64, 128)])
def test_gemm_rows_swiglu_equals_product_then_swiglu(M, N, K, tile):
    """The fused SwiGLU is the separate kernel's arithmetic: same bits."""
    from lollm_amd import ops
    print(f"case gemm rows swiglu M={M} N={N} K={K} tile={tile}", flush=True)
    x, W = case(M, N, K, seed=M + N)
    W = (W.float() * 4).bfloat16().cuda()
    x = x.cuda()
    got = ops.gemm_rows(x, ops.gemm_tile_weights(W, ops.GEMM_SWIGLU), N, K, ops.GEMM_SWIGLU, tile)
    ref = ops.swiglu(ops.gemm_rows(x, ops.gemm_tile_weights(W), N, K, ops.GEMM_NONE, tile))
    assert torch.equal(got, ref)


@pytest.mark.gpu
def test_gemm_rows_several_tiles_per_workgroup_and_row_independence():
    """More tiles than CUs: a workgroup's next tile is loaded during its last one.  Every tile
    shape, and a call over a part of the rows, gives a row the same bits."""
    from lollm_amd import ops
    M, N, K = 2100, 12352, 128
    print(f"case gemm rows many tiles M={M} N={N} K={K}", flush=True)
    x, W = case(M, N, K, seed=3)
    t, xd = ops.gemm_tile_weights(W.cuda()), x.cuda()
    outs = [ops.gemm_rows(xd, t, N, K, ops.GEMM_NONE, tile) for tile in TILES]
    close(outs[0], x.float() @ W.float().t())
    for o in outs[1:]:
        assert torch.equal(o, outs[0])
    part = ops.gemm_rows(xd[700:877].contiguous(), t, N, K, ops.GEMM_NONE, 24)
    assert torch.equal(part, outs[0][700:877])


@pytest.mark.gpu
def test_projection_takes_the_rows_kernel_and_keeps_gradients():
    from lollm_amd.qwen3_5.blocks import Projection
    x, W = case(1200, 8192, 256, seed=4)
    p = Projection(W.cuda())
    xd = x.cuda()
    assert p.rows_plan(xd, 1200)[0] and not p.rows_plan(xd.float(), 1200)[0]
    close(p(xd), x.float() @ W.float().t())
    xg = xd.clone().requires_grad_()
    p(xg).float().sum().backward()
    assert xg.grad is not None


@pytest.mark.gpu
def test_projection_keeps_weight_gradients_and_tangents():
    """Past 64 rows a trainable weight gets its gradient and its updated values are used (also
    without grad mode), and a forward-mode tangent passes: F.linear's, by exact equality."""
    from torch.autograd import forward_ad
    from lollm_amd.qwen3_5.blocks import Projection
    print("case projection weight gradient and tangent", flush=True)
    x, W = case(1200, 8192, 256, seed=6)
    xd, Wd = x.cuda(), W.cuda()
    wp = torch.nn.Parameter(Wd.clone())
    p = Projection(wp)
    p(xd).float().sum().backward()
    want = torch.nn.Parameter(Wd.clone())
    torch.nn.functional.linear(xd, want).float().sum().backward()
    assert torch.equal(wp.grad, want.grad)
    with torch.no_grad():
        wp.mul_(2)
        assert torch.equal(p(xd), torch.nn.functional.linear(xd, wp))
    plain, dx = Projection(Wd), x.flip(0).cuda()
    with forward_ad.dual_level():
        tangent = forward_ad.unpack_dual(plain(forward_ad.make_dual(xd, dx))).tangent
    assert torch.equal(tangent, torch.nn.functional.linear(dx, Wd))


class _Recorded(torch.Tensor):
    pass


def test_opaque_call_rule():
    """Each way in which PyTorch follows an operator keeps F.linear (on the CPU: the rule is
    asked inside the transform, and the projection there equals F.linear's own result)."""
    from torch.autograd import forward_ad
    from torch.fx.experimental.proxy_tensor import make_fx
    from lollm_amd.qwen3_5.blocks import Projection, opaque_call_ok
    x, W = case(70, 64, 128, seed=7)
    p = Projection(W)
    asked = []

    def f(a):
        asked.append(opaque_call_ok(a, W))
        return p(a)

    want = torch.nn.functional.linear(x, W)
    assert torch.equal(f(x), want) and asked == [True]
    with torch.inference_mode():
        f(x)
    with torch.no_grad():
        f(x.clone().requires_grad_())
    assert asked == [True] * 3
    del asked[:]
    assert not opaque_call_ok(x, torch.nn.Parameter(W))
    assert f(x.clone().requires_grad_()).requires_grad
    assert f(x.as_subclass(_Recorded)).shape == want.shape
    batched = torch.func.vmap(f)(torch.stack([x, -x]))
    torch.testing.assert_close(batched[1], -want)
    assert torch.equal(torch.func.jvp(f, (x,), (x,))[1], want)
    with forward_ad.dual_level():
        assert torch.equal(forward_ad.unpack_dual(f(forward_ad.make_dual(x, x))).tangent, want)
    assert torch.equal(make_fx(f)(x)(-x), torch.nn.functional.linear(-x, W))
    assert torch.equal(torch.jit.trace(f, (x,), check_trace=False)(-x), torch.nn.functional.linear(-x, W))
    assert asked == [False] * len(asked) and len(asked) >= 7


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,splits,epi", [(65, 320, 1536, 12, 0), (129, 256, 512, 4, 0), (257, 1088, 384, 3, 0),
                                              (96, 4096, 8192, 16, 0), (100, 448, 256, 2, 1), (300, 8192, 256, 2, 0),
                                              (300, 8192, 512, 4, 0)])
def test_gemm_rows_split_k(M, N, K, splits, epi):
    """K in parts: each part's fp32 sums added in order, one rounding at the end.  The last case
    has more (tile, part) pairs than CUs, so that workgroups go from one to the next."""
    from lollm_amd import ops
    if splits == 4 and M == 300:
        assert -(-M // 128) * -(-N // 256) * splits > torch.cuda.get_device_properties(0).multi_processor_count
    print(f"case gemm rows split M={M} N={N} K={K} splits={splits} epi={epi}", flush=True)
    x, W = case(M, N, K, seed=M + K)
    W, xd = (W.float() * 3).bfloat16().cuda(), x.cuda()
    got = ops.gemm_rows(xd, ops.gemm_tile_weights(W, epi), N, K, epi, 24, splits)
    one = ops.gemm_rows(xd, ops.gemm_tile_weights(W, epi), N, K, epi, 24)
    if not epi:
        close(got, x.float() @ W.float().cpu().t())
    # another order of the same fp32 sums: a bf16 rounding (two with SwiGLU) may flip
    assert (got != one).float().mean() <= 2e-2
    torch.testing.assert_close(got.float(), one.float(), rtol=2 ** -6, atol=2e-3)
    from lollm_amd import _lib
    rc = _lib.lib().lollm_gemm_rows(xd.data_ptr(), K, 16, got.data_ptr(), N, M, N, K, 0, 24, splits, xd.data_ptr(),
                                    4 * splits * M * N - 1, None)
    assert rc == 1      # a short workspace is refused before any launch


def test_rows_splits_rule():
    from lollm_amd import ops
    f = ops.gemm_rows_splits
    assert f(96, 4096, 12288, 0, 256) == 16 and f(200, 4096, 12288, 0, 256) == 8
    assert f(512, 4096, 8192, 0, 256) == 4 and f(700, 4096, 8192, 0, 256) == 1
    assert f(96, 4096, 4096, 0, 256) == 1 and f(96, 24576, 12288, 1, 256) == 1
    for M in range(65, 3000, 37):
        for N, K in ((4096, 12288), (4096, 8192), (1024, 8192), (151936, 8192)):
            s = f(M, N, K, 0, 256)
            assert (K // 128) % s == 0 and (s == 1 or -(-M // 128) * -(-N // 256) * s <= 256)


def test_rows_tile_rule():
    """A pure function of the shape; the library keeps what leaves CUs idle or is one full round
    of its 256 x 256 tiles."""
    from lollm_amd import ops
    assert ops.gemm_rows_tile(128, 4096, 4096, 0, 256) == 0
    assert ops.gemm_rows_tile(1024, 1024, 3072, 0, 256) == 0
    assert ops.gemm_rows_tile(3998, 4096, 4096, 0, 256) == 0
    assert ops.gemm_rows_tile(3998, 4096, 4096, 1, 256) == 44
    assert ops.gemm_rows_tile(4500, 4096, 12288, 0, 256) == 34
    assert ops.gemm_rows_tile(2048, 18432, 4096, 0, 256) == 43
    assert ops.gemm_rows_tile(1847, 4096, 4096, 0, 256) == 24
    for M in range(65, 9000, 97):
        for N, K in ((12352, 4096), (18432, 4096), (24576, 4096), (4096, 12288), (1024, 3072)):
            assert ops.gemm_rows_tile(M, N, K, 0, 256) in (0, *TILES)


def test_gemm_rows_refuses_bad_arguments():
    """Before any HIP call, so without a device."""
    from lollm_amd import _lib
    f = _lib.lib().lollm_gemm_rows
    ok = (16, 128, 16, 16, 64, 1, 64, 128, 0, 44, 1, None, 0, None)
    for i, v in ((0, None), (2, None), (3, None), (5, 0), (6, 96), (7, 64), (1, 64), (1, 132), (4, 32), (8, 2), (0, 8), (10, 0), (10, 2)):
        a = list(ok)
        a[i] = v
        assert f(*a) == 1, (i, v)
