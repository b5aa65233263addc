"""GroupNorm in one launch (csrc/kernels/groupnorm.hip) against 64 bits: alone, of two sources, and behind a split-K convolution."""
import pytest
import torch

from shai_amd import native, ops

pytestmark = pytest.mark.gpu


def rnd(*shape, scale=1.0):
    return (torch.randn(*shape, device="cuda") * scale).to(torch.bfloat16)


def norm64(x, gamma, beta, groups, eps, silu):
    N, C = x.shape[0], x.shape[-1]
    g = x.double().reshape(N, -1, groups, C // groups)
    g = g - g.mean((1, 3), keepdim=True)
    y = (g * torch.rsqrt((g * g).mean((1, 3), keepdim=True) + eps)).reshape(x.shape) * gamma.double() + beta.double()
    return y * torch.sigmoid(y) if silu else y


def off(y, want):
    """bf16 outputs: half a unit in the last place of 8 bits is 2^-9 of a value; the mean over them is below that."""
    return ((y.double() - want).norm() / want.norm()).item()


# pixels and channels (32 groups): groups of 4, 6, 10, 12, 20, 30, 40, 60 and 80 channels, one workgroup each or two groups together;
# 1, 2, 4, 8 and 16 vectors a thread, whole and with a remainder; one pixel
@pytest.mark.parametrize("hw,C", [(1, 1280), (3, 128), (64, 1280), (63, 192), (81, 320), (144, 960), (256, 960), (256, 384), (256, 2560), (576, 640),
                                  (1024, 640), (1024, 1920), (2304, 640), (4096, 512), (1023, 1920)])
def test_alone(cuda, hw, C):
    torch.manual_seed(hw + C)
    for N, silu, mean in ((1, True, 0.0), (3, False, 8.0)):
        x, gamma, beta = (rnd(N, hw, C) + mean).bfloat16(), rnd(C), rnd(C)
        assert ops.groupnorm_one_ok(x, hw, C, 32)
        assert off(ops.groupnorm_one(x, gamma, beta, 32, 1e-5, silu), norm64(x, gamma, beta, 32, 1e-5, silu)) < 2 ** -8
    assert off(ops.groupnorm_one(x, None, None, 32, 1e-5), norm64(x, torch.ones(C, device="cuda"), torch.zeros(C, device="cuda"), 32, 1e-5, False)) < 2 ** -8


@pytest.mark.parametrize("hw,C1,C2", [(64, 1280, 640), (256, 640, 320), (500, 320, 640), (16, 8, 120)])
def test_two_sources(cuda, hw, C1, C2):
    """The border lies inside a group (1920 / 32 = 60 channels) or between two; groups of 30 channels go two to a workgroup, 8 vectors a
    thread at the most (500 pixels; ``test_refused`` has 1024)."""
    torch.manual_seed(C1)
    x, x2, gamma, beta = rnd(2, hw, C1), (rnd(2, hw, C2) - 3).bfloat16(), rnd(C1 + C2), rnd(C1 + C2)
    y = ops.groupnorm_one(x, gamma, beta, 32, 1e-5, True, x2=x2)
    assert off(y, norm64(torch.cat([x, x2], -1), gamma, beta, 32, 1e-5, True)) < 2 ** -8


def test_refused(cuda):
    """Odd and narrow groups, and images that registers do not hold, keep the other kernels."""
    x = rnd(1, 64, 96)
    for hw, C, groups in ((64, 96, 32), (64, 224, 32), (1024, 960, 32), (64, 2 * 4, 2 * 2), (70000, 128, 32), (64, 100, 32)):
        assert not ops.groupnorm_one_ok(x, hw, C, groups)
    with pytest.raises(RuntimeError):
        ops.groupnorm_one(x, None, None, 32, 1e-5)


# a split-K choice is folded by the norm's launch, an unsplit one is not; the residual, the image's bias as columns of a wider tensor
@pytest.mark.parametrize("cfg,splits", [(3, 4), (4, 3), (18, 8), (9, 2), (16, 1), (4, 1)])
@pytest.mark.parametrize("side,cin,cout", [(16, 128, 640), (8, 192, 1280), (12, 64, 320)])
def test_after_convolution(cuda, cfg, splits, side, cin, cout):
    torch.manual_seed(side + splits)
    N = 2
    x, b, res = rnd(N, side, side, cin), rnd(cout), rnd(N, side, side, cout)
    w4 = (torch.randn(cout, cin, 3, 3, device="cuda") * (9 * cin) ** -0.5).bfloat16()
    w, temb, gamma, beta = ops.pack_conv_weight(w4), rnd(N, cout + 64)[:, 16:16 + cout], rnd(cout), rnd(cout)
    M, K = N * side * side, 9 * cin
    native.ops().gemm_tuning_import([f"1:{M},{cout},{K},b1,g0|{N},{side},{side},{cin},{cin},3,1,0,0={cfg},{splits}"])
    want = torch.nn.functional.conv2d(x.double().permute(0, 3, 1, 2).cpu(), w4.double().cpu(), b.double().cpu(), padding=1).permute(0, 2, 3, 1).cuda()
    want = want + temb.double()[:, None, None, :]
    for keep in (True, False):
        out, y = ops.conv2d(x, w, b, 3, 3, 1, 1, temb=temb, residual=res if keep else None, gn=(gamma, beta, 32, 1e-5, True), keep=keep)
        raw = want + res.double() if keep else want
        # the norm is of the rounded convolution: 2^-9 of a value, and 2^-9 of its own result
        assert off(y, norm64(raw, gamma, beta, 32, 1e-5, True)) < 2 ** -7
        assert out is None if not keep else off(out, raw) < 2 ** -8
        if keep:
            assert off(y, norm64(out, gamma, beta, 32, 1e-5, True)) < 2 ** -8
            plain = ops.conv2d(x, w, b, 3, 3, 1, 1, temb=temb, residual=res)
            assert torch.equal(out, plain)      # the fold's sums in its order
    # which launch folds: without keep the convolution itself is written only where its K is not split
    raw = torch.full((N, side, side, cout), 7.0, device="cuda", dtype=torch.bfloat16)
    native.ops().conv2d(x, None, w, raw, b, temb, None, None, None, 0, 3, 3, 1, 1, False, 0, 1.0, gn_gamma=gamma, gn_beta=beta,
                        gn_out=torch.empty_like(raw), gn_groups=32, gn_silu=True, keep_out=False)
    assert bool((raw == 7).all()) == (splits > 1)


# 81920 values of a group's parts and more: the fold and the norm are two launches.  Groups of 4 n channels and two groups to a workgroup,
# images of whole segments and of uneven ones (25 x 25: 157, 157, 157, 154 pixels), an image that has 16 segments, and the border below
@pytest.mark.parametrize("N,side,cout,splits", [(2, 32, 640, 4), (1, 32, 640, 8), (2, 16, 1280, 8), (2, 32, 320, 8), (1, 16, 960, 16), (2, 25, 640, 8),
                                                (1, 28, 1280, 3), (2, 16, 1280, 7)])
def test_large_fold(cuda, N, side, cout, splits):
    """Against the unfused convolution's own output, a last bit of y (its mean square is combined from segments, 2^-20); the same with an
    offset of 50 standard deviations, where E[x^2] - mean^2 in fp32 would lose 2500 x 2^-24."""
    torch.manual_seed(side + splits)
    cin = 1024 * splits // 16
    x, b, res = rnd(N, side, side, cin), rnd(cout), rnd(N, side, side, cout)
    w = (torch.randn(cout, 9 * cin, device="cuda") * (9 * cin) ** -0.5).bfloat16()
    gamma, beta, M, K = rnd(cout), rnd(cout), N * side * side, 9 * cin
    native.ops().gemm_tuning_import([f"1:{M},{cout},{K},b1,g0|{N},{side},{side},{cin},{cin},3,1,0,0=18,{splits}"])
    for far in (0, 50):
        r = (res + far).bfloat16()
        plain = ops.conv2d(x, w, b, 3, 3, 1, 1, residual=r)
        for silu in (True, False):
            out, y = ops.conv2d(x, w, b, 3, 3, 1, 1, residual=r, gn=(gamma, beta, 32, 1e-5, silu))
            assert torch.equal(out, plain)
            assert off(y, norm64(out, gamma, beta, 32, 1e-5, silu)) < 2 ** -8
    raw = torch.full((N, side, side, cout), 7.0, device="cuda", dtype=torch.bfloat16)
    native.ops().conv2d(x, None, w, raw, b, None, None, None, None, 0, 3, 3, 1, 1, False, 0, 1.0, gn_gamma=gamma, gn_beta=beta,
                        gn_out=torch.empty_like(raw), gn_groups=32, keep_out=False)
    two = side * side * cout // 32 * splits >= 81920
    assert bool((raw == 7).any()) != two


# which folds take two launches: narrow groups of many pixels, wide ones of few, both sides of the border, and no more than 64 workgroups of the one
@pytest.mark.parametrize("N,side,cout,splits,two", [(1, 24, 640, 4, True), (2, 40, 320, 3, True), (2, 16, 960, 12, True), (2, 16, 960, 8, False),
                                                    (1, 12, 2560, 8, False), (2, 20, 1280, 4, False), (3, 16, 1280, 8, False),
                                                    (4, 16, 1280, 8, False), (4, 24, 640, 8, False)])
def test_which_folds_take_two(cuda, N, side, cout, splits, two):
    cin, M = 64, N * side * side
    x, b, gamma, beta = rnd(N, side, side, cin), rnd(cout), rnd(cout), rnd(cout)
    w = rnd(cout, 9 * cin, scale=(9 * cin) ** -0.5)
    native.ops().gemm_tuning_import([f"1:{M},{cout},{9 * cin},b1,g0|{N},{side},{side},{cin},{cin},3,1,0,0=18,{splits}"])
    raw, y = torch.full((N, side, side, cout), 7.0, device="cuda", dtype=torch.bfloat16), torch.empty(N, side, side, cout, device="cuda", dtype=torch.bfloat16)
    native.ops().conv2d(x, None, w, raw, b, None, None, None, None, 0, 3, 3, 1, 1, False, 0, 1.0, gn_gamma=gamma, gn_beta=beta, gn_out=y,
                        gn_groups=32, keep_out=False)
    assert bool((raw == 7).all()) != two     # the one launch leaves the convolution unwritten
    plain = ops.conv2d(x, w, b, 3, 3, 1, 1)
    assert off(y, norm64(plain, gamma, beta, 32, 1e-5, False)) < 2 ** -8
