"""Hooks run on the GPU too, where fused forms stand for most calls (test_module_calls_cpu.py)."""
import pytest
import torch

from shai_amd import ops
from shai_amd.models import t5, unet2d, vit
from shai_amd.models.layers import GroupNorm, LayerNorm, init_random_

pytestmark = pytest.mark.gpu


def _scale(m, a, y):
    return y * torch.linspace(0, 2, y.shape[-1], device=y.device).bfloat16()


@pytest.mark.parametrize("kind", [t5.RMSNorm, t5.RowParallelLinear, t5.T5Block])
def test_t5(cuda, kind):
    m = init_random_(t5.T5EncoderModel(t5.T5Config.tiny()).to(cuda), 1)
    run = lambda: m(torch.arange(12, device=cuda).view(2, 6), lens=torch.tensor([6, 4], dtype=torch.int32, device=cuda))  # noqa: E731
    want, names = run(), [n for n, s in m.named_modules() if isinstance(s, kind)]
    for n in names:
        h = m.get_submodule(n).register_forward_hook(_scale)
        assert not torch.equal(run(), want), n
        h.remove()
    assert names and torch.equal(run(), want)


@pytest.mark.parametrize("of", ["", "vit", "vit.patch", "vit.layers.0", "vit.layers.0.attention", "vit.layers.1.layernorm_before"])
def test_uint8_images(cuda, of):
    from shai_amd.engines.encoders import ImageClassifierEngine
    eng = ImageClassifierEngine(vit.ViTConfig.tiny(), device="cuda:0", seed=1, use_graphs=False)
    x = torch.randint(0, 256, (2, 64, 64, 3), dtype=torch.uint8).cuda()
    want = eng.logits_u8(x)
    h = eng.model.get_submodule(of).register_forward_hook(_scale)
    assert not torch.equal(eng.logits_u8(x), want)
    h.remove()
    assert torch.equal(eng.logits_u8(x), want)


def test_small_images(cuda):
    """A hooked GroupNorm takes the call back from the convolution in front of it; the rest of the pass is unchanged within bf16."""
    m = init_random_(unet2d.UNet2DConditionModel(unet2d.UNetConfig.tiny()).to(cuda), 1)
    x, t, kv = torch.randn(1, 16, 16, 4, device=cuda).bfloat16(), torch.tensor([3.0], device=cuda), None
    kv = m.context_kv(torch.randn(1, 5, 64, device=cuda).bfloat16())
    want = m(x, t, kv).float()
    ran = []
    for n in ("mid_block.attentions.0.norm", "down_blocks.0.attentions.0.norm", "conv_norm_out"):
        s = m.get_submodule(n)
        assert isinstance(s, GroupNorm)
        h = s.register_forward_hook(lambda mod, a, y, n=n: ran.append(n))
        got = m(x, t, kv).float()
        h.remove()
        assert ran and ran[-1] == n and ((got - want).norm() / want.norm()).item() < 2e-2


def _at(t, elements):
    """``t`` at an address so many elements behind an aligned one."""
    room = torch.empty(t.numel() + 16, dtype=t.dtype, device=t.device)
    v = room[elements:elements + t.numel()].view(t.shape)
    v.copy_(t)
    return v


def test_parameters_at_other_addresses(cuda):
    """Norms and tokens take parameters at any address of 4 bytes, as views of one large buffer are: by the kernels that ask for none."""
    torch.manual_seed(0)
    rnd = lambda *s: torch.randn(*s, device=cuda).bfloat16()      # noqa: E731
    a, w, r, ln = rnd(40, 256), rnd(64, 256) / 16, rnd(40, 64), LayerNorm(64).to(cuda)
    gn, img = GroupNorm(8, 64).to(cuda), rnd(2, 9, 9, 64)
    args = (rnd(2, 6, 64), rnd(1, 1, 64), rnd(1, 3, 64), rnd(1, 10, 64))
    for m in (ln, gn):
        m.weight.data, m.bias.data = rnd(64), rnd(64)
    assert gn.one_ok(img, 81, 64)
    want = *ops.linear_norm(a, w, None, r, ln), gn(img, silu=True), ops.tokens(*args)[0]
    ln.weight.data, gn.bias.data = _at(ln.weight.data, 4), _at(gn.bias.data, 2)
    assert not gn.one_ok(img, 81, 64)
    got = *ops.linear_norm(a, w, None, r, ln), gn(img, silu=True), ops.tokens(args[0], _at(args[1], 2), *args[2:])[0]
    for x, y in zip(got, want):      # other kernels: the sums of another order, rounded to bf16
        assert ((x.float() - y.float()).norm() / y.float().norm()).item() < 5e-3
