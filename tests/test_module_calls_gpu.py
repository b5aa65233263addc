"""Hooks run on the GPU too, where fused forms stand for most calls (test_module_calls_cpu.py)."""
import pytest
import torch

from shai_amd.models import t5, unet2d, vit
from shai_amd.models.layers import GroupNorm, init_random_

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
