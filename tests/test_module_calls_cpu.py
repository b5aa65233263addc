"""Blocks of the encoders and the UNet as modules: a call of one takes and returns what it always did, and what hooks into a call runs
although fused forms stand for most of them."""
import pytest
import torch

from shai_amd.models import clip, t5, unet2d, vit
from shai_amd.models.attention import CrossAttention
from shai_amd.models.layers import LayerNorm, Linear, init_random_
from shai_amd.utils import calls as module_calls
from shai_amd.utils.calls import as_called, then_norm


def _rand(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).bfloat16()


def _clip():
    m = clip.CLIPTextModel(clip.CLIPTextConfig(vocab_size=100, hidden_size=64, intermediate_size=128, num_hidden_layers=2, num_attention_heads=2))
    return m, lambda: m(torch.arange(12).view(2, 6))


def _t5():
    m = t5.T5EncoderModel(t5.T5Config.tiny())
    return m, lambda: m(torch.arange(12).view(2, 6), lens=torch.tensor([6, 4], dtype=torch.int32))


def _vit(**kw):
    m = vit.ViTEncoderModel(vit.ViTConfig.tiny())
    return m, lambda: m(_rand(1, 64, 64, 3), **kw)


def _unet():
    m = unet2d.UNet2DConditionModel(unet2d.UNetConfig.tiny())
    return m, lambda: m(_rand(1, 16, 16, 4), torch.tensor([3.0]), m.context_kv(_rand(1, 5, 64, seed=1)))


MODELS = {"clip": _clip, "t5": _t5, "vit": _vit, "vit_cls": lambda: _vit(cls_only=True), "unet": _unet}


def _names(model, *kinds):
    return [n for n, m in model.named_modules() if isinstance(m, kinds)]


@pytest.mark.parametrize("name", MODELS)
def test_hooks_run_and_change_nothing_else(name, monkeypatch):
    """A hook on any block, attention, MLP, product or LayerNorm / RMSNorm that the forward pass reaches by a call of the module without
    fused forms is run by the pass with them, with the same input and output."""
    model, run = MODELS[name]()
    init_random_(model, 1)
    want = run()
    kinds = (Linear, LayerNorm, t5.RMSNorm, t5.RowParallelLinear, clip.CLIPMLP, clip.CLIPEncoderLayer, t5.T5Block, vit.ViTLayer, CrossAttention,
             vit.FusedSelfAttention, unet2d.BasicTransformerBlock)
    calls, seen = {}, {}

    def record(into):
        return [m.register_forward_hook(lambda mod, a, y, n=n: into.setdefault(n, []).append((a[0].clone(), y.clone())))
                for n, m in model.named_modules() if isinstance(m, kinds)]
    with monkeypatch.context() as mp:      # nothing fused: the calls that there are
        mp.setattr(module_calls, "as_called", lambda *a: False)
        mp.setattr(vit, "as_called", lambda *a: False)
        handles = record(calls)
        assert torch.equal(run(), want)
        for h in handles:
            h.remove()
    assert any("norm" in n or "ln_" in n for n in calls) and len(calls) >= 8
    handles = record(seen)
    assert torch.equal(run(), want)
    for h in handles:
        h.remove()
    assert seen.keys() == calls.keys()
    for n in calls:
        assert len(seen[n]) == len(calls[n])
        for (a, y), (a2, y2) in zip(calls[n], seen[n]):
            assert torch.equal(a, a2) and torch.equal(y, y2), n


@pytest.mark.parametrize("name,kind", [("t5", t5.RMSNorm), ("clip", LayerNorm), ("vit", Linear), ("t5", t5.RowParallelLinear), ("clip", clip.CLIPEncoderLayer),
                                       ("vit", vit.FusedSelfAttention)])
def test_one_hook_alone(name, kind):
    """Every module of a kind by itself: its hook's output is what the pass goes on with."""
    model, run = MODELS[name]()
    init_random_(model, 1)
    want = run()
    for n in _names(model, kind):
        h = model.get_submodule(n).register_forward_hook(lambda m, a, y: y * torch.linspace(0, 2, y.shape[-1]).bfloat16())
        assert not torch.equal(run(), want), n
        h.remove()
    assert torch.equal(run(), want)


def test_calls_of_blocks():
    x, lens, bias = _rand(2, 6, 64), torch.tensor([6, 3], dtype=torch.int32), torch.zeros(2, 6, 6).bfloat16()
    layer = init_random_(_clip()[0], 2).layers[0]
    assert layer(x).shape == x.shape and not torch.equal(layer(x), layer(x, kv_lens=lens))
    assert layer.mlp(x, x).shape == x.shape
    block = init_random_(t5.T5EncoderModel(t5.T5Config.tiny()), 2).blocks[0]
    y = _rand(2, 6, 128)
    assert block(y, bias, lens).shape == y.shape
    v = init_random_(vit.ViTEncoderModel(vit.ViTConfig.tiny()), 2).layers[0]
    assert v(x).shape == x.shape and torch.equal(v.forward_cls(x), v.forward_cls(x, n=v.layernorm_before(x)))
    cross = init_random_(CrossAttention(64, 32, 2), 2)
    kv = cross.context_kv(_rand(2, 6, 32))
    got, cut = cross(x, kv, residual=x, kv_lens=lens), cross(x[1:], kv[1:, :3], residual=x[1:])
    assert torch.equal(got[1:], cut) and not torch.equal(got, cross(x, kv, residual=x))


def test_what_is_not_a_plain_call():
    class Other(Linear):
        def forward(self, x, residual=None):
            return super().forward(x, residual=residual) + 1

    lin, norm, x = init_random_(Linear(64, 64), 1), LayerNorm(64), _rand(3, 64)
    assert as_called(lin, norm) and not as_called(Other(64, 64))
    other = Other(64, 64)
    other.load_state_dict(lin.state_dict())
    y, n = then_norm(other, norm, x, residual=x)
    assert torch.equal(y, lin(x, residual=x) + 1) and torch.equal(n, norm(y))
    norm.forward = lambda x: x
    assert not as_called(norm)
    handle = torch.nn.modules.module.register_module_forward_hook(lambda m, a, y: None)
    try:
        assert not as_called(lin)
    finally:
        handle.remove()
    assert as_called(lin)
