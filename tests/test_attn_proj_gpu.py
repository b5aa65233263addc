"""Attention of short sequences with its output projection and the next norm, in two launches, against fp64."""
import pytest
import torch

from shai_amd import ops
from shai_amd.models.layers import LayerNorm, RMSNorm

pytestmark = pytest.mark.gpu


def problem(cuda, B, Sq, Skv, H, N, causal, bias, lens, rms, seed=0):
    g = torch.Generator(device=cuda).manual_seed(seed + Sq + Skv)
    rand = lambda *s: torch.randn(*s, generator=g, device=cuda).bfloat16()
    qkv = rand(B, max(Sq, Skv), 3 * H * 64)
    q, k, v = (t.view(B, -1, H, 64) for t in qkv.split(H * 64, -1))
    norm = (RMSNorm(N, 1e-6) if rms else LayerNorm(N, 1e-5)).to(cuda)
    with torch.no_grad():
        norm.weight.copy_(rand(N))
        if not rms:
            norm.bias.copy_(rand(N))
    kw = dict(scale=1.0 if bias else None, causal=causal, attn_bias=rand(H, Sq, Skv) if bias else None,
              kv_lens=torch.tensor(lens, dtype=torch.int32, device=cuda) if lens else None)
    w, b = (torch.randn(N, H * 64, generator=g, device=cuda) / (8 * H ** 0.5)).bfloat16(), None if bias else rand(N)
    q = q * 0.25 if bias else q      # scores of a scale of 1
    return (q[:, :Sq], k[:, :Skv], v[:, :Skv], w, b, rand(B, Sq, N), norm), kw


def wanted(args, kw):
    """y in fp64; attention's output rounded to bf16, as it is between the two products."""
    q, k, v, w, b, res, _ = args
    s = torch.einsum("bqhd,bkhd->bhqk", q.double(), k.double()) * (kw["scale"] or 0.125)
    if kw["attn_bias"] is not None:
        s = s + kw["attn_bias"].double()
    key = torch.arange(k.shape[1], device=q.device)
    if kw["kv_lens"] is not None:
        s = s.masked_fill(key >= kw["kv_lens"].view(-1, 1, 1, 1), float("-inf"))
    if kw["causal"]:
        s = s.masked_fill(key > torch.arange(q.shape[1], device=q.device)[:, None], float("-inf"))
    o = torch.einsum("bhqk,bkhd->bqhd", torch.nan_to_num(torch.softmax(s, -1)), v.double())
    y = o.flatten(2).bfloat16().double() @ w.double().T + res.double()
    return y if b is None else y + b.double()


@pytest.mark.parametrize("B,Sq,Skv,H,N,causal,bias,lens,rms", [
    (1, 1, 1, 1, 16, False, False, None, False),             # one query, one key, one tile of columns
    (1, 32, 32, 16, 1024, False, True, [29], True),
    (2, 17, 17, 2, 272, False, True, [17, 0], True),         # rows of the bias at any address; a sequence without keys
    (2, 77, 77, 16, 1024, True, False, None, False),
    (1, 64, 65, 3, 784, False, False, None, False),          # columns that end in a workgroup's second tile
    (3, 65, 64, 2, 256, True, False, [64, 5, 33], False),    # a second block of queries with one row
    (1, 128, 128, 4, 512, False, True, [128], True),
    (1, 197, 197, 12, 768, False, False, None, False),
    (1, 60, 256, 4, 320, False, True, [251], False)])
def test_attention_linear_norm(cuda, monkeypatch, B, Sq, Skv, H, N, causal, bias, lens, rms):
    """P is bf16 (2^-9 of a value each, averaged over the keys), attention's output and y are; the products' sums are fp32."""
    args, kw = problem(cuda, B, Sq, Skv, H, N, causal, bias, lens, rms)
    assert ops._attention_linear_fits(*args, kw["attn_bias"])
    seen = []
    monkeypatch.setattr(ops, "linear_norm", lambda *a, **k: seen.append(a))   # the general path is not taken
    y, n = ops.attention_linear_norm(*args, **kw)
    assert not seen
    want = wanted(args, kw)
    assert (y.double() - want).norm() <= 2 ** -8 * want.norm()
    assert torch.equal(n, args[-1](y)) or (n.double() - args[-1](y).double()).norm() <= 2 ** -8 * n.double().norm()


def test_what_does_not_fit_takes_the_general_path(cuda):
    """More partial sums than pay, heads that lie apart (refused, as attention refuses them), a weight whose rows are not 16 bytes apart, norm
    parameters at odd addresses."""
    args, kw = problem(cuda, 2, 33, 33, 4, 256, False, False, None, False)
    q, k, v, w, b, res, norm = args
    odd = LayerNorm(256).to(cuda)
    odd.weight = torch.nn.Parameter(torch.randn(257, device=cuda).bfloat16()[1:], requires_grad=False)
    apart = torch.randn(2, 33, 4, 128, device=cuda).bfloat16()[..., :64]
    long = problem(cuda, 8, 64, 64, 16, 1024, False, False, None, False)[0]
    wide = (torch.randn(256, 260, device=cuda) * 0.05).bfloat16()[:, :256]
    assert ops._attention_linear_fits(*args, None)
    for a in (long, (q, k, v, w, b, res, odd), (apart, apart, apart, w, b, res, norm), (q, k, v, wide, b, res, norm)):
        assert not ops._attention_linear_fits(*a, None)
    with pytest.raises(RuntimeError, match="packed"):
        ops.attention_linear_norm(apart, apart, apart, w, b, res, norm)
    for a in (long, (q, k, v, w, b, res, odd)):
        want = wanted(a, kw)
        y, n = ops.attention_linear_norm(*a)
        assert (y.double() - want).norm() <= 2 ** -8 * want.norm()
        assert (n.double() - a[-1](y).double()).norm() <= 2 ** -8 * n.double().norm()


def test_what_attention_takes_is_not_refused(cuda):
    """A bias with a batch dimension of one and lengths of more sequences than there are, which attention takes: the general path."""
    args, kw = problem(cuda, 2, 33, 33, 4, 256, False, True, [20, 33], True)
    want = wanted(args, kw)
    bias, lens = kw["attn_bias"], kw["kv_lens"]
    assert ops._attention_linear_fits(*args, bias) and not ops._attention_linear_fits(*args, bias[None])
    for change in (dict(attn_bias=bias[None]), dict(kv_lens=torch.cat([lens, lens]))):
        y, n = ops.attention_linear_norm(*args, **{**kw, **change})
        assert (y.double() - want).norm() <= 2 ** -8 * want.norm()
        assert (n.double() - args[-1](y).double()).norm() <= 2 ** -8 * n.double().norm()
