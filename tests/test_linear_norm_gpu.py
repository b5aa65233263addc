"""A product, its residual and the row norm behind it (ops.linear_norm) against the same in fp32, and the split forms' y against the
separate fold's, bit for bit.

Tolerance: y is rounded to bf16 once (2.3e-3 rms); its norm is taken of the rounded values and rounded again: 2^0.5 of that, 5e-3 with
the statistics' share."""
import pytest
import torch

from shai_amd import ops
from shai_amd.models.layers import LayerNorm, RMSNorm

pytestmark = pytest.mark.gpu


def _rel(a, b):
    a, b = a.float().cpu(), b.float().cpu()
    return ((a - b).norm() / b.norm()).item()


def _norm(kind, n, dev):
    m = (LayerNorm if kind == "layer" else RMSNorm)(n, 1e-6).to(dev)
    m.weight.data.normal_(1.0, 0.2)
    if kind == "layer":
        m.bias.data.normal_(0.0, 0.2)
    return m


def _problem(M, N, K, dev):
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    make = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    return make(M, K).bfloat16(), (make(N, K) / K ** 0.5).bfloat16(), make(N).bfloat16(), make(M, N).bfloat16()


def _want(y, norm):
    y = y.float().cpu()
    if isinstance(norm, RMSNorm):
        return y * torch.rsqrt((y * y).mean(-1, keepdim=True) + norm.eps) * norm.weight.float().cpu()
    return torch.nn.functional.layer_norm(y, y.shape[-1:], norm.weight.float().cpu(), norm.bias.float().cpu(), norm.eps)


# one row, spare lanes in the last chunk, every number of chunks, more parts than are in flight, more than there are K-tiles
@pytest.mark.parametrize("M,N,K", [(1, 8, 512), (3, 264, 512), (32, 1024, 2816), (33, 520, 520), (50, 1280, 640), (197, 768, 3072), (20, 2048, 512)])
@pytest.mark.parametrize("kind", ["layer", "rms"])
@pytest.mark.parametrize("force", [1001, 1003, 1008, 3116, 3216, 3516, 3319])
def test_split_forms(cuda, M, N, K, kind, force):
    if force < 3000 and M > 64:
        pytest.skip("the skinny kernel takes up to 64 rows")
    norm = _norm(kind, N, cuda)
    a, w, b, r = _problem(M, N, K, cuda)
    y, h = (torch.full((M + 1, N), 7.0, device=cuda, dtype=torch.bfloat16) for _ in range(2))
    ops._K().gemm_norm(a, w, y[:M], b, r, norm.weight, getattr(norm, "bias", None), h[:M], norm.eps, kind == "rms", force)
    assert _rel(y[:M], a.float() @ w.float().t() + b.float() + r.float()) < 4e-3
    assert _rel(h[:M], _want(y[:M], norm)) < 5e-3
    assert bool((y[M] == 7).all()) and bool((h[M] == 7).all())
    if force >= 3000:
        apart = torch.empty_like(r)
        ops.gemm_into(a, w, apart, b, residual=r, force_cfg=force)
        assert torch.equal(apart, y[:M])


# the rule: both sides of the largest output, and a width that goes the separate way
@pytest.mark.parametrize("shape,N,K", [((2, 77), 1024, 1024), ((1, 1024), 1024, 256), ((1, 1025), 1024, 256), ((5,), 2056, 256)])
@pytest.mark.parametrize("kind", ["layer", "rms"])
def test_rule(cuda, shape, N, K, kind):
    norm = _norm(kind, N, cuda)
    a, w, b, r = _problem(torch.Size(shape).numel(), N, K, cuda)
    y, h = ops.linear_norm(a.view(*shape, K), w, None, r.view(*shape, N), norm)
    assert y.shape == h.shape == (*shape, N)
    want = (a.float() @ w.float().t() + r.float()).view(*shape, N)
    assert _rel(y, want) < 4e-3 and _rel(h, _want(y, norm)) < 5e-3


# a residual whose rows lie apart (the function goes the separate way, the op folds it as it lies), and one in place of the output
@pytest.mark.parametrize("force", [3216, 1003, 3116])
def test_residuals(cuda, force):
    norm, (a, w, b, r) = _norm("rms", 264, cuda), _problem(33, 264, 512, cuda)
    y, h = torch.empty_like(r), torch.empty_like(r)
    op = lambda y, res: ops._K().gemm_norm(a, w, y, b, res, norm.weight, None, h, norm.eps, True, force)  # noqa: E731
    op(y, r)
    want = y.clone(), h.clone()
    assert _rel(y, a.float() @ w.float().t() + b.float() + r.float()) < 4e-3 and _rel(h, _want(y, norm)) < 5e-3
    wide = torch.full((33, 272), 9.0, device=cuda, dtype=torch.bfloat16)
    wide[:, :264] = r
    for out, res in ((torch.empty_like(r), wide[:, :264]), (r.clone(), None)):
        op(out, out if res is None else res)
        assert torch.equal(out, want[0]) and torch.equal(h, want[1])
    y2, h2 = ops.linear_norm(a, w, b, wide[:, :264], norm)
    assert _rel(y2, want[0]) < 4e-3 and _rel(h2, _want(y2, norm)) < 5e-3
    three = a.view(3, 11, 512).transpose(0, 1)          # an input that is copied first
    y3, h3 = ops.linear_norm(three, w, b, r.view(3, 11, 264).transpose(0, 1).contiguous(), norm)
    assert _rel(y3, want[0].view(3, 11, 264).transpose(0, 1)) < 4e-3 and _rel(h3, _want(y3, norm)) < 5e-3


def test_refusals(cuda):
    a, w, b, r = _problem(16, 64, 64, cuda)
    y, h = torch.empty_like(r), torch.empty_like(r)
    for bad in (dict(w=w[:60]), dict(residual=r[:8]), dict(gamma=b[:8]), dict(y=torch.empty(16, 128, device=cuda, dtype=torch.bfloat16)[:, :64]),
                dict(rms=True), dict(force=1065)):
        args = dict(w=w, y=y, residual=r, gamma=b, rms=False, force=-1, **{}) | bad
        with pytest.raises(RuntimeError, match="gemm_norm"):
            ops._K().gemm_norm(a, args["w"], args["y"], b, args["residual"], args["gamma"], b, h, 1e-5, args["rms"], args["force"])


# what ops.linear refuses (rows that do not begin at 16 bytes) is refused here too, by the op and by the function; what it takes is taken
def test_strides(cuda):
    norm, (a, w, b, r) = _norm("layer", 64, cuda), _problem(16, 64, 512, cuda)
    wide = lambda t, ld: torch.cat([t, t[:, :ld - t.shape[1]]], 1)[:, :t.shape[1]]  # noqa: E731
    y, h = ops.linear_norm(a, w, b, r, norm)
    for x, v in ((wide(a, 520), w), (a, wide(w, 520))):
        y2, h2 = ops.linear_norm(x, v, b, r, norm)
        assert torch.equal(y, y2) and torch.equal(h, h2)
    for x, v in ((wide(a, 514), w), (a, wide(w, 514))):
        for call in (lambda: ops.linear(x, v, b, residual=r), lambda: ops.linear_norm(x, v, b, r, norm),
                     lambda: ops._K().gemm_norm(x, v, y, b, r, norm.weight, norm.bias, h, 1e-6, False, 3216)):
            with pytest.raises(RuntimeError, match="stride not 16B aligned"):
                call()


# rows for which a choice is known by their number of 64-row tiles, or only the plain product's, by its bucket or exactly: that one,
# without a tuning; else one of its own
@pytest.mark.parametrize("M,key,cfg", [(90, 96, "|mbucket=17,2"), (91, 96, "|mbucket=3,1"), (40, 40, "=1000,3"), (150, 192, "|m64|norm=18,2"),
                                       (92, None, None)])
def test_choice_of_the_plain_product(cuda, M, key, cfg):
    N, K = (328, 520) if key else (336, 520)
    name = lambda m: f"0:{m},{N},{K},b1,g0|0,0,0,0,0,0,0,0,0"  # noqa: E731
    if key:
        ops._K().gemm_tuning_import([name(key) + cfg])
    norm, (a, w, b, r) = _norm("rms", N, cuda), _problem(M, N, K, cuda)
    y, h = ops.linear_norm(a, w, b, r, norm)
    assert _rel(y, a.float() @ w.float().t() + b.float() + r.float()) < 4e-3 and _rel(h, _want(y, norm)) < 5e-3
    own = [e.split("=")[1] for e in ops._K().gemm_tuning_export() if e.startswith(name(M)) and "|norm" in e]
    assert len(own) == 1 if key is None else own == (["18,2"] if "m64" in cfg else [])


# up to 64 rows a choice known by their number of 16-row tiles is taken, with the norm and without, and is filed under the rows
@pytest.mark.parametrize("M,tile", [(1, 16), (16, 16), (17, 32), (49, 64), (64, 64)])
def test_choice_by_sixteen_rows(cuda, M, tile):
    N, K = 344, 520
    name = lambda m: f"0:{m},{N},{K},b1,g0|0,0,0,0,0,0,0,0,0"  # noqa: E731
    ops._K().gemm_tuning_import([name(tile) + "|m16=1000,2", name(tile) + "|m16|norm=1000,4"])
    norm, (a, w, b, r) = _norm("rms", N, cuda), _problem(M, N, K, cuda)
    y, h = ops.linear_norm(a, w, b, r, norm)
    want = a.float() @ w.float().t() + b.float() + r.float()
    assert _rel(y, want) < 4e-3 and _rel(h, _want(y, norm)) < 5e-3
    assert _rel(ops.linear(a, w, b, residual=r), want) < 4e-3
    have = ops._K().gemm_tuning_export()
    assert name(M) + "|norm=1000,4" in have and name(M) + "=1000,2" in have
