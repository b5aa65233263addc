"""Small tiles with a deep ring (csrc/kernels/gemm_deep.hip) against fp32 PyTorch, each config forced.

Tolerance: inputs are bf16, sums fp32, outputs rounded to bf16 once: a relative error of at most 2^-8 / sqrt(3) rms = 2.3e-3; 4e-3
leaves room for the activations' approximations and the residual's cancellation."""
import os
import subprocess
import sys

import pytest
import torch

from shai_amd import ops

pytestmark = pytest.mark.gpu
CFGS = [16, 17, 18]                      # 64 x 64 and 128 x 64 with waves along K, 128 x 128
TOL = 4e-3


def _rel(a, b):
    a, b = a.float().cpu(), b.float().cpu()
    return ((a - b).norm() / b.norm()).item()


def _problem(M, N, K, dev):
    torch.manual_seed(M + N + K)
    a = torch.randn(M, K, device=dev).bfloat16()
    w = (torch.randn(N, K, device=dev) / K ** 0.5).bfloat16()
    return a, w, torch.randn(N, device=dev).bfloat16(), torch.randn(M, N, device=dev).bfloat16()


# one row and column, edges of every tile, K below one K-tile, fewer K-tiles than the ring holds, a K tail
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (64, 64, 64), (65, 63, 72), (127, 129, 128), (129, 128, 192), (197, 768, 776),
                                   (512, 1280, 1280), (1000, 200, 2816)])
@pytest.mark.parametrize("cfg", CFGS)
def test_bias_residual(cuda, M, N, K, cfg):
    a, w, b, r = _problem(M, N, K, cuda)
    out = torch.full((M + 1, N), 7.0, device=cuda, dtype=torch.bfloat16)
    ops.gemm_into(a, w, out[:M], b, residual=r, force_cfg=cfg)
    assert _rel(out[:M], a.float() @ w.float().t() + b.float() + r.float()) < TOL
    assert bool((out[M] == 7).all())


@pytest.mark.parametrize("splits", [2, 3, 8])
@pytest.mark.parametrize("cfg", CFGS)
def test_split_k(cuda, splits, cfg):
    a, w, b, r = _problem(197, 330, 1544, cuda)
    out = torch.empty_like(r)
    ops.gemm_into(a, w, out, b, act="gelu", residual=r, force_cfg=3000 + 100 * splits + cfg)
    assert _rel(out, torch.nn.functional.gelu(a.float() @ w.float().t() + b.float()) + r.float()) < TOL


@pytest.mark.parametrize("act", ["silu", "gelu", "gelu_tanh"])
@pytest.mark.parametrize("cfg", CFGS)
def test_glu(cuda, act, cfg):
    a, w, b, _ = _problem(77, 2 * 148, 320, cuda)
    out = torch.empty(77, 148, device=cuda, dtype=torch.bfloat16)
    ops.gemm_into(a, w, out, b, act=act, glu=True, force_cfg=cfg)
    y = a.float() @ w.float().t() + b.float()
    f = {"silu": torch.nn.functional.silu, "gelu": torch.nn.functional.gelu,
         "gelu_tanh": lambda t: torch.nn.functional.gelu(t, approximate="tanh")}[act]
    assert _rel(out, y[:, 0::2] * f(y[:, 1::2])) < TOL


@pytest.mark.parametrize("cfg", CFGS)
def test_batched_strided(cuda, cfg):
    a = torch.randn(3, 100, 256, device=cuda).bfloat16()
    w = (torch.randn(136, 256, device=cuda) / 16).bfloat16()
    j = torch.zeros(3, 110, 136, device=cuda).bfloat16()
    ops.gemm_into(a, w, j[:, 10:], force_cfg=cfg)
    assert _rel(j[:, 10:], a.float() @ w.float().t()) < TOL and j[:, :10].abs().sum().item() == 0


# widths where a lane's 8 columns are whole, cut by 4 or by single ones, and rows whose stride allows 16-byte, 8-byte or 2-byte
# accesses only: columns beside the output stay as they were
@pytest.mark.parametrize("N,ld,glu", [(128, 136, False), (132, 136, False), (132, 132, False), (72, 76, False), (70, 72, False),
                                      (330, 338, False), (128, 136, True), (132, 68, True), (140, 74, True), (68, 34, True)])
@pytest.mark.parametrize("cfg", [3, 4] + CFGS)
def test_epilogue_widths(cuda, cfg, N, ld, glu):
    M, K, n = 131, 128, N // (2 if glu else 1)
    a, w, b, _ = _problem(M, N, K, cuda)
    r = torch.randn(M, ld, device=cuda).bfloat16()[:, :n]
    gate = torch.randn(3, ld, device=cuda).bfloat16()[:, :n]
    per_image = torch.randn(2, N, device=cuda).bfloat16()
    out = torch.full((M, ld), 7.0, device=cuda, dtype=torch.bfloat16)
    ops._K().gemm(a, w, out[:, :n], b, per_image, 100, r, 0.5, 2.0, ops.act_id("silu"), glu, gate, 50, cfg)
    y = 0.5 * (a.float() @ w.float().t()) + b.float() + per_image.float().repeat_interleave(100, 0)[:M]
    y = y[:, 0::2] * torch.nn.functional.silu(y[:, 1::2]) if glu else torch.nn.functional.silu(y)
    assert _rel(out[:, :n], y * gate.float().repeat_interleave(50, 0)[:M] + 2.0 * r.float()) < TOL
    assert bool((out[:, n:] == 7).all())


# a folded LayerNorm at a cut row tile, column tails of 4 and fewer; the product of the normalised rows comes out as the
# difference of two larger terms, in fp32
@pytest.mark.parametrize("M,N,K", [(1, 64, 64), (131, 132, 128), (197, 330, 776), (300, 768, 768)])
@pytest.mark.parametrize("cfg", [0, 1, 2, 3, 4] + CFGS)
def test_folded_layernorm(cuda, cfg, M, N, K):
    a, w, b, r = _problem(M, N, K, cuda)
    mean, rstd, s = torch.randn(M, device=cuda), torch.rand(M, device=cuda) + 0.5, w.float().sum(1)
    out = torch.empty_like(r)
    ops._K().gemm(a, w, out, b, None, 1, r, 1.0, 1.0, ops.act_id("gelu"), False, None, 1, cfg, -1.0, None,
                  torch.stack([mean, rstd], 1).contiguous(), s)
    y = rstd[:, None] * (a.float() @ w.float().t() - mean[:, None] * s) + b.float()
    assert _rel(out, torch.nn.functional.gelu(y) + r.float()) < TOL


# K parts and their fold do not know a LayerNorm: a forced split is refused; the W-stationary kernel runs whole whatever is asked
@pytest.mark.parametrize("cfg", [0, 1, 2, 3, 4, 9, 10] + CFGS)
def test_folded_layernorm_is_not_split(cuda, cfg):
    a, w, b, _ = _problem(300, 640, 320, cuda)
    mr = torch.stack([torch.randn(300, device=cuda), torch.rand(300, device=cuda) + 0.5], 1)
    s, y = w.float().sum(1), torch.empty(300, 640, device=cuda, dtype=torch.bfloat16)
    run = lambda force: ops._K().gemm(a, w, y, b, None, 1, None, 1.0, 1.0, 0, False, None, 1, force, -1.0, None, mr, s)
    with pytest.raises(RuntimeError, match="runs unsplit"):
        run(3200 + cfg)
    want = mr[:, 1:] * (a.float() @ w.float().t() - mr[:, :1] * s) + b.float()
    for force in (3100 + cfg, 3215):
        y.zero_()
        run(force)
        assert _rel(y, want) < TOL


CONV_SCRIPT = r"""
import sys, torch
sys.path.insert(0, {root!r})
import shai_amd.ops as ops
from shai_amd.ops import reference as ref
torch.manual_seed(0)
# images, side, channels, outputs, kernel, stride, padding, upsampled, channels of a second source
cases = [(2, 8, 1280, 1280, 3, 1, 1, False, 0), (1, 16, 64, 96, 3, 2, 1, False, 0), (2, 8, 128, 64, 3, 1, 1, True, 0),
         (2, 7, 64, 64, 1, 1, 0, False, 0), (1, 9, 64, 128, 3, 1, 1, False, 192), (2, 8, 640, 320, 3, 1, 1, True, 640),
         (1, 9, 64, 64, 5, 2, 2, False, 64), (1, 10, 64, 64, 6, 1, 0, False, 0), (2, 7, 128, 32, 3, 1, 3, False, 0),
         (2, 16, 96, 64, 3, 1, 1, False, 0)]  # the last: 96 channels, which these configs do not take
worst = 0.0
for N, H, C, Co, k, stride, pad, up, c2 in cases:
    x = torch.randn(N, H, H, C, device="cuda").bfloat16()
    x2 = torch.randn(N, H, H, c2, device="cuda").bfloat16() if c2 else None
    w = ops.pack_conv_weight((torch.randn(Co, C + c2, k, k, device="cuda") / ((C + c2) * k * k) ** 0.5).bfloat16())
    b = torch.randn(Co, device="cuda").bfloat16()
    y = ops.conv2d(x, w, b, k, k, stride, pad, upsample=up, x2=x2, act="silu")
    want = ref.conv2d(x.cpu(), w.cpu(), b.cpu(), k, k, stride, pad, upsample=up, x2=None if x2 is None else x2.cpu(), act="silu").float()
    worst = max(worst, ((y.float().cpu() - want).norm() / want.norm()).item())
print("WORST", worst)
assert worst < {tol}, worst
"""


@pytest.mark.parametrize("splits", [1, 4])
@pytest.mark.parametrize("cfg", [0, 2, 3, 4] + CFGS)    # 6 x 6 taps are more than a lane's mask holds
def test_conv(cuda, cfg, splits):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, SHAI_GEMM_FORCE=str(cfg), SHAI_GEMM_FORCE_SPLITS=str(splits))
    r = subprocess.run([sys.executable, "-c", CONV_SCRIPT.format(root=root, tol=TOL)], env=env, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-3000:]
