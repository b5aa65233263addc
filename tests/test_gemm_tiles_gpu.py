"""Tiles with two groups of waves along K (gemm_deep.hip), and tiles that the rows end in (gemm_8ph.hip, gemm_w4.hip), against fp32
PyTorch, each config forced.

Tolerance: inputs are bf16, sums fp32, outputs rounded to bf16 once: a relative error of at most 2^-8 / sqrt(3) rms = 2.3e-3; 4e-3
leaves room for the activations' approximations and the residual's cancellation."""
import os
import subprocess
import sys

import pytest
import torch

from shai_amd import ops
from test_gemm_deep_gpu import CONV_SCRIPT

pytestmark = pytest.mark.gpu
GROUPS = [16, 17, 18, 19, 20, 21]        # 64 x 64, 128 x 64, 128 x 128; 192 x 128 and 128 x 128 with two wave groups, 192 x 128 two to a CU
WHOLE = [9, 10, 11, 12, 13]              # eight phases (256 and 320 wide, persistent), four waves
ACTS = {None: lambda t: t, "silu": torch.nn.functional.silu, "gelu": torch.nn.functional.gelu,
        "gelu_tanh": lambda t: torch.nn.functional.gelu(t, approximate="tanh")}
TOL = 4e-3


def _close(a, b):
    a, b = a.float().cpu(), b.float().cpu()
    return ((a - b).norm() / b.norm()).item() < TOL


def _problem(M, N, K, dev):
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    make = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    return make(M, K).bfloat16(), (make(N, K) / K ** 0.5).bfloat16(), make(N).bfloat16(), make(M, N).bfloat16()


# M: one row, a tile's edges, a second tile of one row; N: inside a tile, and whole tiles; K: fewer K-tiles than the ring holds
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (129, 63, 72), (192, 128, 64), (193, 256, 192), (257, 330, 776), (511, 640, 1280)])
@pytest.mark.parametrize("cfg", GROUPS + WHOLE)
def test_in_place_residual(cuda, M, N, K, cfg):
    a, w, b, r = _problem(M, N, K, cuda)
    want = a.float() @ w.float().t() + b.float() + r.float()
    out = torch.full((M + 1, N), 7.0, device=cuda, dtype=torch.bfloat16)
    out[:M] = r
    ops.gemm_into(a, w, out[:M], b, residual=out[:M], force_cfg=cfg)
    assert _close(out[:M], want)
    assert bool((out[M] == 7).all())


@pytest.mark.parametrize("M", [100, 300, 513])
@pytest.mark.parametrize("act", ["silu", "gelu", "gelu_tanh"])
@pytest.mark.parametrize("cfg", GROUPS + WHOLE)
def test_glu(cuda, M, act, cfg):
    a, w, b, _ = _problem(M, 1280, 320, cuda)
    out = torch.full((M + 1, 640), 7.0, device=cuda, dtype=torch.bfloat16)
    ops.gemm_into(a, w, out[:M], b, act=act, glu=True, force_cfg=cfg)
    y = a.float() @ w.float().t() + b.float()
    assert _close(out[:M], y[:, 0::2] * ACTS[act](y[:, 1::2]))
    assert bool((out[M] == 7).all())


@pytest.mark.parametrize("cfg", GROUPS + WHOLE[:4])
def test_folded_layernorm(cuda, cfg):
    M, N, K = 300, 640, 768
    a, w, b, _ = _problem(M, N, K, cuda)
    mean, rstd, s = torch.randn(M, device=cuda), torch.rand(M, device=cuda) + 0.5, w.float().sum(1)
    out = torch.empty(M, N, device=cuda, dtype=torch.bfloat16)
    ops._K().gemm(a, w, out, b, None, 1, None, 1.0, 1.0, ops.act_id("gelu"), False, None, 1, cfg, -1.0, None,
                  torch.stack([mean, rstd], 1).contiguous(), s)
    assert _close(out, ACTS["gelu"](rstd[:, None] * (a.float() @ w.float().t() - mean[:, None] * s) + b.float()))


# rows of a time embedding: the last tile's rows lie in the last image, whose row is the last there is
@pytest.mark.parametrize("cfg", WHOLE)
def test_rows_of_images(cuda, cfg):
    M, N, K = 384, 1280, 128
    a, w, b, r = _problem(M, N, K, cuda)
    per_image = torch.randn(3, N, device=cuda).bfloat16()
    out = torch.empty_like(r)
    ops._K().gemm(a, w, out, b, per_image, 128, r, 0.5, 2.0, ops.act_id("silu"), False, None, 1, cfg)
    y = 0.5 * (a.float() @ w.float().t()) + b.float() + per_image.float().repeat_interleave(128, 0)
    assert _close(out, ACTS["silu"](y) + 2.0 * r.float())


@pytest.mark.parametrize("cfg", [19, 20])
def test_wave_groups_up_to_8192_rows(cuda, cfg):
    a, w, b, r = _problem(8193, 64, 64, cuda)
    out = torch.empty_like(r)
    with pytest.raises(RuntimeError, match="bad force_cfg"):
        ops.gemm_into(a, w, out, b, force_cfg=cfg)
    ops.gemm_into(a[:8192], w, out[:8192], b, force_cfg=cfg)
    assert _close(out[:8192], a[:8192].float() @ w.float().t() + b.float())


@pytest.mark.parametrize("splits", [2, 5])
@pytest.mark.parametrize("cfg", GROUPS)
def test_split_k(cuda, splits, cfg):
    a, w, b, r = _problem(197, 330, 1544, cuda)
    out = torch.empty_like(r)
    ops.gemm_into(a, w, out, b, act="gelu", residual=r, force_cfg=3000 + 100 * splits + cfg)
    assert _close(out, ACTS["gelu"](a.float() @ w.float().t() + b.float()) + r.float())


@pytest.mark.parametrize("splits", [1, 4])
@pytest.mark.parametrize("cfg", GROUPS)
def test_convolution(cuda, cfg, splits):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, SHAI_GEMM_FORCE=str(cfg), SHAI_GEMM_FORCE_SPLITS=str(splits))
    r = subprocess.run([sys.executable, "-c", CONV_SCRIPT.format(root=root, tol=TOL)], env=env, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-3000:]


# counts of parts that are no powers of two, 45 k-tiles: 15, 9, 7 and 3, and 4 with a last part of one
@pytest.mark.parametrize("splits", [3, 5, 7, 12, 15])
@pytest.mark.parametrize("cfg", [0, 1, 2, 3, 4, 9, 10, 11, 12] + GROUPS)
def test_convolution_in_parts(cuda, cfg, splits):
    g = torch.Generator(device=cuda).manual_seed(splits)
    make = lambda *s: torch.randn(*s, generator=g, device=cuda)  # noqa: E731
    x, w4, b, r = make(2, 9, 11, 320).bfloat16(), (make(328, 320, 3, 3) / 2880 ** 0.5).bfloat16(), make(328).bfloat16(), make(2, 9, 11, 328).bfloat16()
    ops._K().gemm_tuning_import([f"1:198,328,2880,b1,g0|2,9,11,320,320,3,1,0,0={cfg},{splits}"])
    y = ops.conv2d(x, ops.pack_conv_weight(w4), b, 3, 3, 1, 1, residual=r)
    want = torch.nn.functional.conv2d(x.double().permute(0, 3, 1, 2).cpu(), w4.double().cpu(), b.double().cpu(), padding=1).permute(0, 2, 3, 1)
    assert _close(y, want + r.double().cpu())


# products that keep one order of sums (packed prompts): every tile that they may take gives the same bits, the others are refused
@pytest.mark.parametrize("N,K,glu", [(512, 1024, False), (320, 320, False), (1536, 776, False), (1024, 512, True)])
def test_one_order(cuda, N, K, glu):
    M = 4100
    a, w, _, _ = _problem(M, N, K, cuda)
    r = torch.randn(M, N // 2 if glu else N, device=cuda).bfloat16()
    run = lambda rows, cfg: ops._K().gemm(a[:rows], w, y[:rows], None, None, 1, r[:rows], 1.0, 1.0, ops.act_id("silu" if glu else None), glu,  # noqa: E731
                                          force_cfg=cfg, one_order=True)
    y, seen = torch.empty_like(r), {}
    for cfg in range(22):
        try:
            run(M, cfg)
        except RuntimeError as e:
            assert "bad force_cfg" in str(e)
            continue
        seen[cfg] = y.clone()
    assert {0, 3, 9, 12, 18, 21} <= set(seen) and not {16, 17, 19, 20} & set(seen)
    for cfg, out in seen.items():
        assert torch.equal(out, seen[3]), cfg
    for cfg in (16, 19):                  # fewer rows: any tile
        run(4095, cfg)
    for cfg in (3203, 3410):              # and no split where the rows keep the order
        run(M, cfg)
        assert torch.equal(y, seen[3])


@pytest.mark.parametrize("N,K,glu,rms", [(512, 1024, False, None), (768, 512, False, 1e-5), (2048, 512, True, 1e-5)])
def test_rows_do_not_depend_on_how_many(cuda, N, K, glu, rms):
    """Rows of a packed prompt beside few others and many, on both sides of the sizes where tiles change; also where the shipped or an
    earlier choice for the rows cuts K."""
    a, w, _, _ = _problem(16000, N, K, cuda)
    call = lambda rows: ops.linear(a[:rows], w, act="silu" if glu else None, glu=glu, rms_eps=rms, one_order=True)  # noqa: E731
    for rows, choice in ((4096, "19,1"), (4864, "10,4"), (9364, "3,2"), (16000, "17,1")):
        ops._K().gemm_tuning_import([f"0:{rows},{N},{K},b1,g{int(glu)}|0,0,0,0,0,0,0,0,0{t}={choice}" for t in ("", "|lib")])
    want = call(16000)
    for rows in (4096, 4864, 9364):
        assert torch.equal(call(rows), want[:rows])


# four waves of 128 x 128 and of 128 x 96: columns that end inside the tile (by eights, and not), in a wave's first and second half; the
# latter's folded LayerNorm, whose factors the products' sums take before bias and activation
@pytest.mark.parametrize("act,glu", [(None, False), ("gelu", False), ("gelu_tanh", True)])
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (257, 192, 64), (255, 200, 72), (130, 388, 128), (513, 456, 776)])
@pytest.mark.parametrize("cfg", [13, 14])
def test_four_waves(cuda, cfg, M, N, K, act, glu):
    if glu and N % 8:
        pytest.skip("gated widths are multiples of 8")
    a, w, b, r = _problem(M, N, K, cuda)
    no = N // 2 if glu else N
    r = r[:, :no].contiguous()
    f = (lambda y: y[:, 0::2] * ACTS[act](y[:, 1::2])) if glu else ACTS[act]
    y = a.float() @ w.float().t()
    out = torch.full((M + 1, no), 7.0, device=cuda, dtype=torch.bfloat16)
    out[:M] = r
    ops.gemm_into(a, w, out[:M], b, act=act, residual=out[:M], glu=glu, force_cfg=cfg)
    assert _close(out[:M], f(y + b.float()) + r.float()) and bool((out[M] == 7).all())
    if cfg == 13:
        return
    g = torch.Generator(device=cuda).manual_seed(N)
    mr, s = torch.rand(M, 2, generator=g, device=cuda) + 0.5, torch.randn(N, generator=g, device=cuda)
    ops._K().gemm(a, w, out[:M], b, None, 1, r, 1.0, 1.0, ops.act_id(act), glu, None, 1, cfg, -1.0, None, mr, s)
    assert _close(out[:M], f(mr[:, 1:] * (y - mr[:, :1] * s) + b.float()) + r.float()) and bool((out[M] == 7).all())
