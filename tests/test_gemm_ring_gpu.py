"""Decode products through a ring in LDS (csrc/lm/gemm_ring.hip) against fp64, at the borders of its rule and of its tiles.

Tolerances, relative 2-norms: fp32 sums of bf16 products 1e-5; one rounding to bf16 (an error spread evenly over
half a unit in the last of 8 bits) at most 2^-8 / sqrt(3) = 2.3e-3."""
import pytest
import torch

from shai_amd.ops import lm

pytestmark = pytest.mark.gpu


def _rel(a, b):
    a, b = a.double().cpu(), b.double().cpu()
    return ((a - b).norm() / b.norm()).item()


def _problem(M, N, K, dev, spare=0):
    g = torch.Generator(device=dev).manual_seed(M * 7 + N + K)
    a = torch.randn(M + 2, K + spare, generator=g, device=dev).bfloat16()[1:M + 1, :K]     # neighbours must not matter
    return a, (torch.randn(N, K, generator=g, device=dev) / K ** 0.5).bfloat16()


# one row more and less than a block, a half, all rows; columns of every workgroup width, ragged ones, more than one round;
# K of a few stages, with half a stage at the end
@pytest.mark.parametrize("M", [9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(512, 512), (516, 576), (8256, 640), (14628, 1088), (17424, 512), (24576, 512), (28676, 576),
                                 (32768, 512), (50180, 576), (512, 1536), (2052, 1472), (4100, 512), (32772, 3072)])
def test_plain(cuda, M, N, K):
    a, w = _problem(M, N, K, cuda, spare=8)
    want = a.double() @ w.double().T
    assert _rel(lm.matmul(a, w, torch.float32), want) < 1e-5
    ld = (N + 23) // 8 * 8
    out = torch.full((M, ld), 3.0, device=cuda, dtype=torch.bfloat16)
    lm.matmul_joint(a, w, out[:, 8:N + 8], 0, 0)
    assert _rel(out[:, 8:N + 8], want) < 2.3e-3
    assert bool((out[:, :8] == 3).all()) and bool((out[:, N + 8:] == 3).all())


# workgroups that begin at different steps of K: 16, 32 and 112 of them, columns that end inside a workgroup, more than one round
@pytest.mark.parametrize("M", [12, 16, 33, 64])
@pytest.mark.parametrize("N,K", [(8200, 2048), (7180, 4096), (7172, 14336), (32772, 4096)])
def test_turned(cuda, M, N, K):
    a, w = _problem(M, N, K, cuda, spare=8)
    assert _rel(lm.matmul(a, w, torch.float32), a.double() @ w.double().T) < 1e-5


@pytest.mark.parametrize("M", [12, 64])
@pytest.mark.parametrize("N,K", [(5632, 1024), (9216, 3072), (8192, 3584), (7168, 7168), (5632, 2112)])
def test_in_order_where_rows_are_not_4_kb(cuda, M, N, K):
    """There the turn is time lost: every workgroup adds K in the same order, so that columns of the same weights are the same bits."""
    a, w = _problem(M, N, K, cuda)
    y = lm.matmul(a, w[:1].expand(N, K).contiguous(), torch.float32)
    assert torch.equal(y, y[:, :1].expand_as(y))


@pytest.mark.parametrize("M", [1, 8, 31, 64])
@pytest.mark.parametrize("N,K", [(512, 512), (2048, 4096), (2048, 12544), (2000, 4160), (1788, 8256), (768, 4160), (4096, 1024), (8192, 576)])
def test_parts(cuda, M, N, K):
    a, w = _problem(M, N, K, cuda, spare=64)
    y = lm.matmul_parts(a, w)
    assert y.shape == (lm.parts(M, N, K), M, N)
    assert _rel(y.sum(0), a.double() @ w.double().T) < 1e-5


@pytest.mark.parametrize("M,N", [(12, 1036), (40, 1036), (12, 5132), (40, 2060)])      # streaming kernel, ring
def test_epilogues(cuda, M, N):
    K = 704
    a, w = _problem(M, N, K, cuda)
    c = a.double() @ w.double().T
    gate, up = c[:, 0::2], c[:, 1::2]
    lim = 0.8
    clamped = gate.clamp(max=lim) * torch.sigmoid(1.702 * gate.clamp(max=lim)) * (up.clamp(-lim, lim) + 1)
    assert _rel(lm.matmul(a, w, epi=lm.EPI_CLAMP_GLU, param=lim), clamped) < 2.3e-3
    gelu = torch.nn.functional.gelu(gate, approximate="tanh") * up
    assert _rel(lm.matmul(a, w, epi=lm.EPI_GELU_GLU), gelu) < 2.3e-3
    assert _rel(lm.matmul(a, w, torch.float32, lm.EPI_SOFTCAP, 2.5), 2.5 * torch.tanh(c / 2.5)) < 1e-5
    out = torch.empty(M, N - 12, device=cuda, dtype=torch.bfloat16)
    side = lm.matmul_joint(a, w, out, 516, 12)
    assert _rel(out[:, :516], torch.relu(c[:, :516]) ** 2) < 2.3e-3
    assert _rel(out[:, 516:], c[:, 516:N - 12]) < 2.3e-3 and _rel(side, c[:, N - 12:]) < 1e-5


def test_residual_norm_of_eight_parts(cuda):
    x = torch.randn(5, 2048, device=cuda)
    d = torch.randn(8, 5, 2048, device=cuda)
    w = torch.rand(2048, device=cuda) + 0.5
    got, h = lm.residual_norm(x.clone(), d, lm.PLAIN, 1.0, None, w, 1e-5, 2048, torch.float32)
    want = x.double() + d.double().sum(0)
    assert _rel(got, want) < 1e-6
    assert _rel(h, want * torch.rsqrt((want * want).mean(-1, keepdim=True) + 1e-5) * w.double()) < 1e-6
