"""The vision encoders' front end (csrc/kernels/vision.hip): uint8 patches, tokens with position embeddings and row moments."""
import pytest
import torch

from shai_amd import ops

pytestmark = pytest.mark.gpu


# one patch; widths that 256 threads do not divide; more than a block's pixels
@pytest.mark.parametrize("B,H,W,P", [(1, 16, 16, 16), (3, 224, 224, 16), (2, 32, 88, 8), (1, 64, 96, 32)])
def test_patches(cuda, B, H, W, P):
    torch.manual_seed(B)
    x = torch.randint(0, 256, (B, H, W, 3), device="cuda", dtype=torch.uint8)
    mean, std = (0.485, 0.456, 0.406), (0.229, 0.224, 0.225)
    assert ops.patches_u8_ok(x, P)
    y = ops.patches_u8(x, P, mean, std)
    want = ((x.double() / 255 - torch.tensor(mean, device="cuda")) / torch.tensor(std, device="cuda"))
    want = want.view(B, H // P, P, W // P, P, 3).transpose(2, 3).reshape(-1, P * P * 3)
    assert (y.double() - want).abs().max().item() <= 2 ** -8 * want.abs().max().item()     # half a unit of bf16
    assert (y != ops.patches_u8(x.cpu(), P, mean, std).cuda()).double().mean().item() < 1e-4   # the same steps in 32 bits


def test_patches_left_alone(cuda):
    x = torch.zeros(2, 32, 32, 3, device="cuda", dtype=torch.uint8)
    flat = torch.zeros(2 * 32 * 32 * 3 + 4, device="cuda", dtype=torch.uint8)[4:].view(2, 32, 32, 3)
    assert not ops.patches_u8_ok(x, 12) and not ops.patches_u8_ok(x[:, :, :24], 8) and not ops.patches_u8_ok(flat, 16)
    assert not ops.patches_u8_ok(x.float(), 16) and not ops.patches_u8_ok(x[:, :20].contiguous(), 16)


# one row; a wave's remainder; widths of one, two and four vectors a lane; with and without detection tokens
@pytest.mark.parametrize("B,n,nd,D", [(1, 1, 0, 64), (2, 196, 0, 768), (3, 5, 7, 192), (1, 9, 2, 1032), (2, 4, 0, 2048)])
def test_tokens(cuda, B, n, nd, D):
    torch.manual_seed(n)
    rnd = lambda *s: torch.randn(*s, device="cuda").bfloat16()       # noqa: E731
    patches, cls, det, pos = rnd(B, n, D), rnd(1, 1, D), rnd(1, nd, D) if nd else None, rnd(1, 1 + n + nd, D) + 20
    x, mr = ops.tokens(patches, cls, det, pos, 1e-6)
    parts = [cls.expand(B, -1, -1), patches] + ([det.expand(B, -1, -1)] if nd else [])
    assert torch.equal(x, (torch.cat(parts, 1).float() + pos.float()).bfloat16())
    rows = x.double().view(-1, D)
    assert (mr[:, 0] - rows.mean(1)).abs().max().item() < 1e-5 * 20
    assert (mr[:, 1] * torch.sqrt(rows.var(1, unbiased=False) + 1e-6) - 1).abs().max().item() < 1e-5
    assert ops.tokens(patches, cls, det, pos)[1] is None
