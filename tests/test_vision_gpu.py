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


# the weight without its padding, beside the images: workgroups that it ends in and whole ones
@pytest.mark.parametrize("D,P", [(1, 8), (192, 16), (768, 16), (3, 24)])
def test_patch_weight(cuda, D, P):
    torch.manual_seed(D)
    x = torch.randint(0, 256, (2, 2 * P, P, 3), device="cuda", dtype=torch.uint8)
    w = torch.randn(D, P * P * 8, device="cuda").bfloat16()
    y, w3 = ops.patches_u8(x, P, (0.5, 0.4, 0.3), (0.2, 0.3, 0.4), w)
    assert torch.equal(y, ops.patches_u8(x, P, (0.5, 0.4, 0.3), (0.2, 0.3, 0.4)))
    assert torch.equal(w3, w.view(D, P * P, 8)[..., :3].reshape(D, -1))
    for bad in (w[:, :-8].contiguous(), w.float()):
        with pytest.raises(RuntimeError):
            ops.patches_u8(x, P, (0.5, 0.4, 0.3), (0.2, 0.3, 0.4), bad)


# graphs follow weights that are loaded in place, in whatever way where nothing is folded: those of batches captured before, and later
# ones
@pytest.mark.parametrize("load", ["load_into", "data", "folded"])
def test_classifier_follows_its_weights(cuda, load, monkeypatch):
    from shai_amd.engines.encoders import ImageClassifierEngine
    from shai_amd.models.vit import ViTConfig
    from shai_amd.weights import load_into
    if load == "folded":
        monkeypatch.setattr(ops, "FOLD_MIN_TILES", 0)
    eng, new = (ImageClassifierEngine(ViTConfig.tiny(), device="cuda:0", seed=s, use_graphs=s == 1) for s in (1, 2))
    g = torch.Generator().manual_seed(3)
    x = {b: torch.randint(0, 256, (b, 64, 64, 3), generator=g, dtype=torch.uint8).cuda() for b in (1, 2, 3)}
    old = {b: eng.logits_u8(x[b]).clone() for b in (1, 2)}
    if load == "data":
        for p, q in zip(eng.model.parameters(), new.model.parameters()):
            p.data.copy_(q)
    else:
        load_into(eng.model, new.model.state_dict())
    for b in (1, 3, 2, 1):
        got = eng.logits_u8(x[b]).clone()
        assert torch.equal(got, new.logits_u8(x[b]))
        assert b not in old or not torch.equal(got, old[b])


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
