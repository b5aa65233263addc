"""The tiled products (csrc/lm/gemm_wide.hip: four waves of 256 x 256; gemm_tile.hip: rings of smaller tiles) against fp64.

Tolerances, relative 2-norms: fp32 sums of bf16 products 1e-5; one rounding to bf16 (an error spread evenly over half a unit in
the last of 8 bits) at most 2^-8 / sqrt(3) = 2.3e-3."""
import pytest
import torch

from shai_amd.ops import lm

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return ((a.double() - b).norm() / b.norm()).item()


def _problem(M, N, K, dev, spare=0):
    g = torch.Generator(device=dev).manual_seed(M * 7 + N + K)
    a = torch.randn(M + 2, K + spare, generator=g, device=dev).bfloat16()[1:M + 1, :K]     # neighbours must not matter
    return a, (torch.randn(N, K, generator=g, device=dev) / K ** 0.5).bfloat16()


# at least 192 tiles: whole ones, a last row, a row missing; columns cut by 4, by 8 and by 252; odd and even counts of k-tiles;
# 258, 288, 351 and 375 tiles, whose last 2, 32, 95 and 119 are cut in quarters, and 391 whose last 135 are not
@pytest.mark.parametrize("M,N", [(4096, 3072), (3073, 3588), (3327, 3336), (257, 24580), (5120, 2820), (257, 32900), (4096, 4608),
                                 (4100, 5636), (3840, 6400), (9900, 2300)])
@pytest.mark.parametrize("K", [1600, 1664])
def test_plain(cuda, M, N, K):
    a, w = _problem(M, N, K, cuda, spare=8)
    want = a.double() @ w.double().T
    ld = (N + 23) // 8 * 8
    out = torch.full((M, ld), 3.0, device=cuda, dtype=torch.bfloat16)
    lm.matmul_joint(a, w, out[:, 8:N + 8], 0, 0)
    assert _rel(out[:, 8:N + 8], want) < 2.3e-3
    assert bool((out[:, :8] == 3).all()) and bool((out[:, N + 8:] == 3).all())


# more than one whole round, tile after tile in a workgroup: two, three and odd counts of k-tiles; a last row and columns that end inside
# a tile, the last round not whole (391 tiles), cut in quarters (544 and 32 more) or with side columns among the quarters (512 and 64); tiles
# with side columns that the whole rounds reach into (510 of 527 tiles without, 391 of 408, 400 of 425)
@pytest.mark.parametrize("M,N,side,act", [(4100, 5640, 0, None), (4352, 8192, 0, 4100), (4096, 8976, 272, None), (8191, 4352, 0, None),
                                           (4100, 7712, 32, None), (4100, 5904, 16, None), (6400, 4104, 8, None)])
@pytest.mark.parametrize("K", [128, 192, 1600])
def test_chain(cuda, M, N, side, act, K):
    a, w = _problem(M, N, K, cuda, spare=8)
    want = a.double() @ w.double().T
    if side:
        main, extra = lm.matmul_with_side(a, w, side)
        assert _rel(main, want[:, :-side]) < 2.3e-3 and _rel(extra, want[:, -side:]) < 1e-5
        return
    out = torch.full((M + 1, N + 16), 3.0, device=cuda, dtype=torch.bfloat16)
    lm.matmul_joint(a, w, out[:M, 8:N + 8], act or 0, 0)
    if act:
        want[:, :act] = want[:, :act].clamp(min=0) ** 2
    assert _rel(out[:M, 8:N + 8], want) < 2.3e-3
    assert bool((out[:, :8] == 3).all()) and bool((out[:, N + 8:] == 3).all()) and bool((out[M] == 3).all())


# smaller tiles: fewer k-tiles than the ring holds, one more, many; 64 x 64, one 128 x 128 tile per CU and more than one
@pytest.mark.parametrize("M,N", [(65, 64), (129, 452), (300, 2052), (1030, 4100), (2100, 4100)])
@pytest.mark.parametrize("K", [64, 192, 256, 320, 2112])
def test_small_tiles(cuda, M, N, K):
    a, w = _problem(M, N, K, cuda, spare=8)
    want = a.double() @ w.double().T
    assert _rel(lm.matmul(a, w, torch.float32), want) < 1e-5
    assert _rel(lm.matmul(a, w), want) < 2.3e-3
    assert _rel(lm.matmul_parts(a, w, torch.float32).double().reshape(-1, M, N).sum(0), want) < 1e-5


# fp32 side columns inside the last tile and over the border of two, of a count that allows 16-byte stores and of one that does not
@pytest.mark.parametrize("side", [4, 20, 33, 257, 300])
def test_side_columns(cuda, side):
    a, w = _problem(3100, 3824 + side, 1600, cuda)
    main, extra = lm.matmul_with_side(a, w, side)
    want = a.double() @ w.double().T
    assert _rel(main, want[:, :-side]) < 2.3e-3 and _rel(extra, want[:, -side:]) < 1e-5


def test_relu2(cuda):
    a, w = _problem(3100, 4092, 1600, cuda)
    want = (a.double() @ w.double().T).clamp(min=0) ** 2
    assert _rel(lm.matmul(a, w, epi=lm.EPI_RELU2), want) < 2.3e-3


# rows by expert, gathered or in place: tiles of few rows, experts without any, one and two k-tiles
@pytest.mark.parametrize("gather", [True, False])
@pytest.mark.parametrize("N,K", [(260, 64), (512, 128), (128, 192)])
def test_grouped(cuda, N, K, gather):
    T, E, top = 1500, 5, 2
    g = torch.Generator(device=cuda).manual_seed(N)
    ids = torch.randint(0, 3, (T, top), generator=g, device=cuda).int()
    ids[:, 1] = 4                                          # experts: 0 .. 2 and 4, none for 3
    plan = lm.plan_experts(ids, E)
    if plan.bm != 256:
        pytest.skip("another tile")
    rows = T if gather else T * top
    a = torch.randn(rows, K, generator=g, device=cuda).bfloat16()
    w = (torch.randn(E, N, K, generator=g, device=cuda) / K ** 0.5).bfloat16()
    c = lm.matmul(a, w, plan=plan, gather=gather)
    off = plan.offsets.tolist()
    for e in range(E):
        s = slice(off[e], off[e + 1])
        x = a[plan.token_of[s].long()] if gather else a[s]
        if off[e + 1] > off[e]:
            assert _rel(c[s], x.double() @ w[e].double().T) < 2.3e-3
