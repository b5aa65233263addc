"""Pugozen through the gfx950 kernels, bf16 and fp32, against the plain oracle."""
import os
import subprocess
import sys

import pugozen_cases as C
import pytest
import torch

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16]
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("dtype", DTYPES, ids=C.name)
@pytest.mark.parametrize("check", C.MECHANISMS, ids=lambda f: f.__name__)
def test_mechanism(cuda, check, dtype):
    check(cuda, dtype)


@pytest.mark.parametrize("dtype", DTYPES, ids=C.name)
@pytest.mark.parametrize("key", sorted(C.SHAPES))
def test_shapes(cuda, tmp_path, key, dtype):
    C.check_shape(tmp_path, cuda, dtype, key)


@pytest.mark.parametrize("dtype", DTYPES, ids=C.name)
@pytest.mark.parametrize("check", C.MODELS, ids=lambda f: f.__name__)
def test_model(cuda, tmp_path, check, dtype):
    check(tmp_path, cuda, dtype)


@pytest.mark.parametrize("kw", [{}, {"use_graphs": False}, {"num_kv_blocks": 7}], ids=["graphs", "eager", "preempt"])
def test_greedy_generation(cuda, tmp_path, kw):
    C.check_greedy(tmp_path, cuda, torch.float32, **kw)


def test_greedy_generation_bf16(cuda, tmp_path):
    C.check_greedy(tmp_path, cuda, torch.bfloat16)


def test_captured_decode_replays_equal_eager(cuda, tmp_path):
    """Decode-program replays, with eager steps and synchronisations between them, against the same steps run eagerly."""
    from shai_amd.engines.llm import LLMEngine
    from shai_amd.models.registry import config_from_path
    c = C.Case(tmp_path, cuda, torch.bfloat16, seed=21)
    mk = lambda g: LLMEngine(config_from_path(c.path), device=cuda, model_path=c.path, max_num_seqs=4, max_model_len=192,
                             use_graphs=g)
    a, b = mk(True), mk(False)
    sa, sb = [[e.open_request() for _ in range(3)] for e in (a, b)]
    toks = [c.tokens(120) for _ in range(3)]
    at = 0
    for i, n in enumerate((9, 1, 1, 2, 1, 1, 1, 30, 1, 1, 1, 1)):
        out = [e.extend([(s, t[at:at + n], [n - 1]) for s, t in zip(ss, toks)]) for e, ss in ((a, sa), (b, sb))]
        at += n
        assert torch.equal(out[0], out[1]), i
        torch.cuda.synchronize()


def test_trace_run_program(cuda, tmp_path):
    c = C.Case(tmp_path, cuda, torch.float32, seed=22)
    toks = c.tokens(32)
    for dtype in DTYPES:
        out = tmp_path / C.name(dtype)
        r = subprocess.run([sys.executable, os.path.join(ROOT, "bin", "trace_run"), "--model", c.path, "--dtype",
                            C.name(dtype), "--out", str(out), "--max-tokens", "128"],
                           input="\n".join(C.replay_lines(c, toks)) + "\n", capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stderr[-2000:]
        said = [ln for ln in r.stdout.splitlines() if ln.startswith("done")]
        C.check_replay_files(c, toks, out, said, dtype)


def test_prompts_in_rounds(cuda, monkeypatch):
    """Heads whose prepared chunks do not fit the workspace together run in several rounds."""
    monkeypatch.setattr(C.lm, "RULE_WORKSPACE", 1)
    C.check_mixers(cuda, torch.bfloat16)
    monkeypatch.setattr(C.lm, "RULE_WORKSPACE", 1 << 20)
    C.check_delta(cuda, torch.bfloat16)
    C.check_retention(cuda, torch.bfloat16)


@pytest.mark.parametrize("rows", [32, 96])
def test_prompts_in_segments(cuda, monkeypatch, rows):
    """Prompts cut into segments that are scanned side by side: at every head size, in batches of unequal lengths."""
    monkeypatch.setattr(C.lm, "rule_segment", lambda *_: rows)
    for check in (C.check_delta, C.check_delta_memory, C.check_retention, C.check_mixers):
        check(cuda, torch.bfloat16)


@pytest.mark.parametrize("B,H,G,d,rule,channels,splits", [
    (1, 4, 1, 128, (4, 2, 128), True, 1), (3, 8, 1, 64, (2, 1, 64), False, 2), (5, 2, 2, 64, (3, 3, 128), True, 1),
    (2, 12, 1, 64, (2, 2, 64), True, 1), (3, 8, 1, 128, (2, 2, 128), True, 2),
    (2, 14, 2, 128, (2, 1, 64), False, 1), (64, 16, 4, 128, (16, 16, 128), True, 1), (1, 4, 4, 128, (2, 2, 256), False, 1),
    (25, 16, 4, 128, (16, 8, 128), False, 1), (26, 16, 4, 128, (16, 16, 64), True, 1)])
def test_mixers_of_a_step_in_one_launch(cuda, B, H, G, d, rule, channels, splits):
    """Attention and delta rule together against one after the other: caches, states and both outputs.  Groups and head sizes that the one
    launch takes and that it does not (12 heads to a group, heads of 256); contexts of one key, of whole blocks and past them; sequences
    without a slot; the most workgroups of the form for few of them, and more.  The sums are the same in the same order, compiled twice: a last bit of the bf16 outputs, 2^-16 of the fp32 states."""
    from types import SimpleNamespace
    lm, (R, K, s) = C.lm, rule
    g = torch.Generator(device=cuda).manual_seed(B * H + s)
    rand = lambda *shape, dtype=torch.bfloat16: torch.randn(*shape, generator=g, device=cuda).to(dtype)
    i32 = lambda t: torch.tensor(t, dtype=torch.int32, device=cuda)
    lens = [(1, 64, 65, 200, 7)[i % 5] for i in range(B)]
    blocks, ch = 4, 2 * K * s + R * s
    batch = SimpleNamespace(is_prefill=False, num_splits=splits, ctx_lens=i32(lens), positions=i32([n - 1 for n in lens]),
                            block_table=i32([[b * blocks + j for j in range(blocks)] for b in range(B)]),
                            slots=i32([-1 if b == 4 else b * blocks * 64 + n - 1 for b, n in enumerate(lens)]),
                            state_slots=i32([-1 if b == 4 else B - 1 - b for b in range(B)]))
    rows = rand(B, (H + G) * d + ch + R * s)
    caches = [rand(B * blocks, G, 64, d) for _ in range(2)]
    state, ring = rand(B, R, s, s, dtype=torch.float32), rand(B, 4, ch)
    turn = lm.HeadTurn(lm.rope_rows(batch.positions, lm.rope_freq(1e4, d // 2).to(cuda)), d, 1e-6, rand(d, dtype=torch.float32),
                       rand(d, dtype=torch.float32))
    f32 = dict(dtype=torch.float32)
    decay, beta = rand(B, R * (s if channels else 1), **f32), rand(B, R, **f32)
    conv, rate, bias, gain = rand(4, ch, **f32), rand(R, **f32).exp(), rand(decay.shape[1], **f32), rand(s, **f32)
    temp, sink = rand(H, **f32), rand(H, **f32)

    def run(together):
        out = torch.zeros(B, H * d + R * s, dtype=torch.bfloat16, device=cuda)
        kc, vc, st, rg = caches[0].clone(), caches[1].clone(), state.clone(), ring.clone()
        r = lm.RuleStep(rows[:, (H + G) * d:(H + G) * d + ch], rows[:, (H + G) * d + ch:], decay, beta, conv, rate, bias, gain, st, rg,
                        out[:, H * d:], lm.RuleShape(K, s, s), 1e-6)
        a = (rows[:, :(H + G) * d], kc, vc, batch, H, lm.WHOLE, d ** -0.5)
        plain = lm.Ungated(temp, sink, out[:, :H * d], 0.7)
        if together:
            lm.attention_beside_rule(*a, turn=turn, plain=plain, rule=r)
        else:
            lm.gated_attention(*a, window=True, turn=turn, plain=plain)
            lm.delta_rule(r.x, r.gate, r.decay, r.beta, r.conv, r.rate, r.bias, r.gain, r.state, r.ring, batch, r.out, r.shape, r.eps)
        return out, kc, vc, st, rg
    one, two = run(True), run(False)
    for i, (a, b) in enumerate(zip(one, two)):
        assert torch.isfinite(b.float()).all()
        assert (a.float() - b.float()).norm() <= (2 ** -16 if a.dtype == torch.float32 else 2 ** -9) * b.float().norm(), i
    assert torch.equal(one[2], two[2]) and torch.equal(one[4], two[4])


@pytest.mark.parametrize("B,H,G,R,K,ranks,splits,one", [
    (1, 16, 4, 16, 16, (128, 128), 1, True), (1, 4, 1, 1, 1, (64, 128), 2, True), (5, 6, 2, 4, 2, (128, 64), 1, True),
    (25, 16, 4, 16, 8, (64, 64), 1, True), (26, 16, 4, 16, 16, (128, 64), 1, True), (76, 16, 4, 16, 16, (64, 128), 1, True),
    (77, 16, 4, 16, 16, (128, 128), 1, False), (2, 16, 4, 4, 4, (192, 64), 1, False)])
def test_logits_made_beside_attention(cuda, B, H, G, R, K, ranks, splits, one):
    """Gate and decay logits made in the launch of a step's two mixers against a product of their own in front of it: both ranks, alike or not,
    the most workgroups of either form, and what the launch does not take.  The logits are the same products in another order (2^-20 of them), which may
    turn the rounding of a gate (bf16), and a decay is e^-(rate softplus), rate up to e^2: outputs to a bf16 rounding, states 2^-14."""
    from types import SimpleNamespace
    lm, s, d = C.lm, 128, 128
    g = torch.Generator(device=cuda).manual_seed(B * H + R)
    rand = lambda *shape, dtype=torch.bfloat16: torch.randn(*shape, generator=g, device=cuda).to(dtype)
    i32 = lambda t: torch.tensor(t, dtype=torch.int32, device=cuda)
    lens = [(1, 64, 65, 200, 7)[i % 5] for i in range(B)]
    blocks, ch, low = 4, 2 * K * s + R * s, sum(ranks)
    batch = SimpleNamespace(is_prefill=False, num_splits=splits, ctx_lens=i32(lens), positions=i32([n - 1 for n in lens]),
                            block_table=i32([[b * blocks + j for j in range(blocks)] for b in range(B)]),
                            slots=i32([-1 if b == 4 else b * blocks * 64 + n - 1 for b, n in enumerate(lens)]),
                            state_slots=i32([-1 if b == 4 else B - 1 - b for b in range(B)]))
    rows = rand(B, (H + G) * d + ch + low)
    caches = [rand(B * blocks, G, 64, d) for _ in range(2)]
    f32 = dict(dtype=torch.float32)
    state, ring = rand(B, R, s, s, **f32), rand(B, 4, ch)
    turn = lm.HeadTurn(lm.rope_rows(batch.positions, lm.rope_freq(1e4, d // 2).to(cuda)), d, 1e-6, rand(d, **f32), rand(d, **f32))
    up = torch.zeros(R * 2 * s, low, dtype=torch.bfloat16, device=cuda)
    up[:R * s, ranks[0]:], up[R * s:, :ranks[0]] = rand(R * s, ranks[1]) / 8, rand(R * s, ranks[0]) / 8
    conv, rate, bias, gain = rand(4, ch, **f32), rand(R, **f32).clamp(max=2).exp(), rand(R * s, **f32), rand(s, **f32)
    beta, temp, sink = rand(B, R, **f32), rand(H, **f32), rand(H, **f32)

    def run(made):
        out = torch.zeros(B, H * d + R * s, dtype=torch.bfloat16, device=cuda)
        kc, vc, st, rg = caches[0].clone(), caches[1].clone(), state.clone(), ring.clone()
        r = lm.RuleStep(rows[:, (H + G) * d:(H + G) * d + ch], rows[:, (H + G) * d + ch:], None, beta, conv, rate, bias, gain, st, rg,
                        out[:, H * d:], lm.RuleShape(K, s, s), 1e-6, up, ranks[0])
        lm.attention_beside_rule(rows[:, :(H + G) * d], kc, vc, batch, H, lm.WHOLE, d ** -0.5, turn=turn,
                                 plain=lm.Ungated(temp, sink, out[:, :H * d], 0.7), rule=r.made() if made else r)
        return out, kc, vc, st, rg
    calls = []
    real = lm._K()
    lm_K = SimpleNamespace(**{n: getattr(real, n) for n in ("attn_beside_rule", "lm_gemm")},
                           attn_beside_rule_low=lambda *a: calls.append(real.attn_beside_rule_low(*a)) or calls[-1])
    with pytest.MonkeyPatch.context() as m:
        m.setattr(lm, "_K", lambda: lm_K)
        got = run(False)
    assert calls == [one]
    for i, (a, b) in enumerate(zip(got, run(True))):
        assert torch.isfinite(b.float()).all()
        assert (a.float() - b.float()).norm() <= (2 ** -14 if a.dtype == torch.float32 else 2 ** -8) * b.float().norm(), i


@pytest.mark.parametrize("M,K,width,N,act,side,parts,source,out", [
    (1, 64, 40, 16, 0, 0, 0, "table", torch.bfloat16), (1, 64, 64, 20, 8, 4, 1, "rows", torch.bfloat16),
    (2, 192, 180, 9000, 0, 0, 4, "rows", torch.float32), (1, 2048, 2048, 17424, 8448, 16, 4, "rows", torch.bfloat16),
    (2, 2048, 2000, 999, 64, 3, 8, "table", torch.bfloat16), (1, 2112, 2112, 8200, 0, 0, 5, "rows", torch.float32),
    (2, 4096, 4096, 333, 0, 0, 3, "rows", torch.float32)])
def test_norm_made_by_its_product(cuda, M, K, width, N, act, side, parts, source, out):
    """A product that makes its input's norm against the two launches: rows of one step of the ring and of many, a K that the waves do not
    share evenly, fewer tiles than workgroups and more, columns that end in a tile.  The residual has the same bits; the norm's mean square
    is summed in another order (2^-20), which may turn a bf16 rounding of h (2^-9 of one of K terms)."""
    lm = C.lm
    g = torch.Generator(device=cuda).manual_seed(K + N)
    rand = lambda *s: torch.randn(*s, generator=g, device=cuda)
    pad = (torch.arange(K, device=cuda) < width).float()
    w, W = (rand(K).abs() + 0.5) * pad, (rand(N, K) / K ** 0.5).bfloat16()
    x, table = rand(M, K) * pad, (rand(50, K) * pad).bfloat16()
    src = x if source == "rows" else lm.Embedding(torch.tensor([49, 7][:M], dtype=torch.int32, device=cuda), table, 3.0)
    delta = rand(parts, M, K) * pad if parts else None
    n = lm.Normed(src, delta, w, 1e-5, width)
    assert lm.normed_fits(n, W)
    got = torch.full((M, N - side), 5.0, dtype=out, device=cuda)
    gx, gs = lm.normed_matmul(n, W, got, act, side)
    wx, h = lm.residual_norm(x.clone() if source == "rows" else src, delta, lm.PLAIN, 1.0, None, w, 1e-5, width, torch.bfloat16)
    c = h.double() @ W.double().T
    c[:, :act] = torch.relu(c[:, :act]) ** 2
    assert torch.equal(gx, wx)
    tol = 2 ** -8 if out == torch.bfloat16 else 2 ** -9
    assert (got.double() - c[:, :N - side]).norm() <= tol * c.norm()
    if side:
        assert (gs.double() - c[:, N - side:]).norm() <= 2 ** -9 * c.norm()


def test_norms_that_stay_apart(cuda):
    """More rows, a wider residual, fp32 weights, sums in bf16 or in more parts, a norm with a bias."""
    lm = C.lm
    W, w = torch.zeros(16, 128, dtype=torch.bfloat16, device=cuda), torch.zeros(128, device=cuda)
    x, d = torch.zeros(2, 128, device=cuda), torch.zeros(4, 2, 128, device=cuda)
    fits = lambda x, d, w, W: lm.normed_fits(lm.Normed(x, d, w, 1e-5, 128), W)
    assert fits(x, d, w, W) and fits(x, None, w, W)
    assert not fits(torch.zeros(3, 128, device=cuda), None, w, W) and not fits(torch.zeros(1, 4160, device=cuda), None, w, W)
    assert not fits(x, d, w, W.float()) and not fits(x, d[0].bfloat16(), w, W) and not fits(x, torch.zeros(9, 2, 128, device=cuda), w, W)
    assert not fits(x, d, lm.Affine(w, w), W)


@pytest.mark.parametrize("T", [1, 3, 300])
@pytest.mark.parametrize("dims", [(2,), (64, 128), (128, 2, 62, 64, 32)])
def test_angles_of_several_tables(cuda, T, dims):
    """Tables of unlike widths in one launch, and more than it takes: the bits of one by one."""
    lm = C.lm
    pos = (torch.arange(T, dtype=torch.int32, device=cuda) * 7919) % 100003
    freqs = [lm.rope_freq(1e4 * (i + 1), d).to(cuda) for i, d in enumerate(dims)]
    for got, f in zip(lm.rope_rows_all(pos, freqs), freqs):
        assert torch.equal(got, lm.rope_rows(pos, f))
