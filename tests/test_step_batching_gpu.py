"""Step-level SD2.1 batching on the GPU (HIP-graph buckets with per-row timesteps + ops.sched_step_rows)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_sched_step_rows_kernel(cuda):
    from shai_amd import ops
    from shai_amd.ops import reference as ref
    torch.manual_seed(0)
    B = 5
    lat = torch.randn(B, 16, 16, 4, device=cuda).bfloat16()
    mo = torch.randn(2 * B, 16, 16, 4, device=cuda).bfloat16()
    rows = torch.tensor([[0.5, 0.6, 0], [-1, 0, 0], [0.2, 0.3, 0], [0.9, 0.95, 0], [-1, 0, 0]], device=cuda)
    for pred in (0, 1):
        got = lat.clone()
        ops.sched_step_rows(mo, got, True, 7.5, pred, rows)
        want = lat.cpu().clone()
        ref.sched_step_rows(mo.cpu(), want, True, 7.5, pred, rows.cpu())
        assert torch.allclose(got.cpu().float(), want.float(), atol=2e-2, rtol=2e-2)
        assert torch.equal(got[1], lat[1]) and torch.equal(got[4], lat[4])


def _batched(eng):
    """Two requests of a batch, one joined in mid-flight, beside the images of generate()."""
    from shai_amd.engines.diffusion import StepBatcher
    eng._graphs.clear()
    sb = StepBatcher(eng, max_batch=4)
    assert sb.warmup() == 4
    a = sb.add("a red fox", 6, seed=1)
    with torch.inference_mode():
        sb.step()
        b = sb.add("a blue hen", 4, seed=2)
        while sb.has_work():
            sb.step()
        assert sb.stats["joined_mid_batch"] == 1
        return [(r.image, eng.generate([p], n, seed=s)[0]) for r, p, n, s in ((a, "a red fox", 6, 1), (b, "a blue hen", 4, 2))]


def test_step_batcher_gpu_matches_generate(cuda):
    """With one form for every product, the same in a batch and alone, the same image.  The forms that the tuner picks by time differ between
    row counts, and so does the order of fp32 sums: this tiny model of random weights, 7.5 times the difference of two nearly equal outputs a
    step, carries a rounding to bf16 as far as 18 to 20 of 255 levels from its fp32 form.  Two images of it then differ by a tenth of that
    at most: 0.3 to 1.7 levels in the mean over 50 sets of forms picked at random."""
    from shai_amd import ops
    from shai_amd.engines.diffusion import SDConfig, StableDiffusionEngine
    eng = StableDiffusionEngine(SDConfig.tiny(), device="cuda")
    for got, want in _batched(eng):
        assert (got.float() - want.float()).abs().mean() < 2.0
    table = list(ops._K().gemm_tuning_export())     # with an entry for every product of this model now
    try:
        ops._K().gemm_tuning_import([e.rsplit("=", 1)[0] + "=4,1" for e in table])
        for got, want in _batched(eng):
            assert torch.equal(got, want)
    finally:
        ops._K().gemm_tuning_import(table)
