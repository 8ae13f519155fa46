"""Positive gates in a prefill act as 0, for every form of the WY build and its anchors, without the
prefill running twice."""
import pytest
import torch

from test_gpu_parity import banner, base_cfg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [{}, dict(bs2=16), dict(bs2=8), dict(diag="lean", diff_clip=20.0),
                                dict(bt=128, bc=64, score_bs=128, bs2=128, wy_eps=1e-2), dict(dot_mode="bf16x3")])
@pytest.mark.parametrize("B,H,L,D", [(1, 2, 300, 128), (2, 5, 129, 64), (3, 33, 384, 64)])   # up to and past 256 chunks
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_same_bits_as_a_clamped_gate_in_one_run(monkeypatch, kw, B, H, L, D, dt):
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")
    from atomic_gdn2 import inference as I
    banner(f"prefill clamp {kw} B{B} H{H} L{L} D{D} {dt}")
    cfg = base_cfg(**kw)
    gen = torch.Generator(device="cuda").manual_seed(L)
    r = lambda: torch.randn(B, H, L, D, generator=gen, device="cuda")  # noqa: E731
    xs = [x.to(dt) for x in (0.1 * r(), 0.1 * r(), r(), r(), torch.sigmoid(r()), 0.1 * r())]     # half the gates positive
    xs[5][0, 0, 7, 3] = float("inf")
    ids = (torch.arange(L, device="cuda") // (2 * cfg.bt)).expand(B, L)
    want = I.chunk_forward_inference(*xs[:5], xs[5].clamp(max=0.0), 0.1, cfg, segment_ids=ids)
    real, runs = I._run_prefill, []
    monkeypatch.setattr(I, "_run_prefill", lambda *a: (runs.append(1), real(*a))[1])
    got = I.chunk_forward_inference(*xs, 0.1, cfg, segment_ids=ids)
    assert runs == [1] and all(torch.equal(a, b) for a, b in zip(got, want))
