"""The order of a prefill's errors: g's domain, a boundary inside a chunk, both id forms, the device, the
tensors' devices."""
import pytest
import torch


def _cfg():
    from atomic_gdn2 import make_cfg
    return make_cfg(bt=64, bc=32, score_bs=64, bs2=32, wy_eps=0.0, dot_mode="highest", solve_dot_mode="highest")


def test_both_id_forms_are_reported_before_their_shapes():
    from atomic_gdn2.inference import chunk_forward_inference
    x = torch.zeros(1, 1, 10, 64)
    with pytest.raises(ValueError, match="not both"):
        chunk_forward_inference(x, x, x, x, x, x, 0.1, _cfg(), segment_ids=torch.zeros(1, 3), cu_seqlens=[0, 10])


@pytest.mark.gpu
def test_the_domain_is_reported_before_the_devices():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")
    from atomic_gdn2.inference import chunk_forward_inference
    x = torch.zeros(1, 2, 150, 64, device="cuda")
    bad = torch.full((1, 2, 150, 64), -1e3)
    mixed = torch.arange(150, device="cuda")[None] // 50
    run = lambda g, **kw: chunk_forward_inference(x, x, x, x, x, g, 0.1, _cfg(), **kw)  # noqa: E731
    with pytest.raises(ValueError, match="outside the layer domain"):
        run(bad)
    with pytest.raises(ValueError, match="inside chunk 0"):
        run(x.cpu(), segment_ids=mixed)
    with pytest.raises(ValueError, match="not both"):
        run(x.cpu(), cu_seqlens=[0, 150], segment_ids=torch.zeros(1, 150))
    with pytest.raises(ValueError, match="g is on cpu"):
        run(x.cpu())
