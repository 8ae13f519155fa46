"""The forward scan with several copies of each slice's chain (few sequences) against the same
sequences inside a batch that fills the chip (one copy): the same bits, for chunk counts around the
copies' strides, resets, damped chunks and training's stored tensors (through the gradients)."""
import pytest
import torch

from test_gpu_parity import banner, base_cfg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")


def _xs(H, L, D, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda: torch.randn(1, H, L, D, generator=gen, device="cuda")  # noqa: E731
    return [0.1 * r(), 0.1 * r(), r(), r(), torch.sigmoid(r()), -0.1 * r().abs()]


@pytest.mark.parametrize("D,small,big", [(128, 3, 17), (128, 9, 17), (64, 5, 33)])   # 4 | 2 | 4 copies, 1
@pytest.mark.parametrize("nc", [1, 2, 3, 4, 5, 6, 9])
@pytest.mark.parametrize("bt", [64, 128])
def test_copies_same_bits(D, small, big, nc, bt):
    from atomic_gdn2 import make_blr_trainable
    from atomic_gdn2.inference import chunk_forward_inference
    banner(f"scan copies D{D} {small} of {big} sequences, {nc} chunks of {bt}")
    cfg = base_cfg(bt=bt, bc=bt // 2, score_bs=bt, wy_eps=0.0 if bt == 64 else 1e-2)
    L = bt * nc
    big_xs = _xs(big, L, D, nc)
    h0 = 0.1 * torch.randn(1, big, D, D, device="cuda")
    cut = lambda t: t[:, :small].contiguous()  # noqa: E731
    fn = make_blr_trainable(cfg, 0.1, state_ckpt=3)

    def grad(xs, h):
        xs = [x.clone().requires_grad_(True) for x in xs + [h]]
        o, hf = fn(*xs)
        return [o.detach(), hf.detach()] + list(torch.autograd.grad((o, hf), xs, (o.detach(), hf.detach())))

    for a, b in zip(grad([cut(x) for x in big_xs], cut(h0)), grad(big_xs, h0)):
        assert torch.equal(a, cut(b))
    ids = (torch.arange(L, device="cuda") // bt >= nc // 2).long()[None]
    a = chunk_forward_inference(*(cut(x) for x in big_xs), 0.1, cfg, h0=cut(h0), segment_ids=ids)
    b = chunk_forward_inference(*big_xs, 0.1, cfg, h0=h0, segment_ids=ids)
    assert all(torch.equal(x, cut(y)) for x, y in zip(a, b))
