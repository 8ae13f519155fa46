"""The WY build with eight waves per chunk (at most 256 chunks) against the four-wave form that larger
launches take: the same sequences alone and inside a batch of 264 chunks, bit for bit."""
import pytest
import torch

from test_gpu_parity import banner, base_cfg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("kw", [dict(), dict(bs2=16), dict(bs2=64, mb=16), dict(score_bs=32, bs2=16, mb=4),
                                dict(dot_mode="bf16x3", solve_dot_mode="bf16x3"), dict(dot_mode="default", wy_eps=1e-2)])
def test_eight_waves_same_bits(D, kw):
    from atomic_gdn2 import make_blr_trainable
    banner(f"wy waves D{D} {kw}")
    H, nc, few = 33, 8, 3
    gen = torch.Generator(device="cuda").manual_seed(D)
    r = lambda: torch.randn(1, H, 64 * nc, D, generator=gen, device="cuda")  # noqa: E731
    big = [0.1 * r(), 0.1 * r(), r(), r(), torch.sigmoid(r()), -0.1 * r().abs()]
    cut = lambda t: t[:, :few].contiguous()  # noqa: E731
    fn = make_blr_trainable(base_cfg(**kw), 0.1, state_ckpt=2)

    def grad(xs):
        xs = [x.clone().requires_grad_(True) for x in xs]
        o, h = fn(*xs)
        return [o.detach(), h.detach()] + list(torch.autograd.grad((o, h), xs, (o.detach(), h.detach())))

    for a, b in zip(grad([cut(x) for x in big]), grad(big)):
        assert torch.equal(a, cut(b))
    with torch.no_grad():
        a, b = fn(*(cut(x.bfloat16()) for x in big)), fn(*(x.bfloat16() for x in big))
    assert torch.equal(a[0], cut(b[0])) and torch.equal(a[1], cut(b[1]))
