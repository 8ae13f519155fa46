"""Several tokens in one gdn2_decode call (the kernel of its own that runs them) against the same
tokens one call at a time, around the depth of its operand ring."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")


@pytest.mark.parametrize("n", [2, 3, 4, 5, 7, 8, 63])
@pytest.mark.parametrize("D,bf_in,bf_state,cap,fuse,zero_state", [
    (64, False, False, False, False, True), (128, False, False, False, False, False), (128, True, False, False, False, True),
    (64, False, True, False, False, False), (128, False, False, True, False, False), (64, True, True, True, False, False),
    (128, False, False, False, True, False), (64, False, False, True, True, False)])
def test_tail_equals_single_tokens(n, D, bf_in, bf_state, cap, fuse, zero_state):
    """The same float32 products and sums in another order: 1e-6 of the values (a bf16 state rounds
    every token, where a last-bit difference can flip a rounding: 2^-8)."""
    from atomic_gdn2.inference import _run_decode
    B, H, ld = 2, 3, n + 2
    gen = torch.Generator(device="cuda").manual_seed(n + D)
    r = lambda *s: torch.randn(s, generator=gen, device="cuda")  # noqa: E731
    xs = [r(B, H, ld, D) for _ in range(6)]
    if not fuse:
        xs[0], xs[1] = (x / x.norm(dim=-1, keepdim=True) for x in xs[:2])
        xs[4], xs[5] = torch.sigmoid(xs[4]), -0.1 * xs[5].abs()
    dt = torch.bfloat16 if bf_in else torch.float32
    xs = [x.to(dt) for x in xs]
    kw = dict(tau=4.0 if cap else None)
    if fuse:
        kw.update(fuse=True, a_log=r(H) - 2.0, dt_bias=r(D))
    sc = torch.bfloat16 if bf_state else torch.float32
    st0 = None if zero_state else (0.3 * r(B, H, D, D)).to(sc)
    flags = (torch.rand(B, n, generator=gen, device="cuda") < 0.2).to(torch.uint8)
    flags[:, 0] = 0
    o = torch.full((B, H, ld, D), 7.0, device="cuda")
    got = _run_decode(xs, int(bf_in), B, H, D, n, ld, 0.3, st0, int(bf_state), o, 0, reset=flags, **kw)
    ref, st = torch.empty_like(o), st0
    for t in range(n):
        one = [x[:, :, t].contiguous() for x in xs]
        ot = torch.empty(B, H, D, device="cuda")
        st = _run_decode(one, int(bf_in), B, H, D, 1, 1, 0.3, st, int(bf_state), ot, 0, reset=flags[:, t].contiguous(), **kw)
        ref[:, :, t] = ot
    tol = 2.0 ** -8 if bf_state else 1e-6
    rel = lambda a, b: float((a.double() - b.double()).norm() / b.double().norm())  # noqa: E731
    assert rel(o[:, :, :n], ref[:, :, :n]) <= tol and rel(got, st) <= tol
    assert bool((o[:, :, n:] == 7.0).all())
