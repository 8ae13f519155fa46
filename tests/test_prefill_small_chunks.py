"""Prefill calls whose chunk the chunk kernels do not run: prompts shorter than a chunk take the token
kernel alone, longer ones raise the descriptor's own message, after the domain of g."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(bt, L, D, seed=0):
    from atomic_gdn2 import make_cfg
    gen = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda: torch.randn(2, 3, L, D, generator=gen, device="cuda")  # noqa: E731
    cfg = make_cfg(bt=bt, bc=bt // 2, score_bs=bt, bs2=bt // 2, mb=2, wy_eps=0.0, g_max=5.0)
    return cfg, [r() / 8, r() / 8, r(), r(), torch.sigmoid(r()), -0.1 * r().abs()]


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")


@pytest.mark.parametrize("bt", [4, 16, 32])
@pytest.mark.parametrize("docs", [False, True])
def test_prompts_shorter_than_a_small_chunk(bt, docs):
    """The same bits as a chunk of 64 gives such a prompt (the chunk size plays no part in it)."""
    from atomic_gdn2.inference import chunk_forward_inference
    L = bt - 1
    cfg, xs = _case(bt, L, 64)
    ids = torch.arange(L, device="cuda").expand(2, L) // 2 if docs else None
    want = chunk_forward_inference(*xs, 0.1, _case(64, L, 64)[0], segment_ids=ids)
    got = chunk_forward_inference(*xs, 0.1, cfg, segment_ids=ids)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("docs", [False, True])
def test_longer_prompts_are_refused_in_order(docs):
    from atomic_gdn2.inference import chunk_forward_inference
    cfg, xs = _case(32, 80, 64)
    ids = torch.zeros(2, 80, dtype=torch.int64, device="cuda") if docs else None
    with pytest.raises(ValueError, match="gdn2_fwd_prefill"):
        chunk_forward_inference(*xs, 0.1, cfg, segment_ids=ids)
    xs[5][0, 0, 0, 0] = -100.0
    with pytest.raises(ValueError, match="outside the layer domain"):
        chunk_forward_inference(*xs, 0.1, cfg, segment_ids=ids)
