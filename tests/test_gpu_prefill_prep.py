"""The prefill's statistics and reset flags in one kernel against the same in torch operations, and the
calls that have to run again or raise after the prefill was already enqueued."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")


@pytest.mark.parametrize("B,H,L,D,bt", [(1, 1, 1, 64, 64), (2, 3, 63, 64, 64), (3, 2, 64, 128, 64), (2, 5, 200, 64, 64),
                                        (2, 2, 640, 128, 256), (5, 3, 1029, 64, 128), (1, 16, 4096, 128, 64)])
@pytest.mark.parametrize("seg_dtype", [None, torch.int32, torch.int64])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_prep_equals_torch(B, H, L, D, bt, seg_dtype, dt):
    from atomic_gdn2 import inference as I
    gen = torch.Generator().manual_seed(L + D)
    g = -torch.rand(B, H, L, D, generator=gen)
    g[-1, -1, -1, -1] = -7.5                       # the extremes at the last and the first element
    g[0, 0, 0, 0] = 0.25
    seg = None
    if seg_dtype is not None:
        seg = torch.cumsum((torch.rand(B, L, generator=gen) < 0.02).long(), 1).to(seg_dtype).cuda() * -3
        if seg_dtype == torch.int64:
            seg[:, L // 2:] += 2 ** 32             # ids that differ above 32 bits only
    for edit in (None, math.nan, math.inf, -math.inf):
        if edit is not None:
            g[0, 0, L // 2, 3] = edit
        x = g.to("cuda", dt)
        a, b = (f(x, seg, seg is not None and L >= bt, B, H, L, D, bt) for f in (I._prep_native, I._prep_torch))
        for u, v in zip(a[:2], b[:2]):
            assert (u is None) == (v is None) and (u is None or torch.equal(u, v.reshape(u.shape)))
        (lo, hi, bad), (lo2, hi2, bad2) = a[2](), b[2]()
        same = lambda p, q: p == q or (math.isnan(p) and math.isnan(q))  # noqa: E731
        assert same(lo, lo2) and same(hi, hi2) and bad == bad2


def test_positive_gates_other_id_types_and_errors():
    from atomic_gdn2 import make_cfg
    from atomic_gdn2.inference import chunk_forward_inference
    cfg = make_cfg(bt=64, bc=32, score_bs=64, bs2=32, wy_eps=0.0, dot_mode="highest", solve_dot_mode="highest")
    gen = torch.Generator(device="cuda").manual_seed(1)
    r = lambda: torch.randn(2, 2, 150, 64, generator=gen, device="cuda")  # noqa: E731
    xs = [r() / 8, r() / 8, r(), r(), torch.sigmoid(r()), 0.1 * r()]           # half of the gates positive
    ids = torch.zeros(2, 150, dtype=torch.int64, device="cuda")
    ids[0, 64:] = 1
    ids[1, 140:] = 4
    o, h = chunk_forward_inference(*xs, 0.125, cfg, segment_ids=ids)
    o2, h2 = chunk_forward_inference(*xs[:5], xs[5].clamp(max=0.0), 0.125, cfg, segment_ids=ids)
    assert torch.equal(o, o2) and torch.equal(h, h2)
    for other in (ids.int(), ids.short(), ids.float(), ids.cpu(), ids.tolist(), ids.t().contiguous().t()):
        o3, h3 = chunk_forward_inference(*xs, 0.125, cfg, segment_ids=other)
        assert torch.equal(o, o3) and torch.equal(h, h3)
    bad = xs[5].clone()
    bad[1, 1, 149, 63] = -1e3
    mixed = ids.clone()
    mixed[1, 70:] = 9
    with pytest.raises(ValueError, match="outside the layer domain"):
        chunk_forward_inference(*xs[:5], bad, 0.125, cfg, segment_ids=mixed)
    with pytest.raises(ValueError, match="inside chunk 1 of batch row 1"):
        chunk_forward_inference(*xs, 0.125, cfg, segment_ids=mixed)
    with pytest.raises(ValueError, match="not both"):
        chunk_forward_inference(*xs, 0.125, cfg, segment_ids=ids, cu_seqlens=[0, 64, 150])
    with pytest.raises(ValueError, match="is on"):
        chunk_forward_inference(*xs[:5], xs[5].cpu(), 0.125, cfg)
    nan = xs[5].clamp(max=0.0)
    nan[0, 0, 3, 3] = math.nan
    o4, _ = chunk_forward_inference(*xs[:5], nan, 0.125, cfg, segment_ids=ids)
    assert torch.isfinite(o4).all() and torch.equal(o4[1], o2[1])
