"""The state carried in place through the C ABI (h_final is h0)."""
import ctypes

import pytest
import torch

from test_gpu_parity import banner, base_cfg


def test_one_workgroup_per_slice_in_place():
    """Several workgroups on a slice's chain each read h0, and one of them writes h_final: in place
    there is one, however few the slices."""
    from atomic_gdn2 import _lib
    copies = _lib.lib().gdn2_debug_scan_copies
    for n_bh, D, nc in [(1, 128, 2), (6, 128, 128), (16, 128, 9), (5, 64, 6), (32, 64, 2)]:
        assert copies(n_bh, D, nc, 1, 256) == 1 < copies(n_bh, D, nc, 0, 256)
    assert copies(0, 128, 4, 0, 256) == copies(4, 96, 4, 0, 256) == copies(4, 64, 0, 0, 256) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("H,L,D", [(3, 256, 128), (9, 320, 128), (5, 576, 64)])
def test_in_place_state_same_bits(H, L, D):
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")
    from atomic_gdn2 import _lib
    banner(f"state in place H{H} L{L} D{D}")
    gen = torch.Generator(device="cuda").manual_seed(0)
    r = lambda: torch.randn(1, H, L, D, generator=gen, device="cuda")  # noqa: E731
    xs = [0.1 * r(), 0.1 * r(), r(), r(), torch.sigmoid(r()), -0.1 * r().abs()]
    h0 = 0.1 * torch.randn(1, H, D, D, generator=gen, device="cuda")
    desc = _lib.make_desc(base_cfg(), 1, H, L, D, 0.1)
    L_ = _lib.lib()

    def run(h, hf):
        o = torch.empty_like(xs[0])
        ws = torch.empty(L_.gdn2_fwd_workspace_bytes(ctypes.byref(desc), 0), dtype=torch.uint8, device="cuda")
        _lib.check(L_.gdn2_fwd(ctypes.byref(desc), *map(_lib.ptr, xs), _lib.ptr(h), _lib.ptr(o), _lib.ptr(hf), None,
                               _lib.ptr(ws), _lib.stream_handle()), "gdn2_fwd")
        return o, hf

    want = run(h0, torch.empty_like(h0))
    h = h0.clone()
    got = run(h, h)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
