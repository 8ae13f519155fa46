"""Rules of the launches that follow the device's CUs: a partition of a card has fewer than 256."""
import ctypes

import pytest

from test_gpu_parity import base_cfg


@pytest.mark.parametrize("cus", [32, 64, 128, 256])
def test_scan_copies_never_take_a_second_round(cus):
    from atomic_gdn2 import _lib
    for D in (64, 128):
        for n_bh in range(1, 80):
            slices = n_bh * D // 16
            n = _lib.lib().gdn2_debug_scan_copies(n_bh, D, 40, 0, cus)
            assert n in (1, 2, 4) and (n == 1 or n * slices <= cus), (n_bh, D)
            assert n == 4 or 2 * n * slices > cus or slices > cus, (n_bh, D)      # and use the CUs there are


@pytest.mark.parametrize("cus", [32, 64, 128, 256])
def test_state_checkpoints_by_rounds_of_the_device(cus):
    """Every chunk's state up to one and a half rounds of two workgroups per CU, then 2 and 3."""
    from atomic_gdn2 import _lib
    rule = _lib.lib().gdn2_debug_state_ckpt
    for D, per in ((64, 1), (128, 2)):
        for wgs in (1, 2 * cus, 3 * cus, 3 * cus + 2, 4 * cus, 4 * cus + 2, 16 * cus):
            d = _lib.make_desc(base_cfg(), 1, 1, 64 * max(1, wgs // per), D, 0.1)
            assert rule(ctypes.byref(d), cus) == (1 if wgs <= 3 * cus else 2 if wgs <= 4 * cus else 3), (D, wgs)


def test_the_rules_ask_the_device():
    """gdn2_default_state_ckpt is the rule of the device at hand (256 CUs without one)."""
    import torch
    from atomic_gdn2 import _lib
    cus = torch.cuda.get_device_properties(0).multi_processor_count if torch.cuda.is_available() else 256
    for H in range(1, 12):
        d = _lib.make_desc(base_cfg(), 4, H, 2048, 128, 0.1)
        assert _lib.lib().gdn2_default_state_ckpt(ctypes.byref(d)) == _lib.lib().gdn2_debug_state_ckpt(ctypes.byref(d), cus)
