"""The WY backward's walk over the score pieces: constant squares for every block size (three of
32 x 32, or the ten 16 x 16 tiles at bs2 = 16) with the anchors of each geometry, against the
float64 oracle, per 64-token chunk."""
import pytest
import torch

from conftest import mk_inputs
from test_gpu_parity import NAMES, banner, base_cfg, compare, hip_grad, oracle_grad

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bt,score_bs,bs2,b3", [
    (64, 64, 16, "highest"), (64, 32, 16, "highest"), (64, 16, 16, "highest"), (64, 64, 16, "bf16x3"),
    (64, 32, 32, "highest"), (64, 64, 64, "highest"), (64, 64, 64, "bf16x3"),
    (128, 128, 64, "highest"), (128, 128, 128, "highest")])
def test_gradients_per_piece_geometry(D, bt, score_bs, bs2, b3):
    """fp32 products: 1e-5 is 20 times the 5e-7 that the operator's fp32 sums show; bf16x3 products
    drop the lo x lo term (2^-16 relative per product): 1e-4."""
    banner(f"pieces D{D} bt{bt} score_bs{score_bs} bs2 {bs2} {b3}")
    cfg = base_cfg(bt=bt, bc=bt // 2, score_bs=score_bs, bs2=bs2, b3_dot_mode=b3)
    arrs = mk_inputs(1, 2 * bt, 3, D, 31, g=0.1, layout="bhld")
    compare(hip_grad(cfg, D ** -0.5, arrs), oracle_grad(cfg, D ** -0.5, arrs),
            1e-5 if b3 == "highest" else 1e-4, names=("o", "h_final") + NAMES)
