"""LMTrain steps whose weight gradients, norms and gates leave the fused small
tiles: one step against the float64 oracle of the same step (the bars of
tests/test_lm_gpu.py: losses 1e-5, gradients 1e-4, norm 1e-5)."""
import pytest

from tests.gpu_util import announce
from tests.test_lm_gpu import _check, _run_case

pytestmark = pytest.mark.gpu

# dim 256 / 128 at the row counts where the separate kernels take over, odd
# widths (ffn not a multiple of 4 leaves no float4 loads), ragged edges of the
# 128x128 and 64x64 tiles, a K remainder (rows not a multiple of 16)
@pytest.mark.parametrize("V,D,L,H,F,B,T", [(300, 256, 1, 4, 516, 16, 64), (130, 136, 2, 4, 275, 61, 64),
                                           (70, 512, 1, 8, 1030, 9, 57), (1500, 320, 3, 5, 644, 7, 61)])
def test_lm_step_large_tiles(V, D, L, H, F, B, T):
    announce("lm large tiles", V, D, L, H, F, B, T)
    gpu, res = _run_case(V, D, L, H, F, B, T, steps=1, lr=0.1, std=0.05, seed=V + D)
    _check(res)
    gpu.close()
