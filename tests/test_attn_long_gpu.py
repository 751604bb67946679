"""LMTrain steps on windows past 64 tokens: attention in one launch per
direction (65 .. 512 tokens, head_dim a multiple of 4 up to 64) and, past those
limits, composed.  One step against the float64 oracle, the bars of
tests/test_lm_gpu.py."""
import pytest

from tests.gpu_util import announce
from tests.test_lm_gpu import _check, _run_case

pytestmark = pytest.mark.gpu


# edges of the 16-row blocks, of four waves' 64 rows and of the 128/256/512-token
# forms; T not a multiple of 4; each head_dim class and partial ones; two layers
@pytest.mark.parametrize("D,H,B,T,causal", [(32, 2, 2, 65, True), (16, 1, 1, 127, True), (64, 2, 1, 128, True),
                                            (48, 1, 2, 129, True), (64, 1, 1, 255, True), (40, 2, 1, 257, True),
                                            (12, 3, 1, 512, True), (64, 1, 1, 80, False), (24, 2, 1, 203, False),
                                            (12, 2, 2, 70, True), (16, 1, 1, 513, True), (136, 2, 1, 72, True)])
def test_lm_step_long_windows(D, H, B, T, causal):
    announce("lm long", D, H, B, T, causal)
    gpu, res = _run_case(60, D, 2, H, 2 * D, B, T, steps=1, lr=0.1, std=0.3, seed=D + T, causal=causal)
    _check(res)
    gpu.close()
