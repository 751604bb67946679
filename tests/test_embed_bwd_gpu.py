"""Embedding scatter at the edges of its scans (2048 ids), column blocks (256),
batches of in-flight rows (16, then 4) and rows per workgroup (4 or 16).

The sum of a row is one chain of fp32 multiply-adds in token order, so it is
compared element by element with the same chain in float32: each of m terms
rounds once to 2^-24 of the running sum, bounded here by the sum of magnitudes.
"""
import numpy as np
import pytest

from lanternl_amd import device
from lanternl_amd._lib import call
from tests.gpu_util import announce, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,V,D", [(0, 5, 8), (1, 1, 1), (17, 3, 256), (2047, 8192, 260), (2049, 8193, 512), (4097, 33, 258),
                                   (5000, 9001, 12)])
@pytest.mark.parametrize("acc", [0, 1])
def test_embed_bwd_edges(n, V, D, acc):
    device.init(0)
    announce("embed_bwd", n, V, D, acc)
    rng = np.random.default_rng(n + V + D)
    ids = np.minimum(rng.geometric(0.3, n) - 1, V + 1).astype(np.int32)   # a few tokens make up most; some out of range
    ids[rng.random(n) < 0.3] = rng.integers(-2, V + 2)
    ids[rng.random(n) < 0.3] = V - 1
    g, base = rng.normal(size=(max(n, 1), D)).astype(np.float32), rng.normal(size=(V, D)).astype(np.float32)
    G, IDS, DT = to_dev(g), to_dev(ids if n else np.zeros(1, np.int32), np.int32), to_dev(base)
    call("lhip_embed_bwd", G.ptr, IDS.ptr, DT.ptr, n, D, V, 0.5, acc)
    ref, mag = base.astype(np.float64) * acc, np.abs(base).astype(np.float64) * acc
    ok = (ids >= 0) & (ids < V)
    np.add.at(ref, ids[ok], 0.5 * g[:n][ok])
    np.add.at(mag, ids[ok], np.abs(0.5 * g[:n][ok]))
    m = np.bincount(ids[ok], minlength=V)[:, None]
    assert (np.abs(DT.download() - ref) <= m * 2.0 ** -24 * mag).all()
