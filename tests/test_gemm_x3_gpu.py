"""The three-term bf16 GEMM (csrc/lhip_gemm_x3.hip) against float64.

Bar: every accumulation rounds to 2^-24 of its partial sum and signs are
random, so the relative 2-norm error grows with the square root of the
accumulations: 2^-24 * (2 + sqrt(K)) leaves about a factor of two.
"""
import numpy as np
import pytest

from lanternl_amd import device
from lanternl_amd._lib import call
from tests.gpu_util import announce, rel_fro, to_dev

pytestmark = pytest.mark.gpu

# (m, n, k): the edges of the 64, 128 and 256 tiles and of the 16-deep stages,
# sizes no tile divides, few tiles over a long K (split), many tiles
SHAPES = [
    (4097, 4095, 65), (4096, 4352, 48),          # 256x256 tiles, one row over / one column short, whole tiles
    (2050, 1999, 33), (1100, 1300, 1025),        # 128x128 tiles, a K remainder of one
    (1024, 1024, 1040), (1025, 1030, 17),        # wave sets with an uneven last round; one stage and one k
    (33, 33, 3000), (20, 20, 5000), (1, 3, 9001),  # one tile, many slices
    (300, 3000, 300), (65, 4099, 2049), (2000, 2100, 5),
    # the last tiles of a round split over K: a few, nearly half a round, with a
    # K remainder, past several rounds
    (2060, 2050, 768), (1999, 2700, 400), (2060, 2050, 531), (4200, 4200, 1056),
]


def _operands(rng, m, n, k, ta, tb, pad=0):
    a = rng.normal(size=(k, m + pad) if ta else (m, k + pad)).astype(np.float32)
    b = rng.normal(size=(n, k + pad) if tb else (k, n + pad)).astype(np.float32)
    return a, b


def _ref(a, b, ta, tb, m, n, k):
    a64 = (a[:, :m].T if ta else a[:, :k]).astype(np.float64)
    b64 = (b[:, :k].T if tb else b[:, :n]).astype(np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        return a64 @ b64


def _run(a, b, ta, tb, m, n, k, c0=None, alpha=1.0, beta=0.0):
    A, B = to_dev(a), to_dev(b)
    C = to_dev(np.full((m, n), np.nan, np.float32) if c0 is None else c0)
    call("lhip_sgemm", ta, tb, m, n, k, alpha, A.ptr, a.shape[1], B.ptr, b.shape[1], beta, C.ptr, n)
    return C.download().astype(np.float64)


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_x3_shapes(m, n, k, ta, tb):
    device.init(0)
    announce("x3", m, n, k, ta, tb)
    rng = np.random.default_rng(m + n + k)
    a, b = _operands(rng, m, n, k, ta, tb, pad=(m + k) % 3)   # leading dimensions of any alignment
    got = _run(a, b, ta, tb, m, n, k)
    assert rel_fro(got, _ref(a, b, ta, tb, m, n, k)) <= 2.0 ** -24 * (2 + np.sqrt(k))


@pytest.mark.parametrize("m,n,k", [(300, 301, 1100), (2050, 2100, 50), (64, 3000, 4100)])
def test_x3_alpha_beta(m, n, k):
    device.init(0)
    announce("x3 alpha beta", m, n, k)
    rng = np.random.default_rng(k)
    a, b = _operands(rng, m, n, k, 0, 1)
    c0 = rng.normal(size=(m, n)).astype(np.float32)
    got = _run(a, b, 0, 1, m, n, k, c0, -0.5, 2.0)
    assert rel_fro(got, -0.5 * _ref(a, b, 0, 1, m, n, k) + 2.0 * c0) <= 2.0 ** -24 * (4 + np.sqrt(k))


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0)])
@pytest.mark.parametrize("k,count", [(512, 3), (48, 2), (500, 2)])   # whole stages; 500: one launch a block
def test_x3_batch_reduce(ta, tb, k, count):
    device.init(0)
    m, n = 1000, 700
    announce("x3 batch reduce", ta, tb, k, count)
    rng = np.random.default_rng(k)
    pairs = [_operands(rng, m, n, k, ta, tb) for _ in range(count)]
    A, B = (to_dev(np.stack([p[i] for p in pairs])) for i in (0, 1))
    C = device.Buffer((m, n))
    call("lhip_sgemm_batched_reduce", ta, tb, m, n, k, 1.0, A.ptr, pairs[0][0].shape[1], pairs[0][0].size, B.ptr,
         pairs[0][1].shape[1], pairs[0][1].size, 0.0, C.ptr, n, count)
    ref = sum(_ref(a, b, ta, tb, m, n, k) for a, b in pairs)
    assert rel_fro(C.download(), ref) <= 2.0 ** -24 * (2 + np.sqrt(k * count))


@pytest.mark.parametrize("batch,m,n,k", [(70, 129, 65, 40), (3, 257, 300, 1000)])
def test_x3_batched(batch, m, n, k):
    device.init(0)
    announce("x3 batched", batch, m, n, k)
    rng = np.random.default_rng(batch)
    a, b = rng.normal(size=(batch, m, k)).astype(np.float32), rng.normal(size=(batch, n, k)).astype(np.float32)
    A, B, C = to_dev(a), to_dev(b), device.Buffer((batch, m, n))
    call("lhip_sgemm_strided_batched", 0, 1, m, n, k, 1.0, A.ptr, k, m * k, B.ptr, k, n * k, 0.0, C.ptr, n, m * n, batch)
    ref = a.astype(np.float64) @ b.astype(np.float64).transpose(0, 2, 1)
    assert rel_fro(C.download(), ref) <= 2.0 ** -24 * (2 + np.sqrt(k))


@pytest.mark.parametrize("m,n,k", [(2100, 2050, 70), (700, 900, 1030), (80, 90, 5003), (4100, 4200, 40)])
def test_x3_values_the_split_cannot_carry(m, n, k):
    """Infinities, NaN, values past the largest bf16 and values below 2^-110
    give what fp32 products give: a tile that meets one is computed in fp32."""
    device.init(0)
    announce("x3 special values", m, n, k)
    rng = np.random.default_rng(m)
    a, b = _operands(rng, m, n, k, 0, 0)
    a[3, 5], a[m - 1, k - 1], a[7, 0] = np.inf, -np.inf, np.nan
    b[5, 11] = 0.0                                     # inf * 0
    a[20, 2], b[2, :] = 3.4e38, np.minimum(np.abs(b[2, :]), 0.5) * 1e-3   # rounds to an infinite bf16
    got, ref = _run(a, b, 0, 0, m, n, k), _ref(a, b, 0, 0, m, n, k)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    np.testing.assert_array_equal(np.isposinf(got), np.isposinf(ref))
    np.testing.assert_array_equal(np.isneginf(got), np.isneginf(ref))
    for rows in (np.arange(m) == 20, np.isfinite(ref).all(1) & (np.arange(m) != 20)):   # 3.4e38 drowns the rest
        assert rel_fro(got[rows], ref[rows]) <= 2.0 ** -24 * (2 + np.sqrt(k))

    a, b = _operands(rng, m, n, k, 0, 0)
    a *= np.float32(1e-35)                             # the terms of such values would be subnormal
    b *= np.float32(1e25)
    assert rel_fro(_run(a, b, 0, 0, m, n, k), _ref(a, b, 0, 0, m, n, k)) <= 2.0 ** -24 * (2 + np.sqrt(k))
