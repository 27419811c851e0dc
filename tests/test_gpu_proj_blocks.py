"""GPU: the 1-bit projections' integer block sums at the edges of their split: rows past a tile,
K of one block, of a partial 512-weight step, of one step a wave, two, and more (K > 16384), one
and two tiles a workgroup; activations with outliers; infinities and NaN.

Tolerance as in test_gpu_proj.py (4e-6 of sum |x| scale): x is rounded to within 2^-28, 2^-29, 2^-30
or 2^-31 (a quarter of the weights each) of the power of two above its 128-weight block's largest
magnitude, at most twice that: 128 * 2 * 15/32 * 2^-28 = 4.5e-7 of the block's largest term."""
import numpy as np
import pytest
import torch

from bitgpu_amd import engine as E
from tests.gpu_helpers import export_k_v, rope_dev, t
from tests.test_gpu_proj import _check_gemv, _dev_weight, _weight

pytestmark = pytest.mark.gpu


def _run(sign, sc, x, h):
    y = E.resid_mm(_dev_weight(sign, sc, sign.shape[1] * 32, sign.shape[0]), t(x), t(h))
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("K,N", [(128, 1), (128, 8209), (512, 17), (640, 8191), (8192, 31), (8320, 15),
                                 (16384, 33), (16512, 47), (25088, 8200)])
def test_block_sums_edges(dev, K, N):
    rng = np.random.default_rng(K + N)
    sign, sc = _weight(rng, N, K)
    x, h = (rng.standard_normal(n).astype(np.float32) for n in (K, N))
    _check_gemv(_run(sign, sc, x, h), x, sign, sc, h)


def test_block_sums_outliers_and_ranges(dev):
    """Outliers in some blocks, blocks of tiny (also denormal) values, a block of zeros: each block
    is rounded against its own largest value, so the bound holds for every block alone."""
    rng = np.random.default_rng(5)
    K, N = 1280, 40
    sign, _ = _weight(rng, N, K)
    x = rng.standard_normal(K).astype(np.float32)
    x[5], x[700] = 3e4, -2e30
    x[128:256] *= np.float32(1e-20)
    x[256:384] = 0
    x[384:512] = rng.integers(-40, 40, 128).astype(np.float32) * np.float32(1e-45)
    for blk in range(K // 128):
        sc = np.zeros((N, K // 128), np.float32)
        sc[:, blk] = 1.5
        _check_gemv(_run(sign, sc, x, np.zeros(N, np.float32)), x, sign, sc)


def test_block_sums_infinities_and_nan(dev):
    rng = np.random.default_rng(6)
    K, N = 1024, 40
    sign, sc = _weight(rng, N, K)
    h = rng.standard_normal(N).astype(np.float32)
    for spots in ({3: np.inf}, {700: -np.inf}, {130: np.inf, 900: np.inf}, {130: np.inf, 131: -np.inf}, {64: np.nan}):
        x = rng.standard_normal(K).astype(np.float32)
        for i, v in spots.items():
            x[i] = v
        w = np.where((sign[:, np.arange(K) // 32] >> (np.arange(K) % 32)) & 1, 1.0, -1.0) * np.repeat(sc, 128, 1)
        with np.errstate(invalid="ignore"):
            want = (w * x).sum(1) + h
        got = _run(sign, sc, x, h)
        assert np.array_equal(np.isnan(got), np.isnan(want)) and not np.isfinite(got).any()
        assert np.array_equal(got[~np.isnan(got)], want[~np.isnan(want)])


@pytest.mark.parametrize("K,N", [(128, 40), (384, 16), (640, 8209), (4224, 40), (8320, 40), (16512, 40)])
@pytest.mark.parametrize("v", [np.inf, -np.inf])
def test_infinity_in_the_last_block(dev, K, N, v):
    """K / 128 no multiple of 4: the last 512-weight step has lanes past the row's end, which load the
    last block again. An infinity there gives the row's own infinity, not NaN."""
    rng = np.random.default_rng(K + N)
    sign, sc = _weight(rng, N, K)
    x, h = (rng.standard_normal(n).astype(np.float32) for n in (K, N))
    x[K - 3] = v
    bit = (sign[:, (K - 3) // 32] >> ((K - 3) % 32)) & 1
    assert np.array_equal(_run(sign, sc, x, h), np.where(bit, v, -v).astype(np.float32))


def test_infinity_in_the_last_block_fused(dev):
    """The same through the fused qkv projection, on the values it appends (keys and queries are
    normalized, so there the infinity is NaN by the norm)."""
    H, KV, D, K, pos = 16, 4, 128, 640, 5
    rng = np.random.default_rng(8)
    sign, sc = _weight(rng, (H + 2 * KV) * D, K)
    x = rng.standard_normal(K).astype(np.float32)
    x[K - 1] = np.inf
    cos, sin, _, _ = rope_dev(1e6, D, 64)
    c = E.KvCache(1, KV, D, "f32", max_seq_len=64, capacity=64)
    g = t(np.ones(D, np.float32))
    E.qkv_proj_prologue(c, 0, t(x), _dev_weight(sign, sc, K, H * D, KV * D, KV * D), H, g, g, 1e-6, cos, sin, D, pos, pos)
    torch.cuda.synchronize()
    _, v, _, _ = export_k_v(c, 0, pos, 1)
    bit = sign[(H + KV) * D:, -1] >> 31
    assert np.array_equal(v.ravel(), np.where(bit, np.inf, -np.inf).astype(np.float32))
    c.close()
