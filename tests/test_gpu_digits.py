"""The sequence body's digit expansion (digits23_4): every value within three quarters of a unit of x * 8323072 / amax (its
fused multiply-add rounds to halves at most, the conversion by half at most), and without a mean error over the tokens
(lanes) in any band of magnitudes (ties taken up by all of them gave 1/4 and 1/8 of a unit in the upper ones)."""
import numpy as np
import pytest
import torch

import stage_hooks as H

pytestmark = pytest.mark.gpu


def _q(x, amax):
    xd = torch.from_numpy(x).cuda()
    q = torch.empty(x.size, dtype=torch.int32, device="cuda")
    H.call("mgt_digits23", H.ptr(xd), x.size // 4, amax, H.ptr(q))
    return q.cpu().numpy().astype(np.float64)


@pytest.mark.parametrize("amax", [1.0, 3.0, 1e-20, 7e25])
@pytest.mark.parametrize("band", [(0.5, 1.0), (0.25, 0.5), (0.125, 0.25), (0.0, 0.125)])
@pytest.mark.parametrize("sign", [1, -1])
def test_rounding(amax, band, sign):
    rng = np.random.default_rng(5)
    n = 1 << 20
    x = (sign * amax * rng.uniform(*band, n)).astype(np.float32)
    inv = np.float64(np.float32(8323072.0) / np.float32(amax))
    err = _q(x, amax) - x.astype(np.float64) * inv
    assert np.abs(err).max() <= 0.75
    # a standard deviation of at most 0.39 of a unit over 2^20 values: 0.0004 on the mean
    assert abs(err.mean()) <= 0.005, err.mean()


def test_ends():
    x = np.array([1, 1, 1, 1, -1, -1, -1, -1, 0, 0, 0, 0, -0.0, -0.0, -0.0, -0.0], np.float32)
    assert np.array_equal(_q(x, 1.0), 8323072.0 * np.sign(x))
    k = np.arange(-40000, 40000, dtype=np.float32)  # whole numbers across every digit's carry
    assert np.array_equal(_q(k, 8323072.0), k)
    big = np.float32(8323072) - np.arange(4096, dtype=np.float32)
    assert np.array_equal(_q(big, 8323072.0), big) and np.array_equal(_q(-big, 8323072.0), -big)
