"""MPX_PREC_FP32 of every NNEDI3 network against the FP64 oracle: ragged tiles, near-flat
windows (variance around the threshold) and full contrast."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wh", [4, 6])
@pytest.mark.parametrize("nns", [16, 32, 64, 128, 256])
def test_fp32_accuracy(nns, wh):
    import mpx
    from oracle.nnedi3 import nnedi3
    rng = np.random.default_rng(nns + wh)
    img = rng.random((37, 70)).astype(np.float32)
    img[:, 20:40] = np.round(img[:, 20:40])                       # black and white noise
    img[:, 40:60] = 0.5 + 3e-4 * rng.standard_normal((37, 20))    # v around 1.2e-7
    img[20:, 50:] = 0.25
    got = mpx.upscale("nnedi3-nns%d-win8x%d" % (nns, wh), torch.from_numpy(img).cuda()).cpu().numpy()
    want = nnedi3(img.astype(np.float64), nns, wh)
    # parts of 11 + 11 bits: the sums' error is about 2^-23 |w| |x'| <= 2^-23 * 9.1 * sqrt(48)
    # = 7.5e-6, and a result moves by at most 5 sd (sd <= 1/2) times half of that per unit of
    # softmax weight, taken twice for the two sums
    assert np.abs(got - want).max() <= 1.9e-5
    # typical error: FP32 rounding of a result near 1/2
    assert np.sqrt(np.mean((got - want) ** 2)) <= 2.0 ** -23
