"""Bucket decisions at their boundaries: planes whose gradient angle sits on (or next to) a
multiple of pi/24 and whose strength sits near the thresholds, where the FP32 hash has to
hand over to its FP64 form, and planes with infinities and NaN, which must not fault."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

VARIANTS = ["ravu-lite-r2", "ravu-lite-ar-r3", "ravu-lite-r4", "ravu-3x-r2", "ravu-3x-r3", "ravu-r2", "ravu-r3",
            "ravu-r4"]


def _ramps(kind):
    """64 x 64 plane in FP32: tiles of 16 x 16, each a ramp of its own angle and slope."""
    rng = np.random.default_rng(5)
    y, x = np.mgrid[0:16, 0:16].astype(np.float64)
    img = np.zeros((64, 64))
    for i in range(16):
        ang = (3 * i + rng.integers(0, 2)) * np.pi / 24 + rng.choice([0, 1e-6, -1e-6, 3e-5, -3e-5])
        s = {"lite": rng.choice([0.004, 0.016, 0.05]), "3x": rng.choice([0.005, 0.02]),
             "log2": 2.0 ** rng.integers(1, 6) / 2000}[kind] * (1 + rng.choice([0, 1e-6, -1e-6, 5e-5]))
        v = 0.5 + s * ((x - 8) * np.cos(ang) + (y - 8) * np.sin(ang))
        img[16 * (i // 4):16 * (i // 4) + 16, 16 * (i % 4):16 * (i % 4) + 16] = v
    return np.clip(img, 0, 1).astype(np.float32)


@pytest.mark.parametrize("name", VARIANTS)
def test_buckets_at_boundaries(name):
    import mpx
    from oracle import ravu
    kind = "lite" if "lite" in name else "3x" if "3x" in name else "log2"
    img = _ramps(kind)
    _, bk = mpx.upscale(name, torch.from_numpy(img).cuda(), buckets=True)
    r = int(name[-1])
    x = img.astype(np.float64)
    if kind == "lite":
        row = ravu.ravu_lite(x, r, ar="-ar-" in name)[1]["row"]
    elif kind == "3x":
        row = ravu.ravu_3x(x, r)[1]["row"]
    else:
        row = ravu.ravu(x, r)[1]["row"]["int11"]   # (the later steps read int11 in FP32)
    got = bk.cpu().numpy().reshape(-1)[:row.size].reshape(row.shape)
    assert np.array_equal(got, row), int((got != row).sum())


@pytest.mark.parametrize("name", ["ravu-lite-ar-r3", "ravu-3x-r3", "ravu-r3", "ravu-zoom-r2"])
def test_nonfinite_samples_stay_local(name):
    """A NaN or an infinity changes only the outputs whose windows see it."""
    import mpx
    img = _ramps("lite")
    bad = img.copy()
    bad[20, 20], bad[40, 41], bad[41, 41] = np.inf, np.nan, -np.inf
    k = 3 if "3x" in name else 2
    a = mpx.upscale(name, torch.from_numpy(img).cuda()).cpu().numpy()
    b = mpx.upscale(name, torch.from_numpy(bad).cuda()).cpu().numpy()
    far = np.ones(img.shape, bool)
    far[10:31, 10:31] = far[30:52, 31:52] = False
    far = np.kron(far, np.ones((k, k), bool))
    assert np.array_equal(a[far], b[far])
