"""The shared FP64 re-decision of a wave: frames on which no, some or all lanes are near a
bucket boundary (exact diagonal ramps, noise, both), at sizes with partly filled tiles."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (33, 9), (70, 21)]


def _frame(w, h, planes):
    rng = np.random.default_rng(w)
    y, x = np.mgrid[0:h, 0:w]
    img = np.empty((planes, h, w))
    for c in range(planes):
        v = ((x + (1 if c % 2 else -1) * y) % 32) / 64.0 + 0.25   # a = d exactly: angle on a boundary
        n = rng.integers(0, 256, size=(h, w)) / 255.0
        img[c] = np.where((x // 11 + y // 5) % 3 == 0, n, v)
    return img.astype(np.float32)


@pytest.mark.parametrize("name", ["ravu-r3", "ravu-r4", "ravu-r2-rgb", "ravu-r3-rgb", "ravu-r4-rgb", "ravu-r4-yuv",
                                  "ravu-zoom-r3", "ravu-zoom-r3-rgb", "ravu-zoom-ar-r2", "ravu-zoom-ar-r2-rgb"])
@pytest.mark.parametrize("w,h", SIZES)
def test_buckets(name, w, h):
    import mpx
    from oracle import ravu
    ch = "rgb" if name.endswith("rgb") else "yuv" if name.endswith("yuv") else "luma"
    img = _frame(w, h, 1 if ch == "luma" else 3)
    img = img[0] if ch == "luma" else img
    r = int(name.split("-r")[1][0])
    x = img.astype(np.float64)
    if "zoom" in name:
        out = (2 * w + 3, 2 * h + 1)
        _, info = ravu.ravu_zoom(x, r, *out, ar="-ar-" in name, channels=ch)
        row, theta = info["row"], info["diag"]["theta"]
    else:
        out = None
        _, info = ravu.ravu(x, r, ch)
        row, theta = info["row"]["int11"], info["diag"]["int11"]["theta"]   # (the later steps read int11 in FP32)
    _, bk = mpx.upscale(name, torch.from_numpy(img).cuda(), target=out, buckets=True)
    got = bk.cpu().numpy().reshape(-1)[:row.size].reshape(row.shape)
    # an angle that is a multiple of pi/24 up to its own last bits is decided by the last bit of
    # atan2, in which the device's and NumPy's library may differ: there the neighbouring
    # angle's bucket (12 or 27 rows away) is as good
    u = theta * 24 / np.pi
    tie = (np.abs(u - np.round(u)) < 1e-13) & (np.abs(got - row) == (12 if "zoom" in name else 27))
    assert np.array_equal(np.where(tie, row, got), row), int((got != row).sum())
