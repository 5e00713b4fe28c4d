"""Buckets of frames with infinities, NaN and values whose squares overflow FP32: windows whose
tensor is not finite take LUT row 0 as in the FP64 oracle, all others their own row."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _frame(planes, kind):
    rng = np.random.default_rng(29)
    img = rng.random((planes, 61, 83)).astype(np.float32)
    if kind == "large":
        return img * np.float32(1e25)
    v = np.float32({"inf": np.inf, "-inf": -np.inf, "nan": np.nan, "max": 3e38}[kind])
    img[0, 20, 30] = img[-1, 45, 61] = v
    img[:, 33, 10] = v
    return img


@pytest.mark.parametrize("kind", ["inf", "-inf", "nan", "max", "large"])
@pytest.mark.parametrize("name", ["ravu-lite-r2", "ravu-lite-r3", "ravu-lite-r4", "ravu-3x-r2", "ravu-3x-r4-rgb",
                                  "ravu-r2", "ravu-r2-rgb", "ravu-r3", "ravu-r3-rgb", "ravu-r4"])
def test_buckets(name, kind):
    import mpx
    from oracle import ravu
    ch = "rgb" if name.endswith("rgb") else "luma"
    img = _frame(3 if ch == "rgb" else 1, kind)
    img = img if ch == "rgb" else img[0]
    x, r = img.astype(np.float64), int(name.split("-r")[1][0])
    with np.errstate(all="ignore"):
        _, info = ravu.ravu_lite(x, r) if "lite" in name else (ravu.ravu_3x if "3x" in name else ravu.ravu)(x, r, ch)
    row = info["row"]["int11"] if isinstance(info["row"], dict) else info["row"]
    _, bk = mpx.upscale(name, torch.from_numpy(img).cuda(), buckets=True)
    got = bk.cpu().numpy().reshape(-1)[:row.size].reshape(row.shape)
    assert np.array_equal(got, row)
