"""Buckets where |b| of the structure tensor meets its threshold beside large a and d: thin crossing
lines (whose b cancels) with faint noise.  There the FP32 hash has the least room between its
error bound and its margin."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _lines(w, h, planes, noise):
    rng = np.random.default_rng(23)
    img = np.full((planes, h, w), 0.1)
    img[:, rng.integers(0, h, h // 7)] = 0.9
    img[:, :, rng.integers(0, w, w // 7)] = 0.9
    img[:, :, w // 2:] *= rng.uniform(0.2, 1.0, (1, 1, w - w // 2))
    return (img + noise * rng.standard_normal(img.shape)).astype(np.float32)


@pytest.mark.parametrize("noise", [0.0, 1e-7, 1e-6])
@pytest.mark.parametrize("name", ["ravu-lite-r2", "ravu-lite-r3", "ravu-lite-r4", "ravu-3x-r3", "ravu-3x-r4-rgb",
                                  "ravu-r2", "ravu-r2-rgb", "ravu-r3", "ravu-r4", "ravu-r4-rgb", "ravu-zoom-r2",
                                  "ravu-zoom-r3", "ravu-zoom-r3-rgb"])
def test_buckets_of_thin_lines(name, noise):
    import mpx
    from oracle import ravu
    ch = "rgb" if name.endswith("rgb") else "luma"
    w, h, r = 203, 131, int(name.split("-r")[1][0])
    img = _lines(w, h, 3 if ch == "rgb" else 1, noise)
    img = img if ch == "rgb" else img[0]
    x = img.astype(np.float64)
    size = (305, 197) if "zoom" in name else None
    if "lite" in name:
        _, info = ravu.ravu_lite(x, r)
        row, theta, step = info["row"], info["diag"]["theta"], 12
    elif "3x" in name:
        _, info = ravu.ravu_3x(x, r, ch)
        row, theta, step = info["row"], info["diag"]["theta"], 9
    elif "zoom" in name:
        _, info = ravu.ravu_zoom(x, r, *size, channels=ch)
        row, theta, step = info["row"], info["diag"]["theta"], 12
    else:
        _, info = ravu.ravu(x, r, ch)
        row, theta, step = info["row"]["int11"], info["diag"]["int11"]["theta"], 27
    _, bk = mpx.upscale(name, torch.from_numpy(img).cuda(), target=size, buckets=True)
    got = bk.cpu().numpy().reshape(-1)[:row.size].reshape(row.shape)
    # an angle that is a multiple of pi/24 up to its own last bits is decided by atan2's last bit
    u = theta * 24 / np.pi
    tie = (np.abs(u - np.round(u)) < 1e-13) & (np.abs(got - row) == step)
    assert int(((got != row) & ~tie).sum()) == 0
