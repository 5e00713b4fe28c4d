"""RAVU kernels' FP64 re-decision of few or many near sites of a wave: the two ways give the same
bits.  A site's decision depends on its window alone, so a crop's interior must equal the
frame's, although the sites fall into other waves (dots, one-code noise and patches of 45-degree
stripes, whose edges are exactly on a boundary)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

W, H, M = 150, 70, 14  # M: farther than an output's window reaches through full RAVU's three steps


def _frame():
    rng = np.random.default_rng(12)
    y, x = np.mgrid[0:H, 0:W]
    img = (rng.random((H, W)) < 0.01).astype(np.float32)
    img[:, 50:95] = ((rng.random((H, 45)) < 0.05) / 255.0).astype(np.float32)
    stripes = ((x + y) // 8 % 2).astype(np.float32)
    img[:, 95:] = stripes[:, 95:]
    img[30:33, 10:40] = stripes[30:33, 10:40]
    return img


@pytest.mark.parametrize("name", ["ravu-r2-rgb", "ravu-r3", "ravu-r3-rgb", "ravu-r4", "ravu-r4-yuv", "ravu-r4-rgb",
                                  "ravu-zoom-r2", "ravu-zoom-ar-r2-yuv", "ravu-zoom-r3", "ravu-zoom-r3-rgb"])
def test_crops_equal_frame(name):
    import mpx
    img = _frame()
    if name.endswith(("rgb", "yuv")):
        img = np.stack([img, img[:, ::-1], img])
    def run(a):
        size = (2 * a.shape[-1], 2 * a.shape[-2])
        return mpx.upscale(name, torch.from_numpy(np.ascontiguousarray(a)).cuda(),
                           target=size if "zoom" in name else None).cpu().numpy()
    full = run(img)
    for dx, dy in ((1, 0), (0, 1), (7, 3), (16, 5), (33, 2)):
        part = run(img[..., dy:, dx:])
        assert np.array_equal(part[..., 2 * M:-2 * M, 2 * M:-2 * M],
                              full[..., 2 * (dy + M):-2 * M, 2 * (dx + M):-2 * M]), (dx, dy)
