"""ravu-zoom's per-pixel weight fetch (ratios whose phases do not fit the plan's table):
phase 0 and its mirror 8 (texel pair 7, 8), the first and last LUT rows, odd sizes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["ravu-zoom-r2", "ravu-zoom-r3", "ravu-zoom-r3-rgb", "ravu-zoom-ar-r2-yuv",
                                  "ravu-zoom-ar-r2"])
@pytest.mark.parametrize("ins,outs", [((31, 20), (279, 180)), ((40, 30), (53, 47)), ((67, 9), (68, 103))])
def test_zoom_fetch(name, ins, outs):
    import mpx
    from oracle.ravu import ravu_zoom
    rng = np.random.default_rng(9)
    ch = "rgb" if name.endswith("rgb") else "yuv" if name.endswith("yuv") else "luma"
    img = rng.random((3, ins[1], ins[0])).astype(np.float32)
    img[:, : ins[1] // 2] = np.round(img[:, : ins[1] // 2])
    img[:, :, : ins[0] // 3] = 0.5   # flat: bucket 0
    if ch == "luma":
        img = img[0]
    got = mpx.upscale(name, torch.from_numpy(img).cuda(), target=outs).cpu().numpy()
    want, _ = ravu_zoom(img.astype(np.float64), int(name.split("-r")[1][0]), outs[0], outs[1], ar="-ar-" in name,
                        channels=ch)
    # FP32 sums of up to 36 taps, weights of four rounded products (the family's bar)
    assert np.abs(got - want).max() <= 2e-5
