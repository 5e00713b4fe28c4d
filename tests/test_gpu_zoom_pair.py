"""ravu-zoom at exactly twice the width (two outputs per thread): edges of the shifted pair grid,
odd sizes, heights at other ratios."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["ravu-zoom-r2", "ravu-zoom-r3-yuv", "ravu-zoom-r3-rgb", "ravu-zoom-ar-r2",
                                  "ravu-zoom-ar-r2-rgb"])
@pytest.mark.parametrize("ins,outs", [((2, 1), (4, 2)), ((31, 20), (62, 40)), ((32, 9), (64, 21)),
                                      ((95, 17), (190, 18))])
def test_zoom_pair(name, ins, outs):
    import mpx
    from oracle.ravu import ravu_zoom
    rng = np.random.default_rng(10)
    ch = "rgb" if name.endswith("rgb") else "yuv" if name.endswith("yuv") else "luma"
    imgs = rng.random((2, 3, ins[1], ins[0])).astype(np.float32)
    imgs[:, :, :, : ins[0] // 3] = 0.5   # flat: bucket 0
    if ch == "luma":
        imgs = imgs[:, 0]
    plan = mpx.default_context().plan(name, *ins, target=outs, max_batch=2)
    for tile in range(plan.tile()["count"]):
        plan.set_tile(tile)
        got = plan.run(torch.from_numpy(imgs).cuda()).cpu().numpy()
        for f in range(2):
            want, _ = ravu_zoom(imgs[f].astype(np.float64), int(name.split("-r")[1][0]), outs[0], outs[1],
                                ar="-ar-" in name, channels=ch)
            # FP32 sums of up to 36 taps, weights of four rounded products (the family's bar)
            assert np.abs(got[f].reshape(want.shape) - want).max() <= 2e-5
