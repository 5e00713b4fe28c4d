"""The resampler's tile edges and its two orders of work (rows kept in LDS, rows filtered
directly under strong downscaling) against the FP64 restatement, for every element type."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# (in size, out size): one pixel, a tile and its neighbours (64 x 8 .. 64 x 32), upscaling by
# a large factor, moderate and strong downscaling (rows past what a tile keeps), one axis of each
SIZES = [((1, 1), (1, 1)), ((5, 3), (65, 33)), ((63, 31), (64, 8)), ((130, 70), (129, 9)), ((33, 17), (640, 330)),
         ((200, 300), (63, 31)), ((90, 2000), (64, 40)), ((2000, 40), (17, 90)), ((700, 700), (20, 7))]


@pytest.mark.parametrize("name,src", [("bilinear", "f16"), ("catmull_rom", "u8"), ("mitchell", "f32"),
                                      ("spline36", "u16"), ("lanczos3", "f16"), ("lanczos3", "u8")])
def test_resample_tiles(name, src):
    import mpx
    from oracle.resample import resample
    rng = np.random.default_rng(11)
    for (w, h), (ow, oh) in SIZES:
        v = rng.integers(0, 256, size=(h, w))
        if src in ("u8", "u16"):
            x = torch.from_numpy(v.astype(np.int32)).to(torch.uint8 if src == "u8" else torch.uint16).cuda()
            ref = v / (255.0 if src == "u8" else 1023.0)
        else:
            ref = (v / 255.0).astype(np.float16 if src == "f16" else np.float32)
            x = torch.from_numpy(ref).cuda()
        got = mpx.resample(x, (ow, oh), offset=(-0.5, 0.25), filter=name, bits=10).float().cpu().numpy()
        want = resample(np.asarray(ref, dtype=np.float64), ow, oh, (-0.5, 0.25), name)
        # FP32 position: |t| <= 2000 has half an ulp 2^-14 after three roundings, moving a
        # weight by at most pi/2 per texel and tap over 2 axes; FP16 output adds 2^-11 |v|
        n = max(w, h, 2)
        tol = 4 * 1.6 * 3 * 2.0 ** (int(np.ceil(np.log2(n))) - 25) + 2e-6
        if src == "f16":
            tol += 2.0 ** -11 * (1 + np.abs(want).max())
        assert np.abs(got - want).max() <= tol, (name, src, (w, h), (ow, oh))
