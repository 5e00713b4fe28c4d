"""ravu-zoom's rounding error against the FP64 oracle is no larger than that of the plain FP32
evaluation: each weight by the two nested interpolations, all taps in one running sum, every step
a fused multiply-add (emulated in FP64, whose product of two FP32 numbers is exact)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

W, H = 200, 120


def _fma(a, b, c):
    return (a.astype(np.float64) * b + c).astype(np.float32)


def _lerp2(lut, g, f, ty):
    """FP32 bilinear fetch of group g's four weights at column phase f and texel row ty."""
    one = np.float32(1)
    tx = np.float32(8) * f
    x0, y0 = np.minimum(np.floor(tx), 7), np.floor(ty)
    ax, ay = (tx - x0)[..., None], (ty - y0)[..., None].astype(np.float32)
    x = 9 * g + x0.astype(int)
    y = np.clip(y0.astype(int), 0, lut.shape[0] - 1), np.clip(y0.astype(int) + 1, 0, lut.shape[0] - 1)
    rows = [_fma(lut[r, x], one - ax, lut[r, x + 1] * ax) for r in y]
    return _fma(rows[0], one - ay, rows[1] * ay)


def _plain(x, r, ow, oh, row):
    from oracle.common import load_lut16
    lut, n = load_lut16("ravu_zoom_lut%d" % r).astype(np.float32), 2 * r
    def phase(o, i, out):
        num = (2 * np.arange(o) + 1) * i - out
        b = num // (2 * out)
        return b, ((num - b * 2 * out).astype(np.float32) / np.float32(2 * out))
    bx, fx = phase(ow, W, ow)
    by, fy = phase(oh, H, oh)
    fx, fy = np.broadcast_to(fx[None, :], (oh, ow)), np.broadcast_to(fy[:, None], (oh, ow))
    acc, half = np.zeros((oh, ow), np.float32), n * n // 2
    def sample(i):
        ys, xs = np.clip(by + i % n - (r - 1), 0, H - 1), np.clip(bx + i // n - (r - 1), 0, W - 1)
        return x[ys[:, None], xs[None, :]]
    for g in range((half + 3) // 4):
        # (the integer row base is kept apart, so the phase keeps its FP32 precision)
        wf = _lerp2(lut, g, fx, 9.0 * row + np.float32(8) * fy)
        wi = _lerp2(lut, g, np.float32(1) - fx, 9.0 * row + np.float32(8) * (np.float32(1) - fy))
        for c in range(min(4, half - 4 * g)):
            p = 4 * g + c
            acc = _fma(sample(n * n - 1 - p), wi[..., c], _fma(sample(p), wf[..., c], acc))
    return np.clip(acc, 0, 1)


@pytest.mark.parametrize("name,size", [("ravu-zoom-r2", (301, 177)), ("ravu-zoom-r3", (301, 177)),
                                       ("ravu-zoom-r2", (300, 180)), ("ravu-zoom-r3", (300, 180))])
def test_no_larger_than_plain_fp32(name, size):
    import mpx
    from oracle.ravu import ravu_zoom
    r = int(name[-1])
    y, x = np.mgrid[0:H, 0:W]
    err = np.zeros(2)
    for seed in range(4):
        v = 0.5 + 0.3 * np.sin(x / (5.0 + seed)) * np.cos(y / 7.0) + 0.01 * np.random.default_rng(seed).standard_normal((H, W))
        img = np.clip(v, 0, 1).astype(np.float32)
        ref, info = ravu_zoom(img.astype(np.float64), r, *size)
        got, bk = mpx.upscale(name, torch.from_numpy(img).cuda(), target=size, buckets=True)
        same = bk.cpu().numpy().reshape(info["row"].shape) == info["row"]
        plain = _plain(img, r, *size, info["row"])
        err += [(((a - ref) * same) ** 2).sum() for a in (got.cpu().numpy().astype(np.float64), plain)]
    assert err[0] <= err[1], np.sqrt(err / (4 * size[0] * size[1]))
