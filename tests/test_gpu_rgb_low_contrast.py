"""rgb hashes on bright frames with faint detail: the luma's rounding in FP32 is then a visible
part of its gradient, so a bucket decided from it differs from the one decided in FP64.  Every
step of full RAVU is compared, steps 2 and 3 from the int11 plane that the device predicted."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _frame(w, h, kind):
    rng = np.random.default_rng(41)
    y, x = np.mgrid[0:h, 0:w]
    base = 0.85 + 0.08 * np.sin(x / 90.0) * np.cos(y / 70.0)
    detail = {"u10": 1.5e-3, "f32": 2e-4}[kind] * rng.standard_normal((h, w))
    img = np.stack([base * k + detail * m for k, m in ((1.0, 1.0), (0.93, 1.1), (0.98, 0.8))])
    return np.round(img * 1023).astype(np.uint16) if kind == "u10" else img.astype(np.float32)


def _check(got, row, theta, step):
    # an angle that is a multiple of pi/24 up to its own last bits is decided by atan2's last bit
    u = theta * 24 / np.pi
    tie = (np.abs(u - np.round(u)) < 1e-13) & (np.abs(got - row) == step)
    assert int(((got != row) & ~tie).sum()) == 0


@pytest.mark.parametrize("kind", ["u10", "f32"])
@pytest.mark.parametrize("name", ["ravu-r2-rgb", "ravu-r3-rgb", "ravu-r4-rgb"])
def test_full(name, kind):
    import mpx
    from oracle import common, ravu
    w, h, n = 460, 300, 2 * int(name[6])
    img = _frame(w, h, kind)
    out, bk = mpx.upscale(name, torch.from_numpy(img).cuda(), bits=10, out_dtype=torch.float32, buckets=True)
    rows = bk.cpu().numpy().reshape(3, h, w)
    x = (img.astype(np.float32) / np.float32(1023) if kind == "u10" else img).astype(np.float64)
    int11 = out.cpu().numpy()[:, 1::2, 1::2].astype(np.float64)
    steps = [ravu._window(x, "rgb", -(n // 2 - 1), n)] + [ravu._lattice_samples(x, int11, "rgb", n, s) for s in (2, 3)]
    for got, (_, lum) in zip(rows, steps):
        a, b, d = common.structure_tensor(lum, n, five_point=True)
        ang, st, co, diag = common.hash_abd(a, b, d, common.STRENGTH_LOG2)
        _check(got, common.lut_row(ang, st, co, 9, 648), diag["theta"], 27)


@pytest.mark.parametrize("kind", ["u10", "f32"])
@pytest.mark.parametrize("name", ["ravu-3x-r2-rgb", "ravu-3x-r3-rgb", "ravu-3x-r4-rgb"])
def test_3x(name, kind):
    import mpx
    from oracle import ravu
    img = _frame(700, 500, kind)
    _, bk = mpx.upscale(name, torch.from_numpy(img).cuda(), bits=10, out_dtype=torch.float16, buckets=True)
    x = (img.astype(np.float32) / np.float32(1023) if kind == "u10" else img).astype(np.float64)
    _, info = ravu.ravu_3x(x, int(name[9]), "rgb")
    _check(bk.cpu().numpy().reshape(info["row"].shape), info["row"], info["diag"]["theta"], 9)


@pytest.mark.parametrize("kind", ["u10", "f32"])
@pytest.mark.parametrize("name,size", [("ravu-zoom-r2-rgb", (800, 600)), ("ravu-zoom-r3-rgb", (800, 600)),
                                       ("ravu-zoom-r3-rgb", (507, 431)), ("ravu-zoom-ar-r2-rgb", (600, 450))])
def test_zoom(name, size, kind):
    import mpx
    from oracle import common, ravu
    w, h, r = 400, 300, 3 if "r3" in name else 2
    img = _frame(w, h, kind)
    _, bk = mpx.upscale(name, torch.from_numpy(img).cuda(), target=size, bits=10, out_dtype=torch.float16,
                        buckets=True)
    x = (img.astype(np.float32) / np.float32(1023) if kind == "u10" else img).astype(np.float64)
    _, info = ravu.ravu_zoom(x, r, *size, ar="-ar-" in name, channels="rgb")
    _check(bk.cpu().numpy().reshape(info["row"].shape), info["row"], info["diag"]["theta"], 12)
