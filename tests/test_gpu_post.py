"""The step after the path on the GPU: tone mapping equals the oracle's
bytes (double-evaluated pow), progressive accumulation of two trace calls
equals the oracle's accumulation of the same two images and the single
render of all their samples to FP32 rounding."""
import math

import numpy as np
import pytest

import vk_cinematic_amd as V
from vk_cinematic_amd import scenes
from test_post import _tonemap, SPO_TX_CR
from _libs import oracle

pytestmark = pytest.mark.gpu


def _render(device, s, cam, w, h, spp, offset, img):
    ctx = V.make_context(cam, s, spp=spp, bounces=3, clamp=0.0,
                         estimator=V.EST_UNBIASED, rng=V.RNG_PCG, seed=9,
                         sample_offset=offset)
    V.path_trace_tiles_device(ctx, V.ComputeTiles(w, h, 64, 64), img)
    return img.download(np.float32, w * h * 4)


def test_tonemap_matches_oracle(device):
    desc = scenes.config1(64, 48)
    s, cam = scenes.load_gpu(device, desc)
    img = device.alloc(64 * 48 * 16)
    px = _render(device, s, cam, 64, 48, 4, 0, img)
    for exposure in (1.0, 0.3):
        got = device.tonemap(img, 64 * 48, exposure, V.TX_DOUBLE)
        assert np.array_equal(got, _tonemap(px, exposure, SPO_TX_CR))
        fast = device.tonemap(img, 64 * 48, exposure, V.TX_FAST)
        assert np.max(np.abs(fast.astype(int) - got.astype(int))) <= 1
    img.free()
    s.close()


def test_progressive_accumulation(device):
    desc = scenes.config1(64, 48)
    s, cam = scenes.load_gpu(device, desc)
    n = 64 * 48
    acc, part, full = device.alloc(n * 16), device.alloc(n * 16), device.alloc(n * 16)
    a = _render(device, s, cam, 64, 48, 2, 0, acc)
    b = _render(device, s, cam, 64, 48, 2, 2, part)
    device.accumulate(acc, part, n, 2, 2)
    got = acc.download(np.float32, n * 4)
    want = a.copy()
    oracle().spo_accumulate(want, np.ascontiguousarray(b), n, 2, 2)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    whole = _render(device, s, cam, 64, 48, 4, 0, full)
    assert np.allclose(got, whole, rtol=1e-5, atol=1e-7)
    for buf in (acc, part, full):
        buf.free()
    s.close()


def _around_steps():
    """Radiances whose c / (1 + c), in float32 as the tone map forms it, lies
    as closely below and above each of the 255 steps of the byte as a float32
    c reaches (the step itself and the float below it wherever they have a c:
    a value just below a power of two often has none), and the floats within
    40 of each step's preimage."""
    picked, tight = [], 0
    for k in range(1, 256):
        def byte(x):   # of the double power, rounded once to float
            g = np.array([math.pow(float(v), float(np.float32(1.0) / np.float32(2.2)))
                          for v in x]).astype(np.float32)
            return np.rint(g * np.float32(255.0))

        at = ((k - 0.5) / 255.0) ** 2.2
        c0 = at / (1.0 - at)
        width = int(60 + 8 * (1 + c0))   # about 1 + c floats c share a value
        c = (np.float32(c0).view(np.int32) + np.arange(-width, width + 1)).astype(np.int32)
        c = c.view(np.float32)
        x = c / (np.float32(1.0) + c)
        above = byte(x) >= k
        assert above.any() and not above.all()
        lo = int(np.argmax(np.where(above, -1.0, x)))    # (x need not rise with c:
        hi = int(np.argmin(np.where(above, x, 2.0)))     # 1 + c rounds too)
        tight += int(x[hi].view(np.int32) - x[lo].view(np.int32) == 1)
        picked += [c[lo], c[hi]]
        picked += list(c[width - 40: width + 41])
    assert tight > 200                   # most steps have both neighbours
    return np.array(picked, np.float32)


@pytest.mark.parametrize("pixels", [1, 255, 257, 2048 * 256 + 3])
def test_tonemap_bytes_at_every_step(device, pixels):
    """Radiances around each of the 255 steps of the byte, and the values
    outside [0, 1): the oracle's bytes exactly.  (The steps themselves are
    pinned float by float on the CPU, tests/test_post.py.)"""
    near = _around_steps()
    odd = np.array([0.0, -0.0, 1e-45, 1e-38, 3e38, np.inf, -np.inf, np.nan, -0.5, -1.0,
                    -2.0, -1e-45, -3e38, 2.0 ** 24, 2.0 ** 25, 1.0], np.float32)
    px = np.resize(np.concatenate([odd, near]), pixels * 4).astype(np.float32)
    img = device.alloc(pixels * 16)
    img.upload(px)
    for exposure in (1.0, 2.0, -1.0):
        got = device.tonemap(img, pixels, exposure, V.TX_DOUBLE)
        assert np.array_equal(got, _tonemap(px, exposure, SPO_TX_CR))
    img.free()
