"""Premultiplied alpha on rows longer than the level, several rows to a workgroup's unit.

Widths from one texel to the widest rows that share a unit of 2048 texels, and
past it, heights of less than a unit, a whole number of units and one row more.
Every texel must equal the oracle's, once premultiplied, and the padding must not
change.
"""
import numpy as np
import pytest

from oracle import orc
from vk_compute_mipmaps_amd import hip_rt
from vk_compute_mipmaps_amd import pyramid as P

pytestmark = pytest.mark.gpu

WIDTHS = [1, 2, 3, 4, 5, 7, 15, 16, 17, 31, 33, 63, 64, 65, 100, 127, 128, 129, 230, 256, 257, 300, 409, 410, 511, 512, 513,
          900]


@pytest.mark.parametrize("fmt", [P.FORMAT_SRGBA8, P.FORMAT_RGBA16F])
@pytest.mark.parametrize("w", WIDTHS)
def test_rows_in_units(w, fmt, stream):
    bpt = P.BYTES_PER_TEXEL[fmt]
    unit = 2048 // w
    for h in sorted({1, 2, max(1, unit - 1), unit, unit + 1, 3 * unit + 1}):
        print(f"premultiply units {w}x{h} format {fmt}", flush=True)
        rng = np.random.default_rng(w * 4099 + h)
        if fmt == P.FORMAT_SRGBA8:
            level0 = rng.integers(0, 256, (h, w, 4), dtype=np.uint8)
            want0 = orc.premultiply_srgba8(level0, exact=True)
        else:
            level0 = rng.uniform(0.0, 4.0, (h, w, 4)).astype(np.float16)
            f = level0.astype(np.float32)
            want0 = level0.copy()
            want0[..., :3] = (f[..., :3] * f[..., 3:]).astype(np.float16)
        pitch = (w + 1 + h % 4) * bpt
        host = np.full((h, pitch), 0x5A, np.uint8)
        want = host.copy()
        host[:, :w * bpt] = level0.view(np.uint8).reshape(h, w * bpt)
        want[:, :w * bpt] = np.ascontiguousarray(want0).view(np.uint8).reshape(h, w * bpt)
        ptr = hip_rt.malloc(host.nbytes)
        try:
            hip_rt.memcpy_htod(ptr, host.ctypes.data, host.nbytes)
            P.premultiply_alpha(stream, fmt, P.make_image(ptr, w, h, 1, [0], [pitch]))
            hip_rt.stream_sync(stream)
            out = np.empty_like(host)
            hip_rt.memcpy_dtoh(out.ctypes.data, ptr, out.nbytes)
        finally:
            hip_rt.free(ptr)
        assert np.array_equal(out, want), f"{w}x{h}"
