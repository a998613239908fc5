"""Premultiplied alpha on rows of every remainder of the four texels a thread takes.

Widths around a thread's four texels and a segment's 2048, tight rows and rows longer than
the level (whose padding must not change) and more rows than workgroups.
"""
import numpy as np
import pytest

from oracle import orc
from vk_compute_mipmaps_amd import hip_rt
from vk_compute_mipmaps_amd import pyramid as P
from vk_compute_mipmaps_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [P.FORMAT_SRGBA8, P.FORMAT_RGBA16F])
@pytest.mark.parametrize("pad", [0, 3])
@pytest.mark.parametrize("w,h", [(1, 1), (3, 5), (5, 2), (1025, 3), (2047, 3), (2048, 2), (2049, 3), (4100, 2), (2, 5000)])
def test_rows_of_every_remainder(w, h, pad, fmt, stream):
    print(f"premultiply {w}x{h} pad {pad} format {fmt}", flush=True)
    bpt = P.BYTES_PER_TEXEL[fmt]
    level0 = synth.srgba8(w, h, 3) if fmt == P.FORMAT_SRGBA8 else synth.rgba16f(w, h, 3)
    if fmt == P.FORMAT_SRGBA8:
        want0 = orc.premultiply_srgba8(level0, exact=True)
    else:
        f = level0.astype(np.float32)
        want0 = level0.copy()
        want0[..., :3] = (f[..., :3] * f[..., 3:]).astype(np.float16)
    pitch = (w + pad) * bpt
    host = np.full(pitch * h + 64, 0x5A, np.uint8)
    want = host.copy()
    for y in range(h):
        host[y * pitch:y * pitch + w * bpt] = level0[y].reshape(-1).view(np.uint8)
        want[y * pitch:y * pitch + w * bpt] = np.ascontiguousarray(want0[y]).reshape(-1).view(np.uint8)
    ptr = hip_rt.malloc(host.nbytes)
    try:
        hip_rt.memcpy_htod(ptr, host.ctypes.data, host.nbytes)
        P.premultiply_alpha(stream, fmt, P.make_image(ptr, w, h, 1, [0], [pitch]))
        hip_rt.stream_sync(stream)
        out = np.empty_like(host)
        hip_rt.memcpy_dtoh(out.ctypes.data, ptr, out.nbytes)
    finally:
        hip_rt.free(ptr)
    assert np.array_equal(out, want)
