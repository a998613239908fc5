"""Two-level general steps on strips (large steps), forced on small levels.

NVPRO_PYRAMID_THIN=0 makes every two-level general step whose first level is at
least 2x2 run strips of 63 second-level columns by 7 or 8 rows.  The sizes put
the second level's edges at, one before and one past a strip's and a group's,
with each remainder of the input's sides modulo 4 (the kernel sizes 2 and 3 of
both levels, and one to three columns at the right edge).  sRGBA8 must equal the
oracle's FP32 emulator bit for bit, the float formats the thin tiles' bytes, and
no byte outside the levels written may change.
"""
import os

import numpy as np
import pytest

from tests import helpers as H
from vk_compute_mipmaps_amd import hip_rt
from vk_compute_mipmaps_amd import pyramid as P
from vk_compute_mipmaps_amd import synth

pytestmark = pytest.mark.gpu

POISON = 0xA5


def _run(w, h, fmt, arith, level0, stream, mode, pad=0, levels=3):
    """Levels 0..2 with rows `pad` texels longer than the levels, in a poisoned buffer with a margin."""
    bpt = P.BYTES_PER_TEXEL[fmt]
    offs, pitches, total = [], [], 0
    for l in range(levels):
        lw, lh = P.level_dims(w, h, l)
        offs.append(total)
        pitches.append((lw + pad) * bpt)
        total += pitches[-1] * lh
    host = np.full(total + 256, POISON, np.uint8)
    for y in range(h):
        host[y * pitches[0]:y * pitches[0] + w * bpt] = level0[y].reshape(-1).view(np.uint8)
    ptr = hip_rt.malloc(host.nbytes)
    old = os.environ.get("NVPRO_PYRAMID_THIN")
    os.environ["NVPRO_PYRAMID_THIN"] = mode
    try:
        hip_rt.memcpy_htod(ptr, host.ctypes.data, host.nbytes)
        image = P.make_image(ptr, w, h, levels, offs, pitches)
        P.nvpro_cmd_pyramid_dispatch(stream, P.pipelines(fmt, False, arith), image, levels)
        hip_rt.stream_sync(stream)
        out = np.empty_like(host)
        hip_rt.memcpy_dtoh(out.ctypes.data, ptr, out.nbytes)
        return out, offs, pitches
    finally:
        if old is None:
            os.environ.pop("NVPRO_PYRAMID_THIN", None)
        else:
            os.environ["NVPRO_PYRAMID_THIN"] = old
        hip_rt.free(ptr)


WIDTHS = [4, 5, 7, 62 * 4 + 1, 63 * 4, 63 * 4 + 1, 63 * 4 + 2, 63 * 4 + 3, 64 * 4 + 3, 126 * 4 + 3, 127 * 4 + 2]
HEIGHTS = [4, 6, 7, 27, 28, 31, 33, 14 * 4 + 3, 16 * 4 + 1]


@pytest.mark.parametrize("w", WIDTHS)
def test_strips_srgba8_against_oracle(w, stream):
    for h in HEIGHTS:
        for pad in (0, 3):
            print(f"strips {w}x{h} pad {pad}", flush=True)
            level0 = synth.srgba8(w, h, w + h)
            out, offs, pitches = _run(w, h, P.FORMAT_SRGBA8, P.ARITH_FP32, level0, stream, "0", pad)
            emu = H.emulate_srgba8(H.host_chain(w, h, level0, 3), w, h, P.plan(w, h, 3, fast=False), 3)
            want = np.full_like(out, POISON)
            for (o, lw, lh), at, pitch in zip(H.level_slices(w, h, 3), offs, pitches):
                rows = emu[o:o + lw * lh * 4].reshape(lh, lw * 4)
                for y in range(lh):
                    want[at + y * pitch:at + y * pitch + lw * 4] = rows[y]
            assert np.array_equal(out, want), f"{w}x{h} pad {pad}"


@pytest.mark.parametrize("fmt,arith", [(P.FORMAT_RGBA16F, P.ARITH_FP32), (P.FORMAT_RGBA16F, P.ARITH_PACKED_FP16),
                                       (P.FORMAT_RGBA32F, P.ARITH_FP32)])
@pytest.mark.parametrize("w", [5, 63 * 4 + 3, 64 * 4 + 2, 127 * 4 + 1])
def test_strips_float_equal_thin_tiles(w, fmt, arith, stream):
    for h in (7, 31, 34, 65):
        print(f"strips {w}x{h} format {fmt} arithmetic {arith}", flush=True)
        rng = np.random.default_rng(w * h)
        level0 = synth.rgba16f(w, h, 7) if fmt == P.FORMAT_RGBA16F else rng.random((h, w, 4), dtype=np.float32)
        strips = _run(w, h, fmt, arith, level0, stream, "0", 1)[0]
        thin = _run(w, h, fmt, arith, level0, stream, "1", 1)[0]
        assert np.array_equal(strips, thin), f"{w}x{h}"
