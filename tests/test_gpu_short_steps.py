"""Two short steps or more in one launch of tiles (before the tail).

Sizes around the tile's edges in each direction: whole and partial last tiles,
every kernel size in the first level, one-texel sides, levels that end with the
tiles (no tail after them), fast and general steps mixed, and the largest that
still take tiles.  sRGBA8 must equal the oracle's FP32 emulator bit for bit;
the float formats must equal the same plan with one launch per step.
"""
import numpy as np
import pytest

from tests import helpers as H
from tests.test_gpu_tail import _step_by_step
from vk_compute_mipmaps_amd import hip_rt
from vk_compute_mipmaps_amd import pyramid as P
from vk_compute_mipmaps_amd import synth

pytestmark = pytest.mark.gpu

SIZES = [(255, 127), (257, 257), (240, 135), (135, 240), (300, 300), (254, 250), (129, 259), (128, 257), (500, 308),
         (4000, 3), (3, 4000), (8191, 1), (1, 8191), (1023, 511), (511, 1023), (1023, 1023), (1000, 500), (1022, 1021)]


def _launches(w, h, level0, fmt, arith, stream, levels):
    chain = P.DeviceMipChain(w, h, fmt)
    try:
        chain.upload_level0(level0)
        chain.dispatch(stream=stream, arithmetic=arith, mip_levels=levels)
        n = P.last_launch_count()
        hip_rt.stream_sync(stream)
        return chain.download(), n
    finally:
        chain.free()


@pytest.mark.parametrize("fast", [True, False])
@pytest.mark.parametrize("w,h", SIZES)
def test_short_steps_srgba8_against_oracle(w, h, fast, stream):
    print(f"short steps {w}x{h} fast {fast}", flush=True)
    level0 = synth.srgba8(w, h, 7 * w + h)
    out = H.gpu_run(w, h, level0, stream, fast=fast)
    emu = H.emulate_srgba8(H.host_chain(w, h, level0), w, h, P.plan(w, h, fast=fast))
    assert np.array_equal(out, emu)


@pytest.mark.parametrize("fmt,arith", [(P.FORMAT_RGBA16F, P.ARITH_FP32), (P.FORMAT_RGBA16F, P.ARITH_PACKED_FP16),
                                       (P.FORMAT_RGBA32F, P.ARITH_FP32)])
def test_short_steps_float_equal_single_steps(fmt, arith, stream):
    for w, h in SIZES:
        print(f"short steps {w}x{h} format {fmt} arithmetic {arith}", flush=True)
        if fmt == P.FORMAT_RGBA16F:
            level0 = synth.rgba16f(w, h, w + h)
        else:
            level0 = np.random.default_rng(w + h).standard_normal((h, w, 4)).astype(np.float32)
        whole = H.gpu_run(w, h, level0, stream, fmt=fmt, arithmetic=arith)
        assert np.array_equal(whole, _step_by_step(w, h, level0, fmt, arith, stream)), f"{w}x{h}"


@pytest.mark.parametrize("w,h", [(255, 127), (1023, 511)])
def test_short_steps_end_with_their_tiles(w, h, stream):
    """Four levels of two steps are one launch."""
    level0 = np.random.default_rng(w).standard_normal((h, w, 4)).astype(np.float32)
    out, launches = _launches(w, h, level0, P.FORMAT_RGBA32F, P.ARITH_FP32, stream, 5)
    full, _ = _launches(w, h, level0, P.FORMAT_RGBA32F, P.ARITH_FP32, stream, 0)
    end = P.chain_bytes(w, h, 5, 16)
    assert launches == 1
    assert np.array_equal(out[:end], full[:end])
