"""The tail kernel (every remaining step of a plan in one workgroup).

Images small enough to be a tail from level 0 on (first output level of at most
1024 texels, two steps or more), at the edges of its range: the most outputs in
each shape, the largest source (2049 x 3), one-texel sides, levels around one
wave's 16 texels, odd and even sides (every kernel size), fast steps, and fast
and general steps mixed.  sRGBA8 must equal the oracle's FP32 emulator bit for
bit; the float formats must equal the same plan with one launch per step, which
partial level counts give (a single remaining step never runs as a tail).
"""
import ctypes

import numpy as np
import pytest

from tests import helpers as H
from vk_compute_mipmaps_amd import hip_rt
from vk_compute_mipmaps_amd import pyramid as P
from vk_compute_mipmaps_amd import synth

pytestmark = pytest.mark.gpu

SIZES = [(2049, 3), (3, 2049), (2049, 1), (1, 2049), (1025, 5), (65, 65), (64, 64), (63, 63), (65, 64), (40, 100),
         (36, 36), (48, 16), (9, 9), (8, 8), (7, 9), (12, 4), (17, 3), (3, 3), (5, 1)]


@pytest.mark.parametrize("fast", [True, False])
@pytest.mark.parametrize("w,h", SIZES)
def test_tail_srgba8_against_oracle(w, h, fast, stream):
    print(f"tail {w}x{h} fast {fast}", flush=True)
    level0 = synth.srgba8(w, h, 5 * w + h)
    out = H.gpu_run(w, h, level0, stream, fast=fast)
    emu = H.emulate_srgba8(H.host_chain(w, h, level0), w, h, P.plan(w, h, fast=fast))
    assert np.array_equal(out, emu)


def _step_by_step(w, h, level0, fmt, arith, stream):
    """The chain with each step of the plan dispatched alone, from its own input level."""
    chain = P.DeviceMipChain(w, h, fmt)
    try:
        chain.upload_level0(level0)
        for s in P.plan(w, h, fmt=fmt):
            # One step: a sub-image whose level 0 is the step's input level.
            lw, lh = P.level_dims(w, h, s.inputLevel)
            n = s.levelCount + 1
            offs = [chain.offsets[s.inputLevel + k] for k in range(n)]
            pitches = [P.level_dims(w, h, s.inputLevel + k)[0] * chain.bpt for k in range(n)]
            image = P.make_image(chain.ptr, lw, lh, n, offs, pitches)
            kind = s.pipeline

            def record(cmd, state, count=s.levelCount, kind=kind):
                return count if P.lib().nvproPyramidCmdDispatch(cmd, kind, count, 1) == 0 else 0

            one = P.DISPATCHER(lambda cmd, state: record(ctypes.c_void_p(cmd), state))
            none = P.DISPATCHER(lambda cmd, state: 0)
            P.nvpro_cmd_pyramid_dispatch_custom(stream, P.pipelines(fmt, True, arith), image, n,
                                                none if kind == P.PIPELINE_FAST else one,
                                                one if kind == P.PIPELINE_FAST else none)
        hip_rt.stream_sync(stream)
        return chain.download()
    finally:
        chain.free()


@pytest.mark.parametrize("fmt,arith", [(P.FORMAT_RGBA16F, P.ARITH_FP32), (P.FORMAT_RGBA16F, P.ARITH_PACKED_FP16),
                                       (P.FORMAT_RGBA32F, P.ARITH_FP32)])
def test_tail_float_equals_single_steps(fmt, arith, stream):
    for w, h in SIZES:
        print(f"tail {w}x{h} format {fmt} arithmetic {arith}", flush=True)
        rng = np.random.default_rng(w + h)
        if fmt == P.FORMAT_RGBA16F:
            level0 = synth.rgba16f(w, h, w + h)
        else:
            level0 = rng.standard_normal((h, w, 4)).astype(np.float32)
            level0[0, 0] = [np.inf, -np.inf, np.nan, np.float32(1e-42)]
        whole = H.gpu_run(w, h, level0, stream, fmt=fmt, arithmetic=arith)
        steps = _step_by_step(w, h, level0, fmt, arith, stream)
        if fmt == P.FORMAT_RGBA32F:  # a NaN's sign and payload are not the filter's
            a, b = whole.view(np.float32), steps.view(np.float32)
            assert np.array_equal(np.isnan(a), np.isnan(b)), f"{w}x{h}"
            whole, steps = np.where(np.isnan(a), 0, a).view(np.uint32), np.where(np.isnan(b), 0, b).view(np.uint32)
        assert np.array_equal(whole, steps), f"{w}x{h}"
