"""Fast steps with so many tiles that tiles x tiles per row passes 2^32 many times
over: the rows of tiles, found by multiplication, at the far end of wide and of
square levels, for steps of one, two and three levels.  sRGBA8 must equal the
oracle's FP32 emulator bit for bit.  (tests/test_fast_tile_rows.py has every
width on the CPU.)
"""
import numpy as np
import pytest

from tests import helpers as H
from vk_compute_mipmaps_amd import pyramid as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,levels", [(53984, 12, 2), (65532, 24, 2), (64408, 68, 3), (65528, 132, 3),
                                        (6596, 6596, 3), (65408, 520, 4)])
def test_wide_fast_steps_against_oracle(w, h, levels, stream):
    print(f"wide tiles {w}x{h} levels {levels}", flush=True)
    steps = P.plan(w, h, levels)
    assert len(steps) == 1 and steps[0].pipeline == P.PIPELINE_FAST and steps[0].levelCount == levels - 1
    level0 = np.random.default_rng(w + h).integers(0, 256, (h, w, 4), dtype=np.uint8)
    out = H.gpu_run(w, h, level0, stream, mip_levels=levels, levels=levels)
    emu = H.emulate_srgba8(H.host_chain(w, h, level0, levels), w, h, steps, levels)
    assert np.array_equal(out, emu)
