"""Fast steps whose tiles are found by multiplication and whose groups outnumber
the workgroups: one tile a row, one row of tiles, a last group of few tiles, the
smallest that stream their input and the fewest groups that give a workgroup
more than one.  sRGBA8 must equal the oracle's FP32 emulator bit for bit.
"""
import numpy as np
import pytest

from tests import helpers as H
from vk_compute_mipmaps_amd import pyramid as P
from vk_compute_mipmaps_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(64, 8192), (8192, 64), (16, 65520), (8, 65528), (65528, 8), (1024, 1024),
                                 (1088, 1024), (1056, 1120), (1072, 1008), (2600, 2008), (4800, 1120)])
def test_fast_tiles_srgba8_against_oracle(w, h, stream):
    print(f"fast tiles {w}x{h}", flush=True)
    level0 = synth.srgba8(w, h, w + 3 * h)
    out = H.gpu_run(w, h, level0, stream)
    emu = H.emulate_srgba8(H.host_chain(w, h, level0), w, h, P.plan(w, h))
    assert np.array_equal(out, emu)
