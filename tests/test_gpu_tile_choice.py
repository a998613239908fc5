"""Thin tiles and strips for the same large two-level step, in the wide formats.

Three levels, so that the step is launched alone whatever its size: one launch,
and NVPRO_PYRAMID_THIN decides how it runs.  Sizes of many strips and rows of
groups; the default, which takes one or the other by size, must give the same.
"""
import os

import numpy as np
import pytest

from tests import helpers as H
from vk_compute_mipmaps_amd import pyramid as P
from vk_compute_mipmaps_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,arith", [(P.FORMAT_RGBA16F, P.ARITH_FP32), (P.FORMAT_RGBA16F, P.ARITH_PACKED_FP16),
                                       (P.FORMAT_RGBA32F, P.ARITH_FP32)])
@pytest.mark.parametrize("w,h", [(645, 389), (1001, 513), (2046, 1023)])
def test_thin_tiles_and_strips_agree(w, h, fmt, arith, stream, monkeypatch):
    print(f"tile choice {w}x{h} format {fmt} arithmetic {arith}", flush=True)
    if fmt == P.FORMAT_RGBA16F:
        level0 = synth.rgba16f(w, h, 23)
    else:
        level0 = np.random.default_rng(23).random((h, w, 4), dtype=np.float32) * np.float32(4.0)
    out = {}
    for mode in ("", "0", "1"):
        monkeypatch.setenv("NVPRO_PYRAMID_THIN", mode)
        out[mode] = H.gpu_run(w, h, level0, stream, fmt=fmt, fast=False, mip_levels=3, levels=3, arithmetic=arith)
        assert P.last_launch_count() == 1
    assert np.array_equal(out["0"], out["1"])
    assert np.array_equal(out[""], out["1"])
