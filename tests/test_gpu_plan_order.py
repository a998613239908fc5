"""Plans of a custom dispatcher whose steps go back a level or start inside the
step before: every level must equal the oracle's FP32 emulator, run on one step
after the other, bit for bit.
"""
import ctypes

import numpy as np
import pytest

from tests import helpers as H
from vk_compute_mipmaps_amd import pyramid as P
from vk_compute_mipmaps_amd import synth

pytestmark = pytest.mark.gpu

F, G = P.PIPELINE_FAST, P.PIPELINE_GENERAL


def _emulate(side, level0, steps):
    """Each step on the levels from its input on, as an image of its own."""
    chain = H.host_chain(side, side, level0)
    offsets, total = P.packed_layout(side, side)
    offsets.append(total)
    for s in steps:
        a, b = offsets[s.inputLevel], offsets[s.inputLevel + s.levelCount + 1]
        own, first = side >> s.inputLevel, P.NvproPyramidStep(s.pipeline, 0, s.levelCount)
        chain[a:b] = H.emulate_srgba8(chain[a:b], own, own, [first], s.levelCount + 1)
    return chain


@pytest.mark.parametrize("side,plan", [
    (128, [(F, 0, 3), (F, 1, 3), (F, 4, 3)]),
    (128, [(F, 0, 3), (F, 3, 1), (F, 3, 2), (F, 5, 2)]),
    (128, [(F, 0, 3), (G, 3, 1), (F, 3, 2), (F, 5, 2)]),
    (128, [(F, 0, 4), (G, 3, 2), (G, 5, 2)]),
    (128, [(F, 0, 3), (G, 3, 2), (G, 5, 2)]),
    (1024, [(F, 0, 6), (F, 4, 3), (G, 6, 2), (G, 8, 2)])])
def test_steps_in_any_order(side, plan, stream):
    print(f"plan order {side} {plan}", flush=True)

    def record(cmd, state):
        for kind, level, count in plan:
            if P.lib().nvproPyramidCmdDispatch(cmd, kind, level << P.INPUT_LEVEL_SHIFT | count, 1):
                return 0
        return state.contents.remainingLevels

    cb = P.DISPATCHER(lambda cmd, state: record(ctypes.c_void_p(cmd), state))
    steps = P.plan(side, side, general_dispatcher=cb, fast_dispatcher=cb)
    assert [(s.pipeline, s.inputLevel, s.levelCount) for s in steps] == plan
    level0 = synth.srgba8(side, side, len(plan))
    out = H.gpu_run(side, side, level0, stream, general_dispatcher=cb, fast_dispatcher=cb)
    assert np.array_equal(out, _emulate(side, level0, steps))
