"""The batch queue taking two items at a time (16-byte texels, many items for each
workgroup): every chain equals its own dispatch, over repeated launches and for
even and odd numbers of items.
"""
import numpy as np
import pytest

from vk_compute_mipmaps_amd import hip_rt
from vk_compute_mipmaps_amd import pyramid as P

pytestmark = pytest.mark.gpu


def _sizes(count):
    return [(64 + 67 * (k % 7), 48 + 91 * (k % 5)) for k in range(count)]


@pytest.mark.parametrize("count", [79, 80, 83])
def test_batch_runs_equal_dispatch_rgba32f(count, stream):
    chains = [P.DeviceMipChain(w, h, P.FORMAT_RGBA32F) for w, h in _sizes(count)]
    try:
        rng = np.random.default_rng(11)
        want = []
        for c in chains:
            c.upload_level0(rng.uniform(0.0, 4.0, (c.height, c.width, 4)).astype(np.float32))
            c.dispatch(stream=stream)
            hip_rt.stream_sync(stream)
            want.append(c.download())
        batch = P.PyramidBatch(P.pipelines(P.FORMAT_RGBA32F), [c.image for c in chains],
                               config=P.batch_config(mode=P.BATCH_MODE_QUEUE, workgroups_per_cu=1))
        try:
            info = batch.info()
            print(f"batch runs, {info.itemCount} items on {info.workgroups} workgroups", flush=True)
            assert info.itemCount >= 8 * info.workgroups
            for rep in range(3):
                for c in chains:
                    c.poison(stream=stream)
                batch.launch(stream)
                hip_rt.stream_sync(stream)
                assert batch.read_errors() == 0
                for k, c in enumerate(chains):
                    assert np.array_equal(c.download(), want[k]), f"launch {rep}, image {k} {c.width}x{c.height}"
        finally:
            batch.destroy()
    finally:
        for c in chains:
            c.free()
