"""A batch whose pools could not grow (hvr_batch_run_async): the old buffers are
gone by then, so neither a captured launch nor a capacity may still speak of
them.  The batch renders and counts on with pools of the sizes it had before."""

import numpy as np
import pytest

import scenes

pytestmark = pytest.mark.gpu

SMALL, LARGE = (64, 64), (200, 200)


@pytest.fixture(autouse=True)
def disarm():
    from pyvr_amd.hip_renderer import _lib

    yield
    _lib.inject_fault(None)


@pytest.fixture
def batch(hip):
    from pyvr_amd.hip_renderer.batch import BatchRenderer, DeviceBlobVolume

    b = BatchRenderer(scalar_format="f16", normal_format="f16x3", pipeline=1)
    vol, ctf = DeviceBlobVolume(shape=(40, 30, 50), seed=1), scenes.c0(size=8, image=8).ctf
    otf = scenes.seeded_otf(5, seed=1, y_max=0.6)

    def run(size, count=False, lut_size=256):
        b.clear()
        b.add(vol, scenes.standard_camera(0.3, 0.2, 3.0), ctf, otf, *size, lut_size=lut_size)
        b.run(count=count)
        return b.counts(0) if count else b.result(0)

    yield run
    b.close()


def _fails(run, after, *args, **kwargs):
    from pyvr_amd.hip_renderer import _lib

    _lib.inject_fault("hvr_batch_grow", after=after)
    with pytest.raises(RuntimeError, match="injected fault in hvr_batch_grow"):
        run(*args, **kwargs)


def test_counts_that_could_not_grow(batch):
    want = batch(SMALL, count=True)
    _fails(batch, 1, LARGE, count=True)              # the images' pool grew, the counts' did not
    assert np.array_equal(batch(SMALL, count=True), want)
    assert batch(LARGE, count=True).shape[0] == LARGE[1]


def test_graphs_of_a_block_that_moved_before_a_failure(batch):
    want = batch(SMALL)
    _fails(batch, 0, SMALL, lut_size=2000)           # no staged block
    _fails(batch, 1, LARGE)                          # one of the old size again, but no images' pool
    assert batch(SMALL) == want
    assert batch(SMALL) == want
    assert len(batch(LARGE)) == 4 * LARGE[0] * LARGE[1]
