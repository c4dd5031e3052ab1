"""Captured launches of a batch (hvr_batch_run_async): batches whose sizes cross
the lanes rule's lines choose other kernels, and come back to graphs that are
still there; more shapes than are kept, grown pools and failed captures are
captured again.  Every replay against the same request alone."""

import pytest

import scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def disarm():
    from pyvr_amd.hip_renderer import _lib

    yield
    _lib.inject_fault(None)


# 4, 2 and 1 lanes per ray on 256 compute units
SIZES = [(300, 300), (700, 700), (1200, 1200)]


@pytest.fixture(scope="module")
def scene():
    from pyvr_amd.hip_renderer.batch import DeviceBlobVolume

    vols = [DeviceBlobVolume(shape=(40, 30, 50), seed=1), DeviceBlobVolume(shape=(33, 40, 20), seed=2)]
    return vols, scenes.c0(size=8, image=8).ctf, [scenes.seeded_otf(5, seed=s, y_max=0.6) for s in (1, 2)]


def _run(b, scene, size, k=0, lut_size=256):
    vols, ctf, otfs = scene
    b.clear()
    b.add(vols[k % 2], scenes.standard_camera(0.3 * k, 0.2, 3.0), ctf, otfs[k // 2 % 2], *size, lut_size=lut_size)
    b.run()
    return b.result(0)


def test_sizes_across_the_lines_keep_their_graphs(hip, scene):
    from pyvr_amd.hip_renderer import _lib
    from pyvr_amd.hip_renderer.batch import BatchRenderer

    b = BatchRenderer(scalar_format="f16", normal_format="f16x3", pipeline=1)
    try:
        b.reserve(4, 1 << 21, 4096)
        for size in SIZES:
            _run(b, scene, size)
        sizes = SIZES + SIZES[::-1] + [(301, 280), (705, 690), (1100, 1201)]
        want = [_run_alone(scene, size, k) for k, size in enumerate(sizes)]
        _lib.inject_fault("hvr_batch_capture", code=-2)
        assert [_run(b, scene, size, k) for k, size in enumerate(sizes)] == want
        with pytest.raises(RuntimeError, match="injected fault in hvr_batch_capture"):
            _run(b, scene, SIZES[0], 0, lut_size=700)       # another LDS size: a shape of its own
        for k, size in enumerate(SIZES):                    # and on after the failure
            assert _run(b, scene, size, k, lut_size=700) == _run_alone(scene, size, k, lut_size=700)
    finally:
        b.close()


def _run_alone(scene, size, k, lut_size=256):
    from pyvr_amd.hip_renderer.batch import BatchRenderer

    b = BatchRenderer(scalar_format="f16", normal_format="f16x3", pipeline=1)
    try:
        return _run(b, scene, size, k, lut_size)
    finally:
        b.close()


def test_more_shapes_than_are_kept(hip, scene):
    """Twelve shapes (three kernels, four LDS sizes) in turn, twice, then pools that
    grow, which takes every graph's staging away."""
    from pyvr_amd.hip_renderer.batch import BatchRenderer

    b = BatchRenderer(scalar_format="f16", normal_format="f16x3", pipeline=1)
    shapes = [(size, n) for n in (256, 300, 700, 1000) for size in SIZES]
    try:
        want = {s: _run_alone(scene, s[0], 1, s[1]) for s in shapes}
        for _ in range(2):
            for s in shapes:
                assert _run(b, scene, s[0], 1, s[1]) == want[s]
        b.reserve(256, 1 << 22, 1 << 16)
        for s in shapes[::-1]:
            assert _run(b, scene, s[0], 1, s[1]) == want[s]
    finally:
        b.close()
