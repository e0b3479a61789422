"""Thinning passes queued whole: masks whose re-check does not settle within the
queued launches (long chains of dependent deletions along the raster order),
masks at addresses the 16-byte scan cannot take, and sizes around the scan's
block; bit for bit against the oracle."""
import numpy as np
import pytest

from tiralib_amd._lib import C, DeviceArray, call

pytestmark = pytest.mark.gpu


def _thin(vol, shift=0):
    host = np.concatenate([np.zeros(shift, np.uint8), vol.reshape(-1)])
    d, it = DeviceArray.from_host(host), C.c_uint()
    try:
        call("tira_lee_thin3_u8", d.ptr + shift, *vol.shape, C.byref(it))
        return d.to_host()[shift:].reshape(vol.shape), int(it.value)
    finally:
        d.free()


def _check(oracle, vol, shift=0):
    ref, it_ref = oracle.lee_thin3(vol)
    got, it = _thin(vol, shift)
    assert it == it_ref
    np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("shape", [(1, 200, 200), (2, 150, 300), (40, 3, 170), (3, 3, 700), (12, 60, 80)])
def test_long_chains(hip, oracle, shape):
    """Plates and bars two voxels thick: every candidate depends on its neighbour in
    raster order, so a decision travels along the whole face."""
    _check(oracle, np.ones(shape, np.uint8))
    rng = np.random.default_rng(sum(shape))
    _check(oracle, (rng.random(shape) < 0.97).astype(np.uint8))


@pytest.mark.parametrize("shift", [0, 1, 8, 15])
@pytest.mark.parametrize("shape", [(16, 16, 16), (5, 29, 113), (17, 61, 64)])
def test_unaligned_masks_and_block_edges(hip, oracle, shift, shape):
    rng = np.random.default_rng(shift + shape[1])
    _check(oracle, (rng.random(shape) < 0.6).astype(np.uint8), shift)
