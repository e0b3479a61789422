"""Tables that the library keeps in its workspace between calls: after a release the
next buffers may lie at the old addresses with other contents, so every table has to
be uploaded again. Memory of the tables' sizes is overwritten between the release
and the next call."""
import numpy as np
import pytest

from tiralib_amd import _lib, api, synth

pytestmark = pytest.mark.gpu


def _overwrite():
    """Leaves other bytes in freed device memory of the sizes of the tables."""
    held = [_lib.DeviceArray.from_host(np.full(1 << k, 0xA5, np.uint8)) for k in range(12, 25) for _ in range(4)]
    for d in held:
        d.free()


@pytest.mark.parametrize("call", ["closed", "sum", "atv", "table", "table_stick", "per_pair"])
def test_tables_are_uploaded_again_after_a_release(hip, call):
    shape, w = (20, 33, 40), 9
    f = synth.tubes_sheets_volume(shape, n_straight=2, n_helix=1, n_sheets=2, seed=3).reshape(shape + (9,))
    d, o = _lib.DeviceArray.from_host(np.ascontiguousarray(f, np.float32)), _lib.DeviceArray(shape + (9,))
    net = api.PlateMLP(1.5, 0.0, 1, 64, seed=3)
    net.train(nsamples=1 << 13, epochs=1, batch=1024, seed=5)

    def vote():
        if call in ("closed", "sum"):
            api.tensorvote3_async(d, o, shape, 1.5, 0.0, w, 1, samples=20,
                                  plate_mode=_lib.PLATE_CLOSED if call == "closed" else _lib.PLATE_SUM)
        elif call == "atv":
            api.tensorvote3_atv_async(d, o, shape, 1.5, w)  # below 32^3 voxels: the gather and its table
        else:
            net.vote(d, o, shape, w, stick=call == "table_stick", tol=1e30,
                     method=_lib.MLP_PER_PAIR if call == "per_pair" else _lib.MLP_TABLE)
        _lib.call("tira_hip_synchronize")
        return o.to_host()

    try:
        first = vote()
        assert np.isfinite(first).all() and np.abs(first).max() > 0
        for _ in range(3):
            _lib.call("tira_hip_release_workspace")
            _overwrite()
            np.testing.assert_array_equal(vote(), first)
    finally:
        net.close()
        d.free()
        o.free()
