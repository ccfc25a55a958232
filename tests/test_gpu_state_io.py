"""Caller arrays to and from the device (deme_upload_state, deme_download_state): every field comes back as it went, at
sizes around the pinned slots the arrays pass through in chunks, whole or only some of the arrays, also written twice
over resident records."""
import ctypes as C

import numpy as np
import pytest

from deme_amd import scenes
from deme_amd.abi import STATE_FIELDS, DeviceSystem, make_state_struct

pytestmark = pytest.mark.gpu


def _random_state(n, rng):
    st = {}
    for k, t in STATE_FIELDS.items():
        st[k] = (rng.integers(0, np.iinfo(t).max, n, dtype=t, endpoint=True) if np.issubdtype(t, np.integer)
                 else rng.normal(size=n).astype(t))
    return st


# 79 bytes an owner: the calling thread alone takes halves of a slot (1 MiB, near 13,273 owners) up to 8 MiB (near 106,184);
# beyond, 2 MiB slots end near multiples of 26,546 owners, and 400,001 take more chunks than there are slots
@pytest.mark.parametrize("n", [1, 2, 63, 13_272, 13_274, 26_545, 26_547, 106_180, 106_190, 400_001])
def test_states_come_back_as_they_went(n):
    rng = np.random.default_rng(n)
    g = np.arange(n)
    side = int(np.ceil(n ** (1 / 3)))
    xyz = np.stack([g % side, (g // side) % side, g // (side * side)], 1) * 0.01
    L = max(side * 0.01 + 0.02, 0.1)
    sc = scenes.spheres_scene(xyz - L / 2 + 0.01, 0.004, (L, L, L))
    dev = DeviceSystem(sc)
    got = dev.get_state()
    for k in ("voxelID", "locX", "oriQw", "family", "vX"):
        assert np.array_equal(got[k], sc.state[k]), k
    full = _random_state(sc.n_owners, rng)
    dev.set_state(full)
    got = dev.get_state()
    for k in STATE_FIELDS:
        assert np.array_equal(got[k], full[k]), k
    # some arrays only: the others keep their values
    part = {k: v for k, v in _random_state(sc.n_owners, rng).items() if k in ("locY", "oriQz", "omgX", "alphaY", "family")}
    dev.set_state(part)
    full.update(part)
    out = {k: np.zeros(sc.n_owners, STATE_FIELDS[k]) for k in ("voxelID", "locZ", "omgX", "alphaY", "vZ", "family")}
    s = make_state_struct(out)
    assert dev.lib.deme_download_state(dev.ctx, C.byref(s)) == 0
    for k, v in out.items():
        assert np.array_equal(v, full[k]), k
    got = dev.get_state()
    for k in STATE_FIELDS:
        assert np.array_equal(got[k], full[k]), k
