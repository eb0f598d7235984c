"""The fill's slabs and sample order: where rays ended before their neighbours
(opaque ones still have samples in the tile's slabs, past ones have none), on
ragged tile edges, and where steps near the rounding of t leave bin midpoints
unordered.  Index work is the oracle's bit for bit."""
import numpy as np
import pytest

from frustumvolumecaching_amd import lib
from frustumvolumecaching_amd import synthetic as S

pytestmark = pytest.mark.gpu


def _opaque():
    wl = S.small_plain(27, 18, stepsize_setup=lib.stepsize_setup)
    wl.step = S.stepsize_info(0.0, 3 ** 0.5 / 128, 0.1, 8.0)
    wl.params = S.make_params(wl.net, table_range=30.0)  # log sigma from -9 to 11
    return wl


def _ragged():
    wl = S.unbounded_1080p(43, 21)
    wl.step = S.stepsize_info(1.0 / 64, 3 ** 0.5 / 128, 0.1, 60.0)
    return wl


def _unordered():
    wl = S.small_plain(8, 8, stepsize_setup=lib.stepsize_setup)
    dt = 2.0 ** -20  # half the spacing of floats in [16, 32)
    wl.step = S.stepsize_info(0.0, dt, 0.1, 17.0 + 160 * dt)
    wl.cam2world = S.look_at((18.0, 0.01, 0.02), (0.0, 0.01, 0.02))
    wl.fov = 0.001
    return wl


@pytest.mark.parametrize("case", [_opaque, _ragged, _unordered])
def test_fill_equals_oracle(oracle_mod, case):
    wl = case()
    lib.stepsize_setup(wl.step, wl.scene)
    if case is not _ragged:
        wl.occupancy = np.ones_like(wl.occupancy)
    model, ref = lib.NerfNetwork.from_workload(wl), oracle_mod.Model.from_workload(wl)
    r = lib.Renderer(model)
    st = r.initCacheBlockwise(wl.rm())
    oc = ref.cache_fill(wl.rm(), oracle_mod.EMU16)
    assert st.n_samples_evaluated == oc.stats.n_samples_evaluated > 0
    # (the oracle also counts a last round whose samples all belong to tiles
    # that end in it and are dropped)
    assert 0 <= oc.stats.n_subiters - st.n_subiters <= 1
    assert st.n_bricks_set == oc.stats.n_bricks_set
    assert np.array_equal(r.brick_table(), oc.brick_table())
    assert np.array_equal(r.known_ranges().view(np.uint32), oc.known_ranges().view(np.uint32))
    assert np.array_equal(r.pool()["isset"], oc.pool()[..., 9])
    if case is _opaque:  # rays end inside the scene
        full = S.small_plain(27, 18, stepsize_setup=lib.stepsize_setup)
        full.step, full.occupancy = wl.step, wl.occupancy
        assert st.n_samples_evaluated < ref_samples(full)
    r.close()
    model.close()


def ref_samples(wl):
    """Samples of a fill in which no ray is opaque."""
    model = lib.NerfNetwork.from_workload(wl)
    r = lib.Renderer(model)
    n = r.initCacheBlockwise(wl.rm()).n_samples_evaluated
    r.close()
    model.close()
    return n
