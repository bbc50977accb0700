"""GPU parity of the row and column stages that AUTO runs where no plane kernel
covers the grid: the edges of their lengths (16 and 256), odd x (rows in
pairs, the last one unpaired), x lengths without a compiled transform, rows
that do not fill a block, 0/1, core-weighted and Laplace-filtered inputs.

Bar: best LCC within 1e-4 of the FP64 oracle; rotation indices identical
where the oracle's winner leads by more than 1e-4; the same maps bit for bit
in any batch, chunk, range, replayed graph or allocation-free call.
"""
import numpy as np
import pytest

from oracle import correlator as oc
from powerfit_amd import HipCorrelator, _lib
from powerfit_amd.rotations import rotations_for_angle
from powerfit_amd.synth import Workload, make_case

from parity import assert_scan_parity

pytestmark = pytest.mark.gpu


def case(shape, laplace=False, core=False, seed=8200):
    return make_case(Workload("rows", min(shape), 2.0, 500, 8.0, 20.0, laplace=laplace,
                              core_weighted=core, seed=seed, shape=shape))


def scan(c, R, batch=8, mode="auto", **kw):
    corr = HipCorrelator(c.target.astype(np.float64), laplace=c.laplace, mode=mode, batch=batch,
                         **kw)
    corr.template = c.template
    corr.mask = c.mask
    corr.rotations = R
    corr.scan()
    return corr


CASES = [
    ((16, 256, 256), {}),
    ((18, 189, 105), {"core": True}),              # odd x, odd y
    ((25, 225, 81), {"laplace": True}),
    ((27, 144, 130), {"laplace": True, "core": True}),   # x / 2 = 65: run-time planned rows
    ((20, 245, 77), {}),                           # odd x with a factor 11
    ((243, 150, 112), {"core": True}),
]


@pytest.mark.parametrize("shape,kw", CASES, ids=[str(s) for s, _ in CASES])
def test_rows_vs_oracle(shape, kw):
    c = case(shape, **kw)
    R = rotations_for_angle(20.0)[:6]
    corr = scan(c, R)
    assert not corr.fused_rt_available and not corr.fused_available
    ref = oc.parallel_scan(c.target.astype(np.float64), c.template, c.mask, R,
                           laplace=c.laplace, nproc=6)
    err, dec = assert_scan_parity(corr.lcc, corr.rot, ref)
    old = scan(c, R, mode="batched")
    e_new = np.abs(corr.lcc - ref.best).max()
    e_old = np.abs(old.lcc - ref.best).max()
    print(f"rows {shape}: {e_new:.2e}, unfused {e_old:.2e}, {dec} decisive", flush=True)


def test_rows_same_in_any_batch_range_graph_and_noalloc():
    c = case((24, 150, 135), core=True)
    R = rotations_for_angle(20.0)[:10]
    corr = scan(c, R, batch=10)
    whole = (corr.lcc.copy(), corr.rot.copy())

    def same(what):
        lcc, rot = corr.result()
        assert np.array_equal(lcc, whole[0]) and np.array_equal(rot, whole[1]), what

    corr.batch = 3
    corr.set_tuning(1, 2)
    corr.reset()
    corr.enqueue_scan(4, 6)
    corr.enqueue_scan(0, 4)
    same("ranges in batches of 3")
    for i in range(3):
        corr.reset()
        corr.enqueue_scan_graph(0, 10)
        same(f"replay {i}")
    lib = _lib.load()
    corr.reset()
    _lib.check(lib.pf_scan_noalloc(corr._ctx, 0, 10, 5, _lib.MODES["auto"]), "pf_scan_noalloc")
    same("allocation-free")


def test_rows_w2_as_its_own_grid():
    c = case((20, 160, 126))
    R = rotations_for_angle(20.0)[:5]
    ref = oc.parallel_scan(c.target.astype(np.float64), c.template, c.mask, R, nproc=5)
    assert_scan_parity(*(lambda k: (k.lcc, k.rot))(scan(c, R, binary_shortcut=False)), ref)


def test_rows_nearest_mask_at_half_voxel_coordinates():
    """Rotations of the 28 degree set put voxels within one rounding of -1/2,
    where the fraction above the floor rounds to 1/2; one misplaced mask voxel
    of N moves the map by about 1 / N of it (2e-6 here).  Bar: 2 eps sqrt(log2 V),
    the FP32 transforms' own noise with a factor of two."""
    c = make_case(Workload("rows", 112, 1.1, 15000, 4.5, 28.0, core_weighted=True, seed=8300,
                           shape=(112, 140, 120)))
    R = rotations_for_angle(28.0)[[263, 303, 319]]
    corr = scan(c, R)
    assert not corr.fused_rt_available
    ref = oc.parallel_scan(c.target.astype(np.float64), c.template, c.mask, R, nproc=3)
    rel = np.linalg.norm(corr.lcc - ref.best) / np.linalg.norm(ref.best)
    bar = 2.0 * np.finfo(np.float32).eps * np.sqrt(np.log2(c.target.size))
    assert rel <= bar, (rel, bar)


@pytest.mark.parametrize("shape", [(40, 40, 40), (40, 41, 40), (24, 130, 130)])
def test_result_on_either_side_of_the_device_decode(shape):
    """The result read back is the same through the host decode (small maps, or no work
    buffer yet: an allocation-free scan) and the device decode, and when read twice."""
    c = case(shape)
    R = rotations_for_angle(20.0)[:4]
    corr = HipCorrelator(c.target.astype(np.float64), batch=4)
    corr.template = c.template
    corr.mask = c.mask
    corr.rotations = R
    lib = _lib.load()
    corr.reset()
    _lib.check(lib.pf_scan_noalloc(corr._ctx, 0, 4, 4, _lib.MODES["auto"]), "pf_scan_noalloc")
    host = [a.copy() for a in corr.result()]      # no work buffer: host decode
    corr.scan()
    for _ in range(2):
        lcc, rot = corr.result()
        assert np.array_equal(lcc, host[0]) and np.array_equal(rot, host[1])
    assert (host[0] > 0).any() and (host[1] > 0).any()
