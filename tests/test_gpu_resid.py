"""GPU parity of the run-time planned pipeline's stages by row residue: every
number of residues (1, 2, 3, 4, 5) with even and odd x, rows of two and three
x stages, y parts of one and two radices, odd row counts (the last packed pair
half empty), 0/1, core-weighted and W^2 as its own grid.

Bar: best LCC within 1e-4 of the FP64 oracle; rotation indices identical where
the oracle's winner leads by more than 1e-4; the same maps bit for bit in any
batch, chunk, range, replayed graph or allocation-free call of the same stages.
"""
import numpy as np
import pytest

from oracle import correlator as oc
from powerfit_amd import HipCorrelator, _lib
from powerfit_amd.rotations import rotations_for_angle
from powerfit_amd.synth import Workload, make_case

from parity import assert_scan_parity

pytestmark = pytest.mark.gpu


def case(shape, laplace=False, core=False, seed=8400):
    return make_case(Workload("resid", min(shape), 2.0, 500, 8.0, 20.0, laplace=laplace,
                              core_weighted=core, seed=seed, shape=shape))


def scan(c, R, batch=8, mode="fused_rt", **kw):
    corr = HipCorrelator(c.target.astype(np.float64), laplace=c.laplace, mode=mode, batch=batch,
                         **kw)
    corr.template = c.template
    corr.mask = c.mask
    corr.rotations = R
    corr.scan()
    return corr


CASES = [
    ((16, 16, 16), {}),                               # the smallest lengths, one residue
    ((24, 20, 27), {"core": True}),                   # one residue, odd x
    ((20, 72, 98), {"core": True}),                   # two residues
    ((18, 64, 75), {"laplace": True}),                # two residues, odd x
    ((25, 81, 105), {}),                              # three residues, odd x, odd row count
    ((21, 81, 100), {"core": True}),                  # three residues
    ((28, 120, 120), {"laplace": True, "core": True}),   # four residues
    ((16, 100, 125), {"core": True}),                 # four residues, three x stages
    ((27, 125, 112), {}),                             # five residues
    ((18, 250, 63), {"core": True}),                  # five residues, odd x
    ((16, 60, 245), {}),                              # the longest odd row
    ((20, 60, 256), {"core": True}),                  # the longest even row
    ((16, 50, 250), {}),                              # rows of three x stages
]


@pytest.mark.parametrize("shape,kw", CASES, ids=["x".join(map(str, s)) for s, _ in CASES])
def test_resid_vs_oracle(shape, kw):
    c = case(shape, **kw)
    R = rotations_for_angle(20.0)[:10]
    ref = oc.parallel_scan(c.target.astype(np.float64), c.template, c.mask, R,
                           laplace=c.laplace, nproc=5)
    corr = scan(c, R)
    assert corr.fused_rt_available
    err, dec = assert_scan_parity(corr.lcc, corr.rot, ref)
    corr.set_schedule(1)
    corr.scan()
    assert_scan_parity(corr.lcc, corr.rot, ref)
    own = scan(c, R, binary_shortcut=False)
    assert_scan_parity(own.lcc, own.rot, ref)
    rel = np.linalg.norm(own.lcc - ref.best) / np.linalg.norm(ref.best)
    print(f"{shape}: max {err:.1e}, rel {rel:.1e}, {dec} decisive", flush=True)


@pytest.mark.parametrize("shape", [(24, 96, 112), (25, 81, 105)], ids=["four", "three"])
def test_resid_same_in_any_batch_range_graph_and_noalloc(shape):
    c = case(shape, core=True)
    R = rotations_for_angle(20.0)[:24]
    corr = scan(c, R, batch=24)
    whole = (corr.lcc.copy(), corr.rot.copy())

    def same(what):
        lcc, rot = corr.result()
        assert np.array_equal(lcc, whole[0]) and np.array_equal(rot, whole[1]), what

    corr.batch = 8
    corr.set_tuning(3, 2)
    corr.reset()
    corr.enqueue_scan(10, 14)
    corr.enqueue_scan(0, 10)
    same("ranges")
    for i in range(3):
        corr.reset()
        corr.enqueue_scan_graph(0, 24)
        same(f"replay {i}")
    lib = _lib.load()
    corr.reset()
    _lib.check(lib.pf_scan_noalloc(corr._ctx, 0, 24, 8, _lib.MODES["fused_rt"]),
               "pf_scan_noalloc")
    same("allocation-free")


def test_one_rotation_per_launch_gives_the_same_map():
    """One rotation of residue tiles takes more room than its packed spectra: the
    launches stay the same kernels and the result the same bits."""
    c = case((25, 81, 105))
    R = rotations_for_angle(20.0)[:12]
    a = scan(c, R, batch=12)
    b = scan(c, R, batch=1)
    assert np.array_equal(a.lcc, b.lcc) and np.array_equal(a.rot, b.rot)


@pytest.mark.parametrize("shape,kw", [((24, 130, 135), {"core": True}), ((20, 144, 144), {}),
                                      ((27, 160, 150), {"laplace": True}),
                                      ((112, 140, 120), {"core": True})],
                         ids=["five odd", "four", "five", "half voxels"])
def test_auto_beyond_the_plane_kernels(shape, kw):
    """Grids whose planes are beyond the plane kernels, through AUTO: no further
    from the oracle than the unfused kernels that ran there (a tenth more for the
    FP32 transforms' own scatter), with rotations that put voxels within one
    rounding of half a voxel."""
    c = case(shape, seed=8500, **kw)
    R = rotations_for_angle(28.0)[[0, 5, 263, 303, 319]]
    ref = oc.parallel_scan(c.target.astype(np.float64), c.template, c.mask, R,
                           laplace=c.laplace, nproc=5)
    new, old = (scan(c, R, mode=m) for m in ("auto", "batched"))
    assert not new.fused_rt_available and not new.fused_available
    assert_scan_parity(new.lcc, new.rot, ref)
    e = [np.linalg.norm(k.lcc - ref.best) / np.linalg.norm(ref.best) for k in (new, old)]
    print(f"{shape}: rel {e[0]:.2e}, unfused {e[1]:.2e}", flush=True)
    assert e[0] <= 1.1 * max(e[1], 2.0 * np.finfo(np.float32).eps)


@pytest.mark.parametrize("n,core", [(48, True), (72, False), (80, True), (96, False), (144, True),
                                    (160, False)])
def test_auto_at_compiled_sizes_vs_compiled(n, core):
    """Sizes where AUTO takes the residue stages: the oracle's map, and the compiled
    kernels' to FP32 rounding of both (the parity bar)."""
    c = case((n, n, n), core=core, seed=8600)
    R = rotations_for_angle(20.0)[:4]
    ref = oc.parallel_scan(c.target.astype(np.float64), c.template, c.mask, R, nproc=4)
    auto, fused = (scan(c, R, mode=m) for m in ("auto", "fused"))
    assert auto.fused_available
    assert_scan_parity(auto.lcc, auto.rot, ref)
    assert_scan_parity(fused.lcc, fused.rot, ref)
    assert not np.array_equal(auto.lcc, fused.lcc)
