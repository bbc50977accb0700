"""Rotations per block: the automatic choice (many small blocks, fuller last chunks)
changes no bit of a result, whatever the range leaves over."""
import numpy as np
import pytest

from powerfit_amd import HipCorrelator, rotations_for_angle

pytestmark = pytest.mark.gpu


def _case(shape):
    rng = np.random.default_rng(sum(shape))
    grids = np.meshgrid(*[np.fft.fftfreq(n, 1.0 / n) for n in shape], indexing="ij")
    mask = (sum(g * g for g in grids) <= (0.3 * min(shape)) ** 2).astype(float)
    return rng.standard_normal(shape), rng.random(shape) * mask, mask


# one rotation, a ragged last chunk, a full batch and a short one after it
@pytest.mark.parametrize("count", [1, 100, 256, 301])
# compiled planes, residue stages of one, two and four residues, rows and columns
@pytest.mark.parametrize("shape", [(64, 64, 64), (48, 48, 48), (60, 64, 75), (96, 96, 96),
                                   (24, 168, 180)])
def test_automatic_chunks_change_nothing(shape, count):
    target, template, mask = _case(shape)
    R = rotations_for_angle(20.0)[:count]
    assert len(R) == count
    out = []
    for chunk in (0, 1, 7, 64):
        print(f"{shape} {count} rotations, chunk {chunk}", flush=True)
        corr = HipCorrelator(target)
        corr.set_tuning(chunk, chunk)
        corr.template = template
        corr.mask = mask
        corr.rotations = R
        corr.scan()
        out.append((corr.lcc.copy(), corr.rot.copy()))
    for lcc, rot in out[1:]:
        assert np.array_equal(lcc, out[0][0])
        assert np.array_equal(rot, out[0][1])
