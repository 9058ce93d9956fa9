"""Receivers and sources of a step in one launch of several blocks, against the
launches that record and add one after the other."""
import numpy as np
import pytest

from cases import small_case

pytestmark = pytest.mark.gpu


# one block up to 256 receivers or from 17 sources on; several otherwise, with
# receivers on the source cells in the first and in the last block
@pytest.mark.parametrize("nrec", [255, 256, 257, 600])
@pytest.mark.parametrize("nsrc", [1, 16, 17])
@pytest.mark.parametrize("prec", [0, 2])
def test_receivers_on_source_cells(gpu_ctx, nrec, nsrc, prec):
    from seiscl_amd import Model
    csts, p, (sp, s, rp) = small_case(ND=3, N=(28, 26, 30), L=1, NT=30, nab=8, seisout=3)
    csts["FP16"] = prec
    dh = csts["dh"]
    rng = np.random.default_rng(5)
    cells = rng.integers([9, 9, 9], [17, 15, 18], (nrec, 3))      # x, y, z
    rec = np.zeros((8, nrec), np.float32)
    rec[:3] = cells.T * dh
    src = np.zeros((5, nsrc), np.float32)
    src[:3] = np.concatenate([rec[:3, :1], rec[:3, -(nsrc - 1):]], 1)[:, :nsrc] if nsrc > 1 \
        else rec[:3, :1]
    src[3] = np.arange(nsrc)
    src[4] = np.array([100, 0, 2])[np.arange(nsrc) % 3]
    wave = (rng.standard_normal((30, nsrc)) * np.abs(s).max()).astype(np.float32)
    m = Model(gpu_ctx, p, **csts)
    out = m.forward(src, wave, rec)
    m.set_profiling(True)
    want = m.forward(src, wave, rec)
    m.set_profiling(False)
    m.close()
    for a, b in zip(out, want):
        assert np.abs(b).max() > 0 and np.array_equal(a, b)
