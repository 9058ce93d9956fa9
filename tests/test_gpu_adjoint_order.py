"""3D adjoint steps whose tiles go along x (planes of 2.25 MB and more), bit for
bit against the oracle: slabs dealt to the XCDs and not, odd sizes, and planes just
under the line.  Every cell is updated on its own, so the order changes no result."""
import numpy as np
import pytest

from cases import small_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", [
    dict(N=(128, 128, 24)), dict(N=(131, 101, 25)), dict(N=(128, 96, 24)),
    dict(N=(131, 69, 27), FDORDER=8), dict(N=(190, 189, 24), L=1),
    dict(N=(190, 192, 24), L=2, freesurf=1)], ids=str)
def test_tile_orders(oracle_lib, gpu_ctx, case):
    from seiscl_amd import Model
    csts, p, (sp, s, rp) = small_case(ND=3, NT=36, nab=8, **case)
    rng = np.random.default_rng(3)
    res = [rng.standard_normal((36, rp.shape[1])).astype(np.float32) for _ in range(3)]
    ref = oracle_lib.gradient(p, sp, s, rp, res=res, **csts)
    m = Model(gpu_ctx, p, **csts)
    m.grad_zero()
    m.gradient(sp, s, rp, res=res)
    g = m.grad_read()
    m.close()
    for k in ref["grad"]:
        assert np.abs(ref["grad"][k]).max() > 0, k
        np.testing.assert_array_equal(g[k], ref["grad"][k])
