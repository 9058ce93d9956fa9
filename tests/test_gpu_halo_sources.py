"""3D viscoelastic gradients with sources on halo cells (above, below or beside
the grid), which keep what every step's sources add to them, against the oracle."""
import numpy as np
import pytest

from cases import small_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,freesurf", [(1, 0), (2, 1)])
@pytest.mark.parametrize("where", ["z", "y"])
def test_source_on_halo_cell(oracle_lib, gpu_ctx, L, freesurf, where):
    from seiscl_amd import Model
    csts, p, (sp, s, rp) = small_case(ND=3, N=(28, 26, 30), NT=48, nab=8, L=L, freesurf=freesurf)
    dh = csts["dh"]
    for k in range(2):
        if where == "z":
            sp[2, k] = -dh if freesurf or k == 0 else csts["N"][0] * dh
        else:
            sp[1, k] = -dh if k == 0 else csts["N"][1] * dh
    rng = np.random.default_rng(3)
    res = [rng.standard_normal((48, rp.shape[1])).astype(np.float32) for _ in range(3)]
    ref = oracle_lib.gradient(p, sp, s, rp, res=res, **csts)
    m = Model(gpu_ctx, p, **csts)
    m.grad_zero()
    m.gradient(sp, s, rp, res=res)
    g, plan = m.grad_read(), m.grad_plan()
    m.close()
    assert plan["n0"] > 1   # several segments: their history is kept in the same place
    for k in ref["grad"]:
        assert np.abs(ref["grad"][k]).max() > 0, k
        np.testing.assert_array_equal(g[k], ref["grad"][k])
