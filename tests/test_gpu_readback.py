"""Results in the caller's layout: what the GPU transposes and transforms against
the library's other layout and the host's arithmetic."""
import numpy as np
import pytest

from cases import small_case

pytestmark = pytest.mark.gpu


def _ids(c):
    return "-".join(f"{k}{v}" for k, v in c.items())


# sizes around the 32 x 32 tiles of the transposition, one cell over and under
@pytest.mark.parametrize("case", [
    dict(ND=2, N=(32, 33)), dict(ND=2, N=(65, 31), L=1), dict(ND=2, N=(31, 64), L=2, freesurf=1),
    dict(ND=3, N=(33, 24, 32), L=1), dict(ND=3, N=(24, 31, 33))], ids=_ids)
@pytest.mark.parametrize("param_type", [0, 1, 2])
def test_gradient_layouts(gpu_ctx, case, param_type):
    from seiscl_amd import Model
    from seiscl_amd._lib import check, fptr
    from seiscl_amd.engine import from_c_layout
    csts, p, (sp, s, rp) = small_case(NT=40, nab=8, **case)
    csts["param_type"] = param_type
    if param_type == 1:
        p = dict(p, M=p["vp"] ** 2 * p["rho"], mu=p["vs"] ** 2 * p["rho"])
    elif param_type == 2:
        p = dict(p, Ip=p["vp"] * p["rho"], Is=p["vs"] * p["rho"])
    m = Model(gpu_ctx, p, **csts)
    m.grad_zero()
    out = m.forward_save(sp, s, rp)
    m.adjoint(out)
    g = m.grad_read()
    n = int(np.prod(case["N"]))
    flat = np.zeros(5 * n, np.float32)
    check(m.lib.seis_grad_read(m.handle, fptr(flat[:3 * n])))
    if case.get("L"):
        check(m.lib.seis_grad_read_tau(m.handle, fptr(flat[3 * n:])))
    m.close()
    assert len(g) == (5 if case.get("L") else 3)
    for q, k in enumerate(g):
        assert g[k].shape == tuple(case["N"]) and g[k].flags.c_contiguous
        assert np.abs(g[k]).max() > 0
        assert np.array_equal(g[k], from_c_layout(flat[q * n:(q + 1) * n], case["N"]))


@pytest.mark.parametrize("case", [
    dict(ND=2, seisout=1), dict(ND=2, seisout=2), dict(ND=2, seisout=4),
    dict(ND=22, seisout=4), dict(ND=3, seisout=3)], ids=_ids)
@pytest.mark.parametrize("prec", [0, 2, 64])
def test_seismogram_layouts(gpu_ctx, case, prec):
    from seiscl_amd import Model
    csts, p, shot = small_case(NT=37, **case)
    csts["FP16"] = prec
    m = Model(gpu_ctx, p, **csts)
    raw = m.forward(*shot, raw=True)
    out = m.forward(*shot)
    m.bind_shot(*shot)
    m.run_steps(0, 37)
    again = m.read_shot()
    m.close()
    assert np.abs(raw).max() > 0
    for q, o in enumerate(out):
        assert o.shape == (37, shot[2].shape[1]) and o.flags.c_contiguous
        assert np.array_equal(o, raw[q].T) and np.array_equal(again[q], o)
