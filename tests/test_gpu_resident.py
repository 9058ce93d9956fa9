"""2D runs resident on the chip against the step kernels.

Both make the same operations on the same values in the same order, so
seismograms and wavefields are compared bit for bit.  set_profiling(True) makes
a model's steps with the step kernels.
"""
import numpy as np
import pytest

from cases import small_case
from seiscl_amd.workloads import ricker

pytestmark = pytest.mark.gpu

NT = 90
FIELDS = {2: ("vx", "vz", "sxx", "szz", "sxz"), 22: ("vx", "vz", "p")}

# Tiles are at most 64 - 2H cells high and 16, 32, 48 or 80 - 2H columns wide
# (H half the FD order): grids of one tile, one cell more or less than a
# multiple of a tile, and wide enough for every width.
CASES = (
    [dict(ND=2, FDORDER=o, N=n) for o, n in (
        (2, (16, 17)), (2, (60, 18)), (2, (61, 131)), (4, (56, 60)), (4, (57, 61)),
        (8, (48, 40)), (8, (49, 97)), (12, (40, 41)), (12, (91, 67)))]
    + [dict(ND=2, FDORDER=4, N=(120, n), freesurf=1) for n in (900, 1700, 3100)]
    + [dict(ND=2, FDORDER=o, N=(113, 140), L=l, freesurf=f, seisout=4)
       for o in (4, 10) for l in (0, 1, 2) for f in (0, 1)]
    + [dict(ND=2, FDORDER=6, N=(300, 1100), L=l, freesurf=1) for l in (1, 2)]
    + [dict(ND=2, FDORDER=8, N=(300, 1100), L=l) for l in (1, 2)]
    + [dict(ND=2, FDORDER=8, N=(107, 111), abs_type=a, freesurf=f)
       for a in (0, 2) for f in (0, 1)]
    + [dict(ND=22, FDORDER=o, N=n, seisout=4) for o, n in (
        (2, (16, 16)), (4, (57, 200)), (8, (113, 900)), (8, (300, 1500)), (12, (95, 77)))]
    + [dict(ND=22, FDORDER=8, N=(64, 100), abs_type=2)]
)


def _ids(c):
    return "-".join(f"{k}{v}" for k, v in c.items())


def _shot(case, nab=8):
    """Sources that share a cell, on a tile's edge, in the grid's halo and
    outside it; receivers on every kind of cell, some twice."""
    csts, params, (sp, s, rp) = small_case(NT=NT, nab=nab, **case)
    nz, nx = case["N"]
    dh, t = 10.0, 3 if case["ND"] == 22 else 100
    zs = (1 if case.get("freesurf") else nab + 1) * dh
    xs = np.array([nx // 2, nx // 2, nx - 1, 0, nx // 3, nx + 4]) * dh
    zz = np.array([zs, zs, zs, (nz // 2) * dh, -dh if csts["FDORDER"] > 2 else zs, zs])
    typ = np.array([t, 2, 0, t, 2, t], float)
    sp = np.stack([xs, 0 * xs, zz, 0 * xs, typ])
    s = np.stack([ricker(15.0 + 3 * k, NT, csts["dt"], tmin=-0.02) for k in range(6)], 1)
    rx = np.concatenate([np.arange(nx), [nx // 2, nx // 2, nx + 3]]) * dh
    rz = np.concatenate([np.arange(nx) % nz, [int(zs / dh)] * 2, [3]]) * dh
    rec = np.stack([rx, 0 * rx, rz, 0 * rx, np.arange(rx.size) + 1.0, 0 * rx, 0 * rx, 0 * rx])
    if rx.size > 1000:
        rec = rec[:, :: rx.size // 1000 + 1]
    return csts, params, (sp, s.astype(np.float32), rec)


def _state(m, nd):
    return [m.read_field(k) for k in FIELDS[nd]]


@pytest.mark.parametrize("case", CASES, ids=_ids)
def test_resident_equals_steps(gpu_ctx, case):
    from seiscl_amd import Model
    csts, params, shot = _shot(case)
    m = Model(gpu_ctx, params, **csts)
    got, fields = m.forward(*shot), _state(m, case["ND"])
    m.set_profiling(True)
    ref, rfields = m.forward(*shot), _state(m, case["ND"])
    m.close()
    assert any(np.abs(r).max() > 0 for r in ref)
    for a, b in zip(got + fields, ref + rfields):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("case", [CASES[4], CASES[14], CASES[-2]], ids=_ids)
def test_resident_runs_continue(gpu_ctx, case):
    """Runs of any length, resident or too short for it, one after another."""
    from seiscl_amd import Model
    csts, params, shot = _shot(case)
    m = Model(gpu_ctx, params, **csts)
    ref = m.forward(*shot)
    m.bind_shot(*shot)
    t = 0
    for n in (17, 1, 3, 33, 16, NT):
        n = min(n, NT - t)
        m.run_steps(t, n)
        t += n
    got = m.read_shot()
    m.close()
    for a, b in zip(got, ref):
        assert np.array_equal(a, b)


# Adjoint runs hold ten wavefields (elastic) in LDS: tiles 16, 32 or 48 - 2H
# columns wide; viscoelastic ones 16 or 32.
GRADS = (
    [dict(ND=2, FDORDER=o, N=n) for o, n in (
        (2, (36, 37)), (4, (56, 60)), (4, (113, 131)), (8, (49, 97)), (12, (91, 67)),
        (4, (120, 900)), (4, (120, 1700)), (6, (120, 2100)), (8, (120, 2100)))]
    + [dict(ND=2, FDORDER=o, N=(113, 140), L=l, freesurf=f, seisout=so)
       for o, so in ((4, 2), (6, 1), (10, 4)) for l in (0, 1, 2) for f in (0, 1)]
    + [dict(ND=2, FDORDER=4, N=(113, 1100), L=2, freesurf=1)]
    + [dict(ND=2, FDORDER=8, N=(107, 111), abs_type=0, L=l) for l in (0, 2)]
)


def _gradient(m, shot, seed=5):
    rp = shot[2]
    rng = np.random.default_rng(seed)
    m.grad_zero()
    out = m.forward_save(*shot)
    size = max(np.abs(o).max() for o in out)
    res = [(size * rng.standard_normal((NT, rp.shape[1]))).astype(np.float32) for _ in out]
    m.adjoint(res)
    return m.grad_read(), _state(m, 2) if m.csts.L == 0 else []


@pytest.mark.parametrize("case", GRADS, ids=_ids)
def test_resident_adjoint_equals_steps(gpu_ctx, case):
    from seiscl_amd import Model
    csts, params, (sp, s, rp) = _shot(case)
    # receivers on cells of their own (the others stay with the step kernels)
    cells = rp[[0, 2]].astype(int).T
    rp = rp[:, np.unique(cells, axis=0, return_index=True)[1]]
    m = Model(gpu_ctx, params, **csts)
    if case.get("L"):
        m.set_grad_memory((100 << 20) if case["N"][1] > 1000 else 0)
    g, f = _gradient(m, (sp, s, rp))
    m.set_profiling(True)
    r, rf = _gradient(m, (sp, s, rp))
    m.close()
    for k in r:
        assert np.abs(r[k]).max() > 0
        assert np.array_equal(g[k], r[k]), k
    for a, b in zip(f, rf):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("case", [
    dict(ND=2, FDORDER=4, N=(113, 140)), dict(ND=2, FDORDER=8, N=(113, 140), L=1, freesurf=1),
    dict(ND=22, FDORDER=8, N=(70, 90))], ids=_ids)
def test_y_forces(gpu_ctx, case):
    """Source type 1, which has no velocity of its own in 2D, does the same in
    resident runs and step by step: seismograms, and gradients where there are any."""
    from seiscl_amd import Model
    csts, params, (sp, s, rp) = _shot(case)
    sp[4, :2] = 1
    cells = rp[[0, 2]].astype(int).T
    shot = (sp, s, rp[:, np.unique(cells, axis=0, return_index=True)[1]])
    m = Model(gpu_ctx, params, **csts)
    runs = []
    for prof in (False, True):
        m.set_profiling(prof)
        r = list(m.forward(*shot))
        if case["ND"] == 2:
            g, f = _gradient(m, shot)
            r += list(g.values()) + f
        runs.append(r)
    m.close()
    for a, b in zip(*runs):
        assert np.abs(b).max() > 0 and np.array_equal(a, b)


def test_run_that_gives_up_is_made_by_steps(gpu_ctx, monkeypatch):
    """Blocks that do not wait at all: the run ends, the model's state is as
    before it, and the step kernels make the steps."""
    from seiscl_amd import Context, Model
    case = dict(ND=2, FDORDER=4, N=(113, 140), L=1, freesurf=1)
    csts, params, shot = _shot(case)
    m = Model(gpu_ctx, params, **csts)
    m.set_profiling(True)
    ref, rfields = m.forward(*shot), _state(m, 2)
    m.close()
    monkeypatch.setenv("SEIS_RESIDENT_WAIT_MS", "0")
    ctx = Context(0)
    m = Model(ctx, params, **csts)
    got = [m.forward(*shot) + _state(m, 2) for _ in range(2)]
    runs = ctx.resident_runs()
    m.close()
    ctx.close()
    for k in range(2):
        for a, b in zip(got[k], ref + rfields):
            assert np.array_equal(a, b)
    assert runs == dict(made=(0, 0), gave_up=(2, 0))


@pytest.mark.parametrize("L", [0, 1])
def test_adjoint_that_gives_up_is_made_by_steps(gpu_ctx, monkeypatch, L):
    from seiscl_amd import Context, Model
    csts, params, (sp, s, rp) = _shot(dict(ND=2, FDORDER=4, N=(113, 140), L=L, freesurf=1))
    rp = rp[:, :100]
    m = Model(gpu_ctx, params, **csts)
    r, _ = _gradient(m, (sp, s, rp))
    m.close()
    monkeypatch.setenv("SEIS_RESIDENT_WAIT_MS", "0")
    ctx = Context(0)
    m = Model(ctx, params, **csts)
    for _ in range(2):
        g, _ = _gradient(m, (sp, s, rp))
        for k in r:
            assert np.array_equal(g[k], r[k]), k
    m.close()
    ctx.close()
