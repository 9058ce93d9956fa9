"""2D runs resident on the chip against the step kernels.

Both make the same operations on the same values in the same order, so
seismograms and wavefields are compared bit for bit.  set_profiling(True) makes
a model's steps with the step kernels; the context's counts of resident runs say
that the others were none.
"""
import threading

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


def _shot(case, nab=8, nt=NT):
    """Sources that share a cell, on a tile's edge, in the grid's halo and
    outside it; receivers on every kind of cell, some twice."""
    csts, params, (sp, s, rp) = small_case(NT=nt, nab=nab, **case)
    nz, nx = case["N"]
    dh, t = 10.0, 3 if case["ND"] == 22 else 100
    zs = (1 if case.get("freesurf") else nab + 1) * dh
    xs = np.array([nx // 2, nx // 2, nx - 1, 0, nx // 3, nx + 4]) * dh
    zz = np.array([zs, zs, zs, (nz // 2) * dh, -dh if csts["FDORDER"] > 2 else zs, zs])
    typ = np.array([t, 2, 0, t, 2, t], float)
    sp = np.stack([xs, 0 * xs, zz, 0 * xs, typ])
    s = np.stack([ricker(15.0 + 3 * k, nt, csts["dt"], tmin=-0.02) for k in range(6)], 1)
    rx = np.concatenate([np.arange(nx), [nx // 2, nx // 2, nx + 3]]) * dh
    rz = np.concatenate([np.arange(nx) % nz, [int(zs / dh)] * 2, [3]]) * dh
    rec = np.stack([rx, 0 * rx, rz, 0 * rx, np.arange(rx.size) + 1.0, 0 * rx, 0 * rx, 0 * rx])
    if rx.size > 1000:
        rec = rec[:, :: rx.size // 1000 + 1]
    return csts, params, (sp, s.astype(np.float32), rec)


class Runs:
    """Resident runs of a context in a with block: made, gave_up (forward, adjoint)."""

    def __init__(self, ctx):
        self.ctx = ctx

    def __enter__(self):
        self.before = self.ctx.resident_runs()
        return self

    def __exit__(self, *exc):
        now = self.ctx.resident_runs()
        for k in now:
            setattr(self, k, tuple(a - b for a, b in zip(now[k], self.before[k])))


def _state(m, nd):
    return [m.read_field(k) for k in FIELDS[nd]]


@pytest.mark.parametrize("case", CASES, ids=_ids)
def test_resident_equals_steps(gpu_ctx, case):
    from seiscl_amd import Model
    csts, params, shot = _shot(case)
    m = Model(gpu_ctx, params, **csts)
    with Runs(gpu_ctx) as runs:
        got, fields = m.forward(*shot), _state(m, case["ND"])
    m.set_profiling(True)
    with Runs(gpu_ctx) as steps:
        ref, rfields = m.forward(*shot), _state(m, case["ND"])
    m.close()
    assert runs.made == (1, 0) and runs.gave_up == steps.made == (0, 0)
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
    with Runs(gpu_ctx) as runs:
        for n in (17, 1, 3, 33, 16, NT):
            n = min(n, NT - t)
            m.run_steps(t, n)
            t += n
    got = m.read_shot()
    m.close()
    assert runs.made == (4, 0) and runs.gave_up == (0, 0)   # of 17, 33, 16 and 20 steps
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


def _nt(case):
    """Viscoelastic gradients are made in segments: long enough ones to be resident."""
    if not case.get("L"):
        return NT
    return 1500 if case["N"][1] > 1000 else 300


def _gradient(m, shot, seed=5):
    rp, nt = shot[2], m.csts.NT
    rng = np.random.default_rng(seed)
    m.grad_zero()
    out = m.forward_save(*shot)
    size = max(np.abs(o).max() for o in out)
    res = [(size * rng.standard_normal((nt, rp.shape[1]))).astype(np.float32) for _ in out]
    m.adjoint(res)
    return m.grad_read(), _state(m, 2) if m.csts.L == 0 else []


@pytest.mark.parametrize("case", GRADS, ids=_ids)
def test_resident_adjoint_equals_steps(gpu_ctx, case):
    from seiscl_amd import Model
    csts, params, (sp, s, rp) = _shot(case, nt=_nt(case))
    # receivers on cells of their own (the others stay with the step kernels)
    cells = rp[[0, 2]].astype(int).T
    rp = rp[:, np.unique(cells, axis=0, return_index=True)[1]]
    m = Model(gpu_ctx, params, **csts)
    two = _nt(case) == 1500     # memory for a plan of two levels, no more
    if case.get("L"):
        m.set_grad_memory((300 << 20) if two else 0)
    with Runs(gpu_ctx) as runs:
        g, f = _gradient(m, (sp, s, rp))
    levels = m.grad_plan()["levels"]
    m.set_profiling(True)
    with Runs(gpu_ctx) as steps:
        r, rf = _gradient(m, (sp, s, rp))
    m.close()
    assert (levels == 2) == two
    # (ten wavefields at order 8 and 2100 columns do not fit the chip)
    assert runs.made[0] > 0 and (runs.made[1] > 0) == (case["N"][1] < 2100 or case["FDORDER"] < 8)
    assert runs.gave_up == steps.made == (0, 0)
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
    csts, params, (sp, s, rp) = _shot(case, nt=_nt(case))
    sp[4, :2] = 1
    cells = rp[[0, 2]].astype(int).T
    shot = (sp, s, rp[:, np.unique(cells, axis=0, return_index=True)[1]])
    m = Model(gpu_ctx, params, **csts)
    runs, counts = [], []
    for prof in (False, True):
        m.set_profiling(prof)
        with Runs(gpu_ctx) as n:
            r = list(m.forward(*shot))
            if case["ND"] == 2:
                g, f = _gradient(m, shot)
                r += list(g.values()) + f
        runs.append(r)
        counts.append(n)
    m.close()
    grads = int(case["ND"] == 2)
    assert counts[0].made[0] > grads and counts[0].made[1] >= grads
    assert counts[0].gave_up == counts[1].made == (0, 0)
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
    case = dict(ND=2, FDORDER=4, N=(113, 140), L=L, freesurf=1)
    csts, params, (sp, s, rp) = _shot(case, nt=_nt(case))
    rp = rp[:, :100]
    m = Model(gpu_ctx, params, **csts)
    r, _ = _gradient(m, (sp, s, rp))
    m.close()
    monkeypatch.setenv("SEIS_RESIDENT_WAIT_MS", "0")
    ctx = Context(0)
    m = Model(ctx, params, **csts)
    got = [_gradient(m, (sp, s, rp))[0] for _ in range(2)]
    runs = ctx.resident_runs()
    m.close()
    ctx.close()
    for g in got:
        for k in r:
            assert np.array_equal(g[k], r[k]), k
    # every run tried and given up, the adjoint ones as well
    assert runs["made"] == (0, 0) and min(runs["gave_up"]) >= 2


@pytest.mark.parametrize("case", [dict(ND=2, FDORDER=8, N=(100, 100)),
                                  dict(ND=22, FDORDER=12, N=(60, 40))], ids=_ids)
def test_run_longer_than_the_wait(gpu_ctx, monkeypatch, case):
    """More steps than 16 bits number, on grids with blocks of halo cells alone,
    which are at the end of the run long before the others."""
    from seiscl_amd import Context, Model
    csts, params, (sp, s, rp) = small_case(nab=8, NT=70000, **case)
    s = np.random.default_rng(4).standard_normal(s.shape).astype(np.float32)
    monkeypatch.setenv("SEIS_RESIDENT_WAIT_MS", "20")
    ctx = Context(0)
    m = Model(ctx, params, **csts)
    got = m.forward(sp, s, rp[:, :4])
    runs = ctx.resident_runs()
    m.bind_shot(sp, s, rp[:, :4])
    for t in range(0, 70000, 14):    # too short for resident runs
        m.run_steps(t, 14)
    ref, after = m.read_shot(), ctx.resident_runs()
    m.close()
    ctx.close()
    assert runs == after == dict(made=(1, 0), gave_up=(0, 0))
    for a, b in zip(got, ref):
        assert np.abs(b[-100:]).max() > 0 and np.array_equal(a, b)


def test_no_run_beside_another_process(gpu_ctx):
    """While another process (here: another open file) holds the GPU's lock file,
    forward, gradient and batch steps are made by the step kernels."""
    import fcntl
    import glob
    from seiscl_amd import Model
    from seiscl_amd.engine import Batch
    csts, params, (sp, s, rp) = _shot(dict(ND=2, FDORDER=4, N=(113, 140)))
    shot = (sp, s, rp[:, :90])
    m, b = Model(gpu_ctx, params, **csts), Batch(gpu_ctx, 2)

    def run():
        g, f = _gradient(m, shot)
        out = m.forward(*shot)
        m.bind_shot(*shot)
        slot = b.add(m)
        b.step(NT)
        last = m.read_shot()
        b.remove(slot)
        return list(g.values()) + f + out + last

    with Runs(gpu_ctx) as free:
        want = run()
    locks = [open(p) for p in glob.glob("/tmp/seiscl_amd-resident-*.lock")]
    for f in locks:
        fcntl.flock(f, fcntl.LOCK_EX | fcntl.LOCK_NB)
    with Runs(gpu_ctx) as held:
        got = run()
    for f in locks:
        f.close()
    with Runs(gpu_ctx) as again:
        run()
    b.close()
    m.close()
    assert locks and free.made == again.made == (3, 1)
    assert held.made == (0, 0) and free.gave_up == held.gave_up == again.gave_up == (0, 0)
    for x, y in zip(got, want):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("L", [0, 2])
def test_runs_beside_another_context(gpu_ctx, L):
    """Resident runs on grids with blocks of halo cells, beside the kernels of a
    second context's 3D gradient: none gives up."""
    from seiscl_amd import Context, Model
    case = dict(ND=2, FDORDER=8, N=(100, 100), L=L)
    csts, params, (sp, s, rp) = _shot(case, nt=_nt(case))
    rp = rp[:, :90]
    c3, p3, shot3 = small_case(ND=3, N=(64, 60, 66), NT=60, nab=8)
    res3 = [np.ones((60, shot3[2].shape[1]), np.float32)] * 3
    stop, errors, ctx = threading.Event(), [], Context(0)

    def other():
        try:
            m3 = Model(ctx, p3, **c3)
            while not stop.is_set():
                m3.grad_zero()
                m3.gradient(*shot3, res=res3)
            m3.close()
        except Exception as e:
            errors.append(e)

    m = Model(gpu_ctx, params, **csts)
    ref, _ = _gradient(m, (sp, s, rp))
    th = threading.Thread(target=other)
    th.start()
    try:
        with Runs(gpu_ctx) as runs:
            got = [_gradient(m, (sp, s, rp))[0] for _ in range(40)]
    finally:
        stop.set()
        th.join()
        m.close()
        ctx.close()
    for g in got:
        for k in ref:
            assert np.array_equal(g[k], ref[k]), k
    assert not errors and min(runs.made) >= 40 and runs.gave_up == (0, 0)
