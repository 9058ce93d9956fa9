"""Batch steps made as resident runs and by the batch kernels, mixed, against the
same jobs alone, step kernel by step kernel.  The context's counts of resident
runs say which way the steps went."""
import numpy as np
import pytest

from cases import small_case

pytestmark = pytest.mark.gpu

# one large job, small ones of every kind, one with more sources than the
# receivers' launch compares with, one whose receiver table the resident runs refuse,
# one that is better off resident in long runs only
JOBS = [dict(ND=22, FDORDER=8, N=(600, 1500), NT=90), dict(ND=22, FDORDER=8, N=(70, 90), NT=64),
        dict(ND=2, FDORDER=8, N=(65, 129), NT=113), dict(ND=22, FDORDER=2, N=(64, 400), NT=40),
        dict(ND=2, FDORDER=12, N=(90, 120), NT=70), dict(ND=2, FDORDER=4, N=(80, 100), NT=80),
        dict(ND=2, FDORDER=4, N=(433, 1217), NT=90)]


def _job(k, kw):
    csts, p, (sp, s, rp) = small_case(**kw)
    if k == 4:
        sp = np.repeat(sp[:, :1], 17, 1)
        sp[0] += 10 * np.arange(17)
        s = np.repeat(s[:, :1], 17, 1)
        rp[:3, :3] = sp[:3, :3]
    if k == 5:
        rp = np.tile(rp, (1, 1100 // rp.shape[1] + 1))
    rp[:3, 0] = sp[:3, 0]
    return csts, p, (sp, s, rp)


def _alone(ctx, job):
    from seiscl_amd import Model
    csts, p, shot = job
    m = Model(ctx, p, **csts)
    m.set_profiling(True)
    out = m.forward(*shot)
    m.close()
    return out


@pytest.mark.parametrize("chunk", [15, 16, 33, 200])
@pytest.mark.parametrize("jobs", [[0], [1, 2], [0, 5], [6, 5], [0, 1, 2, 3, 4, 5]], ids=str)
@pytest.mark.parametrize("wait", [500, 0])
def test_batch_steps(gpu_ctx, monkeypatch, chunk, jobs, wait):
    from seiscl_amd import Context, Model
    from seiscl_amd.engine import Batch
    resident = chunk >= (200 if 6 in jobs else 16)
    jobs = [_job(k, JOBS[k]) for k in jobs]
    want = [_alone(gpu_ctx, j) for j in jobs]
    monkeypatch.setenv("SEIS_RESIDENT_WAIT_MS", str(wait))   # 0: every resident run gives up
    ctx = Context(0)
    models, b = [], Batch(ctx, 8)
    for csts, p, shot in jobs:
        m = Model(ctx, p, **csts)
        m.bind_shot(*shot)
        models.append(m)
        b.add(m)
        b.step(3)            # later jobs join while the first ones step
    while b.status()[0]:
        b.step(chunk)
    got = []
    for k, m in enumerate(models):
        got.append(m.read_shot())
        b.remove(k)
        m.close()
    b.close()
    runs = ctx.resident_runs()
    ctx.close()
    for g, w in zip(got, want):
        for a, r in zip(g, w):
            assert np.abs(r).max() > 0 and np.array_equal(a, r)
    assert (runs["made"][0] > 0) == (resident and wait > 0)
    assert (runs["gave_up"][0] > 0) == (resident and wait == 0)
    assert runs["made"][1] == runs["gave_up"][1] == 0


def test_model_bound_again_in_the_batch(gpu_ctx):
    """A slot steps the shot it was added with: 1100 receivers stay with the batch
    kernels also when the model is bound to a few of them."""
    from seiscl_amd import Model
    from seiscl_amd.engine import Batch
    csts, p, (sp, s, rp) = small_case(ND=2, FDORDER=4, N=(80, 100), NT=80)
    rp = np.tile(rp, (1, 1100 // rp.shape[1] + 1))
    m, b = Model(gpu_ctx, p, **csts), Batch(gpu_ctx, 2)
    before = gpu_ctx.resident_runs()
    m.bind_shot(sp, s, rp)
    b.add(m)
    m.bind_shot(sp, s, rp[:, :7], init=False)
    b.step(80)
    gpu_ctx.sync()
    field = m.read_field("vx")
    after = gpu_ctx.resident_runs()
    b.close()
    m.set_profiling(True)
    m.forward(sp, s, rp)
    want = m.read_field("vx")
    m.close()
    assert before == after
    assert np.abs(want).max() > 0 and np.array_equal(field, want)
