"""The 2D time loop with the wavefield held on the chip (GPU tests, through
pysit_amd_resident_run): every result equals the one-launch-per-step loop bit
for bit."""
import numpy as np
import pytest

from tests.problems import Synthetic
from tests.test_gpu_graph import _batch, _gradient, _same, _uneven

pytestmark = pytest.mark.gpu


def _pair(probs, dtype, **kw):
    """The same batch on the step kernels and on the resident loop."""
    return _batch(probs, dtype, 0, **kw), _batch(probs, dtype, None, resident=True, **kw)


def _check(probs, dtype, res, segment=None, **kw):
    steps, held = _pair(probs, dtype, **kw)
    assert held.resident_tables() is not None and steps.resident_tables() is None
    ref = _gradient(steps, res, segment=segment)
    for rep in range(2):
        out = _gradient(held, res, segment=segment)
        assert _same(out[0], ref[0]), f"traces, pass {rep}"
        assert _same(out[1], ref[1]), f"images, pass {rep}"
    assert held.resident_tables().epoch.value > 0  # the runs above went through it
    return steps, held


def _residuals(probs, seed=9):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal((p.nt, p.n_rec)) for p in probs]


# (shape, PML widths): strips of every kind -- no room between the x sides, one
# strip per side, a single middle strip, many strips; z rows of one cell more or
# less than whole cells, rows wholly inside the PML, no PML on a side
SHAPES = [((24, 30), ((4, 5), (6, 4))), ((61, 53), ((6, 7), (5, 8))), ((150, 65), ((10, 8), (7, 9))),
          ((90, 260), ((0, 9), (0, 6))), ((333, 41), ((12, 12), (12, 12)))]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("order", [2, 4, 6, 8])
@pytest.mark.parametrize("shape,pml", SHAPES)
def test_resident_loop_equals_step_launches(gpu, dtype, order, shape, pml):
    p = Synthetic(shape, pml, (0.01, 0.012), 83, order, seed=order, n_rec=9)
    print("resident", shape, order, np.dtype(dtype).name, flush=True)
    _check([p], dtype, _residuals([p]))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("segment", [None, 30])
def test_resident_loop_uneven_shots_and_segments(gpu, dtype, segment):
    probs = _uneven()
    print("resident uneven", np.dtype(dtype).name, segment, flush=True)
    _check(probs, dtype, _residuals(probs), segment=segment)


@pytest.mark.parametrize("window", [7, 32])
def test_resident_loop_windows_and_chunks(gpu, window, monkeypatch):
    """FP32 windows that end inside launches and at their ends: the source and
    receiver buffers hold 32 slots here, so a run takes many launches."""
    from pysit_amd import resident
    monkeypatch.setattr(resident, "CHUNK_BYTES", 1)
    p = Synthetic((90, 110), ((10, 10), (10, 10)), (0.01, 0.01), 300, 8, seed=4)
    for seg in (None, 50):
        print("resident window", window, seg, flush=True)
        _check([p], np.float32, _residuals([p], 7), segment=seg, ic_window=window)


@pytest.mark.parametrize("kw", [{"imaging_period": 3}, {"adjoint": "exact"}])
def test_resident_loop_imaging_period_and_exact_adjoint(gpu, kw):
    p = Synthetic((70, 75), ((6, 7), (5, 8)), (0.01, 0.012), 90, 8, seed=2)
    for dtype in (np.float64, np.float32):
        print("resident", kw, np.dtype(dtype).name, flush=True)
        _check([p], dtype, _residuals([p], 1), **kw)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_resident_loop_born_and_groups(gpu, dtype, monkeypatch):
    """Born runs, and shots that run in several groups."""
    from pysit_amd import resident
    probs = [Synthetic((60, 75), ((6, 7), (5, 8)), (0.01, 0.012), 90, 8, seed=s, n_src=1 + s) for s in range(3)]
    for p in probs[1:]:
        p.model, p.Cpad, p.dt = probs[0].model, probs[0].Cpad, probs[0].dt
    plan = resident.plan_groups
    monkeypatch.setattr(resident, "plan_groups", lambda shots, cus: plan(shots, len(shots[0].cut(1e9))))
    print("resident groups", np.dtype(dtype).name, flush=True)
    steps, held = _check(probs, dtype, _residuals(probs))
    assert len(held.resident_tables().group_lds) > 1
    m1 = np.random.default_rng(4).standard_normal(probs[0].model.shape)
    outs = []
    for b in (steps, held):
        b.forward(keep_dw=True, segment=probs[0].nt)
        outs.append([t.cpu().numpy().copy() for t in b.born(m1)])
    assert _same(outs[0], outs[1])


def test_resident_wait_bound_is_an_error(gpu):
    """A wait beyond its bound ends the launch and is reported: the host marks
    the run as one that waited too long, without any kernel that does."""
    from pysit_amd import _native as N
    p = Synthetic((61, 53), ((6, 7), (5, 8)), (0.01, 0.012), 40, 4, seed=3)
    steps, held = _pair([p], np.float64)
    ref = _gradient(steps, _residuals([p]))
    t = held.resident_tables()
    t.err[0] = 1
    with pytest.raises(N.NativeError, match="waited too long"):
        held.forward(keep_dw=True)
    out = _gradient(held, _residuals([p]))
    assert _same(out[0], ref[0]) and _same(out[1], ref[1])


@pytest.mark.parametrize("window", [7, 64])
def test_fp32_window_of_a_shot_that_starts_in_a_short_segment(gpu, window):
    """A shot whose step 0 lies in a segment too short for the resident loop:
    the step kernels leave its FP32 window open, and the window's end lies in
    a segment where the shot takes no step."""
    base = Synthetic((60, 50), ((6, 6), (5, 5)), (0.01, 0.01), 97, 8, seed=3, src_center=(30, 8))
    probs = [base] + [Synthetic((60, 50), ((6, 6), (5, 5)), (0.01, 0.01), nt, 8, seed=40 + nt, model=base.model,
                                dt=base.dt, src_center=(30, 8)) for nt in (5, 7, 36, 68)]
    res = _residuals(probs, 3)
    steps, held = _pair(probs, np.float32, ic_window=window)
    ref = _gradient(steps, res)
    assert all(np.abs(i).max() > 0 for i in ref[1])
    short = []  # lengths of the runs that the step kernels took
    run = held._resident_for
    held._resident_for = lambda b, mode, n: run(b, mode, n) or short.append((mode, n))
    # slots 90 to 96 are a segment of 7: the shots of 5 and 7 steps live in it
    out = _gradient(held, res, segment=30)
    assert (2, 7) in short and held.resident_tables().epoch.value > 0
    assert _same(out[0], ref[0]) and _same(out[1], ref[1])


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_resident_expired_wait_ends_the_launch(gpu, dtype):
    """Waits with a bound of one poll expire in many strips at different
    steps: every launch ends, the run is reported, and the runs after it are
    whole again."""
    import torch
    from pysit_amd import _native as N
    from pysit_amd import resident
    p = Synthetic((333, 141), ((12, 12), (12, 12)), (0.01, 0.01), 200, 8, seed=5)
    steps, held = _pair([p], dtype)
    ref = _gradient(steps, _residuals([p]))
    t = held.resident_tables()
    assert t.n_strips > 8
    t.struct.spin = 1
    print("resident expired wait", np.dtype(dtype).name, flush=True)
    held.forward(keep_dw=True)
    torch.cuda.synchronize()
    assert int(t.err[0]) == 1
    t.struct.spin = resident.SPIN
    with pytest.raises(N.NativeError, match="waited too long"):
        held.forward(keep_dw=True)
    out = _gradient(held, _residuals([p]))
    assert _same(out[0], ref[0]) and _same(out[1], ref[1])


def _one_poll(held):
    """Waits of this batch give up after one poll."""
    held.resident_tables().struct.spin = 1


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_results_of_an_expired_wait_are_nan(gpu, dtype):
    """No trace and no image of a run whose wait expired holds a number, also
    where the host has not seen it yet, and another batch's runs are not
    touched."""
    import torch
    from pysit_amd import _native as N
    p = Synthetic((333, 141), ((12, 12), (12, 12)), (0.01, 0.01), 200, 8, seed=5)
    res = _residuals([p])
    steps, held = _pair([p], dtype)
    other = _batch([p], dtype, None, resident=True)
    ref = _gradient(steps, res)
    _one_poll(held)
    print("resident expired results", np.dtype(dtype).name, flush=True)
    tr = held.forward(keep_dw=True)[0].cpu()
    assert torch.isnan(tr).all()
    held.resident_tables().err[0] = 0  # as if the host had not waited yet
    held.resident_tables().struct.spin = 1 << 20
    ic = held.migrate(res)
    assert torch.isnan(ic).all()
    tr = held.forward(keep_dw=True)[0].cpu()
    assert torch.isnan(tr).all()
    out = _gradient(other, res)
    assert _same(out[0], ref[0]) and _same(out[1], ref[1])
    held.resident_tables().err[0] = 1
    with pytest.raises(N.NativeError, match="waited too long"):
        held.check()
    with pytest.raises(RuntimeError, match="forward"):
        held.migrate(res)  # the history went with the run
    out = _gradient(held, res)
    assert _same(out[0], ref[0]) and _same(out[1], ref[1])


def test_modeling_raises_for_an_expired_wait(gpu, monkeypatch):
    """forward_model raises in the call whose wait expired, and the next call
    is right."""
    import pysit_amd as pa
    from pysit_amd import _native as N
    from pysit_amd import resident
    from tests.problems import c1_setup
    m, shots, solver, model = c1_setup(tf=0.3)
    ref = pa.TemporalModeling(solver, tile_x=8).forward_model(shots[0], model, return_parameters=["simdata"])
    monkeypatch.setattr(resident, "SPIN", 1)
    tools = pa.TemporalModeling(solver)
    print("resident expired forward_model", flush=True)
    with pytest.raises(N.NativeError, match="waited too long"):
        tools.forward_model(shots[0], model, return_parameters=["simdata"])
    out = tools.forward_model(shots[0], model, return_parameters=["simdata"])
    assert np.array_equal(out["simdata"], ref["simdata"])


def test_short_adjoint_segments_precompute_their_sources(gpu):
    """An adjoint run too short for the resident loop reads its sources
    precomputed, as every run of the step kernels does."""
    p = Synthetic((60, 50), ((6, 6), (5, 5)), (0.01, 0.01), 97, 8, seed=3)
    steps, held = _pair([p], np.float32)
    ref = _gradient(steps, _residuals([p]))
    out = _gradient(held, _residuals([p]), segment=30)
    assert _same(out[0], ref[0]) and _same(out[1], ref[1])
    assert held._inj_pre.numel() == 7 * (held.adj_inj[2].numel() - 1)  # slots 90 to 96


def test_evaluate_raises_for_an_expired_wait(gpu, monkeypatch):
    """The objective alone, whose traces never reach the host."""
    import pysit_amd as pa
    from pysit_amd import _native as N
    from pysit_amd import resident
    from tests.problems import c1_setup
    m, shots, solver, model = c1_setup(tf=0.3)
    pa.generate_seismic_data(shots, solver, model)
    trial = solver.ModelParameters(m, {"C": 1.01 * model.C})
    want = pa.TemporalLeastSquares(solver).evaluate(shots, trial)
    assert np.isfinite(want) and want > 0
    monkeypatch.setattr(resident, "SPIN", 1)
    obj = pa.TemporalLeastSquares(solver)
    print("resident expired evaluate", flush=True)
    with pytest.raises(N.NativeError, match="waited too long"):
        obj.evaluate(shots, trial)
    assert obj.evaluate(shots, trial) == want
