"""The chunked kernels of the small models where they can go wrong, against the
oracle: nodes per thread 1..8 and fibres that end at their boundaries, matrices whose
waves are coupled across their boundaries, a dt that changes from step to step,
stimuli on another parameter and through the clamp, the stimulation state machine
over launches and groups of 64 Heun steps, the serial solve's cached factors, and the
reverse sweep's 1..4 nodes per thread.

Bars as elsewhere: relative L2 error of Vm <= 1e-10 for the partitioned solve, bits
for the serial solve and between schedules, 1e-9 for gradients against the dense
reference.
"""
import numpy as np
import pytest

from cases import AM, CM, firing_table, vc_lane_stim_range
from oracle_binding import OracleBatch

pytestmark = pytest.mark.gpu


def _mesh(lengths, h=0.01, seed=1):
    n = np.array(lengths, np.int32)
    rng = np.random.default_rng(seed)
    elem = h * (1.0 + 0.1 * rng.uniform(-1.0, 1.0, int(n.sum()) - n.size))
    return dict(n_nodes=n, element_lengths=elem, prefactor=rng.uniform(3.0, 4.5, n.size) / (AM * CM))


def _pulse(n, amplitude=1200.0, stim_param=0):
    mid = n // 2
    F = n.size
    return dict(stim_begin=np.maximum(mid - 1, 0).astype(np.int32), stim_end=np.minimum(mid + 2, n).astype(np.int32),
                onset=np.random.default_rng(2).uniform(0.0, 0.05, F), duration=np.full(F, 0.1),
                amplitude=np.full(F, amplitude), stim_param=stim_param)


def _rows(n_steps, dt=1e-3, dt1=None):
    t = np.arange(n_steps) * dt
    return np.stack([t, np.full(n_steps, dt), np.full(n_steps, dt / 2),
                     np.full(n_steps, dt) if dt1 is None else np.broadcast_to(dt1, (n_steps,))], 1)


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def _run(mesh, stim, rows, n0D=1, tuning=None, **kw):
    from opendihu_amd.fibers import FiberBatch
    g = FiberBatch(**mesh, **kw)
    g.set_tuning(**(tuning or {}))
    g.set_current_stimulation(**stim)
    g.enable_spike_detection(0.0)
    g.advance_schedule(rows, n0D)
    out = g.get_states(), g.spikes()
    g.close()
    return out


def _oracle(mesh, stim, rows, scheme, n0D=1):
    o = OracleBatch(**mesh, scheme=scheme, threads=8)
    o.set_current_stimulation(**stim)
    o.enable_spike_detection(0.0)
    o.advance_schedule(rows, n0D)
    return o


# 128, 256 and 512 threads per fibre; ends at, before and after thread and wave boundaries
@pytest.mark.parametrize("threads,lengths", [
    (128, [2, 127, 128, 129, 640, 897, 1024]),
    (256, [2, 3, 256, 257, 511, 513, 769, 1025, 1281, 1537, 1793, 2047]),
    (256, [4096, 3585, 2561, 1537, 513, 64]),
])
@pytest.mark.parametrize("scheme", ["CN", "IE"])
def test_nodes_per_thread(threads, lengths, scheme):
    mesh = _mesh(lengths)
    stim = _pulse(mesh["n_nodes"])
    rows = _rows(250)
    states, spikes = _run(mesh, stim, rows, scheme=scheme, kernels="fused", tuning=dict(threads=threads))
    split, _ = _run(mesh, stim, rows, scheme=scheme, kernels="split", tuning=dict(threads=threads))
    o = _oracle(mesh, stim, rows, scheme)
    assert _rel(states[0], o.vm()) <= 1e-10
    np.testing.assert_array_equal(spikes[0], o.spikes()[0])
    if 2 in lengths:  # wholly stimulated, the only fibre to reach the threshold in these steps
        assert (spikes[0] > 0).any()
    np.testing.assert_array_equal(states, split)


@pytest.mark.parametrize("dt1", [0.05, 1.0])
@pytest.mark.parametrize("scheme", ["CN", "IE"])
def test_waves_coupled_across_boundaries(dt1, scheme):
    """a diffusion step of 100 to 7700 squared elements: the separators' reduction
    takes all its levels and the waves' ends depend on each other"""
    mesh = _mesh([2, 63, 65, 200, 257, 700, 1025, 2048], h=0.001)
    stim = _pulse(mesh["n_nodes"])
    rows = _rows(60, dt1=dt1)
    o = _oracle(mesh, stim, rows, scheme)
    for kernels in ("fused", "split"):
        states, _ = _run(mesh, stim, rows, scheme=scheme, kernels=kernels)
        assert np.isfinite(states).all()
        assert _rel(states[0], o.vm()) <= 1e-10, kernels


def test_dt_changes_from_step_to_step():
    """the factored matrix follows dt: equal over some steps, different in the last
    bits, by a factor of two and back"""
    mesh = _mesh([5, 300, 1000, 1500])
    stim = _pulse(mesh["n_nodes"])
    k = np.arange(120)
    dt1 = np.where(k % 7 < 3, 1e-3, 1e-3 * (1.0 + 1e-13 * k)) * np.where(k // 30 == 2, 2.0, 1.0)
    rows = _rows(120, dt1=dt1)
    o = _oracle(mesh, stim, rows, "CN")
    states, _ = _run(mesh, stim, rows, scheme="CN", kernels="fused", tuning=dict(steps_per_launch=50))
    split, _ = _run(mesh, stim, rows, scheme="CN", kernels="split")
    np.testing.assert_array_equal(states, split)
    assert _rel(states[0], o.vm()) <= 1e-10
    serial, _ = _run(mesh, stim, rows, scheme="CN", kernels="fused", thomas="serial")
    np.testing.assert_array_equal(serial[0], o.vm())


@pytest.mark.parametrize("kernels", ["fused", "split"])
def test_serial_solve_at_the_edges(kernels):
    """rows in groups of 8 (fused) and 64 (split) of the recurrence"""
    mesh = _mesh([2, 3, 7, 8, 9, 16, 63, 64, 65, 127, 128, 129, 1025, 2048])
    stim = _pulse(mesh["n_nodes"])
    rows = _rows(120)
    o = _oracle(mesh, stim, rows, "IE")
    states, spikes = _run(mesh, stim, rows, scheme="IE", kernels=kernels, thomas="serial")
    for k in range(4):
        np.testing.assert_array_equal(states[k], o.get_state(k), err_msg=f"state {k}")
    np.testing.assert_array_equal(spikes[0], o.spikes()[0])


def test_flags_of_many_heun_steps_are_bounded():
    """a launch covers fewer steps where its flags (16 bytes per fibre and 64 Heun steps)
    would take more than 64 MiB: 512 steps of 2 x 64 Heun steps are 256 MiB here"""
    import torch
    from opendihu_amd.fibers import FiberBatch
    F, n0D, K = 16384, 64, 512
    mesh = _mesh(np.full(F, 2))
    b = FiberBatch(**mesh, scheme="CN", kernels="fused")
    rows = _rows(K)
    rows[:, 2] /= n0D
    b.advance_schedule(rows[:1], n0D)
    b.synchronize()
    free = torch.cuda.mem_get_info()[0]
    b.advance_schedule(rows, n0D)
    b.synchronize()
    assert free - torch.cuda.mem_get_info()[0] <= 100 << 20
    assert b.launch_counts()["fused"] == 1 + 4


@pytest.mark.parametrize("n,n0D", [(2048, 24350), (2048, 26000), (900, 40000)])
def test_fused_serial_solve_beside_many_heun_steps(n, n0D):
    """the flags of a half step's Heun steps share the LDS with the factored matrix (up
    to 24400 steps at 2048 nodes): past that the solve assembles its rows each time, and
    the states keep the split kernels' bits"""
    mesh = _mesh([n, 5])
    stim = _pulse(mesh["n_nodes"])
    rows = _rows(1)
    rows[:, 2] /= n0D
    fused, _ = _run(mesh, stim, rows, n0D, scheme="CN", kernels="fused", thomas="serial")
    split, _ = _run(mesh, stim, rows, n0D, scheme="CN", kernels="split", thomas="serial")
    assert np.isfinite(fused).all() and np.ptp(fused[0]) > 0
    np.testing.assert_array_equal(fused, split)


@pytest.mark.parametrize("n_fibers,nmax", [(8191, 8), (8192, 8), (8200, 8), (16384, 16), (25000, 24)])
def test_serial_solve_of_many_short_fibres(n_fibers, nmax):
    """one lane or one wave per fibre, whole and partial waves of fibres: the oracle's bits"""
    n = np.random.default_rng(4).integers(2, nmax + 1, n_fibers)
    n[0] = nmax
    mesh = _mesh(n)
    stim = _pulse(mesh["n_nodes"])
    rows = _rows(30)
    o = _oracle(mesh, stim, rows, "CN")
    states, _ = _run(mesh, stim, rows, scheme="CN", kernels="split", thomas="serial")
    for k in range(4):
        np.testing.assert_array_equal(states[k], o.get_state(k), err_msg=f"state {k}")


@pytest.mark.parametrize("stim_param,amplitude", [(0, 1200.0), (1, 400.0), (3, 5.0)])
@pytest.mark.parametrize("n0D", [1, 3])
def test_pulse_on_any_parameter(stim_param, amplitude, n0D):
    mesh = _mesh([3, 150, 700, 1100])
    stim = _pulse(mesh["n_nodes"], amplitude, stim_param)
    rows = _rows(150)
    rows[:, 2] /= n0D
    states, _ = _run(mesh, stim, rows, n0D, scheme="IE", kernels="fused")
    split, _ = _run(mesh, stim, rows, n0D, scheme="IE", kernels="split")
    o = _oracle(mesh, stim, rows, "IE", n0D)
    np.testing.assert_array_equal(states, split)
    assert _rel(states[0], o.vm()) <= 1e-10


@pytest.mark.parametrize("n0D,per_launch", [(1, 512), (1, 13), (3, 45), (5, 7)])
@pytest.mark.parametrize("only", [False, True])
def test_stimulation_state_machine_over_launches(n0D, per_launch, only):
    """repeat windows, jitter lists and the clamp with the flags of a whole launch
    evaluated beforehand: states, spikes and the stimulation log as the split
    kernels', and the oracle's log"""
    from opendihu_amd.fibers import FiberBatch
    mesh = _mesh([40, 301, 600, 130, 257])
    n = mesh["n_nodes"]
    F = n.size
    off = np.concatenate([[0], np.cumsum(n)[:-1]])
    sb, se = vc_lane_stim_range(off, n // 2, n, 4)
    dt, runs = 2e-3, {}
    o = OracleBatch(**mesh, scheme="IE", threads=8)
    batches = {"oracle": o}
    for kernels in ("fused", "split"):
        batches[kernels] = FiberBatch(**mesh, scheme="IE", kernels=kernels)
    batches["fused"].set_tuning(steps_per_launch=per_launch)
    for name, b in batches.items():
        b.set_firing_table_stimulation(sb, se, firing_table(40, 10, 4.0, 0.1, seed=2), (np.arange(F) * 7) % 10 + 1,
                                       call_frequency=20.0, repeat_after_first_call=0.01,
                                       call_enable_begin=0.05 * (np.arange(F) % 3),
                                       jitter_lists=[[0.1, -0.1, 0.05][: f % 4] for f in range(F)], log_capacity=4096)
        b.enable_spike_detection(0.0)
        b.set_only_compute_if_stimulated(only)
        for k0, k in ((0, 100), (100, 151)):
            b.advance(k0 * dt, dt, k, dt0D=dt / 2 / n0D, n0D=n0D)
        times, fibres = b.stimulation_log()
        runs[name] = (b.vm(), b.spikes(), sorted(zip(fibres.tolist(), times.tolist())))
    assert len(runs["oracle"][2]) > F
    assert runs["fused"][2] == runs["split"][2] == runs["oracle"][2]
    np.testing.assert_array_equal(runs["fused"][0], runs["split"][0])
    np.testing.assert_array_equal(runs["fused"][1][0], runs["oracle"][1][0])
    assert _rel(runs["fused"][0], runs["oracle"][0]) <= 1e-10


def _gradients(lengths, scheme, threads, sensors, n_steps):
    """device gradient and dense reference of each fibre"""
    import adjoint_reference as R
    from opendihu_amd.adjoint import AdjointProblem
    from opendihu_amd.fibers import FiberBatch
    mesh = _mesh(lengths)
    n, F = mesh["n_nodes"], len(lengths)
    stim = _pulse(n)
    stim["onset"] = np.linspace(0.0, 0.004, F)
    rows = _rows(n_steps)
    rng = np.random.default_rng(5)
    theta = np.stack([rng.uniform(100, 140, F), rng.uniform(30, 42, F), rng.uniform(0.2, 0.4, F),
                      mesh["prefactor"] * AM * CM], 1)
    sensors = np.stack([sensors(k) for k in n]).astype(np.int32)
    b = FiberBatch(**mesh, scheme=scheme, kernels="fused", thomas="partitioned")
    b.set_current_stimulation(**stim)
    if threads == 256:
        b.set_tuning(adjoint_threads=256)
    prob = AdjointProblem(b, rows, sensors, checkpoint_interval=3)
    tr = prob.forward(theta)
    dtr = np.random.default_rng(6).standard_normal(tr.shape)
    grad = prob.backward(dtr)
    eoff = np.concatenate([[0], np.cumsum(n - 1)])
    for f in range(F):
        fib = R.Fibre(h=mesh["element_lengths"][eoff[f]:eoff[f + 1]], sb=int(stim["stim_begin"][f]),
                      se=int(stim["stim_end"][f]), onset=stim["onset"][f], duration=0.1, amplitude=1200.0,
                      sensors=sensors[f])
        yield f, grad[f], R.gradient(fib, theta[f], rows, scheme == "IE", dtr[:, f, :], AM * CM)


GRADIENT_SIZES = [([2, 65, 130], 256), ([257, 520, 770], 256), ([100, 600, 1025, 1600], 512)]


@pytest.mark.parametrize("scheme", ["CN", "IE"])
@pytest.mark.parametrize("lengths,threads", GRADIENT_SIZES)
def test_gradient_at_the_ends(scheme, lengths, threads):
    """sensors at the first and last node, reaction parameters only: in 8 steps the
    pulse does not reach them (or, with 2 nodes, there is no gradient), and the
    conductivity's derivative, 0 to 1e-20 in 80-bit arithmetic, is below the dense
    reference's rounding of 1e-15"""
    for f, g, ref in _gradients(lengths, scheme, threads, lambda k: np.array([0, k - 1]), 8):
        np.testing.assert_allclose(g[:3], ref[:3], rtol=1e-9, err_msg=f"fibre {f}")


@pytest.mark.parametrize("scheme", ["CN", "IE"])
@pytest.mark.parametrize("lengths,threads", [([65, 130], 256), ([257, 520, 770], 256), ([100, 600, 1025, 1600], 512)])
def test_gradient_nodes_per_thread(scheme, lengths, threads):
    """sensors at the pulse and beside it, all four parameters; the dense reference
    is within 1e-13 of itself in 80-bit arithmetic here"""
    for f, g, ref in _gradients(lengths, scheme, threads, lambda k: k // 2 + np.array([-2, 0, 3]), 12):
        np.testing.assert_allclose(g, ref, rtol=1e-9, err_msg=f"fibre {f}")


@pytest.mark.parametrize("thomas", ["serial", "partitioned"])
def test_recomputed_segments_have_the_forward_bits(thomas):
    """whole tape and checkpoints: the same gradient for either solve"""
    from opendihu_amd.adjoint import AdjointProblem
    from opendihu_amd.fibers import FiberBatch
    mesh = _mesh([30, 300, 700])
    stim = _pulse(mesh["n_nodes"])
    theta = np.stack([np.full(3, 120.0), np.full(3, 36.0), np.full(3, 0.3), mesh["prefactor"] * AM * CM], 1)
    sensors = (mesh["n_nodes"][:, None] // 2 + np.array([[-2, 3]])).astype(np.int32)
    grads = []
    for tape in ("whole", "segments"):
        b = FiberBatch(**mesh, scheme="CN", kernels="fused", thomas=thomas)
        b.set_current_stimulation(**stim)
        prob = AdjointProblem(b, _rows(70), sensors, checkpoint_interval=16, tape=tape)
        tr = prob.forward(theta)
        grads.append(prob.backward(np.random.default_rng(6).standard_normal(tr.shape)))
    assert np.isfinite(grads[0]).all() and (grads[0] != 0).all()
    np.testing.assert_array_equal(grads[0], grads[1])


@pytest.mark.parametrize("exp,vm", [("libm", -2500.0), ("libm", -6900.0), ("approx", -2800.0), ("approx", -10100.0),
                                    ("approx", 24000.0)])
def test_far_from_rest(exp, vm):
    """where the product of the reaction's denominators overflows, its rates stay finite:
    Heun steps so short that the states keep the serial run's values (1e-12), the
    gradient's sums finite"""
    from opendihu_amd.adjoint import AdjointProblem
    from opendihu_amd.fibers import FiberBatch
    mesh = _mesh([2, 70])
    rows = _rows(4)
    rows[:, 2] = 1e-200
    runs = []
    for kernels, thomas in (("fused", "serial"), ("fused", "partitioned"), ("split", "partitioned")):
        b = FiberBatch(**mesh, scheme="CN", kernels=kernels, thomas=thomas, exp_mode=exp)
        b.set_state(0, np.full(72, vm))
        b.advance_schedule(rows)
        runs.append(b.get_states())
    assert np.isfinite(runs[0]).all()
    for r in runs[1:]:
        np.testing.assert_allclose(r, runs[0], rtol=1e-12)
    b = FiberBatch(**mesh, scheme="CN", kernels="fused", thomas="partitioned", exp_mode=exp)
    b.set_state(0, np.full(72, vm))
    b.set_current_stimulation(**_pulse(mesh["n_nodes"]))
    theta = np.stack([np.full(2, 120.0), np.full(2, 36.0), np.full(2, 0.3), mesh["prefactor"] * AM * CM], 1)
    prob = AdjointProblem(b, rows, np.array([[0, 1], [5, 69]], np.int32))
    tr = prob.forward(theta)
    assert np.isfinite(tr).all() and np.isfinite(prob.backward(np.ones_like(tr))).all()


@pytest.mark.parametrize("thomas", ["serial", "partitioned"])
def test_adjoint_leaves_fibres_without_centre_buffer_unstimulated(thomas):
    """point-buffer order: a fibre whose stimulation point lies in none of its buffers is
    never stimulated, in the adjoint's forward and reverse sweep as elsewhere: traces and
    gradients of a batch whose fibre 1 has no pulse, bit for bit"""
    from opendihu_amd.adjoint import AdjointProblem
    from opendihu_amd.fibers import FiberBatch
    mesh = _mesh([301, 301, 301])
    stim = _pulse(mesh["n_nodes"])
    theta = np.stack([np.full(3, 120.0), np.full(3, 36.0), np.full(3, 0.3), mesh["prefactor"] * AM * CM], 1)
    sensors = (mesh["n_nodes"][:, None] // 2 + np.array([[-1, 0, 3]])).astype(np.int32)
    runs = []
    for order in (True, False):
        b = FiberBatch(**mesh, scheme="CN", kernels="fused", thomas=thomas)
        b.set_current_stimulation(**(stim if order else dict(stim, onset=stim["onset"] + np.array([0.0, 1e6, 0.0]))))
        if order:
            b.set_point_buffer_order(4, np.array([150, 10 ** 6, 150], np.int32))
        prob = AdjointProblem(b, _rows(60), sensors, checkpoint_interval=16)
        tr = prob.forward(theta)
        runs.append((tr, prob.backward(np.random.default_rng(6).standard_normal(tr.shape))))
    assert (runs[0][0][-1, 1] < -60).all() and (runs[0][0][-1, 0] > -60).any()   # fibre 1 rests, fibre 0 does not
    np.testing.assert_array_equal(runs[0][0], runs[1][0])
    np.testing.assert_array_equal(runs[0][1], runs[1][1])
