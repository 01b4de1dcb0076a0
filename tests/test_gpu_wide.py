"""Large lattice columns held in the registers of one workgroup (taken for the usual
step of lattices that leave no room in LDS for the padded solve) against the kernel of
512 threads, at 1e-9 of the phase scale with identical vortex counts."""
import numpy as np
import pytest

import pyjjasim_amd as pa

pytestmark = pytest.mark.gpu

# the smallest; an odd count of junctions in the first round (a pair across both), both
# ways; an odd junction count; long sides both ways (15 row parts a mode); the largest
SIZES = [(66, 66), (70, 71), (71, 70), (72, 72), (34, 261), (261, 34), (120, 70), (60, 128), (99, 100), (100, 100)]


def _run(c, block_size, W, Nt, T, beta_time, **kw):
    t = 0.05 * np.arange(Nt)
    drive = pa.SeparableSource(c.current_base(0.0)[:, None] * np.linspace(0.5, 1.3, W), 1.0 + 0.3 * np.sin(t))
    f = 0.1 + 0.02 * np.arange(c.face_count())[:, None, None] / c.face_count() + 0.01 * np.sin(t)[None, None, :]
    if beta_time:
        T = T * (1.0 + 0.5 * np.cos(t))[None, None, :] * np.ones((c.junction_count(), 1, 1))
    return pa.TimeEvolutionProblem(c, solver="lattice", parts=1, block_size=block_size, time_step=0.05,
                                   time_step_count=Nt, external_flux=f, current_sources=drive, temperature=T, seed=3,
                                   store_time_steps=[0, 5, 17, Nt - 1], steps_per_launch=13, **kw).compute()


def _compare(a, b):
    for get in ("get_theta", "get_current", "get_voltage"):
        u, v = getattr(a, get)(), getattr(b, get)()
        assert np.abs(u - v).max() <= 1e-9 * np.abs(u).max(), get
    np.testing.assert_array_equal(a.get_vortex_configuration(), b.get_vortex_configuration())


@pytest.mark.parametrize("n,m", SIZES)
@pytest.mark.parametrize("aniso,beta_l,T,beta_time", [(False, 0.0, 0.02, False), (True, 0.5, 0.0, False),
                                                      (True, 0.0, 0.02, True)])
def test_gpu_wide_matches(n, m, aniso, beta_l, T, beta_time):
    c = pa.SquareArray(n, m)
    x1, y1, x2, y2 = c.get_junction_coordinates()
    c.set_capacitance(np.where(y1 == y2, 1.0, 2.0) if aniso else 1.0)
    if beta_l:
        c.set_inductance(beta_l)
    rng = np.random.default_rng(n + m)
    c.set_critical_current(np.exp(0.1 * rng.standard_normal(c.junction_count())))
    print(f"[wide] {n}x{m} T={T}", flush=True)
    _compare(_run(c, 512, 2, 36, T, beta_time), _run(c, 1024, 2, 36, T, beta_time))


def test_gpu_wide_skips_a_zero_current_source():
    """A current source that counts as zero (np.allclose) is left out of the step, as in the
    general kernels, and still added to the stored current."""
    c = pa.SquareArray(66, 66)
    Is = 9e-9 * np.cos(np.arange(c.junction_count()))[:, None, None] * np.ones((1, 2, 1))
    f = 0.1 + 0.1 * np.random.default_rng(0).random(c.face_count())[:, None, None]
    print("[wide] zero current source", flush=True)
    a, b = (pa.TimeEvolutionProblem(c, solver="lattice", parts=1, block_size=bs, time_step=0.05, time_step_count=36,
                                    external_flux=f, current_sources=Is, store_time_steps=[0, 17, 35]).compute()
            for bs in (512, 1024))
    _compare(a, b)


def _lattice(n, m, aniso):
    c = pa.SquareArray(n, m)
    x1, y1, x2, y2 = c.get_junction_coordinates()
    c.set_capacitance(np.where(y1 == y2, 1.0, 2.0) if aniso else 1.0)
    c.set_critical_current(np.exp(0.1 * np.random.default_rng(n + m).standard_normal(c.junction_count())))
    return c


def _same_bits(a, b):
    return np.array_equal(a.get_theta(), b.get_theta())


# the other combinations of noise and of coefficients that are one value: coefficients of
# their own with noise, a noise amplitude of their own, neither
@pytest.mark.parametrize("aniso,T", [(True, 0.02), (False, "junction"), (False, 0.0)])
def test_gpu_wide_forms_match(aniso, T):
    """The two workgroup sizes agree, and not bit for bit: the large one's columns lay in
    registers (fused multiply-adds; the general kernels' results do not depend on the
    size)."""
    c = _lattice(71, 70, aniso)
    if T == "junction":
        T = 0.01 + 0.02 * np.random.default_rng(5).random((c.junction_count(), 1, 1))
    print("[wide] forms", flush=True)
    a, b = (_run(c, bs, 2, 36, T, False) for bs in (512, 1024))
    _compare(a, b)
    assert not _same_bits(a, b)


def test_gpu_wide_leaves_varying_temperature_to_the_general_kernel():
    c = _lattice(66, 66, True)
    assert _same_bits(*(_run(c, bs, 2, 36, 0.02, True) for bs in (512, 1024)))


def test_gpu_wide_lattices_share_a_plan():
    """Two large lattices of different sizes in one launch: each as alone with workgroups of
    512 threads, and in registers."""
    print("[wide] batch", flush=True)
    problems = []
    for n, m, W, T in ((66, 68, 2, 0.02), (99, 100, 1, 0.0)):
        c = _lattice(n, m, n == 66)
        problems.append(dict(circuit=c, time_step=0.05, time_step_count=30, external_flux=0.1, temperature=T, seed=3,
                             current_sources=c.current_base(0.0)[:, None, None] * np.linspace(0.5, 1.3, W)[None, :, None],
                             store_time_steps=[0, 11, 29], solver="lattice", parts=1, steps_per_launch=13))
    both = pa.TimeEvolutionBatch([pa.TimeEvolutionProblem(block_size=1024, **p) for p in problems], block_size=1024).compute()
    for p, b in zip(problems, both):
        a = pa.TimeEvolutionProblem(block_size=512, **p).compute()
        _compare(a, b)
        assert not _same_bits(a, b)
