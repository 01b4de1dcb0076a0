"""Columns whose whole state stays on chip: workgroups of at most 512 threads keep
their junction pairs in registers (up to three a thread) or in LDS, and give bit
for bit what the general kernels (workgroups of 1024 threads) give, forward and
backward; the padded lattice solve of small stores against the oracle."""
import numpy as np
import pytest

import pyjjasim_amd as pa
from oracle import te_oracle as to

pytestmark = pytest.mark.gpu


def _circuit(kind, n, m, uniform=True):
    c = {"sq": pa.SquareArray, "hc": pa.HoneycombArray, "tri": pa.TriangularArray}[kind](n, m)
    rng = np.random.default_rng(n * 100 + m)
    c.set_critical_current(np.exp(0.1 * rng.standard_normal(c.junction_count())))
    c.set_capacitance(0.7 if uniform else 0.5 + rng.random(c.junction_count()))
    return c


# (lattice, sizes, uniform, workgroup): one pair a thread with pairs to spare and
# exactly full, two, three, and the form with its state in LDS
FORMS = [("sq", 6, 5, True, 64), ("sq", 9, 8, True, 64), ("sq", 9, 8, False, 64), ("hc", 6, 5, True, 64),
         ("sq", 16, 13, True, 128), ("tri", 8, 6, True, 64), ("tri", 12, 9, False, 128), ("sq", 30, 21, True, 256),
         ("tri", 16, 12, True, 512), ("sq", 31, 40, True, 512), ("hc", 14, 12, False, 256)]


@pytest.mark.parametrize("kind,n,m,uniform,bs", FORMS)
def test_gpu_resident_columns_bit_identical(kind, n, m, uniform, bs):
    c = _circuit(kind, n, m, uniform)
    W, Nt = 3, 40
    print(f"[resident] {kind} {n}x{m}, {bs} threads", flush=True)
    t = 0.05 * np.arange(Nt)
    drive = pa.SeparableSource(c.current_base(0.0)[:, None] * np.array([0.4, 0.9, 1.4]), 1.0 + 0.3 * np.sin(t))
    f = 0.1 + 0.02 * np.arange(c.face_count())[:, None, None] / c.face_count() + 0.01 * np.sin(t)[None, None, :]
    runs = [pa.TimeEvolutionProblem(c, time_step=0.05, time_step_count=Nt, external_flux=f, current_sources=drive,
                                    temperature=T, seed=3, store_time_steps=[0, 17, Nt - 1], block_size=b,
                                    steps_per_launch=spl).compute()
            for b, spl, T in ((1024, None, 0.02), (bs, 1, 0.02), (bs, 13, 0.02), (1024, None, 0.0), (bs, None, 0.0))]
    for a, b in ((1, 0), (2, 0), (4, 3)):
        for get in ("get_theta", "get_current", "get_vortex_configuration"):
            np.testing.assert_array_equal(getattr(runs[a], get)(), getattr(runs[b], get)())


@pytest.mark.parametrize("kind,n,m,uniform,bs", FORMS)
def test_gpu_resident_gradients_bit_identical(kind, n, m, uniform, bs):
    torch = pytest.importorskip("torch")
    c = _circuit(kind, n, m, uniform)
    Nj, Nf, W, Nt = c.junction_count(), c.face_count(), 2, 30
    rng = np.random.default_rng(1)
    put = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")
    Ic, f = put(np.exp(0.1 * rng.standard_normal(Nj))), put(0.1 + 0.02 * rng.standard_normal((Nf, W)))
    Is, G = put(np.outer(c.current_base(0.0), [0.5, 1.1])), put(rng.standard_normal((Nj, W, 3)))
    print(f"[resident] gradient {kind} {n}x{m}, {bs} threads", flush=True)
    out = []
    for b in (1024, bs):
        with pa.DifferentiableEvolution(c, time_step=0.05, time_step_count=Nt, problem_count=W, temperature=0.01,
                                        store_time_steps=[0, 11, Nt - 1], checkpoint_every=8, seed=6,
                                        block_size=b) as evo:
            leaves = [v.clone().requires_grad_(True) for v in (Ic, f, Is)]
            (evo(*leaves) * G).sum().backward()
            out.append([v.grad.cpu().numpy() for v in leaves])
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


# sides at and around multiples of 16 modes (one, two and three pairs of blocks),
# the smallest padded lattice, one that is too narrow for it, an elongated one
@pytest.mark.parametrize("n,m", [(9, 9), (8, 12), (17, 18), (33, 34), (34, 65), (66, 20)])
def test_gpu_padded_lattice_solve_matches_oracle(n, m):
    c = _circuit("sq", n, m)
    Nt, ts = 60, [30, 59]
    Is = c.current_base(0.0)[:, None, None] * np.array([0.6, 1.3])[None, :, None]
    print(f"[resident] lattice {n}x{m} vs oracle", flush=True)
    res = pa.TimeEvolutionProblem(c, time_step=0.05, time_step_count=Nt, external_flux=0.21, current_sources=Is,
                                  store_time_steps=ts, solver="lattice", face_store="lds").compute()
    ref = to.evolve(c, dt=0.05, Nt=Nt, f=0.21, Is=Is, store_time_steps=ts)
    th, V = res.get_theta(), res.get_voltage()
    assert np.abs(th - ref["theta"]).max() <= 1e-9 * np.abs(ref["theta"]).max()
    assert np.abs(V - ref["voltage"]).max() <= 1e-9 * np.abs(ref["voltage"]).max()
    np.testing.assert_array_equal(res.get_vortex_configuration(), to.vortex(c.get_cycle_matrix(), ref["theta"]))
