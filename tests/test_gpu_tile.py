"""Lattices of at most 16 by 16 faces, whose face system one wave solves on the matrix
cores, against the staged factor: every shape class of the tile (the smallest lattice,
thin ones, odd and even sides, a full tile), phases, currents and gradients."""
import numpy as np
import pytest

import pyjjasim_amd as pa

pytestmark = pytest.mark.gpu

SIZES = [(3, 3), (3, 9), (17, 3), (5, 4), (8, 8), (9, 6), (10, 10), (12, 9), (16, 17), (17, 17)]


@pytest.mark.parametrize("n,m", SIZES)
@pytest.mark.parametrize("aniso,T,block_size", [(False, 0.02, None), (True, 0.0, None), (False, 0.0, 1024)])
def test_gpu_tile_matches_factor(n, m, aniso, T, block_size):
    c = pa.SquareArray(n, m)
    x1, y1, x2, y2 = c.get_junction_coordinates()
    c.set_capacitance(np.where(y1 == y2, 1.0, 2.0) if aniso else 1.0)
    Nt, W = 40, 3
    t = 0.05 * np.arange(Nt)
    kw = dict(time_step=0.05, time_step_count=Nt, temperature=T, seed=3, store_time_steps=[0, 17, Nt - 1],
              external_flux=0.1 + 0.02 * np.arange(c.face_count())[:, None, None] / c.face_count(),
              current_sources=pa.SeparableSource(c.current_base(0.0)[:, None] * np.array([0.4, 0.9, 1.3]), 1.0 + 0.3 * np.sin(t)))
    print(f"[tile] {n}x{m} T={T}", flush=True)
    a = pa.TimeEvolutionProblem(c, solver="cholesky", parts=1, **kw).compute()
    b = pa.TimeEvolutionProblem(c, solver="lattice", parts=1, block_size=block_size, **kw).compute()
    for get in ("get_theta", "get_current", "get_voltage"):
        u, v = getattr(a, get)(), getattr(b, get)()
        assert np.abs(u - v).max() <= 1e-9 * max(np.abs(u).max(), 1.0), get
    np.testing.assert_array_equal(a.get_vortex_configuration(), b.get_vortex_configuration())


@pytest.mark.parametrize("n,m", [(3, 3), (12, 9), (17, 17)])
def test_gpu_tile_gradients_match_factor(n, m):
    torch = pytest.importorskip("torch")
    c = pa.SquareArray(n, m)
    Nj, Nf, W, Nt = c.junction_count(), c.face_count(), 2, 24
    rng = np.random.default_rng(1)
    put = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")
    Ic, f = put(np.exp(0.1 * rng.standard_normal(Nj))), put(0.1 + 0.02 * rng.standard_normal((Nf, W)))
    Is, G = put(np.outer(c.current_base(0.0), [0.5, 1.1])), put(rng.standard_normal((Nj, W, 3)))
    out = []
    for solver in ("cholesky", "lattice"):
        with pa.DifferentiableEvolution(c, time_step=0.05, time_step_count=Nt, problem_count=W, temperature=0.01,
                                        store_time_steps=[0, 11, Nt - 1], seed=6, solver=solver, parts=1) as evo:
            leaves = [v.clone().requires_grad_(True) for v in (Ic, f, Is)]
            (evo(*leaves) * G).sum().backward()
            out.append([v.grad.cpu().numpy() for v in leaves])
    for a, b in zip(*out):
        assert np.abs(a - b).max() <= 1e-9 * np.abs(a).max()
