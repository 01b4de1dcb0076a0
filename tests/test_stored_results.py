"""Stored results: selected steps and derivatives of ranges, gaps and nothing, and
results turned on the device in several blocks."""
import numpy as np
import pytest

from pyjjasim_amd import engine
from pyjjasim_amd.time_evolution import _apply_derivative, _steps


@pytest.mark.parametrize("index", [[], [4], [4, 5, 6], [3, 5, 8], [3, 4, 8], list(range(3, 12))])
@pytest.mark.parametrize("stencil", [(1.0, -1.0), (1.5, -2.0, 0.5), (11 / 6, -3.0, 1.5, -1 / 3)])
def test_steps_and_derivatives(index, stencil):
    index = np.array(index, dtype=int)
    x = np.random.default_rng(0).standard_normal((5, 3, 12))
    assert np.array_equal(_steps(x, index), x[:, :, index])
    # the formula starts with two terms and takes the third and fourth of longer stencils
    want = stencil[0] * x[:, :, index] + stencil[1] * x[:, :, index - 1]
    if len(stencil) >= 4:
        want = want + stencil[2] * x[:, :, index - 2]
    got = _apply_derivative(x, index, stencil, 0.25)
    assert got.shape == (5, 3, len(index)) and np.array_equal(got, want / 0.25)


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,W", [(4, 3, 1), (7, 5, 3), (30, 2, 2)])
def test_results_in_blocks(nx, ny, W, monkeypatch):
    import pyjjasim_amd as pj
    problem = pj.TimeEvolutionProblem(
        pj.SquareArray(nx, ny), time_step=0.05, time_step_count=40, external_flux=0.1,
        current_sources=pj.SquareArray(nx, ny).current_base(0)[:, None, None] * np.linspace(0.4, 1.2, W)[None, :, None],
        temperature=0.0, store_time_steps=np.arange(40) % 7 < 4)
    whole = problem.compute()
    monkeypatch.setattr(engine, "TURN_BYTES", 3 * 8 * W * 30)     # a few elements at a time
    parts = problem.compute()
    for get in ("get_theta", "get_voltage", "get_current", "get_vortex_configuration"):
        a, b = getattr(whole, get)(), getattr(parts, get)()
        assert a.dtype == b.dtype and a.flags.c_contiguous and np.array_equal(a, b)
        assert np.array_equal(getattr(whole, get)([8]), a[:, :, [list(np.flatnonzero(np.arange(40) % 7 < 4)).index(8)]])
