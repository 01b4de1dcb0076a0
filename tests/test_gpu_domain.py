"""Columns of general circuits as subdomains (one workgroup each, one meeting a
step): the automatic layout of mid-size and large circuits with few columns,
against the staged factor at 1e-9 of the phase scale with identical vortex counts,
forward and backward, and the oracle."""
import numpy as np
import pytest

import pyjjasim_amd as pa
from oracle import te_oracle as to
from pyjjasim_amd import engine

pytestmark = pytest.mark.gpu


def _circuit(kind, n, m, hetero=False):
    c = {"hc": pa.HoneycombArray, "tri": pa.TriangularArray, "sq": pa.SquareArray}[kind](n, m)
    rng = np.random.default_rng(n + m)
    c.set_critical_current(np.exp(0.1 * rng.standard_normal(c.junction_count())))
    c.set_capacitance(0.5 + rng.random(c.junction_count()) if hetero else 0.8)
    if hetero:
        c.set_inductance(0.3)
    return c


# (lattice, sizes, parts, per-junction coefficients): interiors of one cell and of
# many, one to four pairs a thread, 2 to 32 parts
CASES = [("hc", 11, 9, 4, False), ("tri", 9, 8, 8, False), ("tri", 20, 20, 32, False), ("hc", 30, 30, 4, False),
         ("sq", 21, 17, 2, True), ("tri", 40, 40, 4, True), ("tri", 50, 60, 8, False)]


def _forced(monkeypatch, parts):
    monkeypatch.setattr(engine, "domain_parts", lambda *a, **k: parts)


@pytest.mark.parametrize("kind,n,m,parts,hetero", CASES)
def test_gpu_domains_match_factor(monkeypatch, kind, n, m, parts, hetero):
    c = _circuit(kind, n, m, hetero)
    W, Nt = 2, 36
    t = 0.05 * np.arange(Nt)
    drive = pa.SeparableSource(c.current_base(0.0)[:, None] * np.array([0.5, 1.3]), 1.0 + 0.3 * np.sin(t))
    f = 0.1 + 0.02 * np.arange(c.face_count())[:, None, None] / c.face_count() + 0.01 * np.sin(t)[None, None, :]
    for T in (0.0, 0.02):
        kw = dict(time_step=0.05, time_step_count=Nt, external_flux=f, current_sources=drive, temperature=T, seed=3,
                  store_time_steps=[0, 17, Nt - 1], steps_per_launch=13)
        print(f"[domain] {kind} {n}x{m}, {parts} parts, T={T}", flush=True)
        a = pa.TimeEvolutionProblem(c, solver="cholesky", parts=1, **kw).compute()
        _forced(monkeypatch, parts)
        b = pa.TimeEvolutionProblem(c, **kw).compute()
        for get in ("get_theta", "get_current", "get_voltage"):
            u, v = getattr(a, get)(), getattr(b, get)()
            assert np.abs(u - v).max() <= 1e-9 * np.abs(u).max(), get
        np.testing.assert_array_equal(a.get_vortex_configuration(), b.get_vortex_configuration())


@pytest.mark.parametrize("kind,n,m,parts,hetero", CASES)
def test_gpu_domain_gradients_match_factor(monkeypatch, kind, n, m, parts, hetero):
    torch = pytest.importorskip("torch")
    c = _circuit(kind, n, m, hetero)
    Nj, Nf, W, Nt = c.junction_count(), c.face_count(), 2, 24
    rng = np.random.default_rng(1)
    put = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")
    Ic, f = put(np.exp(0.1 * rng.standard_normal(Nj))), put(0.1 + 0.02 * rng.standard_normal((Nf, W)))
    Is, G = put(np.outer(c.current_base(0.0), [0.5, 1.1])), put(rng.standard_normal((Nj, W, 3)))
    print(f"[domain] gradient {kind} {n}x{m}, {parts} parts", flush=True)
    out = []
    for domains in (False, True):
        if domains:
            _forced(monkeypatch, parts)
        kw = {} if domains else {"solver": "cholesky", "parts": 1}
        with pa.DifferentiableEvolution(c, time_step=0.05, time_step_count=Nt, problem_count=W, temperature=0.01,
                                        store_time_steps=[0, 11, Nt - 1], checkpoint_every=7, seed=6, **kw) as evo:
            assert (evo.eng.host.domains is not None) == domains
            leaves = [v.clone().requires_grad_(True) for v in (Ic, f, Is)]
            (evo(*leaves) * G).sum().backward()
            out.append([v.grad.cpu().numpy() for v in leaves])
    for a, b in zip(*out):
        assert np.abs(a - b).max() <= 1e-9 * np.abs(a).max()


def test_gpu_domains_match_oracle(monkeypatch):
    c = _circuit("hc", 14, 13)
    _forced(monkeypatch, 8)
    Nt, ts = 200, [99, 199]
    Is = c.current_base(0.0)[:, None, None] * np.array([0.6, 1.3])[None, :, None]
    p = pa.TimeEvolutionProblem(c, time_step=0.05, time_step_count=Nt, external_flux=0.21, current_sources=Is,
                                store_time_steps=ts)
    res = p.compute()
    ref = to.evolve(c, dt=0.05, Nt=Nt, f=0.21, Is=Is, store_time_steps=ts)
    assert np.abs(res.get_theta() - ref["theta"]).max() <= 1e-9 * np.abs(ref["theta"]).max()
    np.testing.assert_array_equal(res.get_vortex_configuration(), to.vortex(c.get_cycle_matrix(), ref["theta"]))
