"""A forward pass captured into a HIP graph and replayed, with eager passes between the
replays: columns in one workgroup, in row slabs and in subdomains (whose parts count
their exchanges on the device, so that a replay counts on)."""
import numpy as np
import pytest

import pyjjasim_amd as pa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make,parts", [(lambda: pa.SquareArray(12, 12), 1), (lambda: pa.SquareArray(70, 72), 16),
                                        (lambda: pa.HoneycombArray(16, 16), 8)])
def test_forward_replays(make, parts):
    torch = pytest.importorskip("torch")
    c = make()
    W = 2
    rng = np.random.default_rng(0)
    put = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")
    Ic = put(np.exp(0.1 * rng.standard_normal(c.junction_count())))
    f, Is = put(np.full((c.face_count(), W), 0.1)), put(np.outer(c.current_base(0.0), [0.5, 1.1]))
    with pa.DifferentiableEvolution(c, time_step=0.05, time_step_count=15, problem_count=W, temperature=0.01,
                                    store_time_steps=[0, 14], seed=6) as evo:
        print(f"[capture] {c.junction_count()} junctions, {evo.eng.host.parts} parts", flush=True)
        assert (evo.eng.host.parts > 1) == (parts > 1)
        side = torch.cuda.Stream()
        with torch.cuda.stream(side), torch.no_grad():
            for _ in range(2):
                want = evo(Ic, f, Is).clone()
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.no_grad(), torch.cuda.graph(graph, stream=side):
            out = evo(Ic, f, Is)
        for _ in range(4):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
            with torch.cuda.stream(side), torch.no_grad():
                again = evo(Ic, f, Is)
            side.synchronize()
            assert torch.equal(again, want)


def test_column_barriers_refuse_capture():
    """A pass whose parts meet at column barriers is refused while its stream is captured,
    before anything is recorded, and runs as before afterwards."""
    torch = pytest.importorskip("torch")
    from pyjjasim_amd import _native
    c, W = pa.SquareArray(30, 30), 2
    put = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")
    Ic, f = put(np.ones(c.junction_count())), put(np.full((c.face_count(), W), 0.1))
    Is = put(np.outer(c.current_base(0.0), [0.5, 1.1]))
    with pa.DifferentiableEvolution(c, time_step=0.05, time_step_count=12, problem_count=W, store_time_steps=[11], parts=4,
                                    face_store="global", block_size=256) as evo, torch.no_grad():
        print("[capture] column barriers", flush=True)
        want = evo(Ic, f, Is)
        torch.cuda.synchronize()
        with pytest.raises(_native.NativeError, match="captured"):
            with torch.cuda.graph(torch.cuda.CUDAGraph()):
                evo(Ic, f, Is)
        torch.cuda.synchronize()
        assert torch.equal(evo(Ic, f, Is), want)


def _inputs(torch, c, W, seed):
    """Ic, f and Is, the last two without a column axis: the kernels read them in place."""
    rng = np.random.default_rng(seed)
    put = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")
    return (put(np.exp(0.1 * rng.standard_normal(c.junction_count()))), put(0.1 + 0.05 * rng.random(c.face_count())),
            put((0.5 + 0.1 * seed) * c.current_base(0.0)))


PLANS = [(lambda: pa.SquareArray(12, 12), {}), (lambda: pa.SquareArray(70, 72), {"parts": 1}),
         (lambda: pa.SquareArray(70, 72), {}), (lambda: pa.HoneycombArray(16, 16), {})]


@pytest.mark.parametrize("make,opts", PLANS, ids=["resident", "wide", "slabs", "domains"])
@pytest.mark.parametrize("grad", [False, True])
def test_replays_keep_their_inputs(make, opts, grad):
    """Captured on a stream of its own without a pass before it; between the replays eager
    passes, forward and backward, with other tensors on other streams. Every replay gives
    what the captured inputs give (two segments, so the backward pass recomputes phases
    and runs the adjoint twice), and every eager pass what its own give."""
    torch = pytest.importorskip("torch")
    c, W, Nt = make(), 2, 15
    A, B = _inputs(torch, c, W, 1), _inputs(torch, c, W, 2)
    G = torch.tensor(np.random.default_rng(3).standard_normal((c.junction_count(), W, 2)), device="cuda")
    kw = dict(time_step=0.05, time_step_count=Nt, problem_count=W, temperature=0.01, store_time_steps=[3, Nt - 1],
              checkpoint_every=8, seed=6, **opts)

    def run(evo, leaves):
        with torch.set_grad_enabled(grad):
            th = evo(*leaves)
            return (th.detach(),) + (torch.autograd.grad(th, leaves, G) if grad else ())
    leaves = [[x.clone().requires_grad_(grad) for x in X] for X in (A, B)]
    print(f"[capture] {c.junction_count()} junctions, grad={grad}", flush=True)
    with pa.DifferentiableEvolution(c, **kw) as evo:
        want = [[x.clone() for x in run(evo, X)] for X in leaves]
    with pa.DifferentiableEvolution(c, **kw) as evo:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = run(evo, leaves[0])
        for k in range(4):
            graph.replay()
            torch.cuda.synchronize()
            for a, b in zip(out, want[0]):
                assert torch.equal(a, b)
            side = torch.cuda.Stream()
            with torch.cuda.stream(side):
                for X, ref in (zip(leaves, want) if k % 2 else [(leaves[1], want[1])]):
                    for a, b in zip(run(evo, X), ref):
                        assert torch.equal(a, b)
            side.synchronize()


@pytest.mark.parametrize("make", [lambda: pa.SquareArray(70, 72), lambda: pa.HoneycombArray(16, 16)], ids=["slabs", "domains"])
def test_a_replay_that_gave_up_shows(make):
    """Parts that stop waiting for each other (a wait limit of no polls, every kernel still
    running to its end) leave no phases that look valid: the replay's results hold NaN, the
    next call outside the graph raises, and the one after that is exact again."""
    torch = pytest.importorskip("torch")
    from pyjjasim_amd import _native
    c, W = make(), 2
    X = _inputs(torch, c, W, 1)
    with pa.DifferentiableEvolution(c, time_step=0.05, time_step_count=15, problem_count=W, store_time_steps=[14]) as evo, \
            torch.no_grad():
        print(f"[capture] {c.junction_count()} junctions give up", flush=True)
        want = evo(*X)
        torch.cuda.synchronize()
        _native.check(evo.eng.lib.jja_plan_set_wait_limit(evo.eng.handle, 0))
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = evo(*X)
        _native.check(evo.eng.lib.jja_plan_set_wait_limit(evo.eng.handle, 1 << 21))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.isnan(out).any()
        with pytest.raises(_native.NativeError, match="gave up"):
            evo(*X)
        assert torch.equal(evo(*X), want)
