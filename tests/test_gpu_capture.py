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
