"""Subdomains of a circuit's face system (domain_plan.py): the kernel's steps,
emulated on the host from the rows it streams, against a direct sparse solve; every
junction in one part; what does not fit or is not positive definite is left to the
factor."""
import numpy as np
import pytest
import scipy.sparse
import scipy.sparse.linalg

import pyjjasim_amd as pa
from pyjjasim_amd.domain_plan import DomainPlan
from pyjjasim_amd.solver_plan import CircuitPlan, cycle_codes, face_system_matrix


def _system(c):
    cx, cy = c.get_face_centroids()
    jc = cycle_codes(c.get_cycle_matrix(), c._Nf(), c._Nj())[2]
    return face_system_matrix(c, 0.05), np.stack([cx, cy], axis=1), jc


def _disordered():
    c = pa.SquareArray(21, 17)
    rng = np.random.default_rng(2)
    c.set_resistance(np.exp(0.3 * rng.standard_normal(c.junction_count())))
    c.set_capacitance(rng.random(c.junction_count()))
    return c


def _mutual():
    c = pa.SquareArray(14, 13)
    n = c.junction_count()
    c.set_inductance(scipy.sparse.diags([0.1, 1.0, 0.1], [-1, 0, 1], shape=(n, n)).tocsc())
    return c


CIRCUITS = {"honeycomb": (lambda: pa.HoneycombArray(11, 9), 4), "triangular": (lambda: pa.TriangularArray(9, 8), 8),
            "triangular_16": (lambda: pa.TriangularArray(20, 21), 16), "square_R": (_disordered, 2),
            "square_R_32": (_disordered, 32), "mutual": (_mutual, 4)}


@pytest.mark.parametrize("name", sorted(CIRCUITS))
def test_domain_solve_matches_direct(name):
    make, parts = CIRCUITS[name]
    K, xy, jc = _system(make())
    d = DomainPlan(K, xy, jc, parts)
    assert d.ok
    b = np.random.default_rng(1).standard_normal(K.shape[0])
    x = scipy.sparse.linalg.spsolve(K.tocsc(), b)
    assert np.abs(d.emulate(b) - x).max() <= 1e-11 * np.abs(x).max()
    # every junction is present and owned once
    e = d.pair[d.pair >= 0]
    held = np.concatenate([2 * (e[(e >> m) & 1 == 1] >> 4) + m for m in range(2)])
    assert np.array_equal(np.sort(held), np.arange(len(jc) // 2))
    assert np.array_equal((e & 3) << 2, e & 12)
    # every face's flux and gradient belong to one part
    assert np.array_equal(np.sort(d.face_id[d.face_id >= 0]), np.arange(K.shape[0]))


def test_domain_plan_validates():
    """The descriptor of a plan with subdomains passes the library's checks, and a
    changed index does not."""
    import ctypes as C
    from pyjjasim_amd import _native
    c = pa.HoneycombArray(11, 9)
    plan = CircuitPlan(c, 0.05, domains=4)
    assert plan.domains is not None and plan.parts == 4
    lib = _native.lib()
    assert lib.jja_plan_validate(1, C.byref(plan.desc(max_columns=2))) == 0
    for name, value in (("ent_off", 60000), ("pub_at", plan.domains.n_local), ("slice_rows", 1 << 20),
                        ("source", 1 << 20), ("face_code", 4 * plan.domains.pairs), ("pair", 1 << 26)):
        a = getattr(plan.domains, name)
        a = a.reshape(-1)
        at = int(np.flatnonzero(a != a[0])[0]) if name in ("ent_off", "slice_rows") else 0
        old = a[at]
        a[at] = value
        assert lib.jja_plan_validate(1, C.byref(plan.desc(max_columns=2))) != 0, name
        a[at] = old
    assert lib.jja_plan_validate(1, C.byref(plan.desc(max_columns=2))) == 0


def test_domain_plan_leaves_the_rest_to_the_factor():
    K, xy, jc = _system(pa.HoneycombArray(11, 9))
    assert not DomainPlan(-K, xy, jc, 4).ok                    # not positive definite
    K2 = K.copy()
    K2.data[:] = np.nan
    assert not DomainPlan(K2, xy, jc, 4).ok
    assert not DomainPlan(*_system(pa.HoneycombArray(3, 2)), 16).ok    # parts without faces of their own
    # lattices keep the lattice solve, other stencils the factor
    assert CircuitPlan(pa.SquareArray(12, 12), 0.05, domains=4).uses_lattice
    p = CircuitPlan(pa.HoneycombArray(11, 9), 0.05, 4, domains=4)
    assert p.domains is None and p.parts == 1


def test_domain_plans_stand_alone():
    """What the header asks of a descriptor with subdomains is checked: a plan of that
    problem alone, no lattice solve beside them, and faces and junctions to work on."""
    import ctypes as C
    from pyjjasim_amd import _native
    lib = _native.lib()
    make = lambda: CircuitPlan(pa.HoneycombArray(11, 9), 0.05, domains=4)
    plans = [make(), make()]
    both = (_native.ProblemDesc * 2)(*[p.desc(max_columns=2) for p in plans])
    assert lib.jja_plan_validate(1, both) == 0
    assert lib.jja_plan_validate(2, both) == -1                    # JJA_EINVAL
    assert b"domains" in lib.jja_last_error()
    beside = CircuitPlan(pa.SquareArray(12, 12), 0.05).relayout(512, 4)   # a split lattice
    d = beside.desc(max_columns=2)
    assert lib.jja_plan_validate(1, C.byref(d)) == 0
    d.domains = both[0].domains
    assert lib.jja_plan_validate(1, C.byref(d)) == -1
    for name in ("n_junctions", "n_faces"):
        d = make().desc(max_columns=2)
        d.domains = both[0].domains
        setattr(d, name, 0)
        d.n_face_slices = 0
        assert lib.jja_plan_validate(1, C.byref(d)) == -1, name


def test_domain_plan_pickles_and_keeps_its_descriptors():
    """A plan with subdomains pickles after its descriptor was made, as every plan does, and
    a descriptor stays valid when another is made of the same plan."""
    import ctypes as C
    import pickle
    from pyjjasim_amd import _native
    plan = CircuitPlan(pa.HoneycombArray(11, 9), 0.05, domains=4)
    first = plan.desc(max_columns=2)
    head = C.cast(first.domains, C.POINTER(_native.Domains)).contents
    records = head.records
    second = plan.desc(max_columns=3)
    assert first.domains == second.domains and head.records == records
    lib = _native.lib()
    assert lib.jja_plan_validate(1, C.byref(first)) == 0 and lib.jja_plan_validate(1, C.byref(second)) == 0
    copy = pickle.loads(pickle.dumps(plan))
    assert lib.jja_plan_validate(1, C.byref(copy.desc(max_columns=2))) == 0
    b = np.random.default_rng(0).standard_normal(plan.Nf)
    np.testing.assert_array_equal(copy.domains.emulate(b), plan.domains.emulate(b))


@pytest.mark.parametrize("seed", range(4))
def test_domain_programs_match_the_plan_builder(seed):
    """The library's programs for phases given as rows are those of the builder of the
    staged factor, record by record: rows of no entry, of one, of a lane's eight and one
    more, of all lanes' 512 and more; phases without rows and waves without work."""
    import ctypes as C
    from pyjjasim_amd import _native
    rng = np.random.default_rng(seed)
    lens = [rng.permutation([0, 1, 7, 8, 9, 63, 64, 65, 511, 512, 513, 1100, *rng.integers(0, 700, n)])[:n] for n in (0, 1, 5, 150)]
    rows = [rng.permutation(2000)[:len(l)].astype(np.int32) for l in lens]
    kinds = [0, _native.SLICE_BLOCK, _native.SLICE_BLOCK, 0]
    idx = [rng.integers(0, 65536, int(l.sum())).astype(np.int32) for l in lens]
    val = [rng.standard_normal(int(l.sum())) for l in lens]

    class Builder(CircuitPlan):
        def __init__(self):
            self.block_size, self.parts, self.global_store, self.index_bytes = 512, 1, False, 2
            self._build_wave_program([(0, r, np.concatenate(([0], np.cumsum(l))), i, v, k, None, "col", "col")
                                      for r, l, i, v, k in zip(rows, lens, idx, val, kinds)], 8)
    want = Builder()
    ends = lambda counts, t: np.concatenate(([0], np.cumsum(counts))).astype(t)
    given = [ends([4], np.int32), ends([len(l) for l in lens], np.int64), np.array(kinds, np.int32), np.concatenate(rows),
             ends(np.concatenate(lens), np.int64), np.concatenate(idx), np.concatenate(val)]
    sizes = np.zeros(3, np.int64)
    point = lambda *arrays: [a.ctypes.data for a in arrays]
    lib = _native.lib()
    assert lib.jja_domain_programs(1, 8, *point(*given, sizes), *[None] * 5) == 0
    made = [np.empty((sizes[0], 8), np.int32), np.empty(9, np.int32), np.empty(sizes[1]), np.empty(sizes[1], np.uint16),
            np.empty(sizes[2], np.int32)]
    assert lib.jja_domain_programs(1, 8, *point(*given, sizes, *made)) == 0
    np.testing.assert_array_equal(made[0].view(np.int64)[:, :2], [s[:2] for s in want.solve_slices])
    np.testing.assert_array_equal(made[0][:, 4:], [s[2:] for s in want.solve_slices])
    for got, name in zip(made[1:], ("wave_ptr", "ent_val", "ent_off", "slice_rows")):
        np.testing.assert_array_equal(got, getattr(want, name), err_msg=name)
    assert lib.jja_domain_programs(1, 0, *point(*given, sizes), *[None] * 5) == -1
