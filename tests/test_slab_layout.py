"""The row slabs of lattice columns that the automatic layout asks for are ones that fit:
where they do not (long narrow lattices), a column that one workgroup holds stays in
one, and a larger one keeps parts with column barriers, and says so."""
import ctypes as C

import pytest

import pyjjasim_amd as pa
from pyjjasim_amd import _native, engine
from pyjjasim_amd.solver_plan import CircuitPlan


def _plan(n, m):
    c = pa.SquareArray(n, m)
    return CircuitPlan(c, 0.05, block_size=engine.default_block_size(c._Nj(), c._Nf()))


# (array, columns, slabs asked for, whether they fit): mid-size and large ones, as many
# rows a part as there may be, and rows so short that a slab holds too many of them
@pytest.mark.parametrize("n,m,W,parts,fit", [(64, 64, 32, 8, True), (100, 100, 1, 16, True), (256, 256, 16, 16, True),
                                             (18, 257, 1, 16, True), (9, 400, 64, 4, True), (9, 701, 100, 2, False),
                                             (13, 601, 65, 2, False), (11, 1501, 40, 4, False), (1001, 9, 65, 2, False)])
def test_slabs_asked_for_fit_or_are_left(n, m, W, parts, fit):
    host = _plan(n, m)
    assert engine.slab_parts(host, W, 256) == parts
    sliced = engine.slab_layout(host, parts)
    assert (sliced is not None) == (fit or host.global_store)
    if sliced is not None:
        assert sliced.slabs == fit and sliced.parts == parts and sliced.block_size == engine.SLAB_BLOCK
    assert engine.slab_layout(host, 1) is None


def test_slabs_fit_checks_its_problem():
    lib, host = _native.lib(), _plan(64, 64)
    plan = host.relayout(512, 8, slabs=True)
    d = plan.desc()
    assert lib.jja_slabs_fit(C.byref(d)) == 1
    d.lattice_slabs = 0
    assert lib.jja_slabs_fit(C.byref(d)) == 0
    for block, parts in ((1024, 8), (512, 1)):                     # other workgroups, no parts
        other = host.relayout(block, parts, slabs=True)
        assert lib.jja_slabs_fit(C.byref(other.desc())) == 0
    d = plan.desc()
    d.max_columns = 0
    assert lib.jja_slabs_fit(C.byref(d)) == -1                     # JJA_EINVAL


def test_lattice_without_its_column_factor_is_accepted():
    """A lattice descriptor that leaves lattice_gc at 0 (its tables solve it) passes the
    checks and gets no slabs; a wrong one does not pass."""
    lib, host = _native.lib(), _plan(64, 64)
    plan = host.relayout(512, 8, slabs=True)
    d = plan.desc()
    d.lattice_gc = 0.0
    assert lib.jja_plan_validate(1, C.byref(d)) == 0 and lib.jja_slabs_fit(C.byref(d)) == 0
    for wrong in (-1.0, float("nan"), float("inf")):
        d.lattice_gc = wrong
        assert lib.jja_plan_validate(1, C.byref(d)) == -1
