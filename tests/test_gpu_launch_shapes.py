"""Sizes at which the assembly and field kernels change their split of the work: the describe
kernel's two ways to share out row groups (a wavefront or sixteen lanes each, with the groups of many
sources shared by a block), the one- and two-pass CSR layout, the fill's chunks, the field grid's
tiles of 16 points, and an assembly's recording as a graph on its second call in a row. GEPs within
_compare.RTOL of the oracle, fields within 1e-13 of the largest (as in the fields' other tests);
forced chunks and graph replays give the same bits."""

import ctypes as C
import re

import numpy as np
import pytest
import scipy.linalg

import cases
import fem_2d_amd as F
import oracle
from _compare import assert_gep_matches
from fem_2d_amd import _native as N
from fem_2d_amd import workloads as W
from test_gpu_parity import _view_from_arrays
from test_zz_no_alloc import DeviceArrays, check_same, noalloc

pytestmark = pytest.mark.gpu

FIELD_TOL = 1e-13


@pytest.fixture(scope="module")
def ctx():
    return F.Context(0)


def _same_bits(g, ref):
    np.testing.assert_array_equal(g.row_ptr, ref.row_ptr)
    np.testing.assert_array_equal(g.col, ref.col)
    np.testing.assert_array_equal(g.a_val.view(np.uint8), ref.a_val.view(np.uint8))
    np.testing.assert_array_equal(g.b_val.view(np.uint8), ref.b_val.view(np.uint8))


# 1, 2 190 (past the 2 048 where the layout takes its second pass), 4 163, 17 080 and 29 527 groups (the
# last two past two groups a wavefront); 16, 14, 49 and 513 of them have more than 16 sources
@pytest.mark.parametrize("nx,ny,levels", [(1, 1, 0), (22, 12, 2), (32, 16, 2), (64, 32, 2), (64, 32, 3)])
def test_row_groups(ctx, nx, ny, levels):
    print(f"[shapes] waveguide {nx}x{ny} levels={levels}", flush=True)
    dom = F.Domain.from_mesh(W.waveguide_64x32_mesh(nx, ny, order=2, levels=levels))
    gep = F.galerkin_sample_gep_hcurl(dom, (8, 8), F.HierPoly, ctx=ctx)
    rc, ref = oracle.assemble(dom.view(), basis=F.HierPoly.code, glq=(8, 8), n_threads=8)
    assert rc == 0
    assert_gep_matches(gep, ref)


@pytest.mark.parametrize("name", ["waveguide_small", "small_hp_irregular", "deep_corner"])
def test_forced_chunks(ctx, name):
    dom, glq = cases.ALL[name]()
    ref = F.galerkin_sample_gep_hcurl(dom, glq, F.KOLShapeFn, ctx=ctx)
    c = F.Context(0)
    for chunk in (64, 128, 1024, 4096):
        print(f"[shapes] {name} chunk={chunk}", flush=True)
        c.set_fill_chunk(chunk)
        _same_bits(F.galerkin_sample_gep_hcurl(dom, glq, F.KOLShapeFn, ctx=c), ref)
    c.close()


@pytest.mark.parametrize("basis", [0, 1])
@pytest.mark.parametrize("d", [2, 15, 16, 17, 33])
def test_field_tiles(ctx, basis, d):
    """A NaN DoF value reaches the points that it reaches in the oracle's sums."""
    print(f"[shapes] fields basis={basis} d={d}", flush=True)
    dom, _ = cases.small_hp_irregular()
    B = F.KOLShapeFn if basis else F.HierPoly
    sol = np.random.default_rng(d).standard_normal(dom.num_dofs)
    for poison in (False, True):
        if poison:
            sol[dom.num_dofs // 2] = np.nan
        rc, ex, ey = oracle.xy_fields(dom.view(), basis, (d, d), sol)
        assert rc == 0
        for got, exp in zip(F.xy_fields_array(dom, sol, (d, d), B, ctx=ctx), (ex, ey)):
            np.testing.assert_array_equal(np.isnan(got), np.isnan(exp))
            assert np.nanmax(np.abs(got - exp)) <= FIELD_TOL * np.nanmax(np.abs(exp))


def test_recording_order():
    """Launched, recorded and replayed assemblies of two Domains of one context in every order of
    succession, the second one's larger buffers allocated after the first one's recording."""
    print("[shapes] recording order", flush=True)
    c, eager = F.Context(0), F.Context(0)
    eager.set_graphs(False)
    made = [cases.waveguide_small(), cases.small_hp_irregular()]
    refs = [F.galerkin_sample_gep_hcurl(d, q, F.HierPoly, ctx=eager) for d, q in made]
    doms = [F.DeviceDomain(d, c) for d, _ in made]
    for i in (0, 0, 0, 1, 0, 1, 1, 1, 0, 1, 0, 0, 0, 1):
        _same_bits(doms[i].download(doms[i].assemble(made[i][1], F.HierPoly)), refs[i])
    c.close()
    eager.close()


@pytest.mark.parametrize("solve", ["solve_gep_sparse", "solve_gep_dense"])
@pytest.mark.parametrize("nx,ny,order", [(2, 1, 2), (2, 2, 3), (4, 4, 4)])
def test_solve_of_few_dofs(ctx, nx, ny, order, solve):
    """10 and 60 DoFs (one partly filled block, and GMRES steps that exhaust the space) and a few
    hundred: the eigenpair nearest the target, 1e-10 from LAPACK's value, residual below 1e-9 (the
    iteration's own bound is 1e-10)."""
    print(f"[shapes] {solve} {nx}x{ny} order={order}", flush=True)
    dom = F.Domain.from_mesh(W.waveguide_64x32_mesh(nx, ny, order=order, levels=0))
    gep = F.galerkin_sample_gep_hcurl(dom, (8, 8), F.HierPoly, ctx=ctx)
    A, B = (m.toarray() for m in gep.to_scipy())
    lams = scipy.linalg.eigh(A, B, eigvals_only=True)
    lam = lams[lams > 1e-6 * lams[-1]][0]
    pair = getattr(F, solve)(gep, 1.01 * lam, ctx=ctx)
    x = pair.vector
    assert abs(pair.value - lam) <= 1e-10 * lam
    assert np.linalg.norm(A @ x - pair.value * (B @ x)) <= 1e-9 * np.linalg.norm(A @ x)


@pytest.mark.parametrize("basis", [0, 1])
@pytest.mark.parametrize("order", [20, 21, 31, 32, 40, 120])
def test_fields_of_any_order(ctx, basis, order):
    """A view filled by hand may hold any order that a byte does; a Mesh's go up to 20."""
    print(f"[shapes] fields basis={basis} order={order}", flush=True)
    dom, _ = cases.mixed_refinements()
    a = {k: v.copy() if isinstance(v, np.ndarray) else v for k, v in dom.arrays().items()}
    a["bs_i"][::3] = order
    a["bs_j"][1::4] = order
    a["orders"][0] = order
    view, keep = _view_from_arrays(a)
    sol = np.random.default_rng(order).standard_normal(dom.num_dofs)
    d = 17
    rc, ex, ey = oracle.xy_fields(view, basis, (d, d), sol)
    assert rc == 0
    gx, gy = np.empty_like(ex), np.empty_like(ey)
    p = [x.ctypes.data_as(C.POINTER(C.c_double)) for x in (sol, gx, gy)]
    rc = N.load().fem2d_xy_fields(ctx._h, C.byref(view), basis, d, d, p[0], sol.size, p[1], p[2])
    assert rc == N.OK, N.last_error()
    for got, exp in ((gx, ex), (gy, ey)):
        err = np.abs(got - exp).max() / np.abs(exp).max()
        assert err <= FIELD_TOL


def _nested_pair_dof(a):
    """Order-1 arrays with one DoF's specs on an Elem and one of its descendants, by exchanging one
    spec each of two DoFs: columns of its row group receive more than two contributions."""
    a = {k: v.copy() if isinstance(v, np.ndarray) else v for k, v in a.items()}
    elem = np.repeat(np.arange(a["n_elems"]), np.diff(a["bs_offsets"]))
    specs = a["dof_bs"].reshape(-1, 2)

    def below(e, top):
        while e >= 0 and e != top:
            e = a["parent"][e]
        return e == top

    for p, (t0, t1) in enumerate(specs):
        for q, (t2, t3) in enumerate(specs):
            if p != q and below(elem[t3], elem[t0]) and elem[t3] != elem[t0] and elem[t2] != elem[t1]:
                specs[p, 1], specs[q, 1] = t3, t1
                a["bs_dof"][t3], a["bs_dof"][t1] = p, q
                return a
    raise AssertionError("no such pair of DoFs")


# 32 row groups (one a wavefront) and 18 389 (four a wavefront)
@pytest.mark.parametrize("nx,ny,levels", [(4, 2, 2), (64, 32, 3)])
def test_error_while_describing(ctx, nx, ny, levels):
    """An error that the describe kernel itself reports, so that its later blocks start after it."""
    print(f"[shapes] error while describing {nx}x{ny} levels={levels}", flush=True)
    dom = F.Domain.from_mesh(W.waveguide_64x32_mesh(nx, ny, order=1, levels=levels))
    view, keep = _view_from_arrays(_nested_pair_dof(dom.arrays()))
    out = N.GepCsr()
    rc = N.load().fem2d_galerkin_sample_gep_hcurl(ctx._h, C.byref(view), 0, 0, 1, 8, 8, 0, C.byref(out))
    assert rc == N.ERR_INVALID_VIEW and "two contributions" in N.last_error(), (rc, N.last_error())
    gep = F.galerkin_sample_gep_hcurl(dom, (8, 8), F.HierPoly, ctx=ctx)
    rc, ref = oracle.assemble(dom.view(), basis=F.HierPoly.code, glq=(8, 8), n_threads=8)
    assert rc == 0
    assert_gep_matches(gep, ref)


@pytest.mark.parametrize("precision", [F.FP64, F.FP32])
def test_many_rounds_of_chunks(ctx, precision):
    """25.7 M entries in chunks of 64: about 98 rounds a block, past the 64 tickets that the fill's ring
    keeps, against the few rounds that the automatic size makes."""
    print(f"[shapes] many rounds precision={precision}", flush=True)
    w = W.waveguide_64x32()
    dd = F.DeviceDomain(w.domain, ctx)
    ref = dd.download(dd.assemble(w.glq, F.HierPoly, precision=precision))
    ctx.set_fill_chunk(64)
    try:
        got = dd.download(dd.assemble(w.glq, F.HierPoly, precision=precision))
    finally:
        ctx.set_fill_chunk(0)
    assert ref.nnz == 25_704_606
    _same_bits(got, ref)


def test_error_while_counting(ctx):
    """An error that the block path's counting kernel reports: an edge between an Elem with 84
    descendants and its neighbour, with one DoF's second spec moved into a descendant."""
    print("[shapes] error while counting", flush=True)
    mesh = F.Mesh.rect_grid(2, 1, 0.0, 1.0, 0.0, 0.5)
    mesh.set_global_expansion_orders(F.Orders(1, 1))
    leaves = [0]
    for _ in range(3):
        mesh.execute_h_refinements([(e, F.HRef.t()) for e in leaves])
        leaves = [c for e in leaves for c in mesh.elem(e).child_ids()]
    dom = F.Domain.from_mesh(mesh)
    gep = F.galerkin_sample_gep_hcurl(dom, (8, 8), F.HierPoly, ctx=ctx)
    assert ctx.last_timing()["n_large"] > 0
    rc, ref = oracle.assemble(dom.view(), basis=F.HierPoly.code, glq=(8, 8), n_threads=8)
    assert rc == 0
    assert_gep_matches(gep, ref)
    view, keep = _view_from_arrays(_nested_pair_dof(dom.arrays()))
    out = N.GepCsr()
    rc = N.load().fem2d_galerkin_sample_gep_hcurl(ctx._h, C.byref(view), 0, 0, 1, 8, 8, 0, C.byref(out))
    assert rc == N.ERR_INVALID_VIEW and "two contributions" in N.last_error(), (rc, N.last_error())


@pytest.mark.parametrize("precision", [F.FP64, F.FP32, F.FP32R])
@pytest.mark.parametrize("make", [cases.small_hp_irregular, W.waveguide_64x32])
def test_replays_in_every_precision(precision, make):
    """An assembly launched, recorded and replayed twice, with and without block-path row groups, each
    with the bits of a context that launches kernel by kernel and that works in between."""
    print(f"[shapes] replays precision={precision} {make.__name__}", flush=True)
    w = make()
    dom, glq = w if isinstance(w, tuple) else (w.domain, w.glq)
    c, eager = F.Context(0), F.Context(0)
    eager.set_graphs(False)
    dd, ed = F.DeviceDomain(dom, c), F.DeviceDomain(dom, eager)
    ref = ed.download(ed.assemble(glq, F.KOLShapeFn, precision=precision))
    for _ in range(4):
        _same_bits(dd.download(dd.assemble(glq, F.KOLShapeFn, precision=precision)), ref)
        ed.assemble(glq, F.HierPoly, precision=precision)
        eager.synchronize()
    c.close()
    eager.close()


def test_first_row_table_short_of_scratch():
    """A Domain that leaves the no-allocation entry point less of its scratch array than the table of
    the chunks' first rows would take: larger chunks, and the same bits. Orders of 5 instead of 4 on
    more and more Elems use the array up; an absurd capacity has the call say what it needs."""
    print("[shapes] first-row table short of scratch", flush=True)
    ctx = F.Context(0)
    nothing = DeviceArrays(ctx, 100_000, 0, 8)
    absurd = 4096 << 25  # a table of 2^25 + 1 words at least

    def domain(k):
        mesh = W.waveguide_64x32_mesh(76, 43, order=4, levels=0)
        mesh.set_expansion_on_elems(range(k), F.Orders(5, 5))
        return F.Domain.from_mesh(mesh)

    def words_left(dom):
        rc, _ = noalloc(ctx, F.DeviceDomain(dom, ctx), (8, 8), F.HierPoly, F.FP64, nothing, absurd)
        assert rc == N.ERR_UNSUPPORTED, (rc, N.last_error())
        need, size = map(int, re.search(r"needs (\d+) bytes.* has (\d+) ", N.last_error()).groups())
        return (size - (need - 4 * (absurd // 4096 + 1))) // 4

    k, end = 0, 76 * 43  # more than 2 000 words are left at k, fewer at the end
    assert words_left(domain(k)) > 2000 >= words_left(domain(end))
    while end - k > 1:
        mid = (k + end) // 2
        if words_left(domain(mid)) > 2000:
            k = mid
        else:
            end = mid
    dom = domain(k)
    dd = F.DeviceDomain(dom, ctx)
    nnz = dd.assemble((8, 8), F.HierPoly).nnz
    chunk = ctx.last_timing()["fill_chunk"]
    assert nnz // 4096 + 1 < words_left(dom) < nnz // chunk
    for precision in (F.FP64, F.FP32):
        check_same(ctx, dom, (8, 8), F.HierPoly, precision).free()
    nothing.free()
    ctx.close()


# the rule's branches: one chunk a wavefront, 12 rows, 256 entries, five chunks a wavefront
@pytest.mark.parametrize("nx,order,chunk", [(32, 4, 384), (96, 2, 128), (48, 4, 256), (64, 4, 320)])
def test_chunk_rule(ctx, nx, order, chunk):
    """The automatic chunk size (of the 4 096 wavefronts of 256 CUs) and a forced one give the same bits."""
    print(f"[shapes] chunk rule {nx}x{nx // 2} order={order}", flush=True)
    dd = F.DeviceDomain(F.Domain.from_mesh(W.waveguide_64x32_mesh(nx, nx // 2, order=order, levels=2)), ctx)
    got = dd.download(dd.assemble((8, 8), F.HierPoly))
    assert ctx.last_timing()["fill_chunk"] == chunk
    ctx.set_fill_chunk(512)
    try:
        ref = dd.download(dd.assemble((8, 8), F.HierPoly))
    finally:
        ctx.set_fill_chunk(0)
    _same_bits(got, ref)
