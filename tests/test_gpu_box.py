"""GPU parity of the box family (per-orbital cubic boxes) against the
oracle's box family, which itself equals the masked grid formulation."""
import ctypes

import numpy as np
import pytest

import oracle as O
from mgmol_amd import mgx, synth
from tests.gpu_util import relmax, say, to_dev, to_np

pytestmark = pytest.mark.gpu

DT = {"f64": np.float64, "f32": np.float32}
CODE = {"f64": mgx.F64, "f32": mgx.F32}
TOL = {"f64": 1e-12, "f32": 2e-6}


@pytest.fixture(scope="module")
def ctx():
    from tests.gpu_util import ctx as shared
    return shared()


@pytest.fixture(scope="module")
def cfg():
    # ragged edges, boxes wrapping the periodic seam, 3 levels
    return synth.box_config(nbox=24, gdim=48, h=0.3, edges=(8, 12, 16, 20), nwells=6, seed=5, levels=3)


@pytest.fixture(scope="module")
def boxes(ctx, cfg):
    ob = O.Boxes.make(cfg.origin, cfg.edge, cfg.gdim, cfg.h)
    bs = mgx.BoxSet(ctx, cfg.origin, cfg.edge, cfg.gdim, cfg.h, 3)
    yield ob, bs
    bs.close()


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("level", [0, 1])
def test_box_lap(ctx, boxes, dt, kind, level):
    ob, bs = boxes
    rng = np.random.default_rng(kind + 3 * level)
    u = rng.standard_normal(ob.size(level)).astype(DT[dt])
    tu, to = to_dev(u), to_dev(np.zeros_like(u))
    ctx.call("mgx_box_lap", bs.h, level, kind, CODE[dt], mgx.ptr(tu), mgx.ptr(to))
    ref = O.b_lap(ob, level, kind, u)
    assert relmax(to_np(to), ref) <= TOL[dt]


@pytest.mark.parametrize("dt", ["f64", "f32"])
def test_box_hloc(ctx, boxes, cfg, dt):
    ob, bs = boxes
    u = cfg.psi.astype(DT[dt])
    tu, tv, to = to_dev(u), to_dev(cfg.vtot), to_dev(np.zeros_like(u))
    ctx.call("mgx_box_hloc", bs.h, CODE[dt], mgx.ptr(tu), mgx.ptr(tv), mgx.ptr(to))
    ref = O.b_hloc(ob, cfg.vtot, u)
    err = relmax(to_np(to), ref)
    say("box hloc", dt, err)
    assert err <= TOL[dt]


@pytest.mark.parametrize("dt", ["f64", "f32"])
def test_box_jacobi_transfer(ctx, boxes, dt):
    ob, bs = boxes
    rng = np.random.default_rng(21)
    f = rng.standard_normal(ob.size(0)).astype(DT[dt])
    x = rng.standard_normal(ob.size(0)).astype(DT[dt])
    w = np.zeros_like(x)
    jf = O.jacobi_factor(2, list(ob.h))
    tf, tx, tw = to_dev(f), to_dev(x), to_dev(w)
    ctx.call("mgx_box_jacobi", bs.h, 0, 2, CODE[dt], jf, mgx.ptr(tf), mgx.ptr(tx), mgx.ptr(tw))
    xr, wr = x.copy(), w.copy()
    O.b_jacobi(ob, 0, 2, f, xr, wr, jf)
    assert relmax(to_np(tx), xr) <= TOL[dt]
    assert relmax(to_np(tw), wr) <= TOL[dt]
    tc = to_dev(np.zeros(ob.size(1), DT[dt]))
    ctx.call("mgx_box_restrict", bs.h, 0, CODE[dt], mgx.ptr(tf), mgx.ptr(tc))
    assert np.array_equal(to_np(tc), O.b_restrict(ob, 0, f))
    # level 1 -> 2 has odd coarse edges (2, 3, 4, 5): one point per thread
    # there, pairs of points per thread above (all coarse edges even)
    edges = [int(ob.edge[i]) for i in range(ob.nbox)]
    assert any((e >> 2) % 2 for e in edges) and not any((e >> 1) % 2 for e in edges)
    f1 = rng.standard_normal(ob.size(1)).astype(DT[dt])
    tf1, tc1 = to_dev(f1), to_dev(np.zeros(ob.size(2), DT[dt]))
    ctx.call("mgx_box_restrict", bs.h, 1, CODE[dt], mgx.ptr(tf1), mgx.ptr(tc1))
    assert np.array_equal(to_np(tc1), O.b_restrict(ob, 1, f1))
    c = rng.standard_normal(ob.size(1)).astype(DT[dt])
    tc2, tfi = to_dev(c), to_dev(np.zeros(ob.size(0), DT[dt]))
    ctx.call("mgx_box_prolong", bs.h, 0, CODE[dt], mgx.ptr(tc2), mgx.ptr(tfi))
    assert np.array_equal(to_np(tfi), O.b_prolong(ob, 0, c))


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_box_precond(ctx, boxes, prec):
    ob, bs = boxes
    rng = np.random.default_rng(22)
    r = rng.standard_normal(ob.size(0))
    gam = O.gamma(list(ob.h), 2, 0.0, -1.2)
    tr, to = to_dev(r), to_dev(np.zeros_like(r))
    ctx.call("mgx_box_precond_mg", bs.h, 2, 2, gam, CODE[prec], mgx.ptr(tr), mgx.ptr(to))
    ref = O.b_precond(ob, 2, 2, gam, r, dtype=DT[prec])
    err = relmax(to_np(to), ref)
    say("box precond", prec, err)
    assert err <= (1e-12 if prec == "f64" else 1e-5)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("edges,levels", [
    ((4, 8, 12), 1),  # one level below the fine one, of edges 2, 4 and 6
    ((4, 8, 12), 2),  # the last of edge 1
    ((16, 24, 8, 20), 2),  # two points per thread, top edges 12 to 4
    ((16, 32, 8), 3),  # eight points per thread, top edge 16
    ((40, 24), 2),  # the largest top edge that goes from LDS, 20
    ((40, 24), 3),  # with the most LDS, 98 KB in FP64
    ((44,), 1),  # a top edge above it: level by level
    ((48,), 2),  # level 1 (edge 24) by launches, level 2 (edge 12) from LDS
    ((44, 24), 2),  # the same with small boxes: edges 22 and 12, then 11 and 6
    ((48, 24), 3),  # levels 2 and 3 from LDS below a level by launches
])
def test_box_precond_coarse_levels(ctx, edges, levels, prec):
    """The coarse levels from LDS, above the largest top edge level by level,
    and a level by launches above levels from LDS."""
    gdim, h = (104, 104, 104), (0.3, 0.31, 0.29)
    rng = np.random.default_rng(23)
    edge = np.array(edges * 2)[: max(3, len(edges))]
    m = 1 << levels
    origin = rng.integers(0, 104 // m, (len(edge), 3)) * m
    ob = O.Boxes.make(origin, edge, gdim, h)
    bs = mgx.BoxSet(ctx, origin, edge, gdim, h, levels + 1)
    r = rng.standard_normal(ob.size(0))
    for kind, gam in ((0, 0.0), (1, O.gamma(list(ob.h), 1, 0.0, -1.2))):
        tr, to = to_dev(r), to_dev(np.zeros_like(r))
        ctx.call("mgx_box_precond_mg", bs.h, kind, levels, gam, CODE[prec], mgx.ptr(tr), mgx.ptr(to))
        ref = O.b_precond(ob, kind, levels, gam, r, dtype=DT[prec])
        # the tolerances of test_box_precond: the same cycle, one level deeper at most
        assert relmax(to_np(to), ref) <= (1e-12 if prec == "f64" else 1e-5), (kind, gam)
    bs.close()


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("edges,levels", [
    ((40,) + (8,) * 9, 2),  # one large box among small ones, in one launch
    ((24, 32, 40, 16, 36, 28), 2),  # the three size classes (top edges up to 12, 16, 20), in one launch
    ((40, 36, 32, 28, 24) + (8,) * 260, 2),  # more boxes than CUs: a launch per class
    ((40, 28) + (4, 8) * 130, 1),  # the same, the coarse levels one level
    ((32,) * 2 + (16,) * 260, 3),  # the second class and the first, FP64 in two launches
    ((32,) * 2 + (8,) * 520, 1),  # and both types
    ((40, 24) + (8, 12) * 110, 2),  # between the two limits, FP64 by class and FP32 not
])
def test_box_precond_size_classes(ctx, edges, levels, prec):
    """The coarse levels from LDS, in one launch and in one per size class of
    the top edge: every box in its own class, in any order."""
    gdim, h = (96, 96, 96), (0.3, 0.31, 0.29)
    rng = np.random.default_rng(29)
    edge = rng.permutation(np.array(edges))
    m = 1 << levels
    origin = rng.integers(0, 96 // m, (len(edge), 3)) * m
    ob = O.Boxes.make(origin, edge, gdim, h)
    bs = mgx.BoxSet(ctx, origin, edge, gdim, h, levels + 1)
    r = rng.standard_normal(ob.size(0))
    tr, to = to_dev(r), to_dev(np.full_like(r, np.nan))
    ctx.call("mgx_box_precond_mg", bs.h, 1, levels, 0.0, CODE[prec], mgx.ptr(tr), mgx.ptr(to))
    ref = O.b_precond(ob, 1, levels, 0.0, r, dtype=DT[prec])
    # the tolerances of test_box_precond, per box
    off = ob.offsets()
    for j in range(len(edge)):
        a, b = off[j], off[j + 1]
        assert relmax(to_np(to)[a:b], ref[a:b]) <= (1e-12 if prec == "f64" else 1e-5), (j, edge[j])
    bs.close()


@pytest.mark.parametrize("prec", [mgx.PREC_F64, mgx.PREC_SPLIT])
def test_box_gram_h_residual(ctx, boxes, cfg, prec):
    ob, bs = boxes
    hp = O.b_hloc(ob, cfg.vtot, cfg.psi)
    n = ob.nbox
    tp, th = to_dev(cfg.psi), to_dev(hp)
    tS, tH = to_dev(np.zeros((n, n))), to_dev(np.zeros((n, n)))
    ctx.call("mgx_box_gram_h", bs.h, prec, mgx.ptr(tp), mgx.ptr(th), mgx.ptr(tS), mgx.ptr(tH))
    S, H = O.b_gram_h(ob, cfg.psi, hp)
    es, eh = relmax(to_np(tS), S), relmax(to_np(tH), H)
    say("gram/H prec", prec, es, eh)
    # split: FP32 accumulation over 32-point chunks, FP64 beyond
    tol = 1e-13 if prec == mgx.PREC_F64 else 1e-7
    assert es <= tol and eh <= tol
    assert bs.npairs() == len(O.b_pairs(ob)[0])
    th_m = np.linalg.solve(S, H)
    tt = to_dev(np.asfortranarray(th_m).T.copy())
    tr = to_dev(np.zeros_like(cfg.psi))
    ctx.call("mgx_box_residual", bs.h, mgx.ptr(tp), mgx.ptr(th), mgx.ptr(tt), mgx.ptr(tr))
    rref = O.b_residual(ob, cfg.psi, hp, th_m)
    assert relmax(to_np(tr), rref) <= 1e-12
    Sinv = np.linalg.inv(S)
    tI = to_dev(np.asfortranarray(Sinv).T.copy())
    out = ctypes.c_double()
    ctx.call("mgx_box_residual_norm", bs.h, mgx.ptr(tr), mgx.ptr(tI), ctypes.byref(out))
    assert out.value == pytest.approx(O.residual_norm(O.b_diag_dots(ob, rref), Sinv), rel=1e-12)


def _cell_multiplicity(cfg):
    g = np.asarray(cfg.gdim) // 8
    cnt = np.zeros(tuple(g), dtype=int)
    for o, e in zip(cfg.origin, cfg.edge):
        ix = [np.arange(o[d] // 8, (o[d] + e - 1) // 8 + 1) % g[d] for d in range(3)]
        cnt[np.ix_(*ix)] += 1
    return cnt.ravel()


@pytest.mark.parametrize("prec", [mgx.PREC_F64, mgx.PREC_SPLIT])
@pytest.mark.parametrize("crowd", ["mixed", "crowded"])
def test_box_gram_cell_multiplicity(ctx, prec, crowd):
    """Cells covered by 1-4, 5-8, 9-16 and more than 16 boxes take different
    tilings of the cell kernel (row groups packed into the MFMA columns, one
    16-box tile, 2 x 2 tiles); each class is present in one of the two sets."""
    if crowd == "mixed":
        cfg = synth.box_config(nbox=80, gdim=48, h=0.3, edges=(8, 12, 16, 20), nwells=4, seed=5, levels=3)
    else:
        cfg = synth.box_config(nbox=220, gdim=48, h=0.3, edges=(12, 16, 20), nwells=4, seed=7, levels=3)
    k = _cell_multiplicity(cfg)
    if crowd == "mixed":
        assert k.min() <= 4 and np.any((k > 4) & (k <= 8)) and np.any(k > 8)
    else:
        assert k.max() > 16 and k.max() <= 32
    ob = O.Boxes.make(cfg.origin, cfg.edge, cfg.gdim, cfg.h)
    bs = mgx.BoxSet(ctx, cfg.origin, cfg.edge, cfg.gdim, cfg.h, 3)
    try:
        hp = O.b_hloc(ob, cfg.vtot, cfg.psi)
        n = ob.nbox
        tp, th = to_dev(cfg.psi), to_dev(hp)
        tS, tH = to_dev(np.zeros((n, n))), to_dev(np.zeros((n, n)))
        ctx.call("mgx_box_gram_h", bs.h, prec, mgx.ptr(tp), mgx.ptr(th), mgx.ptr(tS), mgx.ptr(tH))
        S, H = O.b_gram_h(ob, cfg.psi, hp)
        es, eh = relmax(to_np(tS), S), relmax(to_np(tH), H)
        say("gram/H", crowd, prec, es, eh)
        tol = 1e-13 if prec == mgx.PREC_F64 else 1e-7
        assert es <= tol and eh <= tol
    finally:
        bs.close()


def test_boxset_rejects_misaligned(ctx):
    with pytest.raises(mgx.MgxError):
        mgx.BoxSet(ctx, [[2, 0, 0]], [8], (32, 32, 32), 0.3, 3)
    with pytest.raises(mgx.MgxError):
        mgx.BoxSet(ctx, [[0, 0, 0]], [16], (32, 32, 32), 0.3, 3)


@pytest.mark.parametrize("prec", [mgx.PREC_F64, mgx.PREC_SPLIT])
def test_box_gram_residual_pair_fallback(ctx, prec):
    """gdim = 36 is not a multiple of the 8^3 cells: the per-pair kernels run."""
    cfg = synth.box_config(nbox=10, gdim=36, h=0.3, edges=(8, 12, 16), nwells=3, seed=8, levels=3)
    ob = O.Boxes.make(cfg.origin, cfg.edge, cfg.gdim, cfg.h)
    bs = mgx.BoxSet(ctx, cfg.origin, cfg.edge, cfg.gdim, cfg.h, 3)
    hp = O.b_hloc(ob, cfg.vtot, cfg.psi)
    n = ob.nbox
    tp, th = to_dev(cfg.psi), to_dev(hp)
    tS, tH = to_dev(np.zeros((n, n))), to_dev(np.zeros((n, n)))
    ctx.call("mgx_box_gram_h", bs.h, prec, mgx.ptr(tp), mgx.ptr(th), mgx.ptr(tS), mgx.ptr(tH))
    S, H = O.b_gram_h(ob, cfg.psi, hp)
    tol = 1e-13 if prec == mgx.PREC_F64 else 1e-7
    assert relmax(to_np(tS), S) <= tol and relmax(to_np(tH), H) <= tol
    th_m = np.linalg.solve(S, H)
    tt = to_dev(np.asfortranarray(th_m).T.copy())
    tr = to_dev(np.zeros_like(cfg.psi))
    ctx.call("mgx_box_residual", bs.h, mgx.ptr(tp), mgx.ptr(th), mgx.ptr(tt), mgx.ptr(tr))
    assert relmax(to_np(tr), O.b_residual(ob, cfg.psi, hp, th_m)) <= 1e-12
    bs.close()
