"""GPU parity of the grid-family entry points (ghosted blocks, packed H psi,
preconditioner) against the oracle, through the C ABI.

Bar: FP64 agrees to 1e-12 relative (max-norm); the transfer operators and
the halo are bit-exact; FP32 agrees to 2e-6 relative.
"""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from mgmol_amd import mgx
from tests.gpu_util import relmax, say, to_dev, to_np

pytestmark = pytest.mark.gpu

DT = {"f64": np.float64, "f32": np.float32}
TOL = {"f64": 1e-12, "f32": 2e-6}


@pytest.fixture(scope="module")
def ctx():
    from tests.gpu_util import ctx as shared
    return shared()


def _grids(dims=(16, 12, 20), ng=2, ll=2.4, bc=(1, 1, 1)):
    h = [ll / d for d in dims]
    return O.Grid.make(dims, ng, h), mgx.Grid.make(dims, ng, h, bc)


# the marching sweeps (periodic and zero boundaries wrapped in the kernel,
# one or more x-segments and y-tiles, several lane groups per thread) and the
# point kernels they fall back to (odd z extent)
MARCH_CASES = [((16, 12, 20), (1, 1, 1)), ((16, 12, 20), (1, 0, 1)), ((24, 20, 96), (0, 1, 0)),
               ((16, 12, 15), (1, 1, 1)), ((40, 36, 8), (1, 1, 1))]


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("kind", [1, 2])
@pytest.mark.parametrize("dims,bc", MARCH_CASES)
def test_jacobi_and_lap_march_cases(ctx, dt, kind, dims, bc):
    og, mg_ = _grids(dims=dims, bc=bc)
    rng = np.random.default_rng(31)
    nf = 3
    f = O.embed(og, rng.standard_normal((nf,) + tuple(og.dim)).astype(DT[dt]))
    x = O.embed(og, rng.standard_normal((nf,) + tuple(og.dim)).astype(DT[dt]))
    w = np.zeros_like(x)
    jf = O.jacobi_factor(kind, list(og.h))
    tf, tx, tw = to_dev(f), to_dev(x), to_dev(w)
    ctx.call("mgx_jacobi", kind, jf, mgx.block(tf, mg_), mgx.block(tx, mg_), mgx.block(tw, mg_))
    xr, wr = x.copy(), w.copy()
    O.jacobi(og, kind, f, xr, wr, jf, bc=bc)
    ex = relmax(O.interior(og, to_np(tx)), O.interior(og, xr))
    ew = relmax(O.interior(og, to_np(tw)), O.interior(og, wr))
    # the stencil on traded ghosts (Dirichlet ghosts zero)
    blk = O.trade(og, x.copy(), bc=bc)
    ti, to = to_dev(blk), to_dev(np.zeros_like(blk))
    ctx.call("mgx_lap_apply", kind, mgx.block(ti, mg_), mgx.block(to, mg_))
    el = relmax(O.interior(og, to_np(to)), O.interior(og, O.lap(og, kind, blk)))
    say("march case", dt, kind, dims, bc, ex, ew, el)
    assert ex <= TOL[dt] and ew <= TOL[dt] and el <= TOL[dt]


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("bc", [(1, 1, 1), (1, 0, 1)])
def test_halo_bit_exact(ctx, dt, bc):
    say("halo", dt, bc)
    og, mg_ = _grids(bc=bc)
    rng = np.random.default_rng(1)
    blk = rng.standard_normal((3,) + og.shape_g).astype(DT[dt])
    t = to_dev(blk)
    ctx.call("mgx_halo", mgx.block(t, mg_))
    ref = O.trade(og, blk.copy(), bc=bc)
    assert np.array_equal(to_np(t), ref)


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("kind", [0, 1, 2])
def test_lap_apply(ctx, dt, kind):
    say("lap", dt, kind)
    og, mg_ = _grids()
    rng = np.random.default_rng(2)
    blk = O.trade(og, O.embed(og, rng.standard_normal((4,) + tuple(og.dim)).astype(DT[dt])))
    ti, to = to_dev(blk), to_dev(np.zeros_like(blk))
    ctx.call("mgx_lap_apply", kind, mgx.block(ti, mg_), mgx.block(to, mg_))
    got = O.interior(og, to_np(to))
    ref = O.interior(og, O.lap(og, kind, blk))
    err = relmax(got, ref)
    say("  rel err", err)
    assert err <= TOL[dt]


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("rg", [0, 1, 2])
def test_rhs_apply(ctx, dt, rg):
    og, mg_ = _grids()
    rng = np.random.default_rng(3)
    blk = O.trade(og, O.embed(og, rng.standard_normal((2,) + tuple(og.dim)).astype(DT[dt])))
    ref = O.rhs_mehr(og, blk, rg)
    go = mgx.Grid.make(og.dim, rg, list(og.h))
    ti, to = to_dev(blk), to_dev(np.zeros_like(ref))
    ctx.call("mgx_rhs_apply", mgx.block(ti, mg_), mgx.block(to, go))
    assert relmax(to_np(to), ref) <= TOL[dt]


def test_pointwise_axpy_mask(ctx):
    og, mg_ = _grids()
    rng = np.random.default_rng(4)
    a = rng.standard_normal((2,) + og.shape_g)
    v = rng.standard_normal(og.shape_g)
    ta, tv, to = to_dev(a), to_dev(v), to_dev(np.zeros_like(a))
    ctx.call("mgx_pointwise_product", mgx.block(ta, mg_), mgx.ptr(tv), mgx.block(to, mg_))
    assert np.array_equal(to_np(to), O.pointwise(og, a, v))
    for dt in (np.float32, np.float64):
        x = rng.standard_normal(1000).astype(dt)
        y = rng.standard_normal(1000).astype(dt)
        tx, ty = to_dev(x), to_dev(y)
        ctx.call("mgx_axpy", mgx.F32 if dt == np.float32 else mgx.F64, 1000, -0.37, mgx.ptr(tx), mgx.ptr(ty))
        assert np.array_equal(to_np(ty), O.axpy(-0.37, x, y.copy()))
    m = (rng.random((2, og.size)) > 0.5).astype(np.uint8)
    tm = to_dev(m)
    ta2 = to_dev(a)
    ctx.call("mgx_mask", mgx.block(ta2, mg_), mgx.ptr(tm))
    assert np.array_equal(to_np(ta2), O.mask(og, a.copy(), m))


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("kind", [1, 2])
def test_jacobi(ctx, dt, kind):
    og, mg_ = _grids()
    rng = np.random.default_rng(5)
    f = O.embed(og, rng.standard_normal((2,) + tuple(og.dim)).astype(DT[dt]))
    x = O.embed(og, rng.standard_normal((2,) + tuple(og.dim)).astype(DT[dt]))
    w = np.zeros_like(x)
    jf = O.jacobi_factor(kind, list(og.h))
    tf, tx, tw = to_dev(f), to_dev(x), to_dev(w)
    ctx.call("mgx_jacobi", kind, jf, mgx.block(tf, mg_), mgx.block(tx, mg_), mgx.block(tw, mg_))
    xr, wr = x.copy(), w.copy()
    O.jacobi(og, kind, f, xr, wr, jf)
    assert relmax(O.interior(og, to_np(tx)), O.interior(og, xr)) <= TOL[dt]
    assert relmax(O.interior(og, to_np(tw)), O.interior(og, wr)) <= TOL[dt]


@pytest.mark.parametrize("dt", ["f64", "f32"])
def test_restrict_prolong_bit_exact(ctx, dt):
    og, mg_ = _grids(dims=(16, 12, 20))
    ogc = og.coarse()
    mgc = mgx.Grid.make(ogc.dim, 2, list(ogc.h))
    rng = np.random.default_rng(6)
    fine = O.trade(og, O.embed(og, rng.standard_normal((3,) + tuple(og.dim)).astype(DT[dt])))
    tf, tc = to_dev(fine), to_dev(np.zeros((3,) + ogc.shape_g, DT[dt]))
    ctx.call("mgx_restrict", mgx.block(tf, mg_), mgx.block(tc, mgc))
    ref = O.restrict(og, fine, ogc)
    assert np.array_equal(O.interior(ogc, to_np(tc)), O.interior(ogc, ref))
    coarse = O.trade(ogc, O.embed(ogc, rng.standard_normal((3,) + tuple(ogc.dim)).astype(DT[dt])))
    tc2, tf2 = to_dev(coarse), to_dev(np.zeros((3,) + og.shape_g, DT[dt]))
    ctx.call("mgx_prolong", mgx.block(tc2, mgc), mgx.block(tf2, mg_))
    ref2 = O.extend(ogc, coarse, og)
    assert np.array_equal(O.interior(og, to_np(tf2)), O.interior(og, ref2))


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("masked", [False, True])
def test_mg_vcycle(ctx, dt, masked):
    say("mg", dt, masked)
    og, mg_ = _grids(dims=(16, 16, 16), ll=4.8)
    rng = np.random.default_rng(7)
    nf = 3
    f = O.embed(og, rng.standard_normal((nf,) + tuple(og.dim)).astype(DT[dt]))
    v = np.zeros_like(f)
    O.axpy(0.02, f, v)
    masks = None
    if masked:
        b = O.Boxes.make([[0, 4, 8], [8, 8, 0], [4, 0, 4]], [8, 8, 4], (16, 16, 16), list(og.h))
        masks = [O.b_masks(b, l) for l in range(3)]
    tv, tf = to_dev(v), to_dev(f)
    tmasks = [to_dev(m) for m in masks] if masks else None
    arr = None
    if tmasks:
        import ctypes
        arr = (ctypes.c_void_p * 3)(*[t.data_ptr() for t in tmasks])
    ctx.call("mgx_mg", 2, 2, mgx.block(tv, mg_), mgx.block(tf, mg_), arr)
    ref = O.mg(og, 2, 2, v.copy(), f, masks=masks)
    err = relmax(O.interior(og, to_np(tv)), O.interior(og, ref))
    say("  rel err", err)
    assert err <= (1e-12 if dt == "f64" else 1e-5)


@pytest.mark.parametrize("kind", [0, 2])
def test_hloc_packed_f64(ctx, kind):
    og, mg_ = _grids(dims=(16, 12, 20), ll=3.0)
    rng = np.random.default_rng(8)
    nf = 4
    psi = rng.standard_normal((nf, og.size))
    v = rng.standard_normal(og.size)
    tp, tv, th = to_dev(psi), to_dev(v), to_dev(np.zeros_like(psi))
    ctx.call("mgx_hloc_apply", kind, mg_, mgx.F64, mgx.ptr(tp), og.size, nf, mgx.ptr(tv), mgx.ptr(th), og.size)
    blk = O.embed(og, psi.reshape((nf,) + tuple(og.dim)))
    ref = O.hloc(og, kind, blk, v)
    err = relmax(to_np(th), ref)
    say("hloc", kind, err)
    assert err <= 1e-12


def test_hloc_packed_f32(ctx):
    og, mg_ = _grids(dims=(16, 12, 20), ll=3.0)
    rng = np.random.default_rng(9)
    psi = rng.standard_normal((2, og.size)).astype(np.float32)
    v = rng.standard_normal(og.size)
    tp, tv, th = to_dev(psi), to_dev(v), to_dev(np.zeros_like(psi))
    ctx.call("mgx_hloc_apply", 2, mg_, mgx.F32, mgx.ptr(tp), og.size, 2, mgx.ptr(tv), mgx.ptr(th), og.size)
    blk = O.trade(og, O.embed(og, psi.reshape((2,) + tuple(og.dim))))
    ref = O.lap4_withpot(og, blk, v)
    assert relmax(to_np(th), ref) <= 2e-6


# output leading dimensions: numpt and numpt + 8 (the FP64 cycle's last
# sweep writes the packed output itself), numpt + 3 (odd: the conversion
# kernel writes it); the padding keeps what it held
@pytest.mark.parametrize("pad", [0, 8, 3])
@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_precond_mg(ctx, prec, pad):
    og, mg_ = _grids(dims=(16, 16, 16), ll=4.8)
    rng = np.random.default_rng(10)
    nf = 2
    res = rng.standard_normal((nf, og.size))
    gam = O.gamma(list(og.h), 2, 0.0, -1.0)
    ldo = og.size + pad
    out = np.full(nf * ldo, 7.25)
    tr, to = to_dev(res), to_dev(out)
    pd = mgx.F32 if prec == "f32" else mgx.F64
    ctx.call("mgx_precond_mg", 2, 2, gam, pd, mg_, mgx.ptr(tr), og.size, nf, None, mgx.ptr(to), ldo)
    got = to_np(to).reshape(nf, ldo)
    ref = O.precond(og, 2, 2, gam, res, dtype=DT[prec])
    err = relmax(got[:, :og.size], ref)
    say("precond", prec, "pad", pad, err)
    assert err <= (1e-12 if prec == "f64" else 1e-5)
    assert np.all(got[:, og.size:] == 7.25)


# the packed V-cycle (no masks) against the general path (masks of ones) and the
# oracle: every operator, one and several levels, tiles of 64 and 32 z-points and
# 8 and 16 rows with remainders, x in one and in several segments, a direction
# shorter than the stencil's reach, levels with and without the one-launch coarse
# cycle, Dirichlet directions, leading dimensions with odd padding, in place.
# The FP64 sums differ in order only (1e-13); FP32 iterates are rounded at the
# same points, a flipped last bit moves on through the cycle (1e-6 of the largest)
@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("lap,dims,nf,levels,bc", [
    (2, (16, 16, 16), 1, 0, (1, 1, 1)), (2, (4, 12, 68), 2, 1, (1, 1, 1)), (0, (36, 20, 100), 3, 2, (1, 1, 1)),
    (1, (24, 40, 40), 2, 3, (1, 1, 1)), (2, (48, 8, 132), 1, 2, (1, 1, 1)), (0, (8, 24, 8), 40, 2, (1, 1, 1)),
    (2, (64, 72, 64), 1, 1, (1, 1, 1)), (2, (16, 24, 36), 2, 2, (0, 1, 1)), (0, (16, 24, 36), 2, 2, (1, 0, 0)),
    (1, (16, 8, 8), 1, 0, (0, 0, 0)), (2, (5, 7, 9), 2, 0, (1, 1, 1))])
def test_precond_packed(ctx, prec, lap, dims, nf, levels, bc):
    og, mg_ = _grids(dims=dims, ll=0.3 * dims[0])
    for i in range(3):
        mg_.h[i] = 0.3
        mg_.bc[i] = bc[i]
        og.h[i] = 0.3
    rng = np.random.default_rng(lap + levels)
    n = og.size
    ld, ldo = n + 3, n + 5
    res = rng.standard_normal((nf, ld))
    gam = O.gamma(list(og.h), levels, 0.0, -1.0)
    pd = mgx.F32 if prec == "f32" else mgx.F64
    tr, to, tg = to_dev(res), to_dev(np.full((nf, ldo), 7.25)), to_dev(np.full((nf, ldo), 7.25))
    ctx.call("mgx_precond_mg", lap, levels, gam, pd, mg_, mgx.ptr(tr), ld, nf, None, mgx.ptr(to), ldo)
    ones = [to_dev(np.ones(nf * (n >> (3 * l)), dtype=np.uint8)) for l in range(levels + 1)]
    masks = (C.c_void_p * (levels + 1))(*[t.data_ptr() for t in ones])
    ctx.call("mgx_precond_mg", lap, levels, gam, pd, mg_, mgx.ptr(tr), ld, nf, masks, mgx.ptr(tg), ldo)
    got, general = to_np(to), to_np(tg)
    assert np.all(got[:, n:] == 7.25)
    tol = 1e-13 if prec == "f64" else 1e-6
    assert relmax(got[:, :n], general[:, :n]) <= tol
    ref = O.precond(og, lap, levels, gam, np.ascontiguousarray(res[:, :n]), dtype=DT[prec], bc=bc)
    assert relmax(got[:, :n], ref) <= (1e-12 if prec == "f64" else 1e-5)
    # in place
    ctx.call("mgx_precond_mg", lap, levels, gam, pd, mg_, mgx.ptr(tr), ld, nf, None, mgx.ptr(tr), ld)
    assert np.array_equal(to_np(tr)[:, :n], got[:, :n])
    assert np.array_equal(to_np(tr)[:, n:], res[:, n:])


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("shift,pad", [(64, 0), (-64, 0), (1, 3), (4096 + 5, 10)])
def test_precond_overlapping_buffers(ctx, prec, shift, pad):
    """Results over a shifted residual, before and behind it, by one value, and
    by a whole function: from a copy of the residual (FP64) or the general path
    (FP32); the tolerances of test_precond_packed."""
    og, mg_ = _grids(dims=(16, 16, 16), ll=4.8)
    n, nf = og.size, 3
    ld = n + pad
    rng = np.random.default_rng(3)
    buf = rng.standard_normal(nf * ld + abs(shift))
    r0 = max(0, -shift)
    res = np.ascontiguousarray(buf[r0:r0 + nf * ld].reshape(nf, ld)[:, :n])
    gam = O.gamma(list(og.h), 2, 0.0, -1.0)
    t = to_dev(buf)
    at = lambda k: C.c_void_p(t.data_ptr() + 8 * k)
    ctx.call("mgx_precond_mg", 2, 2, gam, mgx.F32 if prec == "f32" else mgx.F64, mg_, at(r0), ld, nf, None,
             at(r0 + shift), ld)
    ref = O.precond(og, 2, 2, gam, res, dtype=DT[prec])
    o = r0 + shift
    got = np.concatenate([to_np(t), np.zeros(pad)])[o:o + nf * ld].reshape(nf, ld)
    assert relmax(got[:, :n], ref) <= (1e-12 if prec == "f64" else 1e-5)


def test_precond_refuses_what_it_refused(ctx):
    """Odd dimensions above the coarsest level, too few ghosts for a coarse
    correction, ghosts wider than a coarse level."""
    for dims, ng, levels in [((12, 12, 10), 2, 2), ((16, 16, 16), 0, 1), ((4, 4, 4), 2, 2)]:
        g = mgx.Grid.make(dims, ng, [0.3] * 3)
        n = int(np.prod(dims))
        tr, to = to_dev(np.ones(n)), to_dev(np.zeros(n))
        with pytest.raises(mgx.MgxError):
            ctx.call("mgx_precond_mg", 2, levels, 0.01, mgx.F64, g, mgx.ptr(tr), n, 1, None, mgx.ptr(to), n)


def test_invalid_lap_type_rejected(ctx):
    og, mg_ = _grids()
    t = to_dev(np.zeros((1,) + og.shape_g))
    with pytest.raises(mgx.MgxError):
        ctx.call("mgx_lap_apply", 3, mgx.block(t, mg_), mgx.block(t, mg_))
