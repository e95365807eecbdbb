"""Hops and operators straight from and to the caller's interface buffers
(hop_split_kernel) against the path through internal fields, which a call whose output
overlaps its input still takes, and against the oracle.  Half volumes off the 64-site
chunk (8, 24 and 240 sites), of whole chunks, and t extents on and off the chunk order's
tiles; right-hand sides from one to the most a launch takes."""
import ctypes

import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu

LATS = [(2, 2, 2, 2), (6, 2, 2, 2), (4, 6, 2, 10), (8, 8, 4, 14), (8, 4, 8, 12)]


@pytest.fixture(scope="module")
def q():
    import qcu_cg_inverter_amd as q

    q.init(0)
    return q


def ptrs(bufs):
    return (ctypes.c_void_p * len(bufs))(*[b.ptr for b in bufs])


@pytest.mark.parametrize("L", LATS)
@pytest.mark.parametrize("prec,tol", [(0, 1e-14), (1, 1e-6), (2, 3e-3)])
def test_hop_bits_equal_staged(q, L, prec, tol):
    g = q.Gauge.random(L, seed=41, eps=0.3)
    gref = g.to_numpy()
    vh = q.half_volume(L)
    for recon, nrhs, parity, dag, tb in ((12, 1, 0, 0, 1), (18, 1, 1, 1, -1), (12, 16, 1, 1, -1), (18, 3, 0, 0, -1)):
        vs = [orc.source_gauss(L, 70 + r)[1 - parity] for r in range(nrhs)]
        ins = [q.DeviceBuffer.from_numpy(v) for v in vs]
        outs = [q.DeviceBuffer(vh * 192) for _ in range(nrhs)]
        q.check(q.lib().qcuHopBatch(g.handle, nrhs, ptrs(outs), ptrs(ins), parity, dag, tb, recon, prec))
        direct = [o.to_numpy((vh, 4, 3)) for o in outs]
        q.check(q.lib().qcuHopBatch(g.handle, nrhs, ptrs(ins), ptrs(ins), parity, dag, tb, recon, prec))
        for r in range(nrhs):
            assert np.array_equal(direct[r], ins[r].to_numpy((vh, 4, 3))), (recon, nrhs, r)
        ref = orc.hop(vs[-1], gref, L, parity, s=-1 if dag else 1, tbc=float(tb), recon=recon)
        assert np.linalg.norm(direct[-1] - ref) <= tol * np.linalg.norm(ref), (recon, nrhs)


@pytest.mark.parametrize("L", LATS)
@pytest.mark.parametrize("csw", [0.0, 1.0])
def test_full_operator_bits_equal_staged(q, L, csw):
    g = q.Gauge.random(L, seed=42, eps=0.25)
    gref = g.to_numpy()
    vh = q.half_volume(L)
    v = orc.source_gauss(L, 8)
    A = orc.clover_fields(gref, L, 0.122, csw, recon=18)[0] if csw else None
    for recon, dag, tb in ((12, 0, -1), (18, 1, 1)):
        op = q.Operator(0.122, csw, tb, recon)
        a, o = q.DeviceBuffer.from_numpy(v), q.DeviceBuffer(2 * vh * 192)
        q.check(q.lib().qcuApplyM(g.handle, ctypes.byref(op), o.ptr, a.ptr, dag))
        direct = o.to_numpy((2, vh, 4, 3))
        q.check(q.lib().qcuApplyM(g.handle, ctypes.byref(op), a.ptr, a.ptr, dag))
        assert np.array_equal(direct, a.to_numpy((2, vh, 4, 3))), (recon, dag)
        ref = orc.full_op(v, gref, L, 0.122, A=A, s=-1 if dag else 1, tbc=float(tb), recon=recon)
        assert np.linalg.norm(direct - ref) <= 1e-14 * np.linalg.norm(ref), (recon, dag)
        a = q.DeviceBuffer.from_numpy(v)
        q.check(q.lib().qcuApplyComposite(g.handle, ctypes.byref(op), q.COMP_AINV_D, o.ptr, a.ptr, dag))
        direct = o.to_numpy((2, vh, 4, 3))
        q.check(q.lib().qcuApplyComposite(g.handle, ctypes.byref(op), q.COMP_AINV_D, a.ptr, a.ptr, dag))
        assert np.array_equal(direct, a.to_numpy((2, vh, 4, 3))), (recon, dag)


@pytest.mark.parametrize("L", LATS)
@pytest.mark.parametrize("prec", [0, 1, 2])
def test_split_kernel_bits_equal_pinned_shape(q, L, prec):
    """Hops on internal fields take the leg-split kernel by default and hop_kernel under a
    pinned shape: the same bits from every epilogue (Mhat, Wilson and clover) and, through
    the |out|^2 partials, the same solve to the last bit and iteration."""
    pin = {"block": 128, "rb": 1, "rpt": 1}
    vh = q.half_volume(L)
    b = orc.source_gauss(L, 5)
    for recon, csw in ((12, 0.0), (18, 0.0), (12, 1.0), (18, 1.0)):
        op = q.Operator(0.12, csw, -1, recon)
        sp = q.default_solve_params(tol=1e-9, precision=prec, chunk=4, max_iter=200)

        def results():
            g = q.Gauge.random(L, seed=43, eps=0.2)
            if pinned:
                for p in {0, prec}:
                    q.set_hop_shape(g, p, recon, 1, pin)
            out = [q.apply_mhat(g, op, b[0], dagger=d, precision=prec) for d in (0, 1)]
            x, st = q.solve(g, op, b, sp, raise_on_error=False)
            return out, x, st.iterations, st.true_residual

        # a pinned shape holds for every gauge of this half volume in the process: default first
        pinned = False
        want = results()
        pinned = True
        got = results()
        for a, c in zip(want[0], got[0]):
            assert np.array_equal(a, c), (recon, csw)
        assert np.array_equal(want[1], got[1]) and want[2:] == got[2:], (recon, csw, want[2:], got[2:])
        assert want[3] <= 1e-9


@pytest.mark.parametrize("L", LATS)
@pytest.mark.parametrize("ck", [0.122, 1.0])
def test_clover_built_in_parts(q, L, ck):
    """A, the odd inverse and the even inverse built one after another, as the full
    operator, the Schur operator and the export ask for them, have the bits of one build
    for the export, and the oracle's values; blocks that are not positive definite (they
    occur at ck = 1) are counted once each."""
    vh = q.half_volume(L)
    g = q.Gauge.random(L, seed=44, eps=0.45)
    gref = g.to_numpy()
    op = q.Operator(ck, 1.0, 1, 18)
    v = orc.source_gauss(L, 9)
    q.apply_m(g, op, v)
    q.apply_mhat(g, op, v[0])
    A, Ainv, nf = g.clover(ck, 1.0)
    A1, Ainv1, nf1 = q.Gauge.from_numpy(gref, L).clover(ck, 1.0)
    assert np.array_equal(A, A1) and np.array_equal(Ainv, Ainv1) and nf == nf1
    Aref = orc.clover_A(orc.clover_T(gref, L, recon=18), ck)
    inv_ref, nbad = orc.clover_invert(Aref, chol=True)
    assert nf == nbad
    assert np.abs(A - Aref).max() < 1e-14 * max(1.0, np.abs(Aref).max())
    cond = np.linalg.cond(Aref.reshape(-1, 6, 6)).max()
    assert np.abs(Ainv - inv_ref).max() < 1e-14 * cond * max(1.0, np.abs(inv_ref).max())


@pytest.mark.parametrize("prec", [0, 1])
def test_solves_alternate_gauges(q, prec):
    """Solves that go back and forth between gauges, one of another lattice with the same
    half volume, share a workspace where the lattice is the same; each gives the bits of
    a solve on a gauge of its own, also after the other gauge is gone."""
    b = {L: orc.source_gauss(L, 12) for L in ((8, 4, 8, 8), (4, 8, 8, 8))}
    sp = q.default_solve_params(tol=1e-10, precision=prec)
    op = q.Operator(0.12, 1.0, -1, 12)

    def make(k):
        L = (4, 8, 8, 8) if k == 2 else (8, 4, 8, 8)
        return q.Gauge.random(L, seed=50 + k, eps=0.2)

    alone = {}
    for k in range(3):
        g = make(k)
        alone[k] = q.solve(g, op, b[g.L], sp)[0]
        g.destroy()
    gs = [make(k) for k in range(3)]
    for k in (0, 1, 0, 2, 1, 0):
        assert np.array_equal(q.solve(gs[k], op, b[gs[k].L], sp)[0], alone[k]), k
    gs[1].destroy()
    assert np.array_equal(q.solve(gs[0], op, b[gs[0].L], sp)[0], alone[0])


def test_scalar_steps_change_kernels_mid_solve(q):
    """Sixteen right-hand sides on 16^3x32, checked after every iteration: 16 and 15 take
    their scalar steps in one-block kernels, 14 and fewer in the vector kernels.  Point
    and Gaussian sources converge at different iterations, so the solve goes from one to
    the other; each right-hand side keeps the bits and iterations of its solve alone."""
    L = (16, 16, 16, 32)
    g = q.Gauge.random(L, seed=45, eps=0.2)
    op = q.Operator(0.115, 0.0, -1, 12)
    sp = q.default_solve_params(tol=1e-8, precision=1, chunk=1)
    bs = [q.source_point_device(L, (r, 1, 2, 2 * r), r % 4, r % 3) if r % 3 == 0 else q.source_gaussian_device(L, 60 + r)
          for r in range(16)]
    vh = q.half_volume(L)
    xs = [q.DeviceBuffer(2 * vh * 192) for _ in bs]
    sts = q.solve_batch_device(g, op, xs, bs, sp)
    its = [s.iterations for s in sts]
    assert len(set(its)) >= 2, its
    xa = q.DeviceBuffer(2 * vh * 192)
    for r in range(16):
        sa = q.solve_batch_device(g, op, [xa], [bs[r]], sp)[0]
        assert sa.converged and sa.iterations == its[r], (r, its)
        assert np.array_equal(xa.to_numpy((2, vh, 4, 3)), xs[r].to_numpy((2, vh, 4, 3))), r


@pytest.mark.parametrize("L", [(4, 6, 2, 10), (8, 8, 4, 14)])
@pytest.mark.parametrize("prec", [0, 1, 2])
def test_dropin_import(q, L, prec):
    """The drop-in gauge is imported as rows 0-1 only and its FP32 and FP16 links come from
    those: cg_inverter in each precision on links scaled by 0.12 (at the reference's kappa =
    1 that makes the system as well conditioned as a Wilson solve; row 2 is rebuilt, so it
    scales by 0.12 squared), on a gauge changed in one real of row 1 between calls, and
    indifferent to row 2.  Residuals by the oracle."""
    prm = q.param(L)
    vh = q.half_volume(L)
    b = orc.source_gauss(L, 13)
    bd, xd, yd = q.DeviceBuffer.from_numpy(b), q.DeviceBuffer(2 * vh * 192), q.DeviceBuffer(2 * vh * 192)
    u = 0.12 * orc.gauge_random(L, 46, 0.3)
    gd = q.DeviceBuffer.from_numpy(u)
    sp = q.default_solve_params(tol=1e-10, precision=prec)
    q.check(q.lib().qcuSetDefaultSolve(ctypes.byref(sp)))
    try:
        for step in range(3):
            if step == 1:
                u[2, 1, vh - 1, 1, 2] += 1e-3
            if step == 2:
                u[:, :, :, 2, :] = 7.0
            gd.upload(u)
            q.lib().cg_inverter(bd.ptr, xd.ptr, gd.ptr, ctypes.byref(prm))
            assert q.lib().qcuGetLastError() == 0
            x = xd.to_numpy((2, vh, 4, 3))
            A = orc.clover_fields(u, L, 1.0, 1.0, recon=12)[0]
            r = b - orc.full_op(x, u, L, 1.0, A=A, s=1, tbc=1.0, recon=12)
            assert np.linalg.norm(r) <= 1.01e-10 * np.linalg.norm(b), step
            q.lib().fullDslashQcu(yd.ptr, bd.ptr, gd.ptr, ctypes.byref(prm), 1)
            ref = orc.full_op(b, u, L, 1.0, A=A, s=-1, tbc=1.0, recon=12)
            assert np.linalg.norm(yd.to_numpy((2, vh, 4, 3)) - ref) <= 1e-14 * np.linalg.norm(ref), step
    finally:
        sp = q.default_solve_params(tol=1e-12, precision=0)
        q.check(q.lib().qcuSetDefaultSolve(ctypes.byref(sp)))


@pytest.mark.parametrize("L", LATS)
@pytest.mark.parametrize("prec", [0, 1, 2])
def test_solve_residual_by_oracle(q, L, prec):
    """Residual updates, iterate folds and finishes of slots that converge apart, on half
    volumes off the 64-site chunk: the true residual the solve reports is the oracle's (both
    in FP64, whose rounding of b - M x is below 1e-14 |b|) and is below the tolerance."""
    g = q.Gauge.random(L, seed=45, eps=0.2)
    gref = g.to_numpy()
    for csw in (0.0, 1.0):
        op = q.Operator(0.12, csw, -1, 12)
        A = orc.clover_fields(gref, L, 0.12, csw, recon=12)[0] if csw else None
        bs = [orc.source_gauss(L, 60 + k) for k in range(3)]
        bs[1] = np.zeros_like(bs[1])
        bs[1][0, 0, 1, 2] = 1.0
        sp = q.default_solve_params(tol=1e-9, precision=prec, chunk=3, delta=0.3, max_iter=400)
        xs, sts = q.solve_batch(g, op, bs, sp)
        for b, x, st in zip(bs, xs, sts):
            r = b - orc.full_op(x, gref, L, 0.12, A=A, s=1, tbc=-1.0, recon=12)
            res = np.linalg.norm(r) / np.linalg.norm(b)
            assert st.converged and res <= 1e-9 + 1e-14
            assert abs(res - st.true_residual) <= 1e-14
            assert st.reliable_updates >= 1


@pytest.mark.parametrize("prec,nrhs", [(0, 5), (2, 7)])
def test_lds_hop_chunk_order_bits(q, prec, nrhs):
    """Past the Infinity Cache a batch takes the LDS kernel, which orders the chunks of a
    lattice whose planes are no whole chunks (20^2 / 2 = 200 sites) by eighths of Lt, with
    eight waves a block in FP64 clover: the bits of right-hand sides solved alone."""
    L = (20, 20, 24, 24)
    g = q.Gauge.random(L, seed=46, eps=0.2)
    op = q.Operator(0.12, 1.0, -1, 12)
    sp = q.default_solve_params(tol=1e-12, precision=prec, chunk=4, max_iter=8)
    bs = [orc.source_gauss(L, 80 + k) for k in range(2)]
    bs += [bs[k % 2] * (1.0 + k) for k in range(2, nrhs)]
    xs, sts = q.solve_batch(g, op, bs, sp, raise_on_error=False)
    for k in (0, 1, nrhs - 1):
        x, st = q.solve(g, op, bs[k], sp, raise_on_error=False)
        assert np.array_equal(x, xs[k]) and st.iterations == sts[k].iterations
        assert st.true_residual == sts[k].true_residual
