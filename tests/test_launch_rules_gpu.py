"""The kernels that a rule on sizes picks, against the general ones, on the GPU.

* the wave-per-hop hopping kernel of small lattices gives the bits of the thread-per-site kernel, for lattices that
  do not fill a block of 64 sites or a link tile, plain, with the Aee epilogue and in the fused CG step;
* the staggered multi-RHS kernel with two right-hand sides per thread gives the single-field kernel's bits where the
  last block is not full, and fields that are not 16-byte aligned take the one-per-thread kernel;
* MdagM_eo equals its two D_KS_eo and the elementwise saxpby bit for bit;
* the streaming multi-shift update agrees with numpy;
* stage 2 of the reductions sums every one of many partials once;
* the work order of large multi-RHS fields, slabs that split y, visits every site: site order's bits;
* cl2_scalar_get returns what the stream wrote, on both sides of the mailbox's size and of the time the host watches it,
  and refuses what a copy refuses;
* the lockstep steps take arrays that overlap;
* tuning keys and the autotuner leave other launches' shapes alone, and the size rules pick what they say.
"""
import ctypes

import numpy as np
import pytest

import oracle as O
from cl2qcd_amd import abi
from fields import random_su3_field

pytestmark = pytest.mark.gpu

FORMATS = [(abi.GAUGE_F64_18, abi.F64), (abi.GAUGE_F64_12, abi.F64), (abi.GAUGE_F32_12, abi.F32),
           (abi.GAUGE_F16_12, abi.F16)]
KAPPA, MUBAR = 0.16, 0.0016
NAMES = {abi.GAUGE_F64_18: "f64_18", abi.GAUGE_F64_12: "f64_12", abi.GAUGE_F32_12: "f32_12", abi.GAUGE_F16_12: "f16_12"}


def chosen(ctx, what, fmt, nrhs=None):
    """What the launch rules pick for links of format fmt on this context."""
    return ctx.lib.cl2_tune_get(ctx.handle, ".".join([what, NAMES[fmt]] + ([str(nrhs)] if nrhs else [])).encode())


@pytest.mark.parametrize("phases", [dict(theta_t=1.0), dict(theta_t=1.0, theta_s=0.3, cp_im=0.2)],
                         ids=["real-spatial-weights", "complex-weights"])
@pytest.mark.parametrize("ns,nt", [(2, 2), (6, 10), (8, 4)])  # 8, 1080 and 1024 eo sites
@pytest.mark.parametrize("fmt,prec", FORMATS)
def test_wave_per_hop_matches_thread_per_site(fmt, prec, ns, nt, phases):
    lat = O.lattice(ns, nt, **phases)
    results = []
    for block in (None, 256):
        with abi.Context(ns, nt, **phases) as ctx:
            if block:
                ctx.tune_set(b"hop.block", block)
            assert chosen(ctx, "hop.block", fmt) == (block or 64)
            rng = np.random.default_rng(7)
            gf = ctx.gauge(random_su3_field(4 * O.volume(lat), 8), fmt)
            src, r0 = rng.standard_normal((ctx.veo, 24)), rng.standard_normal((ctx.veo, 24))
            a, b, r = ctx.spinor(prec).upload(src), ctx.spinor(prec), ctx.spinor(prec).upload(r0)
            tmp = ctx.buffer(2 * ctx.lib.cl2_field_bytes(ctx.handle, abi.FIELD_SPINOR_EO, prec))
            got = []
            for evenodd in (abi.EVEN, abi.ODD):
                ctx.dslash_eo(b.ptr, a.ptr, gf.ptr, fmt, evenodd, KAPPA)
                got.append(b.download())
            ctx.fermionmatrix_eo(abi.OP_AEE_MINUS_AND_GAMMA5, b.ptr, a.ptr, gf.ptr, fmt, abi.ACTION_TWISTEDMASS, KAPPA,
                                 MUBAR, tmp.ptr)
            got.append(b.download())
            s = ctx.scalars(10)
            s.store([O.norm2(r0)] + [0.0] * 9)
            ctx.fermionmatrix_eo_cg_step(abi.OP_QPLUSQMINUS_EO, r.ptr, a.ptr, gf.ptr, fmt, abi.ACTION_TWISTEDMASS,
                                         KAPPA, MUBAR, tmp.ptr, s.at(0), s.at(2), s.at(4), s.at(6))
            results.append((got, r.download(), s.get()))
    (got, res, sc), (ref, rres, rsc) = results
    for x, y in zip(got, ref):
        assert np.array_equal(x, y)
    # the norms are the same terms grouped by component pairs: FP64 sums; for FP16 each group is a float chain of 4
    # instead of 24 terms, 24 * 2^-24 relative
    tol = 1.5e-6 if prec == abi.F16 else 1e-13
    assert abs(sc[2] - rsc[2]) <= tol * rsc[2]
    if prec == abi.F16:
        # alpha follows pAp within tol; r_new is requantised to 2^-11 of the site's largest entry
        assert np.abs(res - rres).max() <= 2.0 ** -10 * np.abs(rres).max()
    else:
        bound = 1e-12 if prec == abi.F64 else 4 * 2.0 ** -23
        assert np.abs(res - rres).max() <= bound * np.abs(rres).max()
    assert abs(sc[6] - rsc[6]) <= (2e-3 if prec == abi.F16 else 1e-6) * rsc[6]


@pytest.mark.parametrize("nrhs", [8, 12, 16])
@pytest.mark.parametrize("offset", [0, 8])
def test_staggered_pairs_match_single(nrhs, offset):
    ns, nt, mass = 6, 10, 0.1  # 1080 eo sites: 33 blocks of 32 sites and a rest of 24
    with abi.Context(ns, nt, theta_t=1.0) as ctx:
        lat = O.lattice(ns, nt, theta_t=1.0)
        assert chosen(ctx, "stagg.pairs", abi.GAUGE_F32_12, nrhs) == 1  # with the aligned offset, 0
        gf = ctx.gauge(random_su3_field(4 * O.volume(lat), 3)).converted(abi.GAUGE_F32_12)
        rng = np.random.default_rng(nrhs)
        one = ctx.lib.cl2_field_bytes(ctx.handle, abi.FIELD_SU3VEC_EO, abi.F32)
        blk, out = ctx.buffer(nrhs * one + 16), ctx.buffer(nrhs * one + 16)
        bp, op = blk.ptr + offset, out.ptr + offset
        src = [rng.standard_normal((ctx.veo, 6)) for _ in range(nrhs)]
        a, b = ctx.su3vec(abi.F32), ctx.su3vec(abi.F32)
        for r, v in enumerate(src):
            ctx.block_insert_stagg_eo(bp, a.upload(v).ptr, abi.F32, nrhs, r)
        for evenodd in (abi.EVEN, abi.ODD):
            ctx.D_KS_eo_mrhs(op, bp, gf.ptr, abi.GAUGE_F32_12, evenodd, nrhs)
            for r in range(nrhs):
                ctx.D_KS_eo(b.ptr, a.upload(src[r]).ptr, gf.ptr, abi.GAUGE_F32_12, evenodd)
                got = ctx.su3vec(abi.F32)
                ctx.block_extract_stagg_eo(got.ptr, op, abi.F32, nrhs, r)
                assert np.array_equal(got.download(), b.download())
        # the fused step's sums: |D p|^2 + (m^2 + sigma) |p|^2 per right-hand side, against numpy
        s = ctx.scalars(10 * nrhs)
        s.store(np.concatenate([np.ones(2 * nrhs), np.zeros(8 * nrhs)]))
        rb, tb = ctx.buffer(nrhs * one + 16), ctx.buffer(nrhs * one + 16)
        sigma = (ctypes.c_double * nrhs)(*np.linspace(0.0, 1.0, nrhs))
        ctx.MdagM_eo_mrhs_cg_step(rb.ptr + offset, bp, gf.ptr, abi.GAUGE_F32_12, mass, abi.EVEN, sigma, tb.ptr + offset,
                                  nrhs, s.at(0), s.at(nrhs), s.at(2 * nrhs), s.at(4 * nrhs), s.at(6 * nrhs))
        pap = s.get()[2 * nrhs:4 * nrhs:2]
        for r in range(nrhs):
            p = a.upload(src[r]).download()
            ctx.D_KS_eo(b.ptr, a.ptr, gf.ptr, abi.GAUGE_F32_12, abi.ODD)
            ref = (b.download() ** 2).sum() + (mass * mass + sigma[r]) * (p ** 2).sum()
            assert abs(pap[r] - ref) <= 1e-12 * ref


@pytest.mark.parametrize("fmt,prec", FORMATS[:3])
def test_mdagm_is_two_hops_and_saxpby(fmt, prec):
    ns, nt, mass = 6, 10, 0.37
    with abi.Context(ns, nt, theta_t=1.0) as ctx:
        lat = O.lattice(ns, nt, theta_t=1.0)
        gf = ctx.gauge(random_su3_field(4 * O.volume(lat), 4), fmt)
        x = ctx.su3vec(prec).upload(np.random.default_rng(5).standard_normal((ctx.veo, 6)))
        out, w, ref, tmp = (ctx.su3vec(prec) for _ in range(4))
        for upper, first in ((abi.EVEN, abi.ODD), (abi.ODD, abi.EVEN)):
            ctx.MdagM_eo(out.ptr, x.ptr, gf.ptr, fmt, mass, upper, tmp.ptr)
            ctx.D_KS_eo(w.ptr, x.ptr, gf.ptr, fmt, first)
            ctx.D_KS_eo(ref.ptr, w.ptr, gf.ptr, fmt, upper)
            ctx.saxpby_stagg_eo(ref.ptr, x.ptr, ref.ptr, prec, abi.scalar(mass * mass), abi.scalar(-1.0))
            assert np.array_equal(out.download(), ref.download())


def test_streaming_multishift_update():
    n = 60  # FP64 x and FP32 p of 16^3x32: 283 MB, above the 256 MiB where the update starts to stream
    with abi.Context(16, 32) as ctx:
        rng = np.random.default_rng(2)
        r = ctx.su3vec(abi.F32).upload(rng.standard_normal((ctx.veo, 6)))
        xs, ps = [], []
        for k in range(n):
            xs.append(ctx.su3vec(abi.F64))
            ps.append(ctx.su3vec(abi.F32))
            ctx.gaussian_eo(abi.FIELD_SU3VEC_EO, xs[k].ptr, abi.F64, 10 + k)
            ctx.gaussian_eo(abi.FIELD_SU3VEC_EO, ps[k].ptr, abi.F32, 100 + k)
        check = [0, 1, 31, 58, 59]
        before = {k: (xs[k].download(), ps[k].download()) for k in check}
        coef = rng.standard_normal((3, n))
        active = np.ones(n)
        active[[1, 58]] = 0.0
        dev = ctx.scalars(4 * n)
        dev.store(np.concatenate([coef.ravel(), active]))
        ctx.multishift_update_stagg_eo((ctypes.c_void_p * n)(*[x.ptr for x in xs]), abi.F64,
                                       (ctypes.c_void_p * n)(*[p.ptr for p in ps]), r.ptr, abi.F32, n, dev.at(0),
                                       dev.at(n), dev.at(2 * n), dev.at(3 * n))
        R = r.download()
        for k in check:
            x, p = before[k]
            if active[k]:
                x, p = coef[0, k] * p + x, coef[1, k] * R + coef[2, k] * p
            # one product and one sum per element: two roundings of FP64 (x), of FP32 with rounded factors (p)
            assert np.abs(xs[k].download() - x).max() <= 4 * 2.0 ** -53 * np.abs(x).max()
            assert np.abs(ps[k].download() - p).max() <= 6 * 2.0 ** -24 * np.abs(p).max() + 1e-30


def test_many_partial_sums():
    # 8262 partials of 1024 elements: the second stage with eight loads in flight, and a rest of 70
    with abi.Context(24, 102) as ctx:
        f, s = ctx.spinor(abi.F64), ctx.scalars(2)
        ctx.set_cold_eo(f.ptr, abi.F64)
        ctx.squarenorm_eo(s.ptr, f.ptr, abi.F64)
        assert abs(s.get()[0] - 0.5) < 1e-13  # every component is 1 / sqrt(12 V), V twice the eo sites
    # the block form: 8194 partials per right-hand side (one per 32 sites)
    with abi.Context(2, 65552) as ctx:
        one = ctx.lib.cl2_field_bytes(ctx.handle, abi.FIELD_SU3VEC_EO, abi.F32)
        gf = ctx.gauge(fmt=abi.GAUGE_F32_12, seed=1, epsilon=0.0)
        p, r, t, s = ctx.buffer(2 * one), ctx.buffer(2 * one), ctx.buffer(2 * one), ctx.scalars(20)
        s.store([1.0] * 4 + [0.0] * 16)
        f = ctx.su3vec(abi.F32)
        ctx.set_cold_stagg_eo(f.ptr, abi.F32)
        for k in range(2):
            ctx.block_insert_stagg_eo(p.ptr, f.ptr, abi.F32, 2, k)
        ctx.MdagM_eo_mrhs_cg_step(r.ptr, p.ptr, gf.ptr, abi.GAUGE_F32_12, 1.0, abi.EVEN, None, t.ptr, 2, s.at(0), s.at(2),
                                  s.at(4), s.at(8), s.at(12))
        # unit links and a constant field: D_KS_eo cancels, so <p, A p> = |p|^2 = 1/2
        assert np.abs(s.get()[4:8:2] - 0.5).max() < 1e-6


# fields above 32 MiB: slabs of 3 x 6 rows in z and y, 4 x 8 and 5 x 10, and a lattice that no such slab divides
@pytest.mark.parametrize("fmt,prec,nrhs,ns,nt", [
    (abi.GAUGE_F64_18, abi.F64, 12, 12, 18), (abi.GAUGE_F64_12, abi.F64, 16, 16, 6), (abi.GAUGE_F64_18, abi.F64, 4, 20, 12),
    (abi.GAUGE_F32_12, abi.F32, 12, 12, 36), (abi.GAUGE_F32_12, abi.F32, 16, 20, 6), (abi.GAUGE_F32_12, abi.F32, 8, 18, 16)])
def test_slabs_in_y_visit_every_site(fmt, prec, nrhs, ns, nt):
    with abi.Context(ns, nt, theta_t=1.0) as ctx:
        assert chosen(ctx, "mrhs.slab", fmt, nrhs) == {12: 36, 16: 64, 20: 100, 18: 0}[ns]  # rows times ns / 2
        gf = ctx.gauge(random_su3_field(4 * ns ** 3 * nt, 8), fmt)
        one = ctx.lib.cl2_field_bytes(ctx.handle, abi.FIELD_SPINOR_EO, prec)
        src = ctx.spinor(prec).upload(np.random.default_rng(9).standard_normal((ctx.veo, 24)))
        blk, out, got, ref = ctx.buffer(nrhs * one), ctx.buffer(nrhs * one), ctx.spinor(prec), ctx.spinor(prec)
        for r in range(nrhs):
            ctx.block_insert_eo(blk.ptr, src.ptr, prec, nrhs, r)
        for evenodd in (abi.EVEN, abi.ODD):
            ctx.dslash_eo(ref.ptr, src.ptr, gf.ptr, fmt, evenodd, KAPPA)
            for r in (0, nrhs - 1):
                ctx.block_insert_eo(out.ptr, src.ptr, prec, nrhs, r)  # what no block writes would stay the source
            ctx.dslash_eo_mrhs(out.ptr, blk.ptr, gf.ptr, fmt, evenodd, KAPPA, nrhs)
            for r in (0, nrhs - 1):
                ctx.block_extract_eo(got.ptr, out.ptr, prec, nrhs, r)
                assert np.array_equal(got.download(), ref.download())


@pytest.mark.parametrize("fmt,prec,nrhs,ns,nt", [
    (abi.GAUGE_F64_12, abi.F64, 12, 20, 16), (abi.GAUGE_F32_12, abi.F32, 16, 24, 14), (abi.GAUGE_F32_12, abi.F32, 12, 20, 30)])
def test_staggered_slabs_in_y_visit_every_site(fmt, prec, nrhs, ns, nt):
    with abi.Context(ns, nt, theta_t=1.0) as ctx:
        assert chosen(ctx, "stagg.slab", fmt, nrhs) == {20: 100, 24: 144}[ns]
        gf = ctx.gauge(random_su3_field(4 * ns ** 3 * nt, 3)).converted(fmt)
        one = ctx.lib.cl2_field_bytes(ctx.handle, abi.FIELD_SU3VEC_EO, prec)
        src = ctx.su3vec(prec).upload(np.random.default_rng(9).standard_normal((ctx.veo, 6)))
        blk, out, got, ref = ctx.buffer(nrhs * one), ctx.buffer(nrhs * one), ctx.su3vec(prec), ctx.su3vec(prec)
        for r in range(nrhs):
            ctx.block_insert_stagg_eo(blk.ptr, src.ptr, prec, nrhs, r)
        for evenodd in (abi.EVEN, abi.ODD):
            ctx.D_KS_eo(ref.ptr, src.ptr, gf.ptr, fmt, evenodd)
            ctx.D_KS_eo_mrhs(out.ptr, blk.ptr, gf.ptr, fmt, evenodd, nrhs)
            for r in (0, nrhs - 1):
                ctx.block_extract_stagg_eo(got.ptr, out.ptr, prec, nrhs, r)
                assert np.array_equal(got.download(), ref.download())


@pytest.mark.parametrize("n", [1, 63, 64, 65, 200])
def test_scalar_get(n):
    with abi.Context(4, 4) as ctx:
        values = np.random.default_rng(n).standard_normal(n)
        s = ctx.scalars(n)
        for shift in range(3):  # successive reads of the one mailbox
            s.store(values + shift)
            assert np.array_equal(s.get(), values + shift)


@pytest.mark.parametrize("shared", ["pAp", "r2", "active"])
@pytest.mark.parametrize("staggered", [False, True])
def test_lockstep_step_with_shared_arrays(staggered, shared):
    # the step lengths may take the place of the sums, of the old norms or of the active flags: the residual that
    # follows has the bits that separate arrays give
    ns, nt, n, fmt, prec = 6, 10, 8, abi.GAUGE_F64_18, abi.F64
    with abi.Context(ns, nt, theta_t=1.0) as ctx:
        gf = ctx.gauge(random_su3_field(4 * 2 * ctx.veo, 3))
        field = abi.FIELD_SU3VEC_EO if staggered else abi.FIELD_SPINOR_EO
        one = ctx.lib.cl2_field_bytes(ctx.handle, field, prec)
        p, tmp = ctx.buffer(n * one), ctx.buffer(2 * n * one)
        got = []
        for separate in (True, False):
            r, f = ctx.buffer(n * one), ctx.su3vec(prec) if staggered else ctx.spinor(prec)
            insert, extract = ((ctx.block_insert_stagg_eo, ctx.block_extract_stagg_eo) if staggered
                               else (ctx.block_insert_eo, ctx.block_extract_eo))
            for k in range(n):
                ctx.gaussian_eo(field, f.ptr, prec, 10 + k)
                insert(p.ptr, f.ptr, prec, n, k)
                ctx.gaussian_eo(field, f.ptr, prec, 50 + k)
                insert(r.ptr, f.ptr, prec, n, k)
            s = ctx.scalars(8 * n)
            r2, active, pap, norms, alpha = s.at(0), s.at(2 * n), s.at(4 * n), s.at(6 * n), ctx.scalars(2 * n)
            s.store(np.concatenate([np.linspace(0.5, 2.0, 2 * n), np.ones(n - 1), np.zeros(5 * n + 1)]))
            a = alpha.ptr if separate else {"pAp": pap, "r2": r2, "active": active}[shared]
            if staggered:
                ctx.MdagM_eo_mrhs_cg_step(r.ptr, p.ptr, gf.ptr, fmt, 0.1, abi.EVEN, None, tmp.ptr, n, r2, active, pap, a,
                                          norms)
            else:
                ctx.fermionmatrix_eo_mrhs_cg_step(abi.OP_QPLUSQMINUS_EO, r.ptr, p.ptr, gf.ptr, fmt,
                                                  abi.ACTION_TWISTEDMASS, KAPPA, MUBAR, None, None, tmp.ptr, n, r2,
                                                  active, pap, a, norms)
            fields = []
            for k in range(n):
                extract(f.ptr, r.ptr, prec, n, k)
                fields.append(f.download())
            got.append((np.stack(fields), s.get()[6 * n:]))
        assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])


def test_scalar_get_behind_queued_work():
    # several milliseconds of hopping terms in front of the sum that is read: past the time the host watches the mailbox
    with abi.Context(24, 48, theta_t=1.0) as ctx:
        gf = ctx.gauge(seed=3, epsilon=0.0)
        a, b, s = ctx.spinor(), ctx.spinor(), ctx.scalars(1)
        ctx.set_cold_eo(a.ptr, abi.F64)
        for reps in (1, 41):  # each time as many as leave the field in `b`
            s.store([-1.0])
            ctx.set_cold_eo(a.ptr, abi.F64)
            for k in range(reps):
                src, dst = (a, b) if k % 2 == 0 else (b, a)
                ctx.dslash_eo(dst.ptr, src.ptr, gf.ptr, abi.GAUGE_F64_18, abi.EVEN if k % 2 == 0 else abi.ODD, 0.125)
            ctx.squarenorm_eo(s.ptr, b.ptr, abi.F64)
            early = s.get()[0]
            ctx.sync()
            assert early == s.get()[0] and early > 0.0


def test_scalar_get_refuses_what_a_copy_refuses():
    # a range beyond its allocation, and host memory: errors, and the next read and the next launch are in order again
    with abi.Context(4, 4) as ctx:
        s = ctx.scalars(4)
        s.store([1.0, 2.0, 3.0, 4.0])
        out, host = np.zeros(64), np.arange(64.0)
        for src, n in ((s.ptr, 64), (s.at(3), 2), (host.ctypes.data, 2)):
            assert ctx.lib.cl2_scalar_get(ctx.handle, out.ctypes.data, src, n) != 0
            assert np.array_equal(s.get(), [1.0, 2.0, 3.0, 4.0])
            ctx.scalar_copy(s.at(1), s.at(1) + 8, 1)
            s.store([1.0, 2.0, 3.0, 4.0])


@pytest.mark.parametrize("block", [128, 256])
@pytest.mark.parametrize("ns,nt", [(6, 10), (12, 28)])  # a last block of 56 sites; with the XCD remap
def test_f64_12_gather_order_keeps_the_bits(ns, nt, block):
    # 12-real FP64 links gather two directions at a time where a wave has a SIMD to itself: the bits of the shape with
    # two hops in flight, plain and with the epilogue
    with abi.Context(ns, nt, theta_t=1.0) as ctx:
        gf = ctx.gauge(seed=3, epsilon=0.35).converted(abi.GAUGE_F64_12)
        a, b = ctx.spinor(), ctx.spinor()
        tmp = ctx.buffer(2 * ctx.lib.cl2_field_bytes(ctx.handle, abi.FIELD_SPINOR_EO, abi.F64))
        ctx.gaussian_eo(abi.FIELD_SPINOR_EO, a.ptr, abi.F64, 5)
        ctx.tune_set(b"hop.block", block)
        got = []
        for occ in (1, 0):
            ctx.tune_set(b"hop.occupancy", occ)
            for evenodd in (abi.EVEN, abi.ODD):
                ctx.dslash_eo(b.ptr, a.ptr, gf.ptr, abi.GAUGE_F64_12, evenodd, KAPPA)
                got.append(b.download())
            ctx.fermionmatrix_eo(abi.OP_AEE_MINUS_AND_GAMMA5, b.ptr, a.ptr, gf.ptr, abi.GAUGE_F64_12,
                                 abi.ACTION_TWISTEDMASS, KAPPA, MUBAR, tmp.ptr)
            got.append(b.download())
        for x, y in zip(got[:3], got[3:]):
            assert np.array_equal(x, y)


# 378 and 648 blocks, which the XCDs share in contiguous ranges, in both orders of the sites
@pytest.mark.parametrize("planes", [0, 2])
@pytest.mark.parametrize("ns,nt", [(12, 28), (24, 6)])
@pytest.mark.parametrize("fmt,prec", FORMATS)
def test_wave_per_hop_work_orders(fmt, prec, ns, nt, planes):
    with abi.Context(ns, nt, theta_t=1.0) as ctx:
        g18 = ctx.gauge(seed=3, epsilon=0.35)
        gf = g18 if fmt == abi.GAUGE_F64_18 else g18.converted(fmt)
        a, b = ctx.spinor(prec), ctx.spinor(prec)
        a.upload(np.random.default_rng(7).standard_normal((ctx.veo, 24)))
        tmp = ctx.buffer(2 * ctx.lib.cl2_field_bytes(ctx.handle, abi.FIELD_SPINOR_EO, prec))
        results = []
        for block, zp in ((64, planes), (256, 0)):
            ctx.tune_set(b"hop.block", block)
            ctx.tune_set(b"hop.zplanes", zp)
            got = []
            for evenodd in (abi.EVEN, abi.ODD):
                ctx.dslash_eo(b.ptr, a.ptr, gf.ptr, fmt, evenodd, KAPPA)
                got.append(b.download())
            ctx.fermionmatrix_eo(abi.OP_QPLUSQMINUS_EO, b.ptr, a.ptr, gf.ptr, fmt, abi.ACTION_TWISTEDMASS, KAPPA, MUBAR,
                                 tmp.ptr)
            results.append(got + [b.download()])
        for x, y in zip(*results):
            assert np.array_equal(x, y)


def test_keys_set_by_hand_shape_only_their_launches():
    with abi.Context(8, 8, theta_t=1.0) as ctx:
        block = lambda: ctx.lib.cl2_tune_get(ctx.handle, b"hop.block.f64_18")
        assert block() == 64  # the wave-per-hop kernel of small lattices
        for key, value in ((b"mrhs.lds", 1), (b"mrhs.lds", 0), (b"mrhs.rb", 2), (b"hop.xcd", 1), (b"hop.zplanes", 2)):
            ctx.tune_set(key, value)
            assert block() == 64
        for key, value, expect in ((b"hop.block", 128, 128), (b"hop.block", 0, 64), (b"hop.occupancy", 1, 256),
                                   (b"hop.block", 64, 64), (b"hop.occupancy", -1, 64)):
            ctx.tune_set(key, value)
            assert block() == expect
        assert ctx.lib.cl2_tune_get(ctx.handle, b"hop.block") == 64
        with pytest.raises(abi.Cl2Error):
            ctx.tune_set(b"hop.block", 100)


def test_autotuner_times_the_default_kernel():
    # 8^4, FP64: the wave-per-hop kernel, which is the default there, takes 2/3 of the time of the next shape
    with abi.Context(8, 8, theta_t=1.0) as ctx:
        gf = ctx.gauge(seed=3, epsilon=0.35)
        out = [ctypes.c_int() for _ in range(5)]
        ms = ctypes.c_double()
        ctx.autotune_dslash(gf.ptr, abi.GAUGE_F64_18, 1, ctypes.byref(ms), *[ctypes.byref(o) for o in out])
        assert ctx.lib.cl2_tune_get(ctx.handle, b"hop.block.f64_18") == 64
        assert out[3].value == 512  # its threads
        ctx.tune_set(b"mrhs.lds", 2)  # another launch's key: the tuned shape stays
        assert ctx.lib.cl2_tune_get(ctx.handle, b"hop.block.f64_18") == 64


@pytest.mark.parametrize("ns,nt,blocks", [(14, 20, (64, 256, 64, 64)), (14, 22, (256, 256, 64, 64)),
                                          (16, 24, (256, 256, 64, 64)), (14, 40, (256,) * 4), (20, 40, (256,) * 4)])
def test_wave_per_hop_limits(ns, nt, blocks):
    # beyond them the kernel is slower where the device is full: one such limit per format
    with abi.Context(ns, nt) as ctx:
        got = tuple(ctx.lib.cl2_tune_get(ctx.handle, b"hop.block." + f) for f in (b"f64_18", b"f64_12", b"f32_12", b"f16_12"))
        assert got == blocks


@pytest.mark.parametrize("ns,nt,planes", [(16, 24, (0, 0)), (16, 64, (0, -1)), (20, 36, (0, -1)), (16, 96, (-1, -1)),
                                          (24, 8, (-1, -1)), (32, 4, (-1, -1))])
def test_site_order_limits(ns, nt, planes):
    # lexicographic order only where t-slices are small, whatever the number of sites
    with abi.Context(ns, nt) as ctx:
        assert tuple(ctx.lib.cl2_tune_get(ctx.handle, b"hop.zplanes." + f) for f in (b"f64_18", b"f64_12")) == planes


def test_single_field_autotuning_leaves_staggered_blocks_alone():
    # a 28^3 block has slabs of 7 planes and 14 rows: whole planes that the autotuner finds for one field must not replace them
    with abi.Context(28, 12, theta_t=1.0) as ctx:
        gf = ctx.gauge(seed=3, epsilon=0.35).converted(abi.GAUGE_F32_12)
        slab = lambda: ctx.lib.cl2_tune_get(ctx.handle, b"stagg.slab.f32_12.16")
        before = slab()
        assert 0 < before < 28 * 14
        ctx.autotune_dks(gf.ptr, abi.GAUGE_F32_12, None, None, None, None, None)
        assert slab() == before
        ctx.tune_set(b"hop.zplanes", 7)  # by hand: as set
        assert slab() == 0
