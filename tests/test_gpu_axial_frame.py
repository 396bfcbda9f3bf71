"""The axial frame the sweeps run in (u0_Z = 1 but on the plane z = ns - 1).

Haar-random links, so that the column products are general SU(3) matrices, on
the smallest extents and on timeslices that are no whole number of tiles or
waves: G and U after a few half-sweeps against the CPU oracle, which keeps
every link.  Rounding of G: a column product is projected onto SU(3) at each
step and enters G twice (G' = G h^dagger and back), a few 1e-16 each; the
bound of 1e-11 is that of the drop-in tests (1e-10) less a decade.  A fix
that needs no sweep leaves G = 1 exactly."""
import numpy as np
import pytest

import gfc
import oracle as orc
from test_gpu_u0_pivot import _haar_su3

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns,nt", [(2, 2), (2, 6), (4, 2), (6, 4), (10, 2), (18, 2)])
def test_frame_matches_oracle(ctx, ns, nt):
    geom = gfc.Geometry(ns, nt)
    V = geom.volume
    U = _haar_su3(np.random.default_rng(ns * 100 + nt), 4 * V).reshape(V, 4, 3, 3)
    k = 11  # past a reunitarization
    p = gfc.Params(tolerance=1e-300, estimate_sweeps_to_gf_progress=100000000,
                   max_sweeps_to_fix=k, sweeps_to_reunitarization=10)
    with gfc.Job(ctx, geom) as job:
        job.upload_config(U)
        assert job.reunitarize() == 0
        rc, rep, tr = job.fix(p, trace_len=k)
        G, Uf = job.download_gauge(), job.download_config()
    Uo, Go = U.copy(), np.zeros((V, 3, 3), np.complex128)
    orc.reunitarize(Uo)
    rc_o, tr_o = orc.gaugefix(Uo, Go, orc.geom(ns, nt),
                              orc.params(tolerance=1e-300, max_sweeps=k, estimate=100000000,
                                         reunit_every=10), trace_len=k)
    assert rc == rc_o == gfc.ENOTCONVERGED and rep.sweeps == k
    dG, dU = np.max(np.abs(G - Go)), np.max(np.abs(Uf - Uo))
    rel = np.max(np.abs(tr - tr_o) / tr_o)
    print(f"{ns}^3x{nt}: max|dG| {dG:.2e}, max|dU| {dU:.2e}, e2 rel {rel:.2e}")
    assert dG < 1e-11 and dU < 1e-11 and rel < 1e-12


@pytest.mark.parametrize("precision", [gfc.PREC_FP64, gfc.PREC_MIXED])
def test_no_sweep_leaves_identity(ctx, precision):
    geom = gfc.Geometry(6, 4)
    one = np.broadcast_to(np.eye(3, dtype=np.complex128), (geom.volume, 3, 3))
    U = gfc.generate_smooth(geom, 3, 0.3)
    bad = U.copy()
    bad[5, 2] = np.nan
    o = gfc.Options(precision=precision)
    with gfc.Job(ctx, geom, precision) as job:
        # a tolerance the input already meets, and a residue that is no number
        for cfg, tol in ((U, 1e6), (bad, 1e-16)):
            job.upload_config(cfg)
            rc, rep = job.fix(gfc.Params(tolerance=tol), o)
            assert rc == 0 and rep.sweeps == 0
            assert np.array_equal(job.download_gauge(), one)


@pytest.mark.parametrize("ns,nt", [(2, 2), (6, 4), (18, 2)])
def test_mixed_stopped_in_fp32(ctx, ns, nt):
    """A mixed fix that ends in its FP32 phase never enters the axial frame: G is
    the FP32 G projected in FP64 (SU(3), and U = G U0 G^dagger, to 1e-13) and
    within 20 sweeps of some 50 FP32 roundings each, 6e-8 * 1000, of the FP64 G."""
    geom = gfc.Geometry(ns, nt)
    U0 = gfc.generate_smooth(geom, 5, 0.3)
    p = gfc.Params(tolerance=1e-300, estimate_sweeps_to_gf_progress=100000000,
                   max_sweeps_to_fix=20)
    out = {}
    for prec in (gfc.PREC_FP64, gfc.PREC_MIXED):
        with gfc.Job(ctx, geom, precision=prec) as job:
            job.upload_config(U0)
            assert job.reunitarize() == 0
            rc, rep = job.fix(p, gfc.Options(precision=prec))[:2]
            assert rc == gfc.ENOTCONVERGED and rep.sweeps == 20
            out[prec] = job.download_gauge(), job.download_config()
    assert rep.sweeps_fp32 == 20
    G, U = out[gfc.PREC_MIXED]
    Gt, Ut = G.reshape(nt, ns, ns, ns, 3, 3), U.reshape(nt, ns, ns, ns, 4, 3, 3)
    dag = lambda m: np.conj(np.swapaxes(m, -1, -2))  # noqa: E731
    assert np.abs(G @ dag(G) - np.eye(3)).max() < 1e-13
    V0 = U0.copy()
    orc.reunitarize(V0)
    V0 = V0.reshape(Ut.shape)
    for mu in range(4):
        assert np.abs(Ut[..., mu, :, :] - Gt @ V0[..., mu, :, :]
                      @ dag(np.roll(Gt, -1, axis=mu))).max() < 1e-13
    assert np.abs(G - out[gfc.PREC_FP64][0]).max() < 1000 * 6e-8


@pytest.mark.parametrize("route", [dict(), dict(slice_group=-1), dict(trace_len=240)])
@pytest.mark.parametrize("ns,nt", [(8, 6), (14, 4)])
def test_drift_off_su3_is_bounded(ctx, ns, nt, route):
    """With rare reunitarizations (R = 1000) the frame still projects G every 50
    half-sweeps, in which a site is updated 25 times at most.  An update biases a
    row's norm by a unit roundoff at most, its square by 2 * 1.1e-16: 5.5e-15 in
    all, and row 2, the product of two, by twice that.  (Not projected, row 1 is
    off by 9e-15 and row 2 by 14e-15 after 240, with one hit and omega 1.7.)  All
    routes keep the same bits."""
    geom = gfc.Geometry(ns, nt)
    p = gfc.Params(tolerance=1e-300, estimate_sweeps_to_gf_progress=100000000,
                   max_sweeps_to_fix=240, sweeps_to_reunitarization=1000, omega_OR=1.7, hits=1)
    out = []
    for r in (dict(), route):
        trace_len = r.get("trace_len", 0)
        o = gfc.Options(**{k: v for k, v in r.items() if k != "trace_len"})
        with gfc.Job(ctx, geom) as job:
            job.generate_smooth(7, 0.3)
            job.reunitarize()
            assert job.fix(p, o, trace_len=trace_len)[0] == gfc.ENOTCONVERGED
            out.append(job.download_gauge())
    assert np.array_equal(out[0], out[1])
    norms = (np.abs(out[0].astype(np.clongdouble)) ** 2).sum(-1).mean(0) - 1
    print(norms)
    assert np.all(np.abs(norms) < [5.5e-15, 5.5e-15, 1.1e-14])
