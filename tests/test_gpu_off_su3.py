"""Links that are not matrices of SU(3) and have not been reunitarized: the
sweeps take each for itself, by its first two rows, whatever it is.

Where only the third rows are wrong, that is the clean configuration, so G must
be the CPU oracle's on the clean links (1e-11, as in the axial frame's test) in
whole-lattice and grouped sweeps, with a trace and with retired timeslices, and a
mixed fix that of the clean links.  A link without its second and third row must
stay a matter of the sites next to it."""
import numpy as np
import pytest

import gfc
import oracle as orc
from test_gpu_u0_pivot import _haar_su3

pytestmark = pytest.mark.gpu


def _links(ns, nt):
    V = ns ** 3 * nt
    U = _haar_su3(np.random.default_rng(ns * 100 + nt), 4 * V).reshape(V, 4, 3, 3)
    orc.reunitarize(U)
    return U


def _params(k, **kw):
    return gfc.Params(tolerance=1e-300, estimate_sweeps_to_gf_progress=100000000,
                      max_sweeps_to_fix=k, sweeps_to_reunitarization=10, **kw)


def _fix(ctx, U, ns, nt, p, precision=gfc.PREC_FP64, trace_len=0, **opts):
    with gfc.Job(ctx, gfc.Geometry(ns, nt), precision) as job:
        job.upload_config(U)
        out = job.fix(p, gfc.Options(precision=precision, **opts), trace_len=trace_len)
        return out[0], out[1], job.download_gauge()


@pytest.mark.parametrize("ns,nt,trace,opts", [
    (2, 2, 0, {}), (6, 4, 0, {}), (6, 4, 45, {}), (10, 2, 0, dict(slice_group=-1)),
    (8, 6, 0, dict(slice_group=2)), (8, 4, 0, dict(retire_slices=1)),
    (8, 4, 45, dict(retire_slices=1))])
def test_third_rows_are_not_read(ctx, ns, nt, trace, opts):
    U = _links(ns, nt)
    k = 45
    G = np.zeros((ns ** 3 * nt, 3, 3), np.complex128)
    orc.gaugefix(U.copy(), G, orc.geom(ns, nt),
                 orc.params(tolerance=1e-300, max_sweeps=k, estimate=100000000, reunit_every=10))
    bad = U.copy()
    bad[::3, :, 2] = 7.0
    bad[1, 1:, 2] *= np.exp(0.1j)  # determinant not 1
    rc, rep, Gb = _fix(ctx, bad, ns, nt, _params(k), trace_len=trace, **opts)
    assert rc == gfc.ENOTCONVERGED and rep.sweeps == k
    assert np.abs(Gb - G).max() < 1e-11


def test_third_rows_in_a_mixed_fix(ctx):
    ns, nt = 8, 4
    U = gfc.generate_smooth(gfc.Geometry(ns, nt), 3, 0.3)
    orc.reunitarize(U)
    bad = U.copy()
    bad[5::7, :, 2] = 0.25
    p = gfc.Params(tolerance=1e-14)
    rc, rep, G = _fix(ctx, U, ns, nt, p, gfc.PREC_MIXED)
    rcb, repb, Gb = _fix(ctx, bad, ns, nt, p, gfc.PREC_MIXED)
    assert rc == rcb > 0 and rep.sweeps_fp32 == repb.sweeps_fp32 < rc
    # the same FP32 sweeps; the FP64 ones differ by their rounding
    assert np.abs(Gb - G).max() < 1e-11


@pytest.mark.parametrize("precision", [gfc.PREC_FP64, gfc.PREC_MIXED])
@pytest.mark.parametrize("mu", [1, 2, 3])
def test_null_rows_stay_local(ctx, mu, precision):
    """After one half-sweep G differs from the clean configuration's at the end
    of the link that was swept, and nowhere else."""
    ns, nt = 6, 2
    U = _links(ns, nt)
    bad = U.copy()
    site = 2 * (ns * ns + ns + 1)  # z, y, x = 2, 2, 2 of the first timeslice
    bad[site, mu, 1:] = 0
    G, Gb = (_fix(ctx, u, ns, nt, _params(1), precision)[2] for u in (U, bad))
    far = np.abs(Gb - G).max(axis=(1, 2)) > (1e-12 if precision == gfc.PREC_FP64 else 1e-5)
    assert list(np.nonzero(far)[0]) == [site]
    assert np.isfinite(Gb).all()


def test_links_rounded_to_fp32_stay_in_the_axial_frame(ctx):
    """A configuration stored in FP32 is near enough: G is that of its links
    projected first, to a few times what the rounding is (6e-8 per number)."""
    ns, nt = 8, 4
    U = _links(ns, nt).astype(np.complex64).astype(np.complex128)
    V = U.copy()
    orc.reunitarize(V)
    G, Gp = (_fix(ctx, u, ns, nt, _params(20))[2] for u in (U, V))
    assert np.abs(G - Gp).max() < 1e-5
