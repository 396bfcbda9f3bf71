"""Small lattices in FP64 (ns <= 10): all sweeps between two host decisions in
one launch, a workgroup per timeslice with its G in LDS.  The result must equal
whole-lattice sweeps bit for bit: timeslices smaller than a wave, ones that
fill a workgroup exactly (ns = 8) or not (ns = 10), any reunitarization period
and hits, odd sweep counts (either parity last), more sweeps than one launch
takes (some 2400), and checks that fall on reunitarization points."""
import numpy as np
import pytest

import gfc

pytestmark = pytest.mark.gpu


def _both(ctx, geom, p):
    with gfc.Job(ctx, geom) as job:
        job.generate_smooth(geom.ns, 0.3)
        job.reunitarize()
        job.save_config()
        out = []
        for grp in (-1, 0):
            job.restore_config()
            rc, rep = job.fix(p, gfc.Options(slice_group=grp))
            out.append((rc, rep.sweeps, rep.residue_final, job.download_gauge(),
                        job.download_config()))
    a, b = out
    assert a[:3] == b[:3]
    assert np.array_equal(a[3], b[3]) and np.array_equal(a[4], b[4])
    return a


@pytest.mark.parametrize("ns,nt", [(2, 2), (4, 6), (6, 2), (8, 4), (10, 6), (10, 260)])
@pytest.mark.parametrize("R,hits,n", [(1, 2, 7), (3, 1, 30), (10, 3, 41), (250, 0, 12)])
def test_slices_equal_whole_lattice(ctx, ns, nt, R, hits, n):
    rc, sweeps, *_ = _both(ctx, gfc.Geometry(ns, nt),
                           gfc.Params(tolerance=1e-300, estimate_sweeps_to_gf_progress=100000000,
                                      max_sweeps_to_fix=n, sweeps_to_reunitarization=R,
                                      hits=hits))
    assert rc == gfc.ENOTCONVERGED and sweeps == n


@pytest.mark.parametrize("R", [1, 7, 2000])
def test_more_sweeps_than_a_launch(ctx, R):
    rc, sweeps, *_ = _both(ctx, gfc.Geometry(4, 4),
                           gfc.Params(tolerance=1e-300, estimate_sweeps_to_gf_progress=100000000,
                                      max_sweeps_to_fix=4003, sweeps_to_reunitarization=R))
    assert sweeps == 4003


@pytest.mark.parametrize("proxy", [gfc.PROXY_E2, gfc.PROXY_THETA])
def test_to_tolerance_with_dense_checks(ctx, proxy):
    rc, *_ = _both(ctx, gfc.Geometry(8, 6),
                   gfc.Params(tolerance=1e-14, estimate_sweeps_to_gf_progress=0, gfix_proxy=proxy,
                              sweeps_to_reunitarization=10))
    assert rc > 0


@pytest.mark.parametrize("ns,nt", [(2, 256), (4, 300), (6, 258), (8, 300), (10, 132), (10, 256)])
@pytest.mark.parametrize("hits", [2, 8])
def test_both_sides_of_the_rule(ctx, ns, nt, hits):
    """More timeslices than CUs and the edges of what runs in one launch."""
    _both(ctx, gfc.Geometry(ns, nt),
          gfc.Params(tolerance=1e-300, estimate_sweeps_to_gf_progress=100000000,
                     max_sweeps_to_fix=23, sweeps_to_reunitarization=10, hits=hits))
