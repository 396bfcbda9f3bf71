"""Kernels that take 256 AoS links at a time through LDS, at the edges of such a
block: the projection onto SU(3) (one matrix to a few blocks, a ragged last one,
a null row in its last matrix) and U = G U0 G(n+mu)^dagger on lattices of fewer
links than a block and of 13.5 blocks.  Gram-Schmidt of matrices within 0.3 of
SU(3) and three products of such: some 20 roundings of 1.1e-16 on entries of at
most 1, so 1e-14."""
import numpy as np
import pytest

import gfc

pytestmark = pytest.mark.gpu


def _noisy(rng, n):
    q, _ = np.linalg.qr(rng.normal(size=(n, 3, 3)) + 1j * rng.normal(size=(n, 3, 3)))
    return q + 0.05 * (rng.normal(size=(n, 3, 3)) + 1j * rng.normal(size=(n, 3, 3)))


def _project(m):
    r0 = m[:, 0] / np.linalg.norm(m[:, 0], axis=-1, keepdims=True)
    r1 = m[:, 1] - (r0.conj() * m[:, 1]).sum(-1, keepdims=True) * r0
    r1 = r1 / np.linalg.norm(r1, axis=-1, keepdims=True)
    return np.stack([r0, r1, np.cross(r0.conj(), r1.conj())], axis=1)


@pytest.mark.parametrize("n", (1, 2, 63, 64, 65, 255, 256, 257, 511, 513, 5000))
def test_projection_blocks(ctx, n):
    m = _noisy(np.random.default_rng(n), n)
    out = m.copy()
    assert gfc.reunitarize_field(ctx, out) == 0
    assert np.abs(out - _project(m)).max() < 1e-14
    bad = m.copy()
    bad[-1, 0] = 0
    assert gfc.reunitarize_field(ctx, bad) == gfc.EPROJECT
    assert np.array_equal(bad[:-1], out[:-1])


@pytest.mark.parametrize("ns,nt", ((2, 2), (2, 4), (6, 4), (10, 2)))
def test_transformed_links(ctx, ns, nt):
    geom = gfc.Geometry(ns, nt)
    U0 = _project(_noisy(np.random.default_rng(ns * 100 + nt), geom.volume * 4))
    with gfc.Job(ctx, geom) as job:
        job.upload_config(U0.reshape(geom.volume, 4, 3, 3))
        job.fix(gfc.Params(tolerance=1e-300, max_sweeps_to_fix=7))
        G, U = job.download_gauge(), job.download_config()
    G = G.reshape(nt, ns, ns, ns, 3, 3)
    U = U.reshape(nt, ns, ns, ns, 4, 3, 3)
    u0 = U0.reshape(U.shape)
    for mu in range(4):
        up = np.conj(np.swapaxes(np.roll(G, -1, axis=mu), -1, -2))
        assert np.abs(U[..., mu, :, :] - G @ u0[..., mu, :, :] @ up).max() < 1e-14
