"""Residues and plaquettes of a configuration, whose kernels take 64 sites at a
time through LDS (one such group per workgroup up to 2^18 sites, four above):
sizes below one group, with a ragged last group, and on both sides of the line
between the two splits, on links that are no SU(3) matrices, against a plain
numpy evaluation.  Both sum V terms of order 1 in FP64: 1e-13 relative to the
sum of their magnitudes."""
import numpy as np
import pytest

import gfc

pytestmark = pytest.mark.gpu


def _shift(a, mu):
    """a(n + mu) for a of shape (t, z, y, x, ...)."""
    return np.roll(a, -1, axis=mu)


def _reference(U, ns, nt):
    V = ns ** 3 * nt
    U = U.reshape(nt, ns, ns, ns, 4, 3, 3)
    dag = lambda m: np.conj(np.swapaxes(m, -1, -2))  # noqa: E731
    D = 0
    F = 0.0
    for mu in (1, 2, 3):
        E = U[..., mu, :, :] - dag(U[..., mu, :, :])
        D = D + E - np.roll(E, 1, axis=mu)
        F += np.trace(U[..., mu, :, :], axis1=-2, axis2=-1).real.sum()
    D = D - np.trace(D, axis1=-2, axis2=-1)[..., None, None] / 3 * np.eye(3)
    A = -0.5j * D
    theta = (np.abs(A) ** 2).sum() / (3 * V)
    # sum_a c_a^2 = 2 Re Tr(A A^dagger) for a traceless Hermitian A
    e2 = 2 * (np.abs(A) ** 2).sum() / V
    plaq = []
    for planes in (((3, 2), (3, 1), (2, 1)), ((0, 1), (0, 2), (0, 3))):
        s = 0.0
        for m, n in planes:
            a = U[..., m, :, :] @ _shift(U[..., n, :, :], m)
            b = U[..., n, :, :] @ _shift(U[..., m, :, :], n)
            s += (a * b.conj()).sum().real / 3
        plaq.append(s / (3 * V))
    return (e2, theta, F / (9 * V)), plaq


@pytest.mark.parametrize("ns,nt", [(2, 2), (2, 6), (4, 2), (6, 2), (10, 4), (16, 64), (16, 66),
                                   # above 2^18 sites: a last group of 48 sites; two
                                   # of the last workgroup's four groups empty
                                   (18, 46), (26, 16)])
def test_against_numpy(ctx, ns, nt):
    geom = gfc.Geometry(ns, nt)
    rng = np.random.default_rng(ns * 1000 + nt)
    U = rng.standard_normal((geom.volume, 4, 3, 3, 2)).view(np.complex128)[..., 0]
    with gfc.Job(ctx, geom) as job:
        job.upload_config(U)
        obs, plaq = job.observables(), job.plaquette()
    ref, rplaq = _reference(U, ns, nt)
    print(obs, ref, plaq, rplaq)
    assert abs(obs[0] / ref[0] - 1) < 1e-13 and abs(obs[1] / ref[1] - 1) < 1e-13
    # terms of either sign: a trace has a magnitude of about 2, a plaquette of 30
    assert abs(obs[2] - ref[2]) < 1e-13 * 2
    assert np.all(np.abs(np.array(plaq) - rplaq) < 1e-13 * 30)
