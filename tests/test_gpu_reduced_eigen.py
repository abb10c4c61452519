"""The reduced-space eigensolver at the edges of its wavefront layout (64 rows per
register, half a wavefront of remaining rows) and with multiplets, whose vectors
one wavefront makes one after another.  Oracle: numpy; bounds as for the solver's
other tests (1e-11 of the largest root, residuals 1e-10 of the largest entry)."""
import numpy as np
import pytest

from et_amd import ccsd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('k,n_want,multiplet', [(4, 4, 3), (33, 8, 3), (34, 5, 2), (63, 9, 4), (64, 64, 3), (65, 12, 5),
                                                (100, 7, 2), (128, 128, 3)])
def test_multiplets_and_layout_edges(k, n_want, multiplet):
    rng = np.random.default_rng(k)
    vals = np.sort(rng.uniform(0.2, 3.0, k))
    vals[1:1 + multiplet] = vals[1]                      # one multiplet among the wanted roots
    Q = np.linalg.qr(rng.normal(size=(k, k)))[0]
    G = (Q * vals) @ Q.T
    print(f'reduced eigen k={k} n_want={n_want} multiplet={multiplet}', flush=True)
    wr, wi, X = ccsd.reduced_eigen(G, n_want)
    assert np.abs(wr - np.sort(vals)).max() < 1e-11 * vals.max()
    assert np.abs(G @ X - X * vals[:n_want]).max() < 1e-10 * np.abs(G).max()
    assert np.abs(np.linalg.norm(X, axis=0) - 1.0).max() < 1e-12
    group = X[:, 1:1 + min(multiplet, n_want - 1)]
    assert np.abs(group.T @ group - np.eye(group.shape[1])).max() < 1e-6


@pytest.mark.parametrize('k,at', [(6, 0), (33, 1), (65, 2), (128, 4)])
def test_pairs_between_real_roots(k, at):
    """Complex pairs (one workgroup) beside real roots (one each), the last pair cut
    by the number of wanted roots."""
    rng = np.random.default_rng(100 + k)
    B = np.diag(np.sort(rng.uniform(0.2, 3.0, k)))
    for j in (at, at + 3):
        B[j, j] = B[j + 1, j + 1]
        B[j, j + 1], B[j + 1, j] = 0.05, -0.05
    S = np.eye(k) + 0.1 * rng.normal(size=(k, k)) / np.sqrt(k)
    G = S @ B @ np.linalg.inv(S)
    ref = np.linalg.eigvals(G)
    ref = ref[np.lexsort((ref.imag, np.round(ref.real, 9)))]
    n_want = at + 4
    print(f'reduced eigen pairs k={k} n_want={n_want}', flush=True)
    wr, wi, X = ccsd.reduced_eigen(G, n_want)
    assert np.abs(np.sort(wr) - np.sort(ref.real)).max() < 1e-10 * np.abs(ref).max()
    j = 0
    while j < n_want:
        if wi[j] == 0.0:
            assert np.linalg.norm(G @ X[:, j] - wr[j] * X[:, j]) < 1e-10 * np.abs(G).max()
            j += 1
            continue
        assert wi[j] < 0.0
        if j + 1 < n_want:
            z = X[:, j] + 1j * X[:, j + 1]
            assert np.linalg.norm(G @ z - (wr[j] - 1j * wi[j]) * z) < 1e-10 * np.abs(G).max() * np.linalg.norm(z)
        j += 2
