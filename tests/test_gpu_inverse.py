"""tg_inverse at the edges of its kernels: panels of 16 (order <= 64, matrix in LDS) and
of 32 columns (two halves; last panel of 1, 15, 16, 17, 31, 32), 1, 2 or 3 row blocks a
wave, windows of 96 and 256 columns, and the batch sizes at which the launch changes.

With eps = 2^-52, Gauss-Jordan with partial pivoting leaves residuals of the order of
n eps |A| |X| (1-norms); 8 n eps |A| |X| bounds them with the growth of random matrices,
and the determinant's relative error by the same number."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -52


def check(A, X, det):
    n = A.shape[0]
    bound = 8 * n * EPS * np.linalg.norm(A, 1) * np.linalg.norm(X, 1)
    assert np.max(np.abs(A @ X - np.eye(n))) < bound, n
    sign, logdet = np.linalg.slogdet(A)
    assert abs(det / (sign * np.exp(logdet)) - 1) < bound, n


@pytest.mark.parametrize("n,count", [
    (1, 3), (2, 3), (15, 3), (16, 3), (17, 3), (33, 3), (48, 600), (49, 3), (49, 513), (63, 512),
    (64, 3), (65, 3), (65, 257), (80, 256), (81, 3), (96, 257), (97, 3), (127, 257), (128, 3),
    (128, 300), (129, 3), (144, 2), (145, 2), (255, 2), (256, 2), (257, 2), (289, 2), (320, 2),
    (353, 2), (383, 2), (384, 2), (385, 2)])
def test_inverse_at_kernel_edges(n, count):
    from taurus_vap_amd import gpu
    rng = np.random.default_rng(n)
    A = (rng.normal(size=(count, n, n)) + 1j * rng.normal(size=(count, n, n))) / np.sqrt(2.0 * n)
    X, det, info = gpu.inverse(A.copy())     # order 1 is inverted in place
    assert np.all(info == 0)
    for k in sorted({0, 1 % count, count // 2, count - 1}):
        check(A[k], X[k], det[k])
    # a permutation times signs: every pivot search ties with zeros, all steps exact
    p = rng.permutation(n)
    P = np.zeros((n, n), complex)
    P[np.arange(n), p] = rng.choice([1, -1, 1j, -1j], size=n)
    X, det, info = gpu.inverse(P)
    assert info == 0 and np.array_equal(X, P.conj().T) and np.allclose(det, np.linalg.det(P), atol=1e-9)
    # equal magnitudes everywhere: the candidates differ by their position alone
    if n > 2:
        E = rng.choice([1.0, -1.0], size=(n, n)) + 0j
        X, det, info = gpu.inverse(E / np.sqrt(n))
        if info == 0:
            check(E / np.sqrt(n), X, det)
    # the first vanishing column is reported, one-based
    for z in sorted({0, n // 2, n - 1}):
        S = A[0].copy()
        S[:, z:] = S[:, z:] * (np.arange(z, n) != z)
        _, det, info = gpu.inverse(S)
        assert info == z + 1 and det == 0, (n, z, info)
