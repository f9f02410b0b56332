"""The numpy divide and conquer that the solver's eigenvector signs are held against."""
import numpy as np
import pytest

from tests.stedc_model import stedc, tridiagonal


@pytest.mark.parametrize("n", [1, 2, 3, 16, 40, 130])
@pytest.mark.parametrize("kind", ["gaussian", "decoupled", "weak"])
def test_model_is_an_eigen_decomposition(kind, n):
    d, e = tridiagonal(kind, n, np.random.default_rng(n))
    T = np.diag(d) + np.diag(e, 1) + np.diag(e, -1)
    w, Z = stedc(d, e)
    nrm = np.abs(T).max()
    assert np.abs(w - np.linalg.eigvalsh(T)).max() <= 1e-13 * nrm * np.sqrt(n)
    assert np.abs(T @ Z - Z * w).max() <= 1e-13 * nrm * np.sqrt(n)
    assert np.abs(Z.T @ Z - np.eye(n)).max() <= 1e-13 * np.sqrt(n)


def test_model_signs_of_two_rows():
    # one merge of two rows, v = [1; sign(e)]: both vectors have v^T x < 0
    for e in (0.5, -0.5):
        w, Z = stedc([0.3, -0.2], [e])
        assert np.all(np.array([1.0, np.sign(e)]) @ Z < 0)
    # uncoupled rows keep the sign of a single row
    w, Z = stedc([0.3, -0.2], [0.0])
    assert np.array_equal(Z, [[0.0, 1.0], [1.0, 0.0]])
