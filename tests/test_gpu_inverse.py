"""adga_inverse_matrix_z over its kernels' ranges: one workgroup up to n = 64 (one to four waves, full and partial
ones), the blocked elimination up to 1536 (every panel shape, block remainders 0, 1 and 15), the LU above; well
and badly conditioned matrices, matrices that pivot in every column, and singular ones.

Bounds: the relative error of an inverse is a modest multiple of cond eps; 50 n eps cond in the max norm covers the
growth of partial pivoting on random matrices by orders of magnitude, where a wrong row or column leaves O(1)."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu
SIZES = [1, 2, 3, 15, 16, 17, 31, 33, 40, 48, 49, 63, 64, 65, 79, 80, 81, 127, 128, 129, 256, 257, 271, 511, 513, 540,
         1024, 1025, 1080, 1535, 1536, 1537]


def _matrix(n, kind, seed=0):
    r = np.random.default_rng([n, seed])
    g = r.normal(size=(n, n)) + 1j * r.normal(size=(n, n))
    if kind == "bse":
        return np.eye(n) + 0.35 / np.sqrt(n) * g
    if kind == "random":
        return g
    # the largest entry of every column far from the diagonal: every column pivots
    return 0.1 * g / np.sqrt(n) + np.roll(np.eye(n), n // 2 + 1, axis=0) * (2 + r.random(n))


@pytest.mark.parametrize("n", SIZES)
def test_gpu_inverse_sizes(n):
    from adga_amd import api
    for kind in ("bse", "random", "pivot"):
        a = _matrix(n, kind)
        print(f"inverse n={n} {kind}", flush=True)
        x, ierr = api.inverse_matrix(a)
        assert ierr == 0
        ref = np.linalg.inv(a)
        bound = 50 * n * 2.2e-16 * np.linalg.norm(a, 2) * np.linalg.norm(ref, 2)
        assert rel_err(x, ref) < bound, (kind, rel_err(x, ref), bound)


@pytest.mark.parametrize("n", [40, 100, 600])
def test_gpu_inverse_badly_conditioned(n):
    from adga_amd import api
    u, _, v = np.linalg.svd(_matrix(n, "random"))
    a = (u * np.logspace(0, -7, n)) @ v
    print(f"inverse n={n} condition 1e7", flush=True)
    x, _ = api.inverse_matrix(a)
    assert rel_err(x, np.linalg.inv(a)) < 50 * n * 2.2e-16 * 1e7


@pytest.mark.parametrize("n", [5, 40, 64, 65, 200, 540])
def test_gpu_inverse_singular(n):
    """A zero column, the identity without its last entry and a NaN column: an error, the matrix left as it is."""
    import ctypes as C
    from adga_amd import _lib
    r = np.random.default_rng(n)
    col = n // 2
    zero = r.normal(size=(n, n)) + 0j
    zero[:, col] = 0
    ident = np.eye(n, dtype=complex)
    ident[:, n - 1] = 0
    nan = r.normal(size=(n, n)) + 0j
    nan[:, 0] = np.nan
    for name, a in (("zero column", zero), ("zero last column", ident), ("nan", nan)):
        m = np.asfortranarray(a)
        ierr = C.c_int(0)
        print(f"singular n={n} {name}", flush=True)
        rc = _lib.lib.adga_inverse_matrix_z(n, m.ctypes.data_as(_lib._dp), C.byref(ierr))
        assert rc == _lib.ADGA_E_SINGULAR and 1 <= ierr.value <= n, (name, rc, ierr.value)
        assert np.array_equal(m, a, equal_nan=True)
