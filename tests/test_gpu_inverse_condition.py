"""adga_inverse_matrix_z on matrices of every condition, on both sides of its one-launch kernel's largest size (64)
and over the blocked elimination's panels: X A and A X are the identity to what an LU leaves.

Bound: the rounding errors of a backward-stable inversion add up over inner products of n terms of size cond eps, at
random: |1 - X A|, |1 - A X| < sqrt(n) cond eps, and never less than 16 sqrt(n) eps, for matrices whose singular
values fall evenly from 1 to 1/cond."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = 2.220446049250313e-16


def _matrix(n, cond, seed):
    r = np.random.default_rng([n, seed])
    u, v = (np.linalg.qr(r.normal(size=(n, n)) + 1j * r.normal(size=(n, n)))[0] for _ in range(2))
    return (u * np.logspace(0, -np.log10(cond), n)) @ v


@pytest.mark.parametrize("n", [33, 64, 65, 80, 81, 100, 131, 300, 513, 1025, 1080])
def test_gpu_inverse_residual_of_both_sides(n):
    from adga_amd import api
    for cond in (1.0, 1e2, 1e4, 1e6, 1e8, 1e11, 1e13):
        for seed in range(3 if n < 200 else 1):
            a = _matrix(n, cond, seed)
            print(f"inverse n={n} condition {cond:.0e}", flush=True)
            x, ierr = api.inverse_matrix(a)
            assert ierr == 0
            for name, p in (("X A", x @ a), ("A X", a @ x)):
                err = np.abs(p - np.eye(n)).max()
                assert err < np.sqrt(n) * EPS * max(cond, 16.0), (name, cond, seed, err)
