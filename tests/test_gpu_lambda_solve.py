"""The lambda solve's end states and counts on the device against the oracle's Brent root: targets
that need the bracket to grow, more evaluations than are queued at once, an iteration limit, a target no lambda
reaches (f > 0 at every lambda tried: a non-positive target), a non-finite susceptibility; and again on the same
handle.  The iteration ends at |S - target| <= 1e-14 max(1, target), so lambda is good to 1e-14 / target of itself
for S about 1 / lambda: 1e-11 from a target of 1e-3 on."""
import numpy as np
import pytest

from adga_amd import synth  # noqa: F401
import adga_oracle as O

pytestmark = pytest.mark.gpu


def _handle(api, npq=257, nw=3, seed=0):
    r = np.random.default_rng(seed)
    v = 0.2 + r.random(npq * nw)
    chi = np.asfortranarray(v.astype(np.complex128).reshape(1, 1, -1))
    loc = np.asfortranarray(np.full((1, 1, nw), 0.5, dtype=np.complex128))
    return api.Lambda(chi, loc, 5.0, npq), v


@pytest.mark.parametrize("target", [2e-3, 0.05, 0.3, 3.0, 400.0])
def test_gpu_lambda_solve_targets(target):
    from adga_amd import api
    h, v = _handle(api)
    with h as lam:
        for _ in range(2):
            x, it = lam.solve(target=target)
            ex = O.lambda_solve(v.astype(complex), 5.0, 257, target, chi0=v[257:514])
            assert abs(x - ex) <= 1e-11 * max(1.0, abs(ex)), (x, ex, it)


def test_gpu_lambda_solve_refusals():
    from adga_amd import api
    h, _ = _handle(api)
    with h as lam:
        for kw in ({"target": 400.0, "maxit": 1}, {"target": 0.0}, {"target": -1.0}):
            with pytest.raises(api.AdgaError) as e:
                lam.solve(**kw)
            assert e.value.code == 4, (kw, e.value.code)
        x, _ = lam.solve(target=0.3)
        assert np.isfinite(x)
