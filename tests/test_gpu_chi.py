"""The contraction of chi and bubble_nl on the matrix cores (three orbitals and more) and its derivative form.

* Forward against the numpy oracle at the repository's 1e-10: every orbital count it takes, one slice of
  frequencies and several uneven ones, steps of four that end inside a slice.
* Derivatives against four-point differences of the GPU's own forward pass along a direction of random inputs
  (step 1e-3 of directions that move C and G by a few at most: an h^4 term below 1e-8 and a round-off below 1e-7 relative, as for the
  other derivative tests, so 1e-6)."""
import dataclasses
import types

import numpy as np
import pytest

from conftest import rel_err
from adga_amd import synth

pytestmark = pytest.mark.gpu


def _workload(n, nk, iwf, noise=1e-2):
    model, par = {3: ("t2g", dict(U=5.0, J=0.75, t=-0.26, tp=-0.08))}.get(
        n, ("rand5", dict(U=4.0, J=0.6, t=0.15)))
    return synth.Workload("chi", n, nk, iwf, 1, 10.0, model=model, seed=7, noise=noise, **par)


# (orbitals, k grid, half box): 2 iwf / 8 slices of frequencies for few points
@pytest.mark.parametrize("n,nk,iwf", [(3, (3, 3, 2), 1), (3, (3, 3, 2), 7), (3, (3, 3, 2), 8), (3, (3, 2, 2), 29),
                                      (4, (3, 2, 2), 9), (4, (2, 2, 2), 1), (5, (2, 2, 2), 1), (5, (2, 2, 2), 13)])
def test_gpu_chi_contraction(n, nk, iwf):
    import adga_oracle
    from adga_amd import api
    inp = synth.build_inputs(_workload(n, nk, iwf))
    pts = [(1, q) for q in range(min(5, inp.wl.nqp))]
    cl = lambda w, c: synth.chi_loc(inp, w, c)  # noqa: E731
    ref = adga_oracle.HotPath(inp).run(pts, cl)
    print(f"n={n} N={inp.wl.maxdim}", flush=True)
    with api.Context(inp) as ctx:
        out = api.run_loop(ctx, pts, cl, "fp64")
    for k in ("chi_d", "chi_m", "bubble_nl"):
        assert rel_err(out[k], ref[k]) < 1e-10, (k, rel_err(out[k], ref[k]))


@pytest.mark.parametrize("n,nk,iwf", [(3, (2, 2, 2), 1), (3, (3, 2, 2), 13), (4, (2, 2, 2), 5), (5, (2, 2, 2), 9)])
def test_gpu_chi_contraction_derivative(n, nk, iwf):
    from adga_amd import api
    inp = synth.build_inputs(_workload(n, nk, iwf))
    rng = np.random.default_rng(3)

    def rnd(a):
        return rng.normal(size=a.shape) + 1j * rng.normal(size=a.shape)

    scale = {"hk": 0.05, "siw": 0.05, "giw": 0.01}
    d = {k: s * rnd(getattr(inp, k)) for k, s in scale.items()}
    dx = {c: 1e-3 * rnd(synth.chi_loc(inp, 1, c)) for c in ("dens", "magn")}
    iq = np.arange(1, inp.wl.nqp + 1)

    def forward(h):
        p = dataclasses.replace(inp, mu=inp.mu + 0.05 * h, **{k: getattr(inp, k) + h * v for k, v in d.items()})
        with api.Context(p) as ctx:
            ctx.set_local_omega(1, *(synth.chi_loc(inp, 1, c) + h * dx[c] for c in ("dens", "magn")))
            return ctx.run_points(iq, "fp64")

    tan = types.SimpleNamespace(dhk=d["hk"][..., None], dsiw=d["siw"][..., None], dgiw=d["giw"][..., None],
                                dmu=np.array([0.05]), du=np.zeros(inp.u.shape + (1,)),
                                du_tilde=np.zeros(inp.u_tilde.shape + (1,)))
    print(f"derivative n={n} N={inp.wl.maxdim}", flush=True)
    with api.Context(inp) as ctx:
        ctx.set_tangents(tan)
        ctx.set_local_omega(1, synth.chi_loc(inp, 1, "dens"), synth.chi_loc(inp, 1, "magn"))
        ctx.set_local_omega_tangent(dx["dens"][..., None], dx["magn"][..., None])
        out = ctx.run_points_tangent(iq)
    f = {s: forward(s * 1e-3) for s in (1, -1, 2, -2)}
    for k in ("chi_d", "chi_m", "bubble_nl"):
        fd = (8 * (f[1][k] - f[-1][k]) - (f[2][k] - f[-2][k])) / 12e-3
        assert rel_err(out["d" + k][..., 0], fd) < 1e-6, (k, rel_err(out["d" + k][..., 0], fd))
