"""The half of gamma^q and m_tot that the EOM reads (nu >= 0) against the numpy oracle's full sums: halves
n^2 iwf one below, at and above the residual product's 32-row tiles, smaller than one tile, every orbital count,
with the EOM by k-grid convolution and as direct sums, with V(q), and with the EOM off.

Bound: the repository's 1e-10 against the oracle."""
import numpy as np
import pytest

from conftest import rel_err
from adga_amd import synth

pytestmark = pytest.mark.gpu

# (orbitals, k grid, half box, points): the first row the EOM reads is n^2 iwf
SIZES = [(1, (2, 2, 2), 1, 3), (1, (4, 4, 4), 31, 6), (1, (4, 4, 4), 32, 6), (1, (4, 4, 4), 33, 6), (2, (3, 3, 3), 17, 9),
         (3, (3, 3, 2), 7, 7), (4, (3, 2, 2), 2, 5), (5, (2, 2, 3), 1, 3), (5, (3, 2, 2), 3, 4)]


@pytest.mark.parametrize("vq", [0.0, 0.4])
@pytest.mark.parametrize("n,nk,iwf,npts", SIZES)
def test_gpu_eom_half(n, nk, iwf, npts, vq):
    import adga_oracle
    from adga_amd import api
    model, par = {1: ("sc1", dict(U=2.0, J=0.0, t=0.25)), 3: ("t2g", dict(U=5.0, J=0.75, t=-0.26, tp=-0.08))}.get(
        n, ("rand5", dict(U=4.0, J=0.6, t=0.15)))
    wl = synth.Workload("half", n, nk, iwf, 1, 10.0, model=model, seed=5, noise=1e-2, vq=vq, **par)
    inp = synth.build_inputs(wl)
    pts = [(w, q) for w in (0, 1) for q in range(npts)]
    cl = lambda w, c: synth.chi_loc(inp, w, c)  # noqa: E731
    ref = adga_oracle.HotPath(inp).run(pts, cl)
    for eom in (1, 0):
        print(f"n={n} N={wl.maxdim} points={npts} vq={vq} eom={eom}", flush=True)
        with api.Context(inp, eom=eom) as ctx:
            out = api.run_loop(ctx, pts, cl, "fp64")
        for k in ("chi_d", "chi_m", "sigma_nl", "sigma_dmft"):
            assert rel_err(out[k], ref[k]) < 1e-10, (eom, k, rel_err(out[k], ref[k]))
    with api.Context(inp, do_eom=0) as ctx:
        out = api.run_loop(ctx, pts, cl, "fp64")
    assert rel_err(out["chi_d"], ref["chi_d"]) < 1e-10
    assert np.abs(out["sigma_nl"]).max() == 0.0
