"""The direct bubble (one k sum per point) where its tiles and splits can go wrong: one to five orbitals, grids of
fewer k points than a workgroup's waves share out and of a partial last step, one point and partial groups of
points, repeated ones included: the frequency sum against NumPy and chi against the bubble by convolution.  All add
nkp products in FP64: 8 eps sqrt(nkp nf) of the largest element covers the order of the bubble's sums, where a wrong
index leaves O(1); chi agrees to the repository's 1e-10."""
import numpy as np
import pytest

from conftest import rel_err
from adga_amd import synth

pytestmark = pytest.mark.gpu

CASES = [(1, (3, 2, 2), 3, 1), (2, (4, 3, 5), 4, 5), (3, (1, 1, 1), 2, 1), (3, (2, 1, 3), 3, 2), (3, (5, 3, 2), 4, 1),
         (3, (7, 5, 3), 40, 13), (3, (4, 4, 2), 64, 9), (4, (3, 3, 4), 5, 3), (4, (5, 2, 7), 50, 11),
         (5, (3, 2, 2), 4, 2), (5, (4, 3, 3), 40, 7)]


@pytest.mark.parametrize("n,nk,iwf,npts", CASES)
def test_gpu_bubble_direct(n, nk, iwf, npts):
    from adga_amd import api
    import adga_oracle
    from adga_amd import api
    nkp = int(np.prod(nk))
    wl = synth.Workload("bub", n, nk, iwf, 1, 10.0, 3.0, 0.4, "sc1" if n == 1 else "rand5", t=0.2, seed=n, noise=1e-3)
    inp = synth.build_inputs(wl)
    qs = np.random.default_rng(npts).integers(0, wl.nqp, size=npts)
    hot = adga_oracle.HotPath(inp)
    chi = {c: synth.chi_loc(inp, 1, c) for c in ("dens", "magn")}
    out = []
    for mode in (0, 1):
        print(f"bubble n={n} {nk} iwf={iwf} points={npts} mode {mode}", flush=True)
        with api.Context(inp, bubble=mode, do_eom=False) as ctx:
            loc = ctx.set_local_omega(1, chi["dens"], chi["magn"])[2]
            out.append(ctx.run_points(qs.astype(np.int32) + 1, "fp64"))
    for j, q in enumerate(qs):
        ref = hot.chi0q(int(q), 1).sum(axis=2) / inp.beta ** 2  # bubble_nl: less the local bubble
        err = np.abs(out[0]["bubble_nl"][:, :, j] + loc - ref).max() / np.abs(ref).max()
        assert err < 8 * 2.2e-16 * np.sqrt(nkp * 2 * iwf), (q, err)
    for k in ("chi_d", "chi_m"):
        assert rel_err(out[0][k], out[1][k]) < 1e-10, (k, rel_err(out[0][k], out[1][k]))
