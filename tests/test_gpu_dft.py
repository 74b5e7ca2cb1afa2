"""The k-grid transforms in LDS (bubble and EOM by convolution) against the direct sums, on grids at the edges of
their range: the shortest and longest axes, even and odd ones, padded fields that just fit the LDS and that do
not (then the passes over HBM), and the one-point axis.  Both sum nkp products in FP64, so they agree to a few
eps sqrt(nkp), well inside the repository's 1e-10."""
import numpy as np
import pytest

from conftest import rel_err
from adga_amd import synth

pytestmark = pytest.mark.gpu

GRIDS = [(1, 1, 2), (2, 1, 1), (24, 1, 2), (3, 24, 1), (1, 2, 24), (25, 2, 1), (23, 5, 2), (7, 11, 13), (17, 19, 4),
         (16, 16, 16), (21, 22, 21), (22, 21, 22), (20, 20, 20), (15, 18, 22)]


@pytest.mark.parametrize("nk", GRIDS, ids=["x".join(map(str, g)) for g in GRIDS])
def test_gpu_dft_equals_direct_sums(nk):
    from adga_amd import api
    wl = synth.Workload("dft", 1, nk, 3, 1, 10.0, 2.0, 0.0, "sc1", t=0.25, seed=3, noise=0.02)
    inp = synth.build_inputs(wl)
    pts = [(1, int(q)) for q in np.unique(np.linspace(0, wl.nqp - 1, 5).astype(int))]
    out = []
    for mode in (1, 0):
        print(f"grid {nk} mode {mode}", flush=True)
        with api.Context(inp, bubble=mode, eom=mode) as ctx:
            out.append(api.run_loop(ctx, pts, lambda w, c: synth.chi_loc(inp, w, c), "fp64"))
    for k in ("chi_d", "chi_m", "sigma_nl"):
        assert rel_err(out[0][k], out[1][k]) < 1e-10, (k, rel_err(out[0][k], out[1][k]))
    assert np.abs(out[0]["bubble_nl"] - out[1]["bubble_nl"]).max() < 1e-13


def test_gpu_dft_derivatives():
    from adga_amd import api
    wl = synth.Workload("dft", 2, (5, 4, 3), 3, 1, 8.0, 3.0, 0.5, "rand5", t=0.15, seed=3)
    inp = synth.build_inputs(wl)
    tan = synth.tangents(inp)
    pts = [(1, q) for q in range(0, 60, 7)]
    out = []
    for mode in (1, 0):
        print(f"derivatives mode {mode}", flush=True)
        with api.Context(inp, bubble=mode, eom=mode) as ctx:
            ctx.set_tangents(tan)
            out.append(api.run_loop_tangent(ctx, pts, lambda w, c: synth.chi_loc(inp, w, c),
                                            lambda w, c: synth.dchi_loc(inp, tan, w)))
    for k in ("dchi_d", "dchi_m", "dsigma_nl"):
        assert rel_err(out[0][k], out[1][k]) < 1e-10, (k, rel_err(out[0][k], out[1][k]))
