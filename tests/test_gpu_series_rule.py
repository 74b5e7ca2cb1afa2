"""The fixed-point iteration's decisions (option series = 1): which points go on, which are solved by an LU, and what
accuracy the refined mode leaves."""
import numpy as np
import pytest

from adga_amd import synth
from test_gpu_series import _workload

pytestmark = pytest.mark.gpu


def _run(wl, npts, precision, change=None, **opt):
    """(results, statistics) of the first npts q points at omega = 1 in one batch"""
    from adga_amd import api
    inp = synth.build_inputs(wl)
    if change:
        change(inp)
    print(f"n={wl.n} N={wl.maxdim} points={npts} noise={wl.noise} {precision} {opt}", flush=True)
    with api.Context(inp, batch=npts, **opt) as ctx:
        ctx.set_local_omega(1, *[synth.chi_loc(inp, 1, c) for c in ("dens", "magn")])
        r = ctx.run_points(np.arange(1, npts + 1, dtype=np.int32), precision)
        st = ctx.stats()
    assert (r["status"] == 0).all()
    return r, st


@pytest.mark.parametrize("noise,tol", [(0.5, 1e-6), (0.6, 1e-6), (0.65, 1e-6), (0.5, 1e-9), (0.55, 1e-9)])
def test_gpu_series_goes_on_above_round_off(noise, tol):
    """N = 400, contractions of 0.5 to 0.7 a step: a residual that falls by less than half a step, a few times above
    the caller's tolerance, is not at round-off; the iteration goes on to the tolerance."""
    st = _run(_workload(1, (4, 4, 4), 200, noise), 64, "refined", refine_tol=tol)[1]
    assert st["n_lu_launches"] == 0 and st["n_fp64_resolved"] == 0
    assert st["refine_resid"] <= tol


@pytest.mark.parametrize("precision,noise", [("fp64", 0.4), ("fp64", 0.45), ("refined", 0.5)])
def test_gpu_series_gets_the_last_steps(precision, noise):
    """41 points of N = 540, where a step costs a hundredth of any LU: points that need a few steps more than foreseen
    get them; neither they nor the batch are factored after some twenty steps."""
    st = _run(_workload(3, (4, 4, 3), 30, noise), 41, precision)[1]
    assert st["n_lu_launches"] == 0 and st["n_fp64_resolved"] == 0
    assert st["refine_resid"] <= (1e-14 if precision == "fp64" else 1e-12)


@pytest.mark.parametrize("precision", ["fp64", "refined"])
def test_gpu_series_slow_point_in_a_small_batch(precision):
    """V(q) strong at one of 48 points: the LU of that point alone costs nearly what the LU of all does, so the batch
    is factored at the first sign of it."""

    def v_q(inp):
        inp.v_q[:, :, 40] = 60.0 * np.eye(4)

    st = _run(_workload(2, (4, 4, 3), 17, 1e-3, vq=0.02), 48, precision, change=v_q)[1]
    assert st["n_lu_launches"] == 1


@pytest.mark.parametrize("n,nk,iwf,npts,noise", [(1, (4, 4, 4), 200, 64, 0.4), (1, (4, 4, 4), 200, 64, 0.5),
                                                 (3, (4, 4, 3), 30, 41, 0.4), (3, (4, 4, 4), 60, 16, 0.5)])
def test_gpu_series_refined_accuracy_at_slow_contraction(n, nk, iwf, npts, noise):
    """At a contraction rho of 0.3 to 0.5 a step the error after the last step is r rho / (1 - rho), which stays within
    a tenth of the tolerance (1.5 for the estimate of rho from the number of products), and chi within that of the
    FP64 LU's."""
    wl = _workload(n, nk, iwf, noise)
    r, st = _run(wl, npts, "refined")
    assert st["n_lu_launches"] == 0 and st["n_fp64_resolved"] == 0
    res = st["refine_resid"]
    rho = res ** (1.0 / st["n_gemm_dominant"])
    assert res * rho / (1 - rho) < 1.5e-13, (res, rho)
    ref = _run(wl, npts, "fp64", series=0)[0]
    for k in ("chi_d", "chi_m"):
        assert np.abs(r[k] - ref[k]).max() < 1e-13 * np.abs(ref[k]).max()


@pytest.mark.parametrize("precision", ["fp64", "refined"])
def test_gpu_series_looks_at_points_all_over_the_batch(precision):
    """V(q) strong at the first eight of 500 points of N = 360, as a neighbourhood of Gamma would have it: they are
    solved by themselves, the rest is iterated."""

    def v_q(inp):
        inp.v_q[:, :, :8] = 60.0 * np.eye(9)[:, :, None]

    r, st = _run(_workload(3, (8, 8, 8), 20, 1e-3, vq=0.02), 500, precision, change=v_q)
    assert st["n_lu_launches"] == 0
    if precision == "refined":
        assert st["n_fp64_resolved"] == 16
    ref = _run(_workload(3, (8, 8, 8), 20, 1e-3, vq=0.02), 500, precision, change=v_q, series=0)[0]
    for k in ("chi_d", "chi_m"):
        assert np.abs(r[k] - ref[k]).max() < (1e-12 if precision == "fp64" else 1e-10) * np.abs(ref[k]).max()


@pytest.mark.parametrize("precision", ["fp64", "refined"])
@pytest.mark.parametrize("noise", [1e-3, 0.03, 0.5])
def test_gpu_batch_dependence(precision, noise):
    """The same points in batches of 100, 13 and 1, the bubble formed one way: by the LU each point has the same bits.
    By the iteration a matrix takes the steps of its batch's slowest, and whether a batch is iterated depends on its
    points: they agree to the accuracy of each mode (1e-12 in FP64, a refined solve's 1e-11)."""
    from adga_amd import api
    inp = synth.build_inputs(_workload(3, (5, 5, 4), 20, noise))
    x = [synth.chi_loc(inp, 1, c) for c in ("dens", "magn")]
    for series in (0, 1):
        ref = None
        for batch in (100, 13, 1):
            print(f"batches of {batch} noise={noise} {precision} series={series}", flush=True)
            with api.Context(inp, batch=batch, bubble=0, series=series) as ctx:
                ctx.set_local_omega(1, *x)
                r = ctx.run_points(np.arange(1, 101, dtype=np.int32), precision)
                out = [r["chi_d"], r["chi_m"], ctx.get_sigma()[0]]
            assert (r["status"] == 0).all()
            ref = ref or out
            for a, b in zip(out, ref):
                if series == 0:
                    assert np.array_equal(a, b)
                else:
                    err = np.abs(a - b).max() / np.abs(b).max()
                    assert err < (1e-12 if precision == "fp64" else 1e-11)


def test_gpu_derivatives_share_one_factorisation():
    """N = 100, five orbitals: the forward solve iterates, but four solves by iteration cost more than one LU and four
    solves with its factors."""
    from adga_amd import api
    wl = _workload(5, (4, 4, 4), 2, 1e-3)
    inp = synth.build_inputs(wl)
    tan = synth.tangents(inp)
    iq = np.arange(1, 63, dtype=np.int32)
    print("one factorisation for all directions", flush=True)
    with api.Context(inp, batch=62) as ctx:
        ctx.set_tangents(tan)
        ctx.set_local_omega(0, *[synth.chi_loc(inp, 0, c) for c in ("dens", "magn")])
        ctx.set_local_omega_tangent(*[synth.dchi_loc(inp, tan, 0) for _ in range(2)])
        ctx.run_points(iq, "fp64")
        assert ctx.stats()["n_lu_launches"] == 0
        ctx.run_points_tangent(iq)
        assert ctx.stats()["n_lu_launches"] == 1
