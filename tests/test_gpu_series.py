"""The fixed-point solve of the BSE systems (option series = 1, the default) against the LU (series = 0) on the
same inputs: sizes at the edges of the residual product's tiles and on both of its tile shapes, every orbital
count, vertices from weak to strong (where the LU is taken), V(q), a batch whose points contract unequally, and
the derivatives.

Bounds.  Both solutions leave a relative residual r; the iteration is only taken where the operator contracts, so
|1 - T|^-1 is a few at most and eta differs by a few r: 1e-12 for the FP64 mode (r <= 1e-14 both), and the
repository's 1e-10 for the refined mode (r <= 1e-12)."""
import numpy as np
import pytest

from conftest import rel_err
from adga_amd import synth

pytestmark = pytest.mark.gpu
BOUND = {"fp64": 1e-12, "refined": 1e-10}


def _workload(n, nk, iwf, noise, vq=0.0, seed=5):
    model, par = {1: ("sc1", dict(U=2.0, J=0.0, t=0.25)), 3: ("t2g", dict(U=5.0, J=0.75, t=-0.26, tp=-0.08))}.get(
        n, ("rand5", dict(U=4.0, J=0.6, t=0.15)))
    return synth.Workload("series", n, nk, iwf, 1, 10.0, model=model, seed=seed, noise=noise, vq=vq, **par)


def _both(wl, npts, precision, omega=1, change=None):
    from adga_amd import api
    inp = synth.build_inputs(wl)
    if change:
        change(inp)
    pts = [(omega, q) for q in range(npts)]
    out, st = [], []
    for series in (1, 0):
        print(f"n={wl.n} N={wl.maxdim} points={npts} noise={wl.noise} {precision} series={series}", flush=True)
        with api.Context(inp, series=series, batch=npts) as ctx:
            out.append(api.run_loop(ctx, pts, lambda w, c: synth.chi_loc(inp, w, c), precision))
            st.append(ctx.stats())
    assert (out[0]["status"] == 0).all() and (out[1]["status"] == 0).all()
    for k in ("chi_d", "chi_m", "sigma_nl"):
        assert rel_err(out[0][k], out[1][k]) < BOUND[precision], (k, rel_err(out[0][k], out[1][k]))
    return st


# (orbitals, k grid, half box, points): N and the columns npts n^2 one below, at and above multiples of 32 and
# 64, K chunks of 16 with every remainder class, and one product large enough for the 64 x 64 tiles
SIZES = [(1, (2, 2, 1), 1, 1), (1, (4, 4, 4), 15, 31), (1, (4, 4, 4), 16, 32), (1, (4, 4, 5), 17, 65),
         (2, (3, 3, 3), 4, 16), (2, (3, 3, 4), 9, 33), (3, (3, 3, 2), 7, 7), (4, (3, 2, 2), 2, 5), (4, (4, 2, 2), 3, 12),
         (5, (2, 2, 3), 1, 3), (5, (3, 2, 2), 3, 11), (3, (9, 9, 9), 32, 720)]


@pytest.mark.parametrize("precision", ["fp64", "refined"])
@pytest.mark.parametrize("n,nk,iwf,npts", SIZES)
def test_gpu_series_equals_lu(n, nk, iwf, npts, precision):
    wl = _workload(n, nk, iwf, 1e-3)
    st = _both(wl, npts, precision)
    assert st[1]["n_lu_launches"] == 1
    if wl.maxdim >= 100:  # the smallest systems allow the iteration few steps: either solve
        assert st[0]["n_lu_launches"] == 0
    assert st[0]["refine_resid"] <= (1e-14 if precision == "fp64" else 1e-12)


@pytest.mark.parametrize("precision", ["fp64", "refined"])
@pytest.mark.parametrize("noise,lu", [(0.03, 0), (3.0, 1)])
def test_gpu_series_rule_over_vertex_strength(noise, lu, precision):
    """A vertex that contracts by about 0.03 a step is iterated, one that does not contract takes the LU."""
    for npts in (20, 90):  # below and above the look at a few points first
        st = _both(_workload(3, (5, 5, 4), 20, noise), npts, precision)
        assert st[0]["n_lu_launches"] == lu


@pytest.mark.parametrize("precision", ["fp64", "refined"])
def test_gpu_series_with_vq(precision):
    st = _both(_workload(2, (4, 4, 3), 17, 1e-3, vq=0.1), 48, precision)
    assert st[0]["n_lu_launches"] == 0


@pytest.mark.parametrize("precision", ["fp64", "refined"])
def test_gpu_series_hands_single_points_to_the_lu(precision):
    """V(q) strong at three q only: their points do not contract and are solved by the complex128 LU, the rest
    of the batch is iterated."""
    strong = [40, 130, 255]

    def v_q(inp):
        inp.v_q[:, :, strong] = 60.0 * np.eye(4)[:, :, None]

    st = _both(_workload(2, (8, 8, 4), 17, 1e-3, vq=0.02), 256, precision, change=v_q)
    assert st[0]["n_lu_launches"] == 0
    if precision == "refined":
        assert st[0]["n_fp64_resolved"] == 2 * len(strong)


def test_gpu_series_derivatives():
    from adga_amd import api
    wl = _workload(3, (4, 4, 3), 8, 1e-3)
    inp = synth.build_inputs(wl)
    tan = synth.tangents(inp)
    pts = [(0, q) for q in range(48)]
    out = []
    for series in (1, 0):
        print(f"derivatives series={series}", flush=True)
        with api.Context(inp, series=series, batch=48) as ctx:
            ctx.set_tangents(tan)
            out.append(api.run_loop_tangent(ctx, pts, lambda w, c: synth.chi_loc(inp, w, c),
                                            lambda w, c: synth.dchi_loc(inp, tan, w)))
    for k in ("dchi_d", "dchi_m", "dsigma_nl", "chi_d", "sigma_nl"):
        assert rel_err(out[0][k], out[1][k]) < 1e-12, (k, rel_err(out[0][k], out[1][k]))


def test_gpu_series_refuses_what_the_lu_refuses():
    """A BSE size above the LU's largest (4096) stays an argument error, also where the iteration would converge."""
    from adga_amd import api
    wl = _workload(5, (2, 1, 1), 82, 1e-3)
    inp = synth.build_inputs(wl)
    assert wl.maxdim == 4100
    with api.Context(inp, batch=1) as ctx:
        ctx.set_local_omega(0, synth.chi_loc(inp, 0, "dens"), synth.chi_loc(inp, 0, "magn"))
        with pytest.raises(api.AdgaError) as e:
            ctx.run_points([1], "fp64")
    assert e.value.code == 1
    assert np.isfinite(inp.mu)


@pytest.mark.parametrize("nk", [(16, 16, 16), (17, 19, 12)], ids=["16x16x16", "17x19x12"])
def test_gpu_large_self_energy_download(nk):
    """A self-energy above 16 MB comes back through pinned chunks, whole and partial ones (16.8 and 16.0 MB in
    chunks of 2 MB): equal to the context's own sum over it, bit for bit on a second read."""
    from adga_amd import api
    wl = _workload(2, nk, 32, 1e-3)
    inp = synth.build_inputs(wl)
    pts = [(1, q) for q in (0, 5, 77)]
    print(f"download {nk}", flush=True)
    with api.Context(inp) as ctx:
        a = api.run_loop(ctx, pts, lambda w, c: synth.chi_loc(inp, w, c), "fp64")["sigma_nl"]
        b = ctx.get_sigma()[0]
        loc = ctx.get_sigma_g_loc()[0]
    assert a.nbytes > 15.5e6 and np.array_equal(a, b)
    mean = a.mean(axis=3)
    for i in range(2):
        mean[i, i] += inp.siw[inp.iwmax - 32:inp.iwmax + 32, i]
    assert rel_err(loc, mean) < 1e-13
