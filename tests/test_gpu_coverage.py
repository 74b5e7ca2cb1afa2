"""Shapes and branches that need more than the smallest workloads: the residual product's 64 x 64 tiles, downloads of
several chunks per host thread, several one-particle frequencies per workgroup, and derivatives whose solve does not
converge by iteration where the forward one does."""
import numpy as np
import pytest

from conftest import rel_err
from adga_amd import synth
from test_gpu_series import _workload

pytestmark = pytest.mark.gpu


def _tiles(rows, cols, channels):
    """64 x 64 tiles of a residual product; from 2048 on they are taken, below 32 x 32 ones"""
    return channels * -(-rows // 64) * -(-cols // 64)


@pytest.mark.parametrize("precision", ["fp64", "refined"])
def test_gpu_large_tiles_equal_lu(precision):
    """N = 666, 720 points: 64 x 64 tiles with remainders of 26 rows, 16 columns and 10 in K, against the LU (the
    bounds of the smaller shapes' test: 1e-12 in FP64, 1e-10 refined)."""
    from adga_amd import api
    wl = _workload(3, (9, 9, 9), 37, 1e-3)
    assert wl.maxdim == 666 and _tiles(666, 720 * 9, 2) >= 2048
    inp = synth.build_inputs(wl)
    x = [synth.chi_loc(inp, 1, c) for c in ("dens", "magn")]
    res = []
    for series in (1, 0):
        print(f"64 x 64 tiles {precision} series={series}", flush=True)
        with api.Context(inp, series=series, batch=720) as ctx:
            ctx.set_local_omega(1, *x)
            r = ctx.run_points(np.arange(1, 721, dtype=np.int32), precision)
            assert (r["status"] == 0).all() and ctx.stats()["n_lu_launches"] == 1 - series
            res.append([r["chi_d"], r["chi_m"], ctx.get_sigma()[0]])
    for a, b in zip(*res):
        assert rel_err(a, b) < (1e-12 if precision == "fp64" else 1e-10)


def test_gpu_large_tiles_equal_small_tiles():
    """1700 points of N = 1080 at once and in batches of 100: every product of the batch, gamma^q's upper half of the
    rows included, on 64 x 64 and on 32 x 32 tiles.  Equal but for the rounding of sums in another order: 1e-12."""
    from adga_amd import api
    assert _tiles(540, 1700 * 9, 1) >= 2048 and _tiles(1080, 100 * 9, 2) < 2048
    wl = _workload(3, (12, 12, 12), 60, 1e-3)
    inp = synth.build_inputs(wl)
    x = [synth.chi_loc(inp, 1, c) for c in ("dens", "magn")]
    iq = np.arange(1, 1701, dtype=np.int32)
    res = []
    for batch in (1700, 100):
        print(f"1700 points in batches of {batch}", flush=True)
        with api.Context(inp, batch=batch) as ctx:
            ctx.set_local_omega(1, *x)
            r = ctx.run_points(iq, "fp64")
            assert (r["status"] == 0).all() and ctx.stats()["n_lu_launches"] == 0
            res.append([r["chi_d"], r["chi_m"], ctx.get_sigma()[0]])
    for a, b in zip(*res):
        assert rel_err(a, b) < 1e-12


@pytest.mark.parametrize("nk,iwf", [((16, 16, 17), 32), ((17, 19, 23), 64)], ids=["17.8MB", "60.9MB"])
def test_gpu_download_in_many_chunks(nk, iwf):
    """Self-energies of 8.5 and 29 chunks of 2 MB for the eight host threads: a partial last chunk, an uneven split, and
    slots used again; equal on a second read, and their k sum is the context's own."""
    from adga_amd import api
    inp = synth.build_inputs(_workload(2, nk, iwf, 1e-3))
    print(f"download {nk}", flush=True)
    with api.Context(inp) as ctx:
        ctx.set_local_omega(1, *[synth.chi_loc(inp, 1, c) for c in ("dens", "magn")])
        ctx.run_points(np.array([1, 6, 78], dtype=np.int32), "fp64")
        a = ctx.get_sigma()[0]
        b = ctx.get_sigma()[0]
        loc = ctx.get_sigma_g_loc()[0]
    assert a.nbytes > 16 << 20 and a.nbytes % (2 << 20) != 0 and np.array_equal(a, b)
    mean = a.mean(axis=3)
    for i in range(2):
        mean[i, i] += inp.siw[inp.iwmax - iwf:inp.iwmax + iwf, i]
    assert rel_err(loc, mean) < 1e-13


@pytest.mark.parametrize("n", [1, 2, 3, 4])
@pytest.mark.parametrize("iwmax", [1024, 1025, 1026, 1027])
def test_gpu_one_particle_sums_of_many_frequencies(n, iwmax):
    """get_giw with four frequencies to a workgroup (n <= 3, from 1024 on) and get_sigma_g_loc with two outside the
    box, last groups of every size, against the oracle: 1e-12 as for the routines' other tests."""
    import adga_oracle
    from adga_amd import api
    nk, iwf = (3, 2, 2), 4
    wl = synth.Workload("onep", n, nk, iwf, 0, 10.0, 3.0, 0.4, "sc1" if n == 1 else "rand5", t=0.2, seed=n, iwmax=iwmax)
    inp = synth.build_inputs(wl)
    rng = np.random.default_rng(iwmax)
    ss = 0.2 * (rng.normal(size=(n, n, wl.nf, 12)) + 1j * rng.normal(size=(n, n, wl.nf, 12)))
    print(f"one-particle sums n={n} iwmax={iwmax}", flush=True)
    with api.Context(inp) as ctx:
        assert rel_err(ctx.get_giw(), adga_oracle.get_giw(inp)) < 1e-12
        sl, gl = ctx.get_sigma_g_loc(ss)
    osl, ogl = adga_oracle.get_sigma_g_loc(inp, ss)
    assert rel_err(sl, osl) < 1e-12 and rel_err(gl, ogl) < 1e-12


def test_gpu_derivative_solves_that_need_the_lu():
    """N = 360 at the iteration's limit: the forward solve and two directions iterate (17 to 19 products each), the third
    direction's right-hand side does not, and its LU factors are formed after the forward pass; with the directions in
    the opposite order they are formed for the first and serve all three.  Against the LU throughout: 1e-12."""
    import dataclasses
    from adga_amd import api
    inp = synth.build_inputs(_workload(3, (4, 4, 3), 20, 0.225))
    tan = synth.tangents(inp)
    x = [synth.chi_loc(inp, 1, c) for c in ("dens", "magn")]
    d = synth.dchi_loc(inp, tan, 1)
    v = np.random.default_rng(3).standard_normal(d.shape[:2] + (1,))
    d = d + 0.03 * (v + v.transpose(1, 0, 2))
    iq = np.arange(1, 49, dtype=np.int32)
    fields = ("dhk", "dsiw", "dgiw", "dmu", "du", "du_tilde")
    for order in (slice(None), slice(None, None, -1)):
        t = dataclasses.replace(tan, **{f: np.ascontiguousarray(getattr(tan, f)[..., order]) for f in fields})
        dx = np.asfortranarray(d[..., order])
        out, products = [], []
        for series in (1, 0):
            print(f"derivatives at the limit, series={series} order {order}", flush=True)
            with api.Context(inp, batch=48, series=series) as ctx:
                ctx.set_tangents(t)
                ctx.set_local_omega(1, *x)
                ctx.set_local_omega_tangent(dx, dx)
                ctx.run_points(iq, "fp64")
                products.append(ctx.stats()["n_gemm_dominant"])
                ctx.reset_sigma()
                r = ctx.run_points_tangent(iq)
                st = ctx.stats()
                products.append(st["n_gemm_dominant"])
                assert (r["status"] == 0).all() and st["n_lu_launches"] == 1 - series
                out.append((r["chi_d"], r["dchi_d"], r["dchi_m"], ctx.get_sigma()[0], ctx.get_sigma_tangent()))
        forward, total = products[:2]
        each = forward - 4
        if order == slice(None):
            assert forward + each <= total < forward + 3 * each, (forward, total)
        else:
            assert total < forward + each, (forward, total)
        for a, b in zip(*out):
            assert rel_err(a, b) < 1e-12
