"""The batched LU by itself (option series = 0): its streams, lane tuning, column groups and sizes, each with the check
that a factorisation ran.  The iteration takes these weak vertices by default."""
import numpy as np
import pytest

from conftest import rel_err
from adga_amd import synth

pytestmark = pytest.mark.gpu


def _run(ctx, inp, omega, qs, precision, box=None, launches=1):
    """set_local_omega and run_points, `launches` factorisations"""
    x = [synth.chi_loc(inp, omega, c) for c in ("dens", "magn")]
    if box is not None and box != inp.wl.iwfmax_small:
        n2, f = inp.n * inp.n, inp.wl.iwfmax_small
        s = slice(n2 * (f - box), n2 * (f + box))
        x = [np.asfortranarray(a[s, s]) for a in x]
    ctx.set_local_omega(omega, *x, box)
    r = ctx.run_points(np.asarray(qs, dtype=np.int32) + 1, precision)
    assert (r["status"] == 0).all() and ctx.stats()["n_lu_launches"] == launches
    return r


@pytest.fixture(scope="module")
def t2g():
    return synth.build_inputs(synth.workload("t2g_k20"))


@pytest.mark.parametrize("precision", ["fp64", "refined"])
def test_gpu_lu_streams_are_identical(t2g, precision):
    """98 points (196 matrices of N = 1080) on one to four streams: parts of 98, 65/65/66 and 49 matrices, equal bits."""
    from adga_amd import api
    qs = range(5, 8000, 82)
    one = None
    for streams in (1, 2, 3, 4):
        print(f"LU on {streams} streams {precision}", flush=True)
        with api.Context(t2g, lu_streams=streams, series=0) as ctx:
            r = _run(ctx, t2g, 1, qs, precision)
            res = [r["chi_d"], r["chi_m"], r["bubble_nl"], ctx.get_sigma()[0]]
        one = one or res
        for a, b in zip(one, res):
            assert np.array_equal(a, b), streams


@pytest.mark.parametrize("precision", ["fp64", "refined"])
def test_gpu_lu_tuned_lanes_are_identical(t2g, precision):
    """Batches of 16: six factorisations of 32 matrices and one of 4 a pass, the first three the timed trials."""
    from adga_amd import api
    qs = range(5, 8000, 82)
    res = []
    for streams in (1, 0):
        with api.Context(t2g, lu_streams=streams, batch=16, series=0) as ctx:
            for _ in range(1 if streams else 2):
                print(f"LU in batches of 16, lu_streams={streams} {precision}", flush=True)
                ctx.reset_sigma()
                r = _run(ctx, t2g, 1, qs, precision, launches=7)
                res.append([r["chi_d"], r["chi_m"], r["bubble_nl"], ctx.get_sigma()[0]])
    for other in res[1:]:
        for a, b in zip(res[0], other):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("precision", ["fp64", "refined"])
def test_gpu_lu_of_the_largest_boxes(precision):
    """N = 4000, 3500 and 2000 in one context, the largest the LU takes (16 rows per thread in the panels, one or two
    right-hand-side columns in LDS): against the iteration."""
    from adga_amd import api
    inp = synth.build_inputs(synth.workload("d5_k16"))
    res = []
    for series in (0, 1):
        res.append([])
        with api.Context(inp, series=series) as ctx:
            for omega, box, qs in ((0, 80, (0, 9)), (5, 70, (1234,)), (-20, 40, (77, 78, 79))):
                print(f"N={50 * box} {precision} series={series}", flush=True)
                r = _run(ctx, inp, omega, qs, precision, box, launches=1 - series)
                assert ctx.stats()["refine_resid"] < (1e-13 if precision == "fp64" else 1e-12)
                res[-1] += [r["chi_d"], r["chi_m"]]
            res[-1].append(ctx.get_sigma()[0])
    for a, b in zip(*res):
        assert rel_err(a, b) < (1e-11 if precision == "fp64" else 1e-10)


@pytest.mark.parametrize("precision", ["fp64", "refined"])
def test_gpu_lu_column_groups_on_a_full_batch(precision):
    """64 points at N = 2000: the solves' 25 columns run in groups (complex64: 3 of 9, complex128: 7 of 4)."""
    from adga_amd import api
    inp = synth.build_inputs(synth.workload("d5_k16", iwfmax_small=40))
    res = []
    for series in (0, 1):
        print(f"64 points N=2000 {precision} series={series}", flush=True)
        with api.Context(inp, series=series, batch=64) as ctx:
            r = _run(ctx, inp, 0, range(64), precision, launches=1 - series)
            res.append([r["chi_d"], r["chi_m"], ctx.get_sigma()[0]])
    for a, b in zip(*res):
        assert rel_err(a, b) < (1e-11 if precision == "fp64" else 1e-10)
