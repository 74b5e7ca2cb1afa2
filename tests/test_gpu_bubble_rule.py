"""The default bubble mode (2): which of the two ways a batch takes, on grids whose transform runs in LDS and on grids
where it does not, and what it does where the tables of every q do not fit the memory.  The two ways add their terms
in different orders, so equal bits say which one ran."""
import dataclasses

import numpy as np
import pytest

from conftest import rel_err
from adga_amd import synth

pytestmark = pytest.mark.gpu
GPU_BYTES = 288 << 30


def _run(inp, npts, mode, chi):
    from adga_amd import api
    with api.Context(inp, bubble=mode, do_eom=False, batch=npts) as ctx:
        ctx.set_local_omega(1, *chi)
        r = ctx.run_points(np.arange(1, npts + 1, dtype=np.int32), "fp64")
    assert (r["status"] == 0).all()
    return r["bubble_nl"]


# axes up to 24 points: from 24 points on by transform with three or five orbitals, 64 otherwise; a longer axis: 64
@pytest.mark.parametrize("n,nk,npts,dft", [(3, (4, 3, 5), 23, 0), (3, (4, 3, 5), 24, 1), (5, (4, 3, 3), 24, 1),
                                           (4, (4, 5, 4), 63, 0), (4, (4, 5, 4), 64, 1), (3, (28, 3, 2), 24, 0),
                                           (3, (28, 3, 2), 63, 0), (3, (28, 3, 2), 64, 1), (5, (25, 3, 1), 30, 0),
                                           (2, (25, 3, 1), 64, 1)])
def test_gpu_bubble_default_rule(n, nk, npts, dft):
    wl = synth.Workload("rule", n, nk, 5, 1, 10.0, 3.0, 0.4, "rand5", t=0.2, seed=n, noise=1e-3)
    inp = synth.build_inputs(wl)
    chi = [synth.chi_loc(inp, 1, c) for c in ("dens", "magn")]
    print(f"bubble rule n={n} {nk} points={npts}", flush=True)
    direct, conv, auto = (_run(inp, npts, m, chi) for m in (0, 1, 2))
    assert not np.array_equal(direct, conv)
    assert np.array_equal(auto, conv if dft else direct)
    assert rel_err(direct, conv) < 1e-10


def test_gpu_bubble_tables_beyond_memory():
    """Five orbitals, 40 frequencies on 80 x 72 x 70 k: two tables of 161 GB.  64 points are summed directly; mode 1
    stays an error, and the context works after it."""
    from adga_amd import _lib, api
    nk, nkp = (80, 72, 70), 80 * 72 * 70
    small = synth.build_inputs(synth.Workload("mem", 5, (2, 2, 2), 20, 1, 10.0, 3.0, 0.4, "rand5", t=0.2, noise=1e-3))
    r = np.random.default_rng(1)
    h = 0.1 * (r.standard_normal((5, 5, nkp)) + 1j * r.standard_normal((5, 5, nkp)))
    inp = dataclasses.replace(small, wl=dataclasses.replace(small.wl, nk=nk), hk=np.asfortranarray(h + h.transpose(1, 0, 2).conj()),
                              q_data=np.arange(1, 65, dtype=np.int32) * 6007, k_data_eom=np.array([1], dtype=np.int32))
    assert 2 * 40 * 625 * nkp * 16 > 1.03 * GPU_BYTES
    chi = [synth.chi_loc(small, 1, c) for c in ("dens", "magn")]
    iq = np.arange(1, 65, dtype=np.int32)
    print("bubble tables beyond the memory", flush=True)
    with api.Context(inp, do_eom=False, batch=64) as ctx:
        ctx.set_local_omega(1, *chi)
        auto = ctx.run_points(iq, "fp64")["bubble_nl"]
        ctx._check(_lib.lib.adga_set_option(ctx.h, b"bubble", 1.0))
        with pytest.raises(api.AdgaError) as e:
            ctx.run_points(iq, "fp64")
        assert e.value.code == 7
        ctx._check(_lib.lib.adga_set_option(ctx.h, b"bubble", 0.0))
        assert np.array_equal(auto, ctx.run_points(iq, "fp64")["bubble_nl"])
