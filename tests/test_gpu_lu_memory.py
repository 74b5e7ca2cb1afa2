"""A batch whose LU factors do not fit the GPU's memory (3 x 20^3-grid workload's size N = 1080: 37.6 MB a point, 8420
points 317 GB of 288 GiB): its points are solved a few at a time, nothing is added to the self-energy twice, and a
smaller batch on the same context works.

Bounds: the same complex128 LU of every point, 1e-12 as between any two FP64 solves here."""
import numpy as np
import pytest

from conftest import rel_err
from adga_amd import synth

pytestmark = pytest.mark.gpu
NPTS = 8420
GPU_BYTES = 288 << 30


def _setup(noise=1e-3):
    wl = synth.Workload("memory", 3, (20, 20, 22), 60, 1, 10.0, model="t2g", seed=4, noise=noise, U=5.0, J=0.75,
                        t=-0.26, tp=-0.08)
    inp = synth.build_inputs(wl)
    return inp, [np.asfortranarray(synth.chi_loc(inp, 1, c)) for c in ("dens", "magn")]


def test_gpu_lu_beyond_memory():
    from adga_amd import _lib, api
    inp, x = _setup()
    iq = np.arange(1, NPTS + 1, dtype=np.int32)
    need = 2 * NPTS * 1080 * 1088 * 16
    assert need > 1.02 * GPU_BYTES
    out = []
    for batch in (NPTS, 2000):
        print(f"LU of {NPTS} points in batches of {batch}", flush=True)
        with api.Context(inp, series=0, batch=batch) as ctx:
            for rep in range(2):
                ctx.reset_sigma()
                ctx.set_local_omega(1, *x)
                r = ctx.run_points(iq, "fp64")
                out.append((r["chi_d"], r["chi_m"], *ctx.get_sigma()[:2]))
                st = ctx.stats()
                assert (r["status"] == 0).all()
                if batch == 2000:
                    break
                assert st["n_lu_launches"] == rep * 5
                # the caller lowers the batch of the same context
                ctx._check(_lib.lib.adga_set_option(ctx.h, b"batch", 2000.0))
    for o in out[:2]:
        for a, b in zip(o, out[2]):
            assert rel_err(a, b) < 1e-12


def test_gpu_derivative_solves_beyond_memory():
    from adga_amd import api
    inp, x = _setup()
    tan = synth.tangents(inp)
    dx = [synth.dchi_loc(inp, tan, 1) for _ in range(2)]
    iq = np.arange(1, NPTS + 1, dtype=np.int32)
    out = []
    for batch, series in ((NPTS, 0), (1700, 1)):
        print(f"derivatives of {NPTS} points in batches of {batch}, series={series}", flush=True)
        with api.Context(inp, series=series, batch=batch) as ctx:
            ctx.set_tangents(tan)
            ctx.set_local_omega(1, *x)
            ctx.set_local_omega_tangent(*dx)
            r = ctx.run_points_tangent(iq)
            out.append((r["dchi_d"], r["dchi_m"], ctx.get_sigma()[0], ctx.get_sigma_tangent()))
    for a, b in zip(*out):
        assert rel_err(a, b) < 1e-12
