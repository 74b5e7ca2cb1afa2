"""get_sigma_g_loc where its split can go wrong: boxes of one frequency and of a wave's lanes less one, exactly and
plus one, a box that fills the frequency range, fewer k points than waves and partial rounds of them, one to five
orbitals, against the oracle.  Bound: 1e-12 relative, as for the routine's other tests."""
import numpy as np
import pytest

from conftest import rel_err
from adga_amd import synth
import adga_oracle

pytestmark = pytest.mark.gpu

CASES = [(1, (1, 1, 1), 1, 2), (1, (3, 2, 2), 63, 90), (2, (2, 1, 1), 64, 64), (3, (5, 4, 3), 65, 70),
         (3, (9, 8, 8), 3, 40), (5, (3, 3, 3), 6, 9)]


@pytest.mark.parametrize("n,nk,iwf,iwmax", CASES)
def test_gpu_sigma_g_loc_box(n, nk, iwf, iwmax):
    from adga_amd import api
    wl = synth.Workload("onep", n, nk, iwf, 0, 10.0, 3.0, 0.4, "sc1" if n == 1 else "rand5", t=0.2, seed=n,
                        iwmax=iwmax)
    inp = synth.build_inputs(wl)
    nkp = int(np.prod(nk))
    rng = np.random.default_rng(iwf)
    ss = 0.2 * (rng.normal(size=(n, n, wl.nf, nkp)) + 1j * rng.normal(size=(n, n, wl.nf, nkp)))
    print(f"sigma_g_loc n={n} {nk} iwf={iwf} iwmax={iwmax}", flush=True)
    with api.Context(inp) as ctx:
        sl, gl = ctx.get_sigma_g_loc(ss)
    osl, ogl = adga_oracle.get_sigma_g_loc(inp, ss)
    assert rel_err(sl, osl) < 1e-12 and rel_err(gl, ogl) < 1e-12
