"""The grouped products and the blocked inverse at the edges of their tiles
(serinv_amd/csrc/gemm_f64.hpp: 32 x 32 blocks, 16-deep k groups, workgroup
tiles of 32 or 64; serinv_amd/csrc/getri_f64.hpp: 64-wide pivot tiles of 16-wide
blocks, one launch per pivot tile up to one tile per CU).

pobtasi (src/serinv/algs/pobtasi.py:92-172) and ddbtasc / ddbtasci
(src/serinv/algs/ddbtasc.py:187-241, ddbtasci.py:187-256) against the oracle at
1e-12 relative (max-norm per output array).
"""

import numpy as np
import pytest

from oracle import dense, generators, serinv_np
from serinv_amd.utils.matrices import bta_spd
from tests._helpers import relerr, to_dev, to_host

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.mark.parametrize("n,b,a", [(3, 15, 1), (3, 16, 16), (3, 31, 33), (3, 32, 32), (3, 33, 31), (3, 47, 0),
                                   (3, 63, 65), (3, 64, 48), (3, 95, 17), (3, 97, 0), (2, 129, 66), (20, 130, 9),
                                   (2, 513, 30)])
def test_selected_inverse_matches_oracle(gpu_device, n, b, a):
    import serinv_amd.algs as algs

    print(f"pobtasi n={n} b={b} a={a}", flush=True)
    D, L, R, T, _ = bta_spd(n, b, a, seed=6100 + n + b + a)
    serinv_np.pobtaf(D, L, R, T)
    g = to_dev(gpu_device, D, L, R, T)
    algs.pobtasi(*g)
    serinv_np.pobtasi(D, L, R, T)
    for name, x, y in zip("DLRT", to_host(*g), (D, L, R, T)):
        assert relerr(x, y) < TOL, name


@pytest.mark.parametrize("b,a,n", [(15, 1, 3), (17, 2, 3), (48, 17, 2), (66, 63, 2), (81, 5, 2), (127, 3, 2),
                                   (191, 65, 2), (193, 1, 2), (1030, 3, 2)])
def test_blocked_inverse_matches_oracle(gpu_device, b, a, n):
    import serinv_amd.algs as algs

    print(f"ddbtasc b={b} a={a} n={n}", flush=True)
    A = generators.dd_bta(b, a, n, np.random.default_rng(6200 + b + a + n))
    arrs = dense.bta_dense_to_arrays_full(A, b, a, n)
    g = to_dev(gpu_device, *arrs)
    o = [x.copy() for x in arrs]
    for step in ("ddbtasc", "ddbtasci"):
        getattr(algs, step)(*g)
        getattr(serinv_np, step)(*o)
        for x, y in zip(to_host(*g), o):
            assert relerr(x, y) < TOL, step
