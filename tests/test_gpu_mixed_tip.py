"""The arrow tip of the mixed factorization is formed and factored in FP64
(rocbta_mpobtaf), for arrows of one 64-row tile and of more, on both pobtaf
algorithms and with both settings of factorize_last_block.

The tip's Schur complement T - sum_i L_{t,i} L_{t,i}^T (src/serinv/algs/pobtaf.py
:143-159) is rebuilt in FP64 on the host from the arrow blocks that the GPU returned,
whose own errors are those of FP32 products, so that what is left is the tip's
arithmetic.  Bounds, relative to the largest entry of the given tip: n b products
of entries below it are summed, 1e-13 (FP32 products leave 1e-8); the factor of
it, well conditioned, 1e-12.
"""

import numpy as np
import pytest

from serinv_amd.utils.matrices import bta_spd
from tests._helpers import relerr, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("last", [True, False])
@pytest.mark.parametrize("algo", ["chain", "loop"])
@pytest.mark.parametrize("n,b,a", [(4, 64, 16), (2, 40, 65), (3, 100, 65), (4, 70, 100), (3, 130, 130)])
def test_tip_is_fp64(gpu_device, monkeypatch, algo, n, b, a, last):
    from serinv_amd.mixed import pobtaf_mixed

    if algo == "loop":
        monkeypatch.setenv("ROCBTA_POBTAF_ALGO", "loop")
    else:
        monkeypatch.delenv("ROCBTA_POBTAF_ALGO", raising=False)
    print(f"mixed tip {algo} n={n} b={b} a={a} last={last}", flush=True)
    D, L, R, T, _ = bta_spd(n, b, a, seed=7100 + n + b + a)
    d, l, r, t = to_dev(gpu_device, D, L, R, T)
    pobtaf_mixed(d, l, r, t, factorize_last_block=last)
    Rg, Tg = to_host(r, t)
    S = T - sum(Rg[i] @ Rg[i].T for i in range(n if last else n - 1))
    if last:
        assert relerr(np.tril(Tg), np.linalg.cholesky(S)) < 1e-12
    else:
        assert np.max(np.abs(np.tril(Tg - S))) < 1e-13 * np.max(np.abs(T))
