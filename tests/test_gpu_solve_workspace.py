"""pobtas through the C ABI with less workspace than the selected sweep uses, for
blocks below 256: what the tile sweep needs, and none for a partial solve, which
its launch-by-launch form does without (src/serinv/algs/pobtas.py:80-159, against
the oracle at 1e-12 relative, max-norm).
"""

import numpy as np
import pytest

from oracle import serinv_np
from serinv_amd.utils.matrices import bta_spd
from tests._helpers import relerr, to_dev, to_host

pytestmark = pytest.mark.gpu
TOL = 1e-12


def _solve(lib, F, x, trans, partial, ws, nbytes):
    import torch

    D, L, R, T = F
    n, b, a = D.shape[0], D.shape[1], R.shape[1]
    ptr = lambda y: y.data_ptr() if y is not None and y.numel() else None  # noqa: E731
    return lib.rocbta_dpobtas(n, b, a, ptr(D), ptr(L), ptr(R), ptr(T), ptr(x), x.shape[1], x.shape[1], trans.encode(),
                              partial, ptr(ws), nbytes, torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("n,b,a,r", [(8, 96, 12, 1), (12, 130, 8, 3), (40, 64, 8, 2), (6, 200, 70, 16)])
def test_solve_in_a_tile_sweep_workspace(gpu_device, monkeypatch, n, b, a, r):
    import torch

    from serinv_amd import _lib

    lib = _lib.load()
    print(f"pobtas n={n} b={b} a={a} r={r} in the tile sweep's workspace", flush=True)
    monkeypatch.setenv("ROCBTA_POBTAS_ALGO", "sweep")
    nbytes = lib.rocbta_workspace_bytes(_lib.OP_POBTAS, n, b, a, r)
    monkeypatch.delenv("ROCBTA_POBTAS_ALGO")
    D, L, R, T, B = bta_spd(n, b, a, seed=7800 + n, n_rhs=r)
    serinv_np.pobtaf(D, L, R, T)
    F, x = to_dev(gpu_device, D, L, R, T), to_dev(gpu_device, B)[0]
    ws = torch.empty(nbytes, dtype=torch.uint8, device=gpu_device)
    for trans in ("N", "C"):
        assert _solve(lib, F, x, trans, 0, ws, nbytes) == 0
        assert int(ws[:4].view(torch.int32).item()) == 0
        serinv_np.pobtas(D, L, R, T, B, trans=trans)
        assert relerr(to_host(x)[0], B) < TOL, trans
    assert _solve(lib, F, x, "N", 0, ws, 4) == _lib.ROCBTA_ERR_WORKSPACE


@pytest.mark.parametrize("n,b,a,r", [(8, 96, 12, 1), (5, 130, 8, 3), (6, 64, 8, 2)])
def test_partial_solve_without_workspace(gpu_device, n, b, a, r):
    from serinv_amd import _lib

    lib = _lib.load()
    print(f"partial pobtas n={n} b={b} a={a} r={r} without workspace", flush=True)
    D, L, R, T, B = bta_spd(n, b, a, seed=7900 + n, n_rhs=r)
    serinv_np.pobtaf(D, L, R, T)
    F, x = to_dev(gpu_device, D, L, R, T), to_dev(gpu_device, B)[0]
    for trans in ("N", "C"):
        assert _solve(lib, F, x, trans, 1, None, 0) == 0
        serinv_np.pobtas(D, L, R, T, B, trans=trans, partial=True)
        assert relerr(to_host(x)[0], B) < TOL, trans
