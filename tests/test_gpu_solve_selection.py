"""The sweep that pobtas selects by the sizes (rocbta_dpobtas), on both sides of its
lines: tile rows of a block, block rows, arrow tiles, columns, partial solves.

pobtas (src/serinv/algs/pobtas.py:80-159) against the oracle at 1e-12 relative
(max-norm), both directions; and calls whose arrow makes the block inverses dear
take no longer than the 64-row-tile sweep.
"""

import numpy as np
import pytest

from oracle import serinv_np
from serinv_amd.utils.matrices import bta_spd
from tests._helpers import relerr, to_dev, to_host

pytestmark = pytest.mark.gpu
TOL = 1e-12

SHAPES = [(9, 64, 3, 1), (10, 64, 64, 1), (39, 64, 70, 1), (40, 64, 65, 1), (15, 64, 3, 4), (16, 64, 3, 2),
          (1, 64, 3, 5), (2, 64, 3, 9), (2, 65, 8, 1), (3, 65, 8, 4), (4, 65, 70, 1), (5, 65, 70, 8), (3, 130, 70, 1),
          (4, 130, 70, 3), (5, 130, 130, 1), (6, 130, 130, 1), (10, 130, 300, 1), (11, 130, 300, 1), (3, 96, 8, 4),
          (7, 96, 8, 2), (8, 96, 8, 4), (6, 96, 300, 4), (7, 96, 300, 4), (2, 96, 130, 16), (3, 96, 130, 16),
          (1, 256, 300, 4), (4, 256, 300, 4), (5, 256, 300, 4), (23, 256, 3, 2), (24, 256, 3, 2), (2, 272, 8, 4),
          (1, 272, 70, 8), (2, 272, 70, 8), (1, 256, 8, 9), (13, 144, 520, 1), (9, 192, 520, 1)]


@pytest.mark.parametrize("n,b,a,r", SHAPES)
def test_selected_solve_matches_oracle(gpu_device, monkeypatch, n, b, a, r):
    import serinv_amd.algs as algs

    monkeypatch.delenv("ROCBTA_POBTAS_ALGO", raising=False)
    print(f"pobtas n={n} b={b} a={a} r={r}", flush=True)
    D, L, R, T, B = bta_spd(n, b, a, seed=7500 + n + b + a + r, n_rhs=r)
    serinv_np.pobtaf(D, L, R, T)
    d, l, rr, t, bb = to_dev(gpu_device, D, L, R, T, B)
    for trans in ("N", "C"):
        serinv_np.pobtas(D, L, R, T, B, trans=trans)
        algs.pobtas(d, l, rr, t, bb, trans=trans)
        assert relerr(to_host(bb)[0], B) < TOL, trans


@pytest.mark.parametrize("n,b,a,r", [(3, 64, 5, 1), (4, 64, 5, 4), (3, 65, 70, 2), (4, 65, 70, 2), (2, 130, 300, 1),
                                     (3, 130, 300, 1), (2, 256, 9, 8), (3, 1040, 70, 1)])
def test_selected_partial_solve_matches_oracle(gpu_device, monkeypatch, n, b, a, r):
    """The tip, which a partial solve leaves alone, holds no factor: NaN."""
    import serinv_amd.algs as algs

    monkeypatch.delenv("ROCBTA_POBTAS_ALGO", raising=False)
    print(f"partial pobtas n={n} b={b} a={a} r={r}", flush=True)
    D, L, R, T, B = bta_spd(n, b, a, seed=7600 + n + b + a + r, n_rhs=r)
    serinv_np.pobtaf(D, L, R, T)
    d, l, rr, t, bb = to_dev(gpu_device, D, L, R, np.full_like(T, np.nan), B)
    for trans in ("N", "C"):
        serinv_np.pobtas(D, L, R, T, B, trans=trans, partial=True)
        algs.pobtas(d, l, rr, t, bb, trans=trans, partial=True)
        assert relerr(to_host(bb)[0], B) < TOL, trans


@pytest.mark.parametrize("n,b,a,r", [(4, 130, 300, 1), (8, 65, 500, 1), (1, 256, 300, 4), (40, 64, 300, 1)])
def test_wide_arrows_are_not_slower_than_the_tile_sweep(gpu_device, monkeypatch, n, b, a, r):
    """1.25 to 1.8 of its time where the inverses were formed all the same."""
    import torch

    import serinv_amd.algs as algs

    monkeypatch.setitem(algs.config, "check_info", False)
    D, L, R, T, B = bta_spd(n, b, a, seed=7700 + n, n_rhs=r)
    F = to_dev(gpu_device, D, L, R, T)
    algs.pobtaf(*F)
    y = to_dev(gpu_device, B)[0]
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    best = {}
    for _ in range(20):
        for form in ("sweep", ""):
            if form:
                monkeypatch.setenv("ROCBTA_POBTAS_ALGO", form)
            else:
                monkeypatch.delenv("ROCBTA_POBTAS_ALGO")
            x = y.clone()
            torch.cuda.synchronize()
            start.record()
            algs.pobtas(*F, x, trans="N")
            algs.pobtas(*F, x, trans="C")
            end.record()
            end.synchronize()
            best[form] = min(best.get(form, float("inf")), start.elapsed_time(end))
    algs.check_status()
    print(f"pobtas n={n} b={b} a={a} r={r}: {best}", flush=True)
    assert best[""] < 1.15 * best["sweep"], best
