"""The block sweep of pobtas at the edges of its two forms
(serinv_amd/csrc/solve_block.hpp): rows of a phase in registers up to b = 1024,
streamed rows beyond.

pobtas (src/serinv/algs/pobtas.py:80-159) with ROCBTA_POBTAS_ALGO=block against
the oracle at 1e-12 relative (max-norm), both directions and the partial
solves, for 1, 4 and 8 columns and ragged groups of them, row groups that end
inside and at a block's edge, and arrows up to the widest the sweep takes.
"""

import numpy as np
import pytest

from oracle import serinv_np
from serinv_amd.utils.matrices import bta_spd
from tests._helpers import relerr, to_dev, to_host

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.mark.parametrize("partial", [False, True])
@pytest.mark.parametrize("n,b,a,r", [(1, 5, 3, 1), (4, 1, 2, 4), (3, 65, 0, 3), (4, 130, 70, 4), (3, 255, 512, 1),
                                     (3, 257, 128, 2), (3, 258, 64, 7), (2, 513, 32, 11), (3, 1023, 9, 1),
                                     (2, 1024, 257, 1), (2, 1028, 5, 4), (3, 1100, 300, 1)])
def test_block_solve_matches_oracle(gpu_device, monkeypatch, n, b, a, r, partial):
    import serinv_amd.algs as algs

    monkeypatch.setenv("ROCBTA_POBTAS_ALGO", "block")
    print(f"block pobtas n={n} b={b} a={a} r={r} partial={partial}", flush=True)
    D, L, R, T, B = bta_spd(n, b, a, seed=5200 + n + b + a + r, n_rhs=r)
    serinv_np.pobtaf(D, L, R, T)
    d, l, rr, t, bb = to_dev(gpu_device, D, L, R, T, B)
    for trans in ("N", "C"):
        serinv_np.pobtas(D, L, R, T, B, trans=trans, partial=partial)
        algs.pobtas(d, l, rr, t, bb, trans=trans, partial=partial)
        assert relerr(to_host(bb)[0], B) < TOL, trans


@pytest.mark.parametrize("n,b,a,r", [(31, 64, 3, 2), (32, 64, 3, 1), (32, 64, 0, 2), (7, 96, 12, 1), (8, 96, 12, 1),
                                     (8, 96, 12, 2), (9, 65, 5, 8), (9, 65, 5, 9), (2, 512, 4, 2), (2, 528, 4, 4),
                                     (2, 528, 4, 5), (32, 64, 600, 1)])
def test_default_solve_matches_oracle(gpu_device, monkeypatch, n, b, a, r):
    """The form the sizes select, on both sides of each line of the rule."""
    import serinv_amd.algs as algs

    monkeypatch.delenv("ROCBTA_POBTAS_ALGO", raising=False)
    print(f"pobtas n={n} b={b} a={a} r={r}", flush=True)
    D, L, R, T, B = bta_spd(n, b, a, seed=5600 + n + b + a + r, n_rhs=r)
    serinv_np.pobtaf(D, L, R, T)
    d, l, rr, t, bb = to_dev(gpu_device, D, L, R, T, B)
    for trans in ("N", "C"):
        serinv_np.pobtas(D, L, R, T, B, trans=trans)
        algs.pobtas(d, l, rr, t, bb, trans=trans)
        assert relerr(to_host(bb)[0], B) < TOL, trans
