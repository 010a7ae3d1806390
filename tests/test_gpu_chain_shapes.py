"""The persistent factorization at ragged last tiles and at arrows of more
than one 64-row tile (serinv_amd/csrc/pobtaf_chain.hpp).

pobtaf (src/serinv/algs/pobtaf.py:69-183) against the oracle at 1e-12
relative (max-norm): block sizes around the 16-column panels and the 64-wide
tiles, arrows around one and two tiles, both settings of
factorize_last_block; and the failing column of a matrix that is not positive
definite, inside a ragged tile.
"""

import numpy as np
import pytest

from oracle import serinv_np
from serinv_amd.utils.matrices import bta_spd
from tests._helpers import relerr, to_dev, to_host

TOL = 1e-12


@pytest.fixture(scope="module")
def algs(gpu_device):
    import serinv_amd.algs as A

    return A


@pytest.mark.gpu
@pytest.mark.parametrize("last", [True, False])
@pytest.mark.parametrize("n,b,a", [(5, 1, 3), (4, 15, 1), (4, 16, 65), (4, 17, 64), (3, 31, 128), (3, 48, 129),
                                   (3, 63, 200), (3, 65, 70), (4, 80, 12), (3, 112, 65), (3, 130, 0), (2, 143, 96),
                                   (1, 64, 70), (1, 70, 130), (2, 192, 100)])
def test_factor_matches_oracle(algs, gpu_device, n, b, a, last):
    print(f"pobtaf n={n} b={b} a={a} last={last}", flush=True)
    D, L, R, T, _ = bta_spd(n, b, a, seed=4100 + 7 * n + b + a)
    d, l, r, t = to_dev(gpu_device, D, L, R, T)
    serinv_np.pobtaf(D, L, R, T, factorize_last_block=last)
    algs.pobtaf(d, l, r, t, factorize_last_block=last)
    got, want = to_host(d, l, r, t), [D, L, R, T]
    if not last:  # blocks that stay symmetric hold their lower triangle
        for x in (got, want):
            x[0], x[3] = x[0].copy(), np.tril(x[3])
            x[0][-1] = np.tril(x[0][-1])
    for name, x, y in zip("DLRT", got, want):
        assert relerr(x, y) < TOL, name


@pytest.mark.gpu
@pytest.mark.parametrize("b,a,block,col", [(70, 3, 1, 66), (130, 70, 0, 129), (17, 0, 2, 16), (33, 5, 2, 0)])
def test_failing_column_in_ragged_tile(algs, gpu_device, b, a, block, col):
    n = 3
    print(f"pobtaf not positive definite b={b} a={a} block={block} col={col}", flush=True)
    D, L, R, T, _ = bta_spd(n, b, a, seed=4200 + b)
    D[block, col, col] = -1.0
    d, l, r, t = to_dev(gpu_device, D, L, R, T)
    with pytest.raises(np.linalg.LinAlgError) as ei:
        if a:
            algs.pobtaf(d, l, r, t)
        else:
            algs.pobtf(d, l)
    assert f"order {block * b + col + 1} " in str(ei.value)


@pytest.mark.parametrize("a", [65, 96, 128, 129, 200])
def test_schedule_of_wide_arrows(a):
    """Task decoding and dependencies for several arrow tiles, on the host."""
    from serinv_amd import _lib

    lib = _lib.load()
    for n in (1, 2, 3, 7):
        for b in (1, 17, 63, 64, 65, 130, 192):
            assert lib.rocbta_dag_selfcheck_arrows(n, b, a) == 0, (n, b, a)
