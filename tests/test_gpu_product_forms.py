"""The grouped products in every storage form of their operands and in launches of
64-wide tiles (serinv_amd/csrc/gemm_f64.hpp: load groups of 16 k, 32 x 32 blocks,
one or two terms).

The A X A^T = B forms of ddbtasc / ddbtasci, natural and permuted
(src/serinv/algs/ddbtasc.py:335-475, 478-710, ddbtasci.py:343-576, 578-845), hold
products with neither, either and both operands transposed, of one and two terms:
against the oracle at 1e-12 relative (max-norm per output array).  Selected
inversions of many block rows launch 64-wide tiles, with lower-triangular and
mirrored outputs: against the oracle at 1e-12, with FP32 products at 1e-5.
"""

import numpy as np
import pytest

from oracle import dense, generators, serinv_np
from serinv_amd.utils.matrices import bta_spd
from tests._helpers import relerr, to_dev, to_host

pytestmark = pytest.mark.gpu
TOL = 1e-12
KEYS = ("B_diagonal_blocks", "B_lower_diagonal_blocks", "B_upper_diagonal_blocks", "B_lower_arrow_blocks",
        "B_upper_arrow_blocks", "B_arrow_tip_block")
BUFS = ("A_lower_buffer_blocks", "A_upper_buffer_blocks", "B_lower_buffer_blocks", "B_upper_buffer_blocks")


def _quadratic_arrays(b, a, n):
    rng = np.random.default_rng(6300 + b + 7 * a + 13 * n)
    A, B = generators.dd_bta(b, a, n, rng), generators.dd_bta(b, a, n, rng)
    generators.symmetrize(B)
    return [list(dense.bta_dense_to_arrays_full(x, b, a, n)) for x in (A, B)]


@pytest.mark.parametrize("b,a,n", [(15, 17, 3), (16, 16, 3), (17, 1, 4), (31, 33, 3), (32, 32, 3), (33, 31, 3),
                                   (47, 5, 3), (48, 50, 3), (63, 64, 3), (80, 15, 3), (97, 66, 3), (144, 48, 3)])
def test_quadratic_forms_match_oracle(gpu_device, b, a, n):
    import serinv_amd.algs as algs

    print(f"quadratic b={b} a={a} n={n}", flush=True)
    A, B = _quadratic_arrays(b, a, n)
    g, gb = to_dev(gpu_device, *A), to_dev(gpu_device, *B)
    rhs = dict(zip(KEYS, gb))
    for step in ("ddbtasc", "ddbtasci"):
        getattr(algs, step)(*g, rhs=rhs, quadratic=True)
        getattr(serinv_np, step + "_quadratic")(*A, *B)
        for x, y in zip(to_host(*g, *gb), A + B):
            assert relerr(x, y) < TOL, step


@pytest.mark.parametrize("b,a,n", [(17, 15, 4), (32, 33, 4), (48, 16, 4), (65, 31, 4), (97, 66, 4)])
def test_permuted_quadratic_forms_match_oracle(gpu_device, b, a, n):
    import serinv_amd.algs as algs

    print(f"permuted quadratic b={b} a={a} n={n}", flush=True)
    A, B = _quadratic_arrays(b, a, n)
    Z = [np.zeros_like(A[1]) for _ in range(4)]
    g, gb, gz = to_dev(gpu_device, *A), to_dev(gpu_device, *B), to_dev(gpu_device, *Z)
    for step in ("ddbtasc", "ddbtasci"):
        getattr(algs, step)(*g, rhs=dict(zip(KEYS, gb)), quadratic=True, buffers=dict(zip(BUFS, gz)))
        getattr(serinv_np, step + "_quadratic_permuted")(*A, *Z[:2], *B, *Z[2:])
        for x, y in zip(to_host(*g, *gb, *gz), A + B + Z):
            assert relerr(x, y) < TOL, step


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n,b,a", [(128, 64, 5), (64, 97, 33), (64, 130, 66), (40, 144, 0), (32, 200, 31)])
def test_selected_inverse_on_wide_tiles(gpu_device, n, b, a, mixed):
    """At least 512 tiles of 64 x 64 in the batched launches."""
    import serinv_amd.algs as algs
    from serinv_amd.mixed import pobtasi_mixed

    print(f"pobtasi n={n} b={b} a={a} mixed={mixed}", flush=True)
    D, L, R, T, _ = bta_spd(n, b, a, seed=6400 + n + b + a)
    serinv_np.pobtaf(D, L, R, T)
    g = to_dev(gpu_device, D, L, R, T)
    (pobtasi_mixed if mixed else algs.pobtasi)(*g)
    serinv_np.pobtasi(D, L, R, T)
    for name, x, y in zip("DLRT", to_host(*g), (D, L, R, T)):
        assert relerr(x, y) < (1e-5 if mixed else TOL), name


def test_transposed_operands_keep_up(gpu_device):
    """The permuted inversion of the quadratic form takes 3.7 times the products of
    the plain one, a third of them with a transposed operand: no more than 4 times
    its time (4.7 where those took half as long again)."""
    import torch

    import serinv_amd.algs as algs

    n, b, a = 6, 1024, 32
    gen = torch.Generator(device=gpu_device).manual_seed(63)

    def dominant():
        rand = lambda *s: torch.rand(s, dtype=torch.float64, device=gpu_device, generator=gen)  # noqa: E731
        D, T = rand(n, b, b), rand(a, a)
        D.diagonal(dim1=1, dim2=2).add_(3 * b + a)
        T.diagonal().add_(n * b + a)
        return [D, rand(n - 1, b, b), rand(n - 1, b, b), rand(n, a, b), rand(n, b, a), T]

    A, B = dominant(), dominant()
    Z = [torch.zeros_like(A[1]) for _ in range(4)]
    algs.ddbtasc(*A, rhs=dict(zip(KEYS, B)), quadratic=True, buffers=dict(zip(BUFS, Z)))
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    best = {}
    for _ in range(6):
        for name in ("plain", "quadratic"):
            A1, B1, Z1 = ([x.clone() for x in y] for y in (A, B, Z))
            start.record()
            if name == "plain":
                algs.ddbtasci(*A1, buffers=dict(zip(BUFS[:2], Z1[:2])))
            else:
                algs.ddbtasci(*A1, rhs=dict(zip(KEYS, B1)), quadratic=True, buffers=dict(zip(BUFS, Z1)))
            end.record()
            end.synchronize()
            best[name] = min(best.get(name, float("inf")), start.elapsed_time(end))
    print(f"ddbtasci permuted n={n} b={b} a={a}: {best}", flush=True)
    assert best["quadratic"] < 4.0 * best["plain"], best


def test_ragged_edges_keep_up(gpu_device):
    """FP32 products at block sizes that are no multiple of the tiles: the selected
    inversion takes no longer with them than with FP64 ones (0.9 of its time; 1.3
    where edge blocks waited for each of their loads)."""
    import torch

    import serinv_amd.algs as algs
    from serinv_amd.mixed import pobtasi_mixed

    n, b, a = 12, 1100, 32
    gen = torch.Generator(device=gpu_device).manual_seed(64)
    rand = lambda *s: torch.rand(s, dtype=torch.float64, device=gpu_device, generator=gen)  # noqa: E731
    D, T = rand(n, b, b), rand(a, a)
    D.diagonal(dim1=1, dim2=2).add_(3 * b + a)
    T.diagonal().add_(n * b + a)
    F = [D, rand(n - 1, b, b), rand(n, a, b), T]
    algs.pobtaf(*F)
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    best = {}
    for _ in range(6):
        for fn in (algs.pobtasi, pobtasi_mixed):
            F1 = [x.clone() for x in F]
            start.record()
            fn(*F1)
            end.record()
            end.synchronize()
            best[fn.__name__] = min(best.get(fn.__name__, float("inf")), start.elapsed_time(end))
    print(f"selected inversion n={n} b={b} a={a}: {best}", flush=True)
    assert best["pobtasi_mixed"] < 1.08 * best["pobtasi"], best
