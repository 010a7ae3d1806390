"""pobtaf with factorize_last_block=False under arrows of more than one 64-row tile:
few tile columns run launch by launch, more of them on the persistent kernel
(rocbta_dpobtaf).

pobtaf (src/serinv/algs/pobtaf.py:143-159) against the oracle at 1e-12 relative
(max-norm) on both sides of the line, in FP64 and, at 1e-5, with FP32 products; and
a call below the line takes no longer than the forced launch-by-launch form.
"""

import numpy as np
import pytest

from oracle import serinv_np
from serinv_amd.utils.matrices import bta_spd
from tests._helpers import relerr, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n,b,a", [(2, 1, 65), (2, 17, 66), (2, 64, 128), (2, 65, 129), (2, 128, 65), (2, 129, 70),
                                   (3, 40, 65), (3, 64, 200), (3, 65, 66), (4, 64, 65), (2, 64, 64), (1, 30, 80)])
def test_open_factor_matches_oracle(gpu_device, monkeypatch, n, b, a, mixed):
    import serinv_amd.algs as algs
    from serinv_amd.mixed import pobtaf_mixed

    monkeypatch.delenv("ROCBTA_POBTAF_ALGO", raising=False)
    print(f"open pobtaf n={n} b={b} a={a} mixed={mixed}", flush=True)
    D, L, R, T, _ = bta_spd(n, b, a, seed=7300 + n + b + a)
    d, l, r, t = to_dev(gpu_device, D, L, R, T)
    (pobtaf_mixed if mixed else algs.pobtaf)(d, l, r, t, factorize_last_block=False)
    serinv_np.pobtaf(D, L, R, T, factorize_last_block=False)
    got, want = to_host(d, l, r, t), [D, L, R, T]
    for x in (got, want):  # blocks that stay symmetric hold their lower triangle
        x[0], x[3] = x[0].copy(), np.tril(x[3])
        x[0][-1] = np.tril(x[0][-1])
    for name, x, y in zip("DLRT", got, want):
        if y.size:
            assert relerr(x, y) < (1e-5 if mixed else 1e-12), name


def test_few_columns_are_not_slower_than_launch_by_launch(gpu_device, monkeypatch):
    """n=2 b=16 a=100: half of the persistent kernel's time (34 of 69 us)."""
    import torch

    import serinv_amd.algs as algs

    monkeypatch.setitem(algs.config, "check_info", False)
    A = to_dev(gpu_device, *bta_spd(2, 16, 100, seed=7400)[:4])
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    best = {}
    for _ in range(40):
        for form in ("loop", "default"):
            if form == "loop":
                monkeypatch.setenv("ROCBTA_POBTAF_ALGO", "loop")
            else:
                monkeypatch.delenv("ROCBTA_POBTAF_ALGO", raising=False)
            F = [x.clone() for x in A]
            torch.cuda.synchronize()
            start.record()
            algs.pobtaf(*F, factorize_last_block=False)
            end.record()
            end.synchronize()
            best[form] = min(best.get(form, float("inf")), start.elapsed_time(end))
    algs.check_status()
    print(f"open pobtaf n=2 b=16 a=100: {best}", flush=True)
    assert best["default"] < 1.5 * best["loop"], best
