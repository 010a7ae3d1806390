"""Workspace sizes of pobtas and pobtaf (rocbta_workspace_bytes), on the host."""

import pytest

from serinv_amd import _lib


@pytest.mark.parametrize("b", [24, 64, 65, 96, 128, 130, 200, 255, 256, 300, 512, 528, 1024, 1040, 1100])
def test_pobtas_workspace_serves_fewer_columns(b):
    """A caller that keeps one workspace for its widest right-hand side solves
    narrower ones in it, whichever sweep the number of columns selects; of blocks
    from 256 on, up to 8 columns."""
    lib = _lib.load()
    for n in (1, 4, 8, 32, 64):
        for a in (0, 8, 70, 300, 600):
            sizes = [lib.rocbta_workspace_bytes(_lib.OP_POBTAS, n, b, a, r) for r in range(1, 72 if b < 256 else 9)]
            assert all(x <= y for x, y in zip(sizes, sizes[1:])), (n, b, a, sizes[:12])


def test_pobtas_workspace_holds_no_unused_transposes():
    """Blocks whose rows a sweep keeps in registers are read where they are: beside
    the block inverses (n b^2) and the scratch of forming them (a quarter of that)
    nothing grows with n b^2."""
    n, b, a = 256, 1024, 32
    size = _lib.load().rocbta_workspace_bytes(_lib.OP_POBTAS, n, b, a, 1)
    assert size < 1.3 * 8 * n * b * b


@pytest.mark.parametrize("n,b,a", [(538, 7, 75), (220, 28, 140), (420, 91, 65), (16, 91, 545), (62, 130, 265)])
def test_pobtaf_of_wide_arrows_fits_the_static_scratch(n, b, a):
    """The largest arrows that the static scratch of rocbta_dpobtaf_noalloc holds
    with five flags and two per tile of a block for each tile column: the flags of
    an arrow's further tiles take no room of their own."""
    lib = _lib.load()
    nt = -(-b // 64)

    def pad(x):
        return -(-x // 256) * 256

    size = (pad(8 * 64 * 64) + 3 * 256 + pad(4 * (n * nt + 2) * (5 + 2 * nt)) + pad(8 * n * nt)
            + pad(8 * 64 * 64 * n * nt) + pad(8 * n * a * a) + pad(8 * b * b) + pad(8 * a * b) + pad(8 * a * a))
    assert lib.rocbta_workspace_bytes(_lib.OP_POBTAF, n, b, a, 0) <= size <= lib.rocbta_noalloc_scratch_bytes()
