"""Host arithmetic of the launches (no GPU): workspace sizes, and how batches are
cut so that every launch stays below HIP's 2^32 work-items."""
import pytest

from gbskernels_amd import _lib


@pytest.mark.parametrize("N", range(14, 30, 2))
@pytest.mark.parametrize("func", ["haf", "lhaf"])
def test_tree_workspace_is_what_the_kernels_write(func, N):
    """One partial (value and double) per include pattern of all but four pairs."""
    for tier, elem in (("fp64", 16), ("kappa", 16), ("certified", 16), ("dd", 32), ("dd_certified", 32)):
        got = _lib.lib().gbs_workspace_bytes(_lib.FUNCS[func], _lib.TIERS[tier], N, 1000)
        assert got == 1000 * 2 ** (N // 2 - 4) * (elem + 8)
