"""Batch.run names the first item at fault in order: tier "auto" or a malformed item."""
import numpy as np
import pytest

from gbskernels_amd.serving import Batch

M = np.eye(2)


@pytest.mark.parametrize("items,message", [
    ([("perm", "auto", M), ("x",)], "auto"), ([("x",), ("perm", "auto", M)], "unpack"),
    ([("perm", "fp64", M), ("perm", "auto", M)], "auto"), ([("perm", "auto", M), ("perm", np.array([1, 2]), M)], "auto"),
    ([("perm", np.array([1, 2]), M), ("perm", "auto", M)], "ambiguous")])
def test_first_fault_is_named(items, message):
    b = Batch.__new__(Batch)  # no device: the checks come first
    b._h = 1
    try:
        with pytest.raises(ValueError, match=message):
            b.run(items)
    finally:
        b._h = None
