"""Strides that the many-row head products read their queries through (no GPU):
whatever view comes in, the strides handed on address its elements, in multiples of
eight."""
import itertools

import pytest
import torch

from voom_amd import ops


@pytest.mark.parametrize("B,H,L,D", [(1, 4, 3, 8), (1, 1, 1, 8), (2, 1, 3, 16), (2, 3, 1, 8)])
def test_strides_of_views(B, H, L, D):
    for odd in itertools.product((3, 8, 1001), repeat=3):
        want = (H * L * D, L * D, D)
        for keep in ((), (0, 1, 2)):  # odd strides of single entries only, or of all
            shape = (B, H, L, D)
            strides = [odd[i] if shape[i] == 1 or i in keep else want[i] for i in range(3)]
            x = torch.arange(1 << 14, dtype=torch.float32).as_strided(shape, (*strides, 1))
            y, s = ops._token_rows(x)
            assert all(v % 8 == 0 for v in s)
            assert torch.equal(y.as_strided(shape, (*s, 1), y.storage_offset()), x)


def test_aligned_views_are_not_copied():
    x = torch.zeros((2, 5, 3, 8)).transpose(1, 2)
    y, s = ops._token_rows(x)
    assert y is x and s == [120, 8, 24]
    y, s = ops._token_rows(torch.zeros((2, 3, 8, 5)).transpose(2, 3))
    assert y.is_contiguous() and s == [120, 40, 8]
