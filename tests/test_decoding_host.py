"""Host-side rules of the decode caches (no GPU)."""

from __future__ import annotations

import numpy as np
import pytest
import torch


@pytest.mark.parametrize("widths", [(128, 128), (128, 128, 128, 128, 64, 64)])
@pytest.mark.parametrize("B", [1, 3])
def test_column_group_takes_slices_of_one_tensor_only(B, widths):
    """Slices of one projection are one view. Tensors of their own that happen to
    lie side by side in memory (one row of 512 bytes each, as a caching allocator
    places them) are not: a view past the first one's storage does not exist."""
    from kch.decoding_cache import _column_group
    x = torch.randn(B, 1, sum(widths))
    g = _column_group(list(x.split(widths, -1)))
    assert g.shape == x.shape and g.data_ptr() == x.data_ptr() and torch.equal(g, x)
    assert _column_group(list(x.split(widths, -1))[::-1]) is None
    if B == 1:
        flat = np.arange(sum(widths), dtype=np.float32)
        at = np.cumsum((0, *widths))
        own = [torch.from_numpy(flat[a:b]).view(1, 1, -1) for a, b in zip(at, at[1:])]
        assert own[1].data_ptr() == own[0].data_ptr() + 4 * widths[0]
        assert _column_group(own) is None
