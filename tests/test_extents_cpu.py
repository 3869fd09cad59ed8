"""Host check of a freqs table's batches and heads: the kernels step through them by stride."""
import pytest
import torch


def test_freqs_extents_rule():
    from pope_amd.hip_pope_flash_attn import _check_freqs_extents
    t = torch.zeros(2, 3, 8, 16)
    _check_freqs_extents(t, 2, 3, 3)
    _check_freqs_extents(t, 1, 2, 2)
    _check_freqs_extents(t[:1, :1], 5, 5, 5)
    _check_freqs_extents(t[:1, :1].expand(2, 3, 8, 16), 5, 5, 5)
    _check_freqs_extents(t[0, 0], 5, 5, 5)
    _check_freqs_extents(t, 2, 6, 3)   # grouped heads: the library's own error
    for B, H in ((3, 3), (2, 4)):
        with pytest.raises(ValueError):
            _check_freqs_extents(t, B, H, H)
