"""The host side of the fp32 operands' fp16 conversion: what the kernel would read through raw pointers is checked
before it is launched."""
import pytest
import torch


class _Library:
    def __init__(self):
        self.casts = 0

    def pope_cast_f16(self, *args):
        self.casts += 1
        return 0


@pytest.mark.parametrize("which", [1, 2])
def test_operands_on_other_devices_never_reach_the_kernel(monkeypatch, which):
    """Checked with meta tensors: an address on another GPU would be a fault where peers cannot be read."""
    from pope_amd import _lib, hip_pope_flash_attn as fa
    library = _Library()
    monkeypatch.setattr(_lib, "lib", lambda: library)
    monkeypatch.setattr(fa, "_stream", lambda t: 0)
    ts = [torch.zeros(1, 2, 3, 8, device="meta" if i == which else "cpu") for i in range(3)]
    with pytest.raises(RuntimeError, match="operand on meta"):
        fa._launch_half(ts, torch.zeros(1, dtype=torch.int32))
    assert library.casts == 0
    fa._launch_half([torch.zeros(1, 2, 3, 8)] * 3, torch.zeros(1, dtype=torch.int32))
    assert library.casts == 1
