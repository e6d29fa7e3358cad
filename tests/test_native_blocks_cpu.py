"""The native host module loads without a GPU, binds to the library and hands back what is not its case."""
import torch

from torchtitan_amd import _lib, ops


def test_module_binds_and_hands_back_cpu_tensors():
    blocks = _lib.blocks()
    x, w = torch.zeros(4, 256, dtype=torch.bfloat16), torch.zeros(256, 256, dtype=torch.bfloat16)
    assert blocks.linear_forward(x, w, 1, 128) is None
    assert blocks.linear_backward(x, w, (256, 128, 256, 0, 0, 4), w, (256, 256, 384, 0, 0, 256), 1, 128, False, False) is None
    assert blocks.linear_apply(x, w, w, (256, 256, 384, 0, 0, 256), 1, False) is None
    assert blocks.ffn_forward(x, w, w, w, 1, 128) is None
    assert not ops.native_block_ok(x, 256, 256)
