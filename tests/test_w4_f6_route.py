"""Which calls come to the six-bit-float kernel of large batches: host arithmetic, no GPU."""
import pytest

import torch

from rumus_amd import nn, ops


# Its preparation gives a row's runs of 32 to a thread each, 512 of them: K counts with its padding to whole groups
@pytest.mark.parametrize("k,g", [(16384, 192), (16384, 320), (16384, 384), (16384, 640), (16384, 768), (16200, 384), (16136, 384),
                                 (14336, 6144), (9224, 9216), (16384, 32768), (11008, 12288), (16385, 64)])
def test_no_k_beyond_16384_once_padded(k, g):
    padded, _ = ops.w4_geometry(k, g)
    assert (padded > 16384) == (not any(ops.qmatmul_int4_block_takes(m, k, n, g) for m in (1500, 4096) for n in (4096, 11008)))


@pytest.mark.parametrize("k,g", [(16384, 64), (16384, 128), (16384, 256), (16320, 192), (16192, 16384), (1024, 64)])
def test_k_up_to_16384_is_taken(k, g):
    assert ops.qmatmul_int4_block_takes(4096, k, 11008, g)


# A decoder block calls a projection of the user's own, whatever it does around the layer
def test_projection_of_another_type_is_not_folded():
    class Own(nn.QLinear):
        pass

    array = lambda *s: torch.zeros(s)
    weight = nn.QuantizedTensor.__new__(nn.QuantizedTensor)
    weight.k, weight.n, weight.group_size, weight.perm = 4096, 4096, 128, None
    weight.packed_tensor, weight.scales_tensor, weight.zp_tensor = array(64), array(64), array(64)
    x = torch.empty(4096, 1)
    assert nn.DecoderBlockW4._folds_rows(nn.QLinear(weight, None), x)
    assert not nn.DecoderBlockW4._folds_rows(Own(weight, None), x)
    assert not nn.DecoderBlockW4._folds_rows(lambda x: x, x)
