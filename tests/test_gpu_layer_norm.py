"""The layer norm in pieces at the edges of its row widths, and the widths beside them that a value at a time takes."""
import pytest
import torch

from test_gpu_lusolix import test_layer_norm_behind_a_gated_add as _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hidden", [8, 1004, 2040, 2048, 2056, 4104, 8192, 8200, 16384])
def test_layer_norm_at_the_edges_of_its_pieces(dt, hidden):
    _check(dt, hidden)
