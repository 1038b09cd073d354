"""The layer norm in pieces at the edges of its row widths, and the widths beside them that a value at a time takes."""
import pytest
import torch

from test_gpu_lusolix import test_layer_norm_behind_a_gated_add as _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hidden", [8, 1004, 2040, 2048, 2056, 4104, 8192, 8200, 16384])
def test_layer_norm_at_the_edges_of_its_pieces(dt, hidden):
    _check(dt, hidden)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("taps,width", [(1, 8), (2, 2056), (3, 40), (4, 2048), (4, 100), (5, 40)])
def test_short_convolution_in_pieces_gives_the_walks_bits(dt, taps, width):
    """Three requests, the first behind rows of its own in the state: rows in pieces, and beside them the widths and the taps
    that take a channel a thread, against the walk over each request's rows."""
    from tokenmill_amd.hip.library import library
    import ctypes
    P, I = lambda t: ctypes.c_void_p(t.data_ptr() if t is not None else None), ctypes.c_int
    lib, code = library(), 1 if dt == torch.bfloat16 else 0
    g = torch.Generator(device="cuda").manual_seed(width + taps)
    lens = [1, 70, 3]
    h = torch.randn(sum(lens), width, generator=g, device="cuda").to(dt)
    w = torch.randn(width, taps, generator=g, device="cuda").to(dt)
    state = torch.randn(4, max(taps - 1, 1), width, generator=g, device="cuda").to(dt)
    cu = torch.tensor([0, 1, 71, 74], dtype=torch.int32, device="cuda")
    slots = torch.tensor([2, 0, 3], dtype=torch.int32, device="cuda")
    seq = torch.repeat_interleave(torch.arange(3, dtype=torch.int32), torch.tensor(lens)).cuda()
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    out, want = torch.full_like(h, float("nan")), torch.full_like(h, float("nan"))
    assert lib.tm_short_conv(P(h), P(out), P(w), P(state), P(cu), P(slots), P(seq), I(len(h)), I(width), I(taps), I(code), stream) == 0
    if taps == 1:
        want = (h.float() + h.float() * w[:, 0].float()).to(dt)
    else:
        assert lib.tm_short_conv_walk(P(h), P(want), P(w), P(state), P(cu), P(slots), I(3), I(width), I(taps), I(code), stream) == 0
    assert torch.equal(out, want)
