"""The wide product of few bfloat16 rows into 32-bit results against 64 bits: columns that fill no tile, K of less than a round, of several with a rest, of an
odd number of steps; a row is the same whatever rows are beside it."""
from __future__ import annotations

import ctypes

import pytest
import torch

from tokenmill_amd.hip.library import library

pytestmark = pytest.mark.gpu
P, I = ctypes.c_void_p, ctypes.c_int


def _product(a, w, lda=None, ldc=None):
    M, (N, K) = a.shape[0], w.shape
    ldc = ldc or N
    out = torch.full((M, ldc), float("nan"), device="cuda")
    rc = library().tm_gemv_bf16(P(a.data_ptr()), I(lda or a.stride(0)), P(w.data_ptr()), P(out.data_ptr()), I(ldc), I(M), I(N), I(K),
                                P(torch.cuda.current_stream().cuda_stream))
    return rc, out


@pytest.mark.parametrize("N,K", [(16384, 32), (16420, 96), (16388, 896), (20000, 928), (16400, 3584)])
def test_against_64_bits_and_the_same_beside_other_rows(N, K):
    g = torch.Generator(device="cuda").manual_seed(N + K)
    wide = torch.randn(16, K + 8, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    ref = wide[:, :K].double() @ w.double().T
    rc, most = _product(wide[:, :K], w, ldc=N + 4)
    assert rc == 0 and most[:, N:].isnan().all()
    # exact products; 32-bit sums of at most about 5, a wavefront's chain of K / (4 x 8) of them and the lanes' inside an instruction
    assert (most[:, :N].double() - ref).abs().max() <= 2.0 ** -24 * 5 * (16 + K ** 0.5)
    for rows in (1, 7, 8, 9):
        rc, out = _product(wide[:rows, :K], w)
        assert rc == 0 and torch.equal(out, most[:rows, :N]), rows


def test_what_it_does_not_take_is_refused():
    a, w = torch.zeros(17, 64, dtype=torch.bfloat16, device="cuda"), torch.zeros(16384, 64, dtype=torch.bfloat16, device="cuda")
    assert _product(a[:16], w)[0] == 0
    for x, m, lda in ((a, w, None), (a[:0], w, None), (a[:4], w[:16380], None), (a[:4], w.view(32768, 32)[:32767], None), (a[:4, 4:], w, None),
                      (a[:4], w, 60), (a[:4], w.view(-1)[:16384 * 48 // 48 * 48].view(16384, 48), None)):
        assert _product(x, m, lda)[0] != 0
