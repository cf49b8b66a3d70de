"""The choice of the tiled products at the ends of the ranges they accept (host code:
no GPU is used)."""
import pytest

from laplace_amd import _lib

F32, F16, BF16, Q2_K, Q5_K = 0, 1, 30, 10, 13


# the longest rows whose 128-row tile offsets stay within 32 bits: 2^25 bytes of weights,
# 2^25 elements of x
@pytest.mark.parametrize("t,longest", [(F32, 1 << 23), (F16, 1 << 24), (BF16, 1 << 24), (Q2_K, 1 << 25), (Q5_K, 1 << 25)])
def test_fact_gemm_row_offsets_fit_32_bits(t, longest):
    L = _lib.lib()
    assert L.lp_gemm_form(t, 2048, longest, 2048, None).startswith(b"fact_gemm ")
    assert L.lp_gemm_form(t, 2048, longest + 256, 2048, None) == b"fact"
