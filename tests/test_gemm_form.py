"""The choice of the tiled products at the ends of the ranges they accept (host code:
no GPU is used)."""
import pytest

from laplace_amd import _lib

F32, F16, Q4_0, Q8_0, Q2_K, Q4_K, Q5_K, Q6_K, BF16 = 0, 1, 2, 8, 10, 12, 13, 14, 30


# the longest rows whose 128-row tile offsets stay within 32 bits: 2^25 bytes of weights,
# 2^25 elements of x
@pytest.mark.parametrize("t,longest", [(F32, 1 << 23), (F16, 1 << 24), (BF16, 1 << 24), (Q2_K, 1 << 25), (Q5_K, 1 << 25)])
def test_fact_gemm_row_offsets_fit_32_bits(t, longest):
    L = _lib.lib()
    assert L.lp_gemm_form(t, 2048, longest, 2048, None).startswith(b"fact_gemm ")
    assert L.lp_gemm_form(t, 2048, longest + 256, 2048, None) == b"fact"


# (type, M, K, N) on a 256-CU part, in pairs on either side of a line
@pytest.mark.parametrize("call,form", [
    ((Q8_0, 12, 1024, 2048), "i8t 32x32x4"), ((Q8_0, 12, 1088, 2048), "i8t 32x32x8"),
    ((Q6_K, 16, 1024, 4096), "i8t 32x32x4"), ((Q6_K, 17, 1280, 4096), "i8t 32x32x8"),
    ((Q6_K, 9, 256, 14336), "i8t 32x128"), ((Q6_K, 9, 512, 14336), "i8t 32x32x4"),
    ((Q4_0, 5, 512, 32768), "i8t 32x128"), ((Q4_0, 5, 576, 32768), "i8t 32x32x4"),
])
def test_short_rows_take_fewer_k_groups(call, form):
    """Where a row has too few stages for eight groups of waves to share."""
    t, M, K, N = call
    assert _lib.lib().lp_gemm_form(t, M, K, N, None).decode() == form


@pytest.mark.parametrize("t,M,K,N,tiled", [
    (BF16, 12, 4096, 2048, False), (BF16, 13, 4096, 2048, True), (BF16, 16, 4096, 2048, True), (BF16, 8, 3072, 3072, False),
    (BF16, 6, 4096, 4096, True), (BF16, 8, 4096, 4096, True),
    (Q5_K, 8, 3072, 3072, False), (Q5_K, 9, 3072, 3072, True), (Q5_K, 6, 3072, 10240, False), (Q5_K, 7, 3072, 10240, True),
    (Q5_K, 8, 2048, 10240, False), (Q5_K, 9, 2048, 10240, True), (Q5_K, 5, 1024, 10240, True), (Q5_K, 6, 4096, 4096, True),
    (Q2_K, 6, 4096, 10240, False), (Q2_K, 7, 4096, 10240, True), (Q2_K, 6, 2048, 14336, False), (Q2_K, 7, 2048, 14336, True),
    (F16, 16, 4096, 3072, False), (F16, 12, 4096, 4096, True), (F16, 16, 8192, 3072, True), (BF16, 8, 8192, 3072, True)])
def test_fact_gemm_lines(t, M, K, N, tiled):
    """The tiled product takes calls where it measured faster than the GEMVs."""
    got = _lib.lib().lp_gemm_form(t, M, K, N, None).decode()
    assert got.startswith("fact_gemm ") if tiled else got == "fact"


@pytest.mark.parametrize("t,M,K,N,tiled", [
    (Q4_K, 33, 4096, 18944, False), (Q4_K, 48, 4096, 32768, True), (Q4_K, 33, 2048, 18944, True), (Q4_K, 33, 4096, 14336, True),
    (Q4_K, 130, 4096, 14336, False), (Q4_K, 192, 4096, 14336, True), (Q4_K, 130, 4096, 12288, True), (Q4_K, 130, 2048, 14336, True),
    (Q4_K, 128, 4096, 14336, True), (Q4_K, 160, 3072, 14336, True), (Q4_K, 130, 3072, 14336, False),
    (Q4_0, 9, 14336, 512, False), (Q4_0, 13, 14336, 512, True), (Q4_0, 12, 18944, 512, False), (Q4_0, 9, 18944, 768, True),
    (Q4_0, 9, 10240, 512, True), (Q4_0, 17, 18944, 512, True)])
def test_int8_product_lines(t, M, K, N, tiled):
    """The tiled int8 product takes calls where it measured faster than the kernels beside it."""
    assert _lib.lib().lp_gemm_form(t, M, K, N, None).decode().startswith("i8t ") == tiled
