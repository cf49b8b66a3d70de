"""The tiled bf16-MFMA product (F32, F16, BF16, Q2_K, Q3_K, Q5_K prompt rows) at the
edges of its tiles and forms, against 64-bit products and the oracle."""
import numpy as np
import pytest

from hip_util import form, normwise
from test_gpu_fact import BF16, BLOCK, F16, F32, FACT, Q2_K, Q3_K, Q5_K, fact_weights, gemm_dev

pytestmark = pytest.mark.gpu
DENSE = {"F32": F32, "F16": F16, "BF16": BF16}

# Per 64 elements (32 of Q5_K) the leading products are summed in fp32: at most 64
# half-ulps of a partial sum, 64 * 2^-25 = 2e-6; the dropped products and the result's
# rounding are below 2^-22. The oracle rounds an fp32 sum K <= 2048 times: with random
# signs ~sqrt(2048) half-ulps, 1.4e-6.
TOL = 4e-6

# (M, N, K): one token and one row past a 32- and 64-tile, K ending 32 elements into
# a 64-element stage (the unquantized types), fewer stages than K groups
SHAPES = [(33, 3001, 256), (65, 1537, 512), (8, 12289, 2304), (127, 900, 2048)]
TAILS = [(33, 3001, 32), (65, 1537, 96), (16, 8190, 288), (127, 801, 1056)]
# M and N that take each form: 32x32 with 8 (6) and 4 K groups, 64x64 with 2 and 1,
# 64x128, 128x128 (and its edges): test_every_form_is_run
FORMS = [(31, 8200, 256), (40, 8200, 256), (33, 14400, 256), (70, 8200, 256), (96, 16500, 256), (200, 24600, 256)]
CASES = [(t, *s) for t in FACT for s in SHAPES + FORMS] + [(t, *s) for t in DENSE for s in TAILS]


def test_every_form_is_run():
    """The cases run each tile form of the product for each type (on 256 CUs)."""
    import torch
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the forms' lines depend on the CU count")
    for name, t in FACT.items():
        got = {form(t, M, K, N) for n, M, N, K in CASES if n == name}
        forms = ("32x32x6", "64x64", "64x128") if name in ("F32", "F16") else ("32x32x8", "32x32x4", "64x64x2", "64x64", "128x128")
        assert got == {f"fact_gemm {f}" for f in forms}, (name, got)


@pytest.mark.parametrize("name,M,N,K", CASES)
def test_fact_gemm_matches_oracle(orc, name, M, N, K):
    print(f"fact gemm {name} M={M} N={N} K={K}", flush=True)
    t = FACT[name]
    assert form(t, M, K, N).startswith("fact_gemm ")
    w = fact_weights(t, K, N, seed=M + N + K + t)
    x = np.random.default_rng(M + 1).standard_normal((M, K)).astype(np.float32)
    x[M // 2, :32] = 0.0
    y = gemm_dev(t, x, w, N)
    rows = np.unique(np.linspace(0, N - 1, 48).astype(int))     # both ends and between
    rb = len(w) // N
    sub = np.concatenate([w[r * rb:(r + 1) * rb] for r in rows])
    assert normwise(y[:, rows], orc.gemm_scalar(t, x, sub, len(rows))) <= TOL


def dense(t, v):
    if t == F16:
        return v.astype(np.float16).astype(np.float32), v.astype(np.float16).view(np.uint8).reshape(-1)
    if t == BF16:
        u = v.view(np.uint32) & 0xffff0000
        return u.view(np.float32), (u >> 16).astype(np.uint16).view(np.uint8).reshape(-1)
    return v, v.view(np.uint8).reshape(-1)


@pytest.mark.parametrize("scale", [1e-35, 1.0, 1e30])
@pytest.mark.parametrize("name", list(DENSE))
def test_fact_gemm_pieces_keep_fp32(name, scale):
    """Every value is multiplied with its 24 bits, at any size: one product per
    output leaves its own rounding and the pieces' last bits."""
    t = DENSE[name]
    M, N, K = 64, 1600, 64
    assert form(t, M, K, N).startswith("fact_gemm ")
    rng = np.random.default_rng(3)
    x = np.zeros((M, K), np.float32)
    x[np.arange(M), np.arange(M)] = ((0.5 + rng.random(M)) * scale).astype(np.float32)
    v, wb = dense(t, rng.standard_normal((N, K)).astype(np.float32))
    y = gemm_dev(t, x, wb, N)
    ref = x.astype(np.float64) @ v.astype(np.float64).T
    assert np.all(np.abs(y - ref) <= 4 * 2.0 ** -24 * np.abs(ref) + 2.0 ** -149)


@pytest.mark.parametrize("name", ["Q2_K", "Q3_K", "Q5_K"])
def test_fact_gemm_quantized_extremes(orc, name):
    """Rows with an infinity, a NaN, values as large and as small as the codes leave room for
    match the oracle; the rows beside them stay as they are."""
    t = FACT[name]
    M, N, K = 40, 1700, 512
    assert form(t, M, K, N).startswith("fact_gemm ")
    w = fact_weights(t, K, N, seed=4)
    x = np.random.default_rng(6).standard_normal((M, K)).astype(np.float32)
    x[1, 7], x[2, 500], x[M - 1, 511] = np.inf, np.nan, -np.inf
    x[3, 9] = 1e36
    x[4] *= 1e-36
    y = gemm_dev(t, x, w, N)
    with np.errstate(all="ignore"):
        ref = orc.gemm_scalar(t, x, w, N)
    assert np.array_equal(np.isnan(y), np.isnan(ref)) and np.array_equal(np.isinf(y), np.isinf(ref))
    for m in range(M):
        f = np.isfinite(ref[m])
        assert np.array_equal(y[m][~f & ~np.isnan(ref[m])], ref[m][~f & ~np.isnan(ref[m])])
        if f.any():
            s = np.abs(ref[m][f]).max()
            assert normwise(y[m][f] / s, ref[m][f] / s) <= TOL, m


@pytest.mark.parametrize("M,N", [(40, 2500), (70, 8200), (200, 24600)])
@pytest.mark.parametrize("name", list(DENSE))
def test_fact_gemm_non_finite(name, M, N):
    """Infinities and NaN on either side, and sums past the fp32 range, come out as
    the plain products give them; all other outputs stay exact."""
    t = DENSE[name]
    K = 96
    rng = np.random.default_rng(5)
    assert form(t, M, K, N).startswith("fact_gemm ")
    x = rng.integers(-4, 5, (M, K)).astype(np.float32)
    v = rng.integers(-4, 5, (N, K)).astype(np.float32)
    x[x == 0] = 1
    v[v == 0] = 1
    x[1, 3], x[2, 90], x[M - 1, 95], x[M - 2, 5] = np.inf, -np.inf, np.nan, np.inf
    v[4, 7], v[N - 1, 0], v[N // 2, 9] = np.inf, -np.inf, np.nan
    x[3, 10], x[4, 10] = 3.4028235e38, -3.38e38
    v, wb = dense(t, v)
    with np.errstate(all="ignore"):
        ref = (x.astype(np.float64)[:, None, :] * v.astype(np.float64)[None, :64]).sum(-1)
        last = (x.astype(np.float64)[:, None, :] * v.astype(np.float64)[None, -64:]).sum(-1)
        mid = (x.astype(np.float64) * v.astype(np.float64)[N // 2]).sum(-1)
    y = gemm_dev(t, x, wb, N)
    for got, want in ((y[:, :64], ref), (y[:, -64:], last), (y[:, N // 2], mid)):
        with np.errstate(all="ignore"):
            want = want.astype(np.float32)
        # a large value beside small ones: those of the sum are lost in either order
        near = np.isclose(got, want, rtol=2.0 ** -22, atol=0, equal_nan=True)
        assert near.all(), np.argwhere(~near)[:5]


@pytest.mark.parametrize("name", ["F16", "BF16"])
def test_fact_gemm_unaligned_weights(name):
    """2-byte aligned weights give the aligned call's bits."""
    import torch
    from hip_util import L, stream, to_dev
    t = FACT[name]
    M, N, K = 40, 2500, 96
    assert form(t, M, K, N).startswith("fact_gemm ")
    w = fact_weights(t, K, N, seed=1)
    x = np.random.default_rng(2).standard_normal((M, K)).astype(np.float32)
    want = gemm_dev(t, x, w, N)
    for off in (2, 6):
        buf = to_dev(np.concatenate([np.zeros(off, np.uint8), w]))
        y = torch.empty(M * N, dtype=torch.float32, device="cuda")
        xd = to_dev(x)
        assert L().lp_gemm_dev(xd.data_ptr(), buf.data_ptr() + off, t, y.data_ptr(), M, K, N, None, 0, stream()) == 0
        torch.cuda.synchronize()
        assert np.array_equal(y.cpu().numpy().reshape(M, N).view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("name", list(FACT))
def test_fact_gemm_line(name):
    """One weight row fewer than the least that takes this product runs on the GEMVs, for
    the fewest rows, for 16 and at short K (where the line is twice as high): the columns
    agree."""
    t = FACT[name]
    rng = np.random.default_rng(8)
    for M, K in ((6 if name in ("F32", "F16") else 5, 4096), (16, 4096), (16, 512)):
        N = next(n for n in range(32, 40000) if form(t, M, K, n) != "fact")
        w = fact_weights(t, K, N, seed=N)
        x = rng.standard_normal((M, K)).astype(np.float32)
        below = gemm_dev(t, x, w[:(N - 1) * (len(w) // N)], N - 1)
        assert normwise(gemm_dev(t, x, w, N)[:, :-1], below) <= TOL


# powers of two of x and of the weights: x (or w) with pieces below 2^-126 beside factors
# that bring the products back to ordinary size, and products near the ends of the range
RANGES = [(-118, 40), (-130, 60), (-145, 100), (-112, 20), (40, -118), (90, -131), (-70, -70), (-60, -62), (100, -100), (-40, 0)]


@pytest.mark.parametrize("ex,ew", RANGES)
@pytest.mark.parametrize("name", list(DENSE))
@pytest.mark.parametrize("M,N", [(40, 2500), (64, 14400), (200, 24600)])
def test_fact_gemm_operand_ranges(name, M, N, ex, ew):
    """Tiny values against large ones keep the bits that fp32 products keep, on either
    side; rows and columns of ordinary size beside them keep theirs."""
    t = DENSE[name]
    if t == F16 and not -24 <= ew <= 14:
        pytest.skip("outside fp16")
    K = 96
    assert form(t, M, K, N).startswith("fact_gemm ")
    rng = np.random.default_rng(200 + ex + 1000 * (200 + ew))
    x = rng.standard_normal((M, K)).astype(np.float32)
    v = rng.standard_normal((N, K)).astype(np.float32)
    x[1], x[M - 1] = x[1] * 2.0 ** ex, 0
    x[3, ::5] *= np.float32(2.0 ** ex)
    x[M - 1, 70] = 1.375 * 2.0 ** ex
    v[5], v[N - 1] = v[5] * 2.0 ** ew, v[N - 1] * 2.0 ** ew
    v[6, ::5] *= np.float32(2.0 ** ew)
    v, wb = dense(t, v)
    y = gemm_dev(t, x, wb, N)
    cols = [0, 5, 6, N // 2, N - 1]
    p = x.astype(np.float64)[:, None] * v.astype(np.float64)[None, cols]
    ref, size = p.sum(-1), np.abs(p).sum(-1)
    # the fp32 dots' own error: at most K roundings of partial sums, denormal ones absolute
    bad = np.abs(y[:, cols] - ref) > 2.0 ** -21 * size + K * 2.0 ** -149
    assert not bad.any(), np.argwhere(bad)[:8]


@pytest.mark.parametrize("name", ["Q2_K", "Q3_K", "Q5_K"])
def test_fact_gemm_tiny_rows_large_scales(name):
    """Rows near 2^-112 with the largest block scales are the ordinary rows' products, scaled:
    the outputs lie near 2^-90."""
    t = FACT[name]
    M, N, K = 40, 2500, 512
    assert form(t, M, K, N).startswith("fact_gemm ")
    w = fact_weights(t, K, N, seed=7)
    _, size, at = BLOCK[t]
    for o in at:
        w.reshape(-1, size)[:, o:o + 2] = np.array([6e4], np.float16).view(np.uint8)
    x = np.random.default_rng(9).standard_normal((M, K)).astype(np.float32)
    plain = gemm_dev(t, x, w, N)
    z = x.copy()
    z[::3] *= np.float32(2.0 ** -112)
    y = gemm_dev(t, z, w, N)
    for m in range(0, M, 3):
        assert normwise(y[m] * np.float32(2.0 ** 112), plain[m]) <= TOL
    rest = [m for m in range(M) if m % 3]
    assert np.array_equal(y[rest].view(np.uint32), plain[rest].view(np.uint32))


@pytest.mark.parametrize("M,N", [(12, 8190), (200, 2500)])
@pytest.mark.parametrize("name", list(FACT))
def test_fact_gemm_all_rows_small(orc, name, M, N):
    """Every output taken the slow way (all of x near 1e-30) is the ordinary product's,
    scaled, and so is one infinite row's sign."""
    t = FACT[name]
    K = 512 if M > 16 else 1024
    assert form(t, M, K, N).startswith("fact_gemm ")
    w = fact_weights(t, K, N, seed=2)
    x = np.random.default_rng(3).standard_normal((M, K)).astype(np.float32)
    y1 = gemm_dev(t, x, w, N)
    y = gemm_dev(t, x * np.float32(2.0 ** -100), w, N)
    for m in range(M):
        assert normwise(y[m] * np.float32(2.0 ** 100), y1[m]) <= TOL
    x[2, 5], x[M - 1] = np.inf, np.nan
    y2 = gemm_dev(t, x, w, N)
    with np.errstate(all="ignore"):
        ref = orc.gemm_scalar(t, x[2:3], w, N)[0]
    assert np.array_equal(y2[2], ref, equal_nan=True) and np.isnan(y2[M - 1]).all()
    rest = [m for m in range(M) if m not in (2, M - 1)]
    assert np.array_equal(y2[rest].view(np.uint32), y1[rest].view(np.uint32))
