"""The tiled int8 MFMA product (Q8_0, Q4_0, Q5_0, Q6_K and Q4_K rows beyond the
small-M kernels) at the edges of its tiles and forms, against the oracle."""
import numpy as np
import pytest

from hip_util import form, gemm_dev, normwise, quantize_dev, synth_weights, synth_x
from oracle.oracle import Q4_0, Q4_K, Q5_0, Q6_K, Q8_0

pytestmark = pytest.mark.gpu
NAMES = {Q8_0: "Q8_0", Q4_0: "Q4_0", Q5_0: "Q5_0", Q6_K: "Q6_K", Q4_K: "Q4_K"}

# Integer block sums are exact on both sides. Each side rounds the scale product
# and the additions of a chain: at most ~(K/32 + 3) half-ulps of the largest
# partial sum, K <= 2048 here: 67 * 2^-25 = 2e-6 normwise, and twice that for two
# sides.
TOL = 4e-6

# (M, N, K): one token and one row past a 32- and 64-tile, K ending inside a
# 128-element stage (64-, 32- and 192-element tails), single-stage K, one stage
# pair and its neighbours, then M and N that take each form (32x128, 32x32 with 8 and
# 4 K groups, 64x64 with 2 and 1, 128x128: test_every_form_is_run)
SHAPES32 = [(9, 31, 64), (12, 33, 192), (17, 1, 1088), (33, 65, 448), (65, 127, 2048), (5, 6555, 1088)]
SHAPES256 = [(17, 33, 256), (33, 31, 512), (65, 129, 1280), (127, 64, 2048)]
FORMS = [(31, 8200, 256), (40, 8200, 512), (33, 14400, 256), (96, 16500, 256), (200, 24600, 256), (500, 8190, 256)]
TAILS = [(500, 8190, 192), (200, 24600, 320)]
SHAPES = {t: SHAPES32 + FORMS + TAILS for t in (Q8_0, Q4_0)}
SHAPES[Q5_0] = [(M, N, K + 32 * (K < 2048)) for M, N, K in SHAPES32 + TAILS] + FORMS
SHAPES[Q6_K] = SHAPES256 + FORMS + [(70, 14400, 512)]
SHAPES[Q4_K] = [(65, 129, 1280), (127, 64, 2048), (96, 4300, 512), (33, 8200, 512), (96, 14400, 256), (130, 16300, 256)]
CASES = [(t, *s) for t in NAMES for s in SHAPES[t]]


def test_every_form_is_run():
    """The cases run each tile form of the product for each type (on 256 CUs)."""
    import torch
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the forms' lines depend on the CU count")
    for t in NAMES:
        got = {form(t, M, K, N) for M, N, K in SHAPES[t]}
        want = {f"i8t {f}" for f in ("32x128", "32x32x8", "32x32x4", "64x64x2", "64x64", "128x128")}
        assert got == want - ({"i8t 32x128"} if t == Q4_K else set()), (NAMES[t], got)


def weights(t, K, N, seed):
    w = synth_weights(t, K, N, seed=seed)
    if t == Q5_0:                                          # finite block scales
        d = np.abs(np.random.default_rng(seed).standard_normal(w.size // 22)) * 0.01
        w.reshape(-1, 22)[:, 0:2] = d.astype(np.float16).view(np.uint8).reshape(-1, 2)
    return w


@pytest.mark.parametrize("t,M,N,K", CASES, ids=[f"{NAMES[c[0]]}-{c[1]}x{c[2]}x{c[3]}" for c in CASES])
def test_i8t_matches_oracle(orc, t, M, N, K):
    print(f"i8t {NAMES[t]} M={M} N={N} K={K}", flush=True)
    w = weights(t, K, N, seed=M + N + K + t)
    assert form(t, M, K, N).startswith("i8t ")
    x = synth_x(M, K, seed=M + 1, outliers=0.01)
    x[M // 2, :32] = 0.0                                   # a block of zeros
    y = gemm_dev(t, x, w, N)
    rows = np.unique(np.linspace(0, N - 1, 48).astype(int))   # both ends and between
    rb = len(w) // N
    ref = orc.gemm_int(t, x, np.concatenate([w[r * rb:(r + 1) * rb] for r in rows]), len(rows))
    assert normwise(y[:, rows], ref) <= TOL


@pytest.mark.parametrize("t", list(NAMES), ids=list(NAMES.values()))
def test_i8t_rows_do_not_depend_on_their_neighbours(orc, t):
    """Every form adds the same 256-element chains in 64 bits, so the first 70
    rows of calls that run on different forms are the same numbers."""
    K, N = 1024, 3000
    w = weights(t, K, N, seed=9 + t)
    x = synth_x(700, K, seed=10, outliers=0.01)
    assert len({form(t, M, K, N) for M in (70, 129, 300, 700)}) >= 3
    first = gemm_dev(t, x[:70], w, N)
    for M in (129, 300, 700):
        y = gemm_dev(t, x[:M], w, N)
        assert np.array_equal(y[:70].view(np.uint32), first.view(np.uint32)), M


@pytest.mark.parametrize("t", list(NAMES), ids=list(NAMES.values()))
def test_i8t_non_finite_rows(orc, t):
    """A NaN or infinity in a row makes that row NaN as the reference's scale
    does, and leaves the others alone."""
    K, N, M = 512, 96, 70
    assert form(t, M, K, N).startswith("i8t ")
    w = weights(t, K, N, seed=20 + t)
    x = synth_x(M, K, seed=21)
    x[3, 40] = np.nan
    x[69, 511] = np.inf
    x[68, 0] = -np.inf
    y = gemm_dev(t, x, w, N)
    ref = orc.gemm_int(t, x, w, N)
    assert np.array_equal(np.isnan(y), np.isnan(ref))
    good = [m for m in range(M) if m not in (3, 68, 69)]
    assert normwise(y[good], ref[good]) <= TOL


# each form, K ending inside a stage where the type allows it
EDGE_SHAPES = [(9, 600, 1216), (17, 33000, 192), (40, 8200, 192), (96, 4300, 320), (70, 14400, 192), (500, 8190, 192)]


@pytest.mark.parametrize("wscale", [None, 2.0 ** -24, 6e4])
@pytest.mark.parametrize("M,N,K", EDGE_SHAPES)
@pytest.mark.parametrize("t", list(NAMES), ids=list(NAMES.values()))
def test_i8t_tiny_rows(orc, t, M, N, K, wscale):
    """Rows down to the smallest fp32 values keep their products' 24 bits, whatever the
    block scales of the weights; the rows beside them keep their bits."""
    print(f"i8t tiny rows {NAMES[t]} M={M} N={N} K={K}", flush=True)
    if t == Q4_K and N == 33000:
        pytest.skip("Q4_K has no 32 x 128 tiles")
    if t in (Q4_K, Q6_K):
        K, M = 1280 if K > 512 else 512, max(M, 17 if t == Q6_K else 70)
    assert form(t, M, K, N).startswith("i8t ")
    w = weights(t, K, N, seed=t).reshape(-1, {Q8_0: 34, Q4_0: 18, Q5_0: 22, Q4_K: 144, Q6_K: 210}[t])
    for at in {Q4_K: [0, 2], Q6_K: [208]}.get(t, [0]):
        if wscale:
            w[:, at:at + 2] = np.array([wscale], np.float16).view(np.uint8)
    w = w.reshape(-1)
    x = synth_x(M, K, seed=32)
    plain = gemm_dev(t, x, w, N)
    scale = {0: 1e-20, 1: 1e-26, 3: 1e-30, 4: 1e-33, 6: 1e-36, 7: 0.0, M - 1: 1e-31}
    for m, s in scale.items():
        x[m] *= np.float32(s)
    y = gemm_dev(t, x, w, N)
    d, _, _, qs = quantize_dev(x)
    X = np.repeat(d.astype(np.float64), 32, axis=1) * qs
    rows = np.unique(np.linspace(0, N - 1, 64).astype(int))
    rb = len(w) // N
    sub = np.concatenate([w[r * rb:(r + 1) * rb] for r in rows])
    W = orc.dequantize(t, sub, len(rows) * K)
    ref = X @ W.astype(np.float64).reshape(len(rows), K).T
    few = list(scale)
    P = np.abs(orc.block_sums(t, sub, qs[few], K, len(rows))).sum(-1).max(-1)
    for i, m in enumerate(few):
        # products of scales below 2^-126 are rounded at 2^-149 (as in fp32), then
        # multiplied with a block sum (of Q6_K times its int8 scale; of Q4_K the 6-bit
        # mins' product too, by a factor up to 2^11 of fp16 dmin)
        quantum = 2.0 ** -149 * (P[i] * (128 if t == Q6_K else 1) + (2048 * K if t == Q4_K else K))
        err = np.abs(y[m, rows] - ref[m]).max()
        assert err <= TOL * np.abs(ref[m]).max() + quantum, (m, scale[m], err, np.abs(ref[m]).max())
    rest = [m for m in range(M) if m not in scale]
    assert np.array_equal(y[rest].view(np.uint32), plain[rest].view(np.uint32))


def positive_weights(t, K, N, seed):
    """Blocks whose codes and sub-scales are all above zero (every block sum with positive
    activations is too), mins of the type zero; returns them with a view of the rows'
    block scales [N, blocks] as fp16 bits."""
    rng = np.random.default_rng(seed)
    size, elems, at = {Q8_0: (34, 32, 0), Q4_0: (18, 32, 0), Q5_0: (22, 32, 0), Q4_K: (144, 256, 0), Q6_K: (210, 256, 208)}[t]
    b = rng.integers(0, 256, (N * (K // elems), size), dtype=np.uint8)
    n = len(b)
    nib = lambda lo, hi, w: (rng.integers(lo, hi, (n, w)) | rng.integers(lo, hi, (n, w)) << 4).astype(np.uint8)
    if t == Q8_0:
        b[:, 2:] = rng.integers(1, 128, (n, 32))
    elif t == Q4_0:
        b[:, 2:] = nib(9, 16, 16)
    elif t == Q5_0:
        b[:, 2:6], b[:, 6:] = 255, nib(1, 16, 16)
    elif t == Q4_K:
        b[:, 2:4], b[:, 16:] = 0, nib(1, 16, 128)
        b[:, 4:8], b[:, 8:12], b[:, 12:16] = 0x41, 0, 0x0f      # scales 1 and 31, mins 0
    else:
        b[:, :128], b[:, 128:192], b[:, 192:208] = nib(1, 16, 128), 0xaa, rng.integers(1, 32, (n, 16))
    d = (0.01 * (0.5 + rng.random(n))).astype(np.float16)
    b[:, at:at + 2] = d.view(np.uint8).reshape(-1, 2)
    return b, b.reshape(N, -1, size)[:, :, at:at + 2].view(np.uint16)[:, :, 0]


@pytest.mark.parametrize("M,N,K", EDGE_SHAPES)
@pytest.mark.parametrize("t", list(NAMES), ids=list(NAMES.values()))
def test_i8t_infinite_block_scales(t, M, N, K):
    """An infinite block scale gives the signed infinity of its product (NaN with a block
    of zeros, or beside an infinity of the other sign), a NaN scale NaN, as at few rows
    (whose kernels multiply a row's last block with zeros once more past its end, which is
    left out here); the other weight rows keep their bits."""
    print(f"i8t infinite scales {NAMES[t]} M={M} N={N} K={K}", flush=True)
    if t == Q4_K and N == 33000:
        pytest.skip("Q4_K has no 32 x 128 tiles")
    if t in (Q4_K, Q6_K):
        K, M = 1280 if K > 512 else 512, max(M, 17 if t == Q6_K else 70)
    assert form(t, M, K, N).startswith("i8t ")
    x = np.abs(synth_x(M, K, seed=31)) + 0.1
    x[2] = 0.0
    w, d = positive_weights(t, K, N, seed=t)
    clean = gemm_dev(t, x, w.reshape(-1), N)
    inf, ninf, nan = 0x7c00, 0xfc00, 0x7e00
    d[4, 0], d[N - 1, -1], d[7, 0], d[7, -1], d[9, 0], d[65, 1] = inf, ninf, inf, ninf, nan, inf
    want = clean.copy()
    want[:, [4, 65]], want[:, N - 1], want[:, [7, 9]] = np.inf, -np.inf, np.nan
    want[2, [4, 65, N - 1]] = np.nan
    if t == Q4_0:                                          # the reference subtracts 8 d sum(x): inf - inf
        want[:, [4, 65, N - 1]] = np.nan
    y = gemm_dev(t, x, w.reshape(-1), N)
    few = gemm_dev(t, x[:3], w.reshape(-1), N)
    special = [4, 7, 9, 65, N - 1]
    assert np.array_equal(few[:, special[:4]], want[:3, special[:4]], equal_nan=True)
    assert np.array_equal(y[:, special], want[:, special], equal_nan=True)
    rest = np.setdiff1d(np.arange(N), special)
    assert np.array_equal(y[:, rest].view(np.uint32), clean[:, rest].view(np.uint32))
