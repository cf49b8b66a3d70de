"""Grouped MoE prompts on the tiled int8 product: each group size (32, 64, 128 pairs)
at the edges of its tiles, uneven experts, dropped pairs, against the oracle."""
import numpy as np
import pytest

from hip_util import L, normwise, stream, synth_weights, synth_x, to_dev
from oracle.oracle import Q4_0, Q4_K, Q6_K, Q8_0
from test_gpu_i8t import positive_weights

pytestmark = pytest.mark.gpu
NAMES = {Q8_0: "Q8_0", Q4_0: "Q4_0", Q6_K: "Q6_K", Q4_K: "Q4_K"}
# exact block sums; each side rounds at most K/32 + 3 <= 27 additions and products of a
# chain: 27 * 2^-25 normwise a side, doubled
TOL = 4e-6


def grouped(t, x, multi, idx, w, E, K, N):
    import torch
    T, topk = idx.shape
    y = torch.full((T * topk, N), 7.0, dtype=torch.float32, device="cuda")
    nb = L().lp_moe_workspace_bytes(T, topk, E, K, multi)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    xd, idd, wd = to_dev(x), to_dev(idx.astype(np.int32)), to_dev(w)
    rc = L().lp_moe_grouped_dev(xd.data_ptr(), multi, idd.data_ptr(), wd.data_ptr(), t, y.data_ptr(), T, topk, E, K, N,
                                ws.data_ptr(), nb, stream())
    assert rc == 0, L().lp_last_error().decode()
    torch.cuda.synchronize()
    return y.cpu().numpy()


def pairs_of(counts, topk, rng):
    """idx of sum(counts) pairs, counts[e] on expert e, in random order."""
    e = rng.permutation(np.repeat(np.arange(len(counts)), counts))
    return e[:len(e) // topk * topk].reshape(-1, topk)


# pairs per expert: means that take groups of 32, 64 and 128 (8 experts), with empty
# experts, one pair, whole groups and one pair past them. Q8_0 and Q4_0 go over to 64 at
# 16 pairs per expert and stay there.
COUNTS = {32: [0, 1, 32, 33, 64, 5, 31, 18], 64: [0, 1, 64, 65, 128, 30, 63, 97], 128: [0, 1, 128, 129, 257, 60, 255, 130]}
SMALL = {**COUNTS, 32: [0, 1, 32, 33, 10, 5, 20, 18]}


def counts_of(t, gs):
    return (SMALL if t in (Q8_0, Q4_0) else COUNTS)[gs]


def check_group(t, idx, E, K, multi, gs):
    want = 64 if t in (Q8_0, Q4_0) and gs == 128 else gs
    assert L().lp_moe_group_pairs(t, *idx.shape, E, K, multi) == want


@pytest.mark.parametrize("multi", [0, 1])
@pytest.mark.parametrize("t", list(NAMES), ids=list(NAMES.values()))
@pytest.mark.parametrize("gs,topk,K,N", [(32, 2, 256, 130), (32, 1, 768, 33), (64, 3, 512, 65), (64, 2, 256, 200),
                                         (128, 2, 512, 129), (128, 1, 256, 31)])
def test_moe_tile_matches_oracle(orc, t, multi, gs, topk, K, N):
    print(f"moe tile {NAMES[t]} groups {gs} topk {topk} K {K} N {N} multi {multi}", flush=True)
    if t in (Q8_0, Q4_0):
        K += 64                                    # K ends inside a 128-element stage
    rng = np.random.default_rng(gs + K + N + t)
    E = 8
    idx = pairs_of(counts_of(t, gs), topk, rng)
    T = idx.shape[0]
    check_group(t, idx, E, K, multi, gs)
    w = synth_weights(t, K, E * N, seed=t + gs)
    x = synth_x(T * topk if multi else T, K, seed=5, outliers=0.01)
    y = grouped(t, x, multi, idx, w, E, K, N)
    rb = len(w) // E
    for e in range(E):
        p = np.flatnonzero(idx.reshape(-1) == e)
        if len(p):
            ref = orc.gemm_int(t, x[p if multi else p // topk], w[e * rb:(e + 1) * rb], N)
            assert normwise(y[p], ref) <= TOL, e


@pytest.mark.parametrize("t", list(NAMES), ids=list(NAMES.values()))
def test_moe_tile_drops_pairs_without_an_expert(t):
    """Pairs whose index names no expert leave their rows as they are; the others
    get the same bits."""
    rng = np.random.default_rng(3)
    E, K, N, topk = 4, 256, 96, 2
    idx = pairs_of([40, 70, 35, 15], topk, rng)
    w = synth_weights(t, K, E * N, seed=8)
    x = synth_x(idx.shape[0], K, seed=9)
    want = grouped(t, x, 0, idx, w, E, K, N)
    bad = idx.copy()
    bad[3, 0], bad[10, 1], bad[-1, 1] = -1, E, 1 << 20
    y = grouped(t, x, 0, bad, w, E, K, N)
    drop = (bad != idx).reshape(-1)
    assert np.all(y[drop] == 7.0)
    assert np.array_equal(y[~drop].view(np.uint32), want[~drop].view(np.uint32))


@pytest.mark.parametrize("multi", [0, 1])
@pytest.mark.parametrize("gs", list(COUNTS))
@pytest.mark.parametrize("t", list(NAMES), ids=list(NAMES.values()))
def test_moe_tile_infinite_block_scales(t, gs, multi):
    """An infinite block scale of an expert's row gives that expert's pairs the signed
    infinity (Q4_0, whose offset is subtracted apart, NaN) and no other output another value;
    a NaN activation row is NaN."""
    rng = np.random.default_rng(gs)
    E, K, N, topk = 8, 512, 70, 2
    idx = pairs_of(counts_of(t, gs), topk, rng)
    check_group(t, idx, E, K, multi, gs)
    P = idx.size
    x = np.abs(synth_x(P if multi else len(idx), K, seed=6)) + 0.1
    w, d = positive_weights(t, K, E * N, seed=gs)
    clean = grouped(t, x, multi, idx, w.reshape(-1), E, K, N)
    d[2 * N + 3, 0], d[4 * N + N - 1, -1] = 0x7c00, 0xfc00
    x[1, 7] = np.nan
    y = grouped(t, x, multi, idx, w.reshape(-1), E, K, N)
    e = idx.reshape(-1)
    want = clean.copy()
    want[e == 2, 3], want[e == 4, N - 1] = (np.nan, np.nan) if t == Q4_0 else (np.inf, -np.inf)
    want[1 if multi else [topk, topk + 1]] = np.nan
    assert np.array_equal(y, want, equal_nan=True)
