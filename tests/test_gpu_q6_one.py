"""The Q6_K GEMV of one activation row: the bits of that row in a call of two."""
import numpy as np
import pytest

from hip_util import L, gemm_dev, synth_weights, synth_x, to_dev
from oracle.oracle import Q6_K

pytestmark = pytest.mark.gpu


# row quads cut off, one super-block, a chunk's last super-block missing, whole chunks
@pytest.mark.parametrize("N,K", [(1, 256), (5, 3840), (63, 4096), (4098, 2048), (33000, 512)])
def test_one_row_is_the_first_of_two(N, K):
    print(f"q6 one row N={N} K={K}", flush=True)
    w = synth_weights(Q6_K, K, N, seed=N + K)
    assert L().lp_gemm_route(Q6_K, 1, K, N, to_dev(w).data_ptr()).decode() == "q6rq"
    x = synth_x(2, K, seed=4, outliers=0.01)
    two = gemm_dev(Q6_K, x, w, N)
    for m in (0, 1):
        one = gemm_dev(Q6_K, x[m:m + 1], w, N)
        assert np.array_equal(one[0].view(np.uint32), two[m].view(np.uint32))
