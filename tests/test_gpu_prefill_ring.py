"""The prefill GEMM's 4- and 8-stage rings (stages of 128 values of K): fewer
stages than the ring, the edges of the passes of 4 stages (10 stages are the
first that take one with 8 in the ring, 6 with 4), every remainder behind them
and partial last stages; bit for bit the oracle's."""
import numpy as np
import pytest

import oracle as O
import uq

pytestmark = pytest.mark.gpu


# 64 rows at up to 64 tokens: 4 workgroups, the ring of 8. 2048 rows at 320
# tokens: 640 workgroups, the ring of 4. 1536 rows at 256: 384, 8 from K 4096 on.
@pytest.mark.parametrize("N,T,K", [(64, 5, 128 * s + p) for s in (1, 2, 7, 8, 9, 10, 11, 12, 13, 14, 17) for p in (0, 32)] +
                         [(2048, 320, 128 * s + p) for s in (3, 5, 6, 7, 8, 9) for p in (0, 96)] +
                         [(1536, 250, 4064), (1536, 250, 4096), (64, 64, 16384)])
def test_ring_edges(gpu, N, T, K):
    raw = uq.synth_quant(uq.KIND_Q8_0, N + K, N, K)
    qs = [O.quant_act(uq.synth_normal(t, K)) for t in range(T)]
    qx, xs = np.stack([q for q, _ in qs]), np.stack([s for _, s in qs])
    y = uq.prefill_gemm(uq.Weight(uq.KIND_Q8_0, K, N, raw), qx, xs)
    assert np.array_equal(y.view(np.uint32), O.prefill_gemm(raw, K, N, xs, qx, T).view(np.uint32))
