"""Host-pointer linears around the size up to which the kernels store their
outputs to pinned host memory themselves (2048 floats over all outputs): the
values, the growth of the pinned buffer between calls, and non-finite values."""
import numpy as np
import pytest

import oracle as O
import uq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,okind", [(uq.KIND_Q8_0, O.Q8_0), (uq.KIND_Q4_K, O.Q4_K), (uq.KIND_Q3_K, O.Q3_K)])
@pytest.mark.parametrize("m", [1, 2047, 2048, 2049, 9001])
def test_matvec_output_sizes(gpu, kind, okind, m):
    n = 512
    raw = uq.synth_quant(kind, m, m, n)
    x = uq.synth_normal(m + 1, n)
    y = uq.matvec(uq.Weight(kind, n, m, raw), x)
    assert np.array_equal(y.view(np.uint32), O.matvec(okind, raw, n, m, x).view(np.uint32))


@pytest.mark.parametrize("ms", [(1024, 512, 512), (1024, 512, 513), (5, 4000, 1)])
def test_batch_output_sizes(gpu, ms):
    n = 768
    raws = [uq.synth_quant(uq.KIND_Q8_0, i, m, n) for i, m in enumerate(ms)]
    x = uq.synth_normal(3, n)
    ys = uq.batch([uq.Weight(uq.KIND_Q8_0, n, m, r) for m, r in zip(ms, raws)], x)
    for m, r, y in zip(ms, raws, ys):
        assert np.array_equal(y.view(np.uint32), O.matvec(O.Q8_0, r, n, m, x).view(np.uint32))


def test_batch_after_a_refused_batch(gpu):
    """A group that holds a kind the int8 linears do not take is refused before
    anything is launched, so that nothing it started stores into the pinned buffer
    of the next call, whose longer x lies where its outputs would have been."""
    short, m = 256, 600  # 1800 outputs: stored to pinned memory by the kernels
    refused = [uq.Weight(k, short, m, uq.synth_quant(k, 5, m, short))
               for k in (uq.KIND_Q8_0, uq.KIND_Q4_K, uq.KIND_IQ4_XS)]
    n = 1536
    raws = [uq.synth_quant(uq.KIND_Q8_0, 9 + i, 600, n) for i in range(3)]
    ws = [uq.Weight(uq.KIND_Q8_0, n, 600, r) for r in raws]
    for seed in range(4):
        with pytest.raises(uq.UqError) as e:
            uq.batch(refused, uq.synth_normal(seed, short))
        assert e.value.status == uq.Error.QUANT_TYPE
        x = uq.synth_normal(100 + seed, n)
        for r, y in zip(raws, uq.batch(ws, x)):
            assert np.array_equal(y.view(np.uint32), O.matvec(O.Q8_0, r, n, 600, x).view(np.uint32))


@pytest.mark.parametrize("m", [2048, 2049, 100000])
def test_linear_output_sizes(gpu, m):
    n = 256
    raw = uq.synth_quant(uq.KIND_IQ4_XS, m, m, n)
    x = uq.synth_normal(m, n)
    y = uq.linear(uq.Weight(uq.KIND_IQ4_XS, n, m, raw), x)
    ref = O.linear(uq.KIND_IQ4_XS, raw, n, m, x)
    assert np.abs(y - ref).max() <= 1e-6 * np.abs(ref).max()


@pytest.mark.parametrize("m", [40, 3000])
def test_non_finite(gpu, m):
    n = 512
    raw = uq.synth_quant(uq.KIND_Q8_0, 1, m, n)
    w = uq.Weight(uq.KIND_Q8_0, n, m, raw)
    x = np.ones(n, np.float32)
    for call in (uq.matvec, uq.linear):
        for bad in (np.nan, np.inf, -np.inf):
            x[n - 1] = bad
            with pytest.raises(uq.UqError) as e:
                call(w, x)
            assert e.value.status == uq.Error.NONFINITE
        x[n - 1] = 1.0
        assert np.isfinite(call(w, x)).all()
    raw[0], raw[1] = 0x00, 0x7C  # an infinite block scale: a non-finite output
    for call in (uq.matvec, uq.linear):
        with pytest.raises(uq.UqError) as e:
            call(uq.Weight(uq.KIND_Q8_0, n, m, raw), x)
        assert e.value.status == uq.Error.NONFINITE
