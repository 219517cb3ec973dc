"""uq_matvec_static where one launch quantizes x and multiplies, and where two
do: bit for bit what uq_quant_act_dev followed by uq_matvec_q_dev gives, over the
kernels (registers, LDS, row blocks), the edges of K and of the rows, both sides
of the line between the two forms, and every x that the entry point takes
(unaligned, over y, non-finite, zero blocks)."""
import numpy as np
import pytest
import torch

import uq

pytestmark = pytest.mark.gpu


def both(w, x, y):
    L = uq.lib()
    q = torch.empty(w.n, dtype=torch.int8, device="cuda")
    s = torch.empty(w.n // 32, dtype=torch.float32, device="cuda")
    ref = torch.full((w.m,), 7.0, device="cuda")
    torch.cuda.synchronize()
    uq._check(L.uq_quant_act_dev(x.data_ptr(), w.n, q.data_ptr(), s.data_ptr(), None))
    uq._check(L.uq_matvec_q_dev(w.handle, q.data_ptr(), s.data_ptr(), ref.data_ptr(), None))
    uq._check(L.uq_matvec_static(w.handle, x.data_ptr(), y.data_ptr(), None))
    L.uq_sync()
    return y.cpu().numpy().view(np.uint32), ref.cpu().numpy().view(np.uint32)


def weight(kind, n, m):
    return uq.Weight(kind, n, m, uq.synth_quant(kind, n + m, m, n))


SHAPES = [(uq.KIND_Q8_0, n, m) for n, m in [(32, 1), (32, 9000), (96, 257), (992, 255), (1536, 4097), (1536, 40000),
                                            (4096, 7000), (4128, 100), (8960, 3), (16352, 64), (16384, 1),
                                            (10240, 70), (10272, 70), (512, 98304), (512, 98320)]]
SHAPES += [(k, n, m) for k in (uq.KIND_Q4_K, uq.KIND_Q3_K)
           for n, m in [(256, 1), (256, 33000), (768, 257), (1536, 4097), (1536, 140000), (4096, 20001), (8960, 100),
                        (8960, 4000), (16384, 5), (1024, 147456), (1024, 147488)]]


@pytest.mark.parametrize("kind,n,m", SHAPES)
def test_equals_two_launches(gpu, kind, n, m):
    w = weight(kind, n, m)
    x = torch.from_numpy(uq.synth_normal(n, n, 0.0, 2.0)).cuda()
    x[: n // 2 : 7] *= 1e-30
    if n >= 64:
        x[32:64] = 0.0
    y, ref = both(w, x, torch.full((m,), 7.0, device="cuda"))
    assert np.array_equal(y, ref)


@pytest.mark.parametrize("kind", [uq.KIND_Q8_0, uq.KIND_Q4_K, uq.KIND_Q3_K])
@pytest.mark.parametrize("form", ["unaligned", "over y", "inside y", "inf", "-inf", "nan"])
def test_any_x(gpu, kind, form):
    n, m = 512, 700
    w = weight(kind, n, m)
    room = torch.from_numpy(uq.synth_normal(5, n + m, 0.0, 1.0)).cuda()
    y = torch.full((m,), 7.0, device="cuda")
    x = room[:n]
    if form == "unaligned":
        x = room[1 : n + 1]
    elif form == "over y":
        y = room[:m]
    elif form == "inside y":
        x, y = room[64 : 64 + n], room[:m]
    else:
        x[300] = float(form)
    y, ref = both(w, x, y)
    nan = np.isnan(ref.view(np.float32))
    assert np.array_equal(nan, np.isnan(y.view(np.float32)))
    assert np.array_equal(y[~nan], ref[~nan])
