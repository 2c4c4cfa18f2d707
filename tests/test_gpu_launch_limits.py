"""Problems of more workgroups than one HIP launch takes (2^32 threads): 70 GB
outputs, of which a few rows are checked."""
import ctypes

import numpy as np
import pytest

import grxcp_amd as g
import oracle as O
from helpers import normwise_rel_err, say, to_dev
from test_gpu_dnn import BF16, dec, enc

pytestmark = pytest.mark.gpu


def big_buffer(libs, nbytes):
    free, total = ctypes.c_size_t(0), ctypes.c_size_t(0)
    g.check_rt(libs.rt.grxMemGetInfo(ctypes.byref(free), ctypes.byref(total)))
    if free.value < nbytes + (4 << 30):
        pytest.skip(f"needs {nbytes >> 30} GiB of GPU memory, {free.value >> 30} free")
    return g.DeviceBuffer(nbytes)


def test_attention_many_heads(gpu, dnn):
    """2^23 heads of 65 keys, Q, K and V of one head broadcast to all: as
    128-query items with split keys they are 2^32 threads."""
    B, H, S, D = 2048, 4096, 65, 64
    r = np.random.default_rng(0)
    q, k, v = (enc(r.standard_normal((S, D)).astype(np.float32), BF16) for _ in range(3))
    o = big_buffer(gpu, B * H * S * D * 2)
    head = S * D
    for first in (0, B * H // 2, B * H - 1):
        o.upload(np.zeros(head, np.uint16), offset=2 * head * first)
    dq, dk, dv = to_dev(q), to_dev(k), to_dev(v)
    one = g.TensorDesc(BF16, [B, H, S, D], [0, 0, D, 1])
    od = g.TensorDesc(BF16, [B, H, S, D])
    say("attention of 2^23 heads")
    s = dnn.attention(g.AttnDesc(False, D ** -0.5), one, dq.p, one, dk.p, one, dv.p, od, o.p)
    assert s == g.SUCCESS, g.STATUS[s]
    g.synchronize()
    ref = O.attention_head(dec(q, BF16).reshape(S, D), dec(k, BF16).reshape(S, D), dec(v, BF16).reshape(S, D),
                           False, D ** -0.5)
    for first in (0, B * H // 2, B * H - 1):
        got = dec(o.download(np.uint16, head, offset=2 * head * first), BF16).reshape(S, D)
        assert normwise_rel_err(got, ref) <= 1e-2, first
    o.close()


def test_softmax_many_unaligned_rows(gpu, dnn):
    """2^23 rows of 4105 elements, in place, one to a 512-thread workgroup."""
    rows, hidden = 1 << 23, 4105
    x = big_buffer(gpu, rows * hidden * 2)
    r = np.random.default_rng(1)
    xe = enc(r.standard_normal((1, hidden)).astype(np.float32), BF16)
    at = (0, rows // 2, rows - 2, rows - 1)
    for i in at:
        x.upload(xe, offset=2 * hidden * i)
    xd = g.TensorDesc(BF16, [rows, hidden])
    say("softmax of 2^23 rows")
    s = dnn.softmax(xd, x.p, xd, x.p)
    assert s == g.SUCCESS, g.STATUS[s]
    g.synchronize()
    ref = O.softmax(dec(xe, BF16).reshape(1, hidden))[0]
    for i in at:
        got = dec(x.download(np.uint16, hidden, offset=2 * hidden * i), BF16)
        assert np.all(np.abs(got - ref) <= 2.0 ** -8 * np.abs(ref)), i
    x.close()


def test_gemm_many_rows_of_few_columns(gpu, blas):
    """2^27 + 16 rows of one column, 16 rows to a 512-thread workgroup of
    gemm_skinny: the wider tiles' kernel."""
    m, n, k = (1 << 27) + 16, 1, 256
    a = big_buffer(gpu, 2 * m * k)
    c = g.DeviceBuffer(4 * m)
    r = np.random.default_rng(2)
    rows = enc(r.standard_normal((64, k)).astype(np.float32), BF16).reshape(64, k)
    b = enc(r.standard_normal((1, k)).astype(np.float32), BF16).reshape(1, k)
    at = (0, m // 2, m - 64)
    for i in at:
        a.upload(rows, offset=2 * k * i)
    db = to_dev(b)
    say("GemmEx of 2^27 + 16 rows and one column")
    s = blas.gemm_ex(1, 0, m, n, k, 1.0, a.p, BF16, k, db.p, BF16, k, 0.0, c.p, g.GRX_R_32F, m)
    assert s == g.SUCCESS, g.STATUS[s]
    g.synchronize()
    ref = dec(rows, BF16).reshape(64, k).astype(np.float64) @ dec(b, BF16).reshape(k).astype(np.float64)
    for i in at:
        assert normwise_rel_err(c.download(np.float32, 64, offset=4 * i), ref) <= 1e-5, i
    c.close()
    a.close()
