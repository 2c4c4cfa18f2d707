"""Row operations on rows off 16-byte boundaries: odd lengths around every
kernel's limits, odd pitches and buffers that start one element off. Rows
there are read and written in chunks at element alignment whose last one is
partial, so the elements around every row (poisoned before the call) must come
back untouched. Bounds as in test_gpu_dnn.py / test_gpu_softmax_gelu.py."""
import ctypes

import numpy as np
import pytest

import grxcp_amd as g
import oracle as O
from helpers import say, to_dev
from test_gpu_dnn import check_norm, dec, enc, nptype
from test_gpu_softmax_gelu import check

pytestmark = pytest.mark.gpu
BF16, F16, F32 = g.GRX_R_16BF, g.GRX_R_16F, g.GRX_R_32F

# (type, rows, hidden): chunks are 8 (16-bit) or 4 (fp32) elements; 64, 256,
# 512, 1024, 2048, 4096 and 8192 of them end a kernel's range
SHAPES = [(BF16, 2050, 999), (F32, 2049, 301), (BF16, 5, 9), (F16, 6, 511), (BF16, 9, 2047), (F16, 3, 2049), (BF16, 4, 4097), (F32, 3, 4095),
          (BF16, 2, 8193), (F32, 2, 8193), (BF16, 2, 16385), (F32, 2, 16383), (F16, 2, 32771),
          (F32, 2, 32001), (BF16, 2, 65531), (F32, 1, 65533), (BF16, 2050, 4099)]


def offset(buf, t):
    return ctypes.c_void_p(buf.p.value + np.dtype(nptype(t)).itemsize)


@pytest.mark.parametrize("op", ["rms", "layer", "softmax", "erf", "tanh"])
@pytest.mark.parametrize("t,rows,hidden", SHAPES)
def test_unaligned_rows(dnn, op, t, rows, hidden):
    r = np.random.default_rng(rows + hidden)
    pitch = hidden + 2 + (hidden & 1)
    x = (2.0 * r.standard_normal((rows, hidden))).astype(np.float32)
    gamma = (1 + 0.1 * r.standard_normal(hidden)).astype(np.float32)
    beta = (0.1 * r.standard_normal(hidden)).astype(np.float32)
    xe, ge, be = (enc(a, t) for a in (x, gamma, beta))
    xq, gq, bq = (dec(a, t) for a in (xe, ge, be))
    poison = np.asarray(0x7FC1 if t != F32 else np.float32(np.nan), nptype(t))
    flat = np.full(1 + rows * pitch, poison, nptype(t))
    src = flat.copy()
    src[1:].reshape(rows, pitch)[:, :hidden] = xe
    dx, dy = to_dev(src), to_dev(flat)
    dg, db = (to_dev(np.concatenate([poison[None], a])) for a in (ge, be))
    xd, wd = g.TensorDesc(t, [rows, hidden], [pitch, 1]), g.TensorDesc(t, [hidden])
    px, py, pg, pb = (offset(b, t) for b in (dx, dy, dg, db))
    say(f"{op} t={t} rows={rows} hidden={hidden} pitch={pitch}, buffers one element off")
    s = {"rms": lambda: dnn.rmsnorm(xd, px, wd, pg, 1e-6, xd, py),
         "layer": lambda: dnn.layernorm(xd, px, wd, pg, pb, 1e-6, xd, py),
         "softmax": lambda: dnn.softmax(xd, px, xd, py),
         "erf": lambda: dnn.gelu(g.GELU_ERF, xd, px, xd, py),
         "tanh": lambda: dnn.gelu(g.GELU_TANH, xd, px, xd, py)}[op]()
    assert s == g.SUCCESS, g.STATUS[s]
    g.synchronize()
    out = dy.download(nptype(t), flat.size)
    body = out[1:].reshape(rows, pitch)
    around = np.concatenate([out[:1], body[:, hidden:].reshape(-1)])
    assert np.array_equal(around.view(np.uint8), np.full(around.size, poison, nptype(t)).view(np.uint8))
    y = dec(np.ascontiguousarray(body[:, :hidden]), t)
    if op == "rms":
        check_norm(y, O.rmsnorm(xq, gq, 1e-6), None, t)
    elif op == "layer":
        check_norm(y, O.layernorm(xq, gq, bq, 1e-6), bq, t)
    elif op == "softmax":
        check(y, O.softmax(xq), t, atol={BF16: 0.0, F16: 6e-8, F32: 1e-30}[t])
    else:
        mode = g.GELU_ERF if op == "erf" else g.GELU_TANH
        check(y, O.gelu(xq, mode).reshape(rows, hidden), t, atol={BF16: 1e-6, F16: 1e-6, F32: 1e-7}[t])


@pytest.mark.parametrize("t,rows,hidden", [(BF16, 3, 5), (F16, 7, 333), (F32, 5, 1001)])
def test_gelu_contiguous_odd_rows(dnn, t, rows, hidden):
    """Contiguous rows of odd length run as one array whose last elements do
    not fill a chunk."""
    x = (3.0 * np.random.default_rng(hidden).standard_normal(rows * hidden)).astype(np.float32)
    xe = enc(x, t)
    guard = np.full(8, 7, nptype(t))
    dx, dy = to_dev(xe), to_dev(np.concatenate([xe, guard]))
    xd = g.TensorDesc(t, [rows, hidden])
    say(f"gelu t={t} {rows}x{hidden} contiguous")
    assert dnn.gelu(g.GELU_ERF, xd, dx.p, xd, dy.p) == g.SUCCESS
    g.synchronize()
    out = dy.download(nptype(t), xe.size + 8)
    assert np.array_equal(out[xe.size:].view(np.uint8), guard.view(np.uint8))
    check(dec(out[:xe.size].copy(), t).reshape(rows, hidden),
          O.gelu(dec(xe, t).reshape(rows, hidden), g.GELU_ERF).reshape(rows, hidden), t,
          atol={BF16: 1e-6, F16: 1e-6, F32: 1e-7}[t])


# Lengths around the chunk (shorter rows take a path of their own), one, two
# and four chunks per lane, and what each leaves for the last chunk.
@pytest.mark.parametrize("layer", [False, True])
@pytest.mark.parametrize("t,hidden", [(BF16, h) for h in (1, 7, 8, 9, 15, 511, 512, 513, 1023, 1025, 2041, 2048, 2049)] +
                         [(F16, h) for h in (3, 10, 505, 1017)] +
                         [(F32, h) for h in (1, 3, 4, 5, 7, 255, 256, 257, 511, 513, 1021, 1024, 1025)])
def test_short_unaligned_norms_in_place(dnn, t, hidden, layer):
    """The last chunk of a row repeats elements of the one before it: they
    count once in the statistics, and in place no chunk reads what another
    has already replaced. A NaN among the repeated elements stays in its row."""
    rows, pitch = 7, hidden + 1
    r = np.random.default_rng(hidden)
    x = (1.5 + 2.0 * r.standard_normal((rows, hidden))).astype(np.float32)
    xe = enc(x, t)
    ge, be = (enc(a.astype(np.float32), t) for a in (1 + 0.1 * r.standard_normal(hidden), r.standard_normal(hidden)))
    xe[4, max(0, hidden - 3)] = 0x7FC1 if t == BF16 else 0x7E01 if t == F16 else np.nan
    poison = np.asarray(0x7FC1 if t != F32 else np.float32(np.nan), nptype(t))
    buf = np.full(1 + rows * pitch, poison, nptype(t))
    buf[1:].reshape(rows, pitch)[:, :hidden] = xe
    dx, dg, db = to_dev(buf), to_dev(np.concatenate([poison[None], ge])), to_dev(np.concatenate([poison[None], be]))
    xd, wd = g.TensorDesc(t, [rows, hidden], [pitch, 1]), g.TensorDesc(t, [hidden])
    p, pg, pb = (offset(b, t) for b in (dx, dg, db))
    say(f"{'layer' if layer else 'rms'}norm t={t} hidden={hidden} in place, one element off")
    s = dnn.layernorm(xd, p, wd, pg, pb, 1e-6, xd, p) if layer else dnn.rmsnorm(xd, p, wd, pg, 1e-6, xd, p)
    assert s == g.SUCCESS, g.STATUS[s]
    g.synchronize()
    out = dx.download(nptype(t), buf.size)
    body = out[1:].reshape(rows, pitch)
    around = np.concatenate([out[:1], body[:, hidden:].reshape(-1)])
    assert np.array_equal(around.view(np.uint8), np.full(around.size, poison, nptype(t)).view(np.uint8))
    y = dec(np.ascontiguousarray(body[:, :hidden]), t)
    assert np.isnan(y[4]).all()
    keep = [i for i in range(rows) if i != 4]
    xq, gq, bq = dec(xe, t)[keep], dec(ge, t), dec(be, t)
    if layer:
        check_norm(y[keep], O.layernorm(xq, gq, bq, 1e-6), bq, t)
    else:
        check_norm(y[keep], O.rmsnorm(xq, gq, 1e-6), None, t)
