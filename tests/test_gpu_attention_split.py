"""Attention problems of few query tiles: items of 128 or 64 queries whose
workgroups split the keys over two or four groups of waves (attn_split), and
causal launches whose heads form one block of the persistent kernel's item
order. Every head against the oracle."""
import ctypes

import numpy as np
import pytest

import grxcp_amd as g
import oracle as O
from helpers import normwise_rel_err, say, to_dev
from test_gpu_dnn import dec, enc, run_attention

pytestmark = pytest.mark.gpu
BF16, F16 = g.GRX_R_16BF, g.GRX_R_16F


def check_heads(dnn, t, B, H, S, D, causal):
    o, q, k, v = run_attention(dnn, t, B, H, S, D, causal, seed=S + D + H)
    assert np.isfinite(o).all()
    for b in range(B):
        for h in range(H):
            ref = O.attention_head(q[b, h], k[b, h], v[b, h], causal, D ** -0.5)
            assert normwise_rel_err(o[b, h], ref) <= 1e-2, (b, h)


# S around the tiles (64 keys), the steps (128 and 256 keys) and the items (64
# and 128 queries): key groups without a tile, partial tiles, one and several
# steps; few heads (64-query items) and more (128-query items)
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,S", [(1, 1, 1), (1, 3, 63), (2, 4, 65), (1, 8, 129), (1, 5, 257), (1, 4, 700),
                                   (1, 24, 200), (2, 16, 300), (3, 20, 130), (1, 32, 517), (1, 8, 1025)])
def test_attention_split(dnn, B, H, S, D, causal):
    check_heads(dnn, BF16, B, H, S, D, causal)


@pytest.mark.parametrize("D", [64, 128])
def test_attention_split_f16(dnn, D):
    check_heads(dnn, F16, 1, 12, 321, D, True)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("case", ["growing", "shrinking"])
def test_attention_split_groups_with_unlike_maxima(dnn, case, D):
    """Key magnitudes that grow or shrink along the sequence: the groups'
    maxima differ by far more than a float's exponent range in their weights,
    so all but one group's contribution underflows."""
    B, H, S = 1, 4, 640
    r = np.random.default_rng(11 + D)
    ramp = np.linspace(0.0, 40.0, S, dtype=np.float32)[None, None, :, None]
    k = r.standard_normal((B, H, S, D)).astype(np.float32) * (ramp if case == "growing" else ramp[:, :, ::-1])
    o, q, kq, v = run_attention(dnn, BF16, B, H, S, D, False, seed=5, k=k)
    assert np.isfinite(o).all()
    for h in range(H):
        ref = O.attention_head(q[0, h], kq[0, h], v[0, h], False, D ** -0.5)
        assert normwise_rel_err(o[0, h], ref) <= 1e-2, h


@pytest.mark.parametrize("H,S,D", [(104, 760, 64), (88, 700, 128)])
def test_attention_heads_in_one_block(dnn, H, S, D):
    """39 and 33 causal items on each XCD's 32 workgroups: one block of all
    its heads, dealt in a snake from the heaviest items on."""
    check_heads(dnn, BF16, 1, H, S, D, True)


# Keys masked by a bias column of K: a tail, one key, the first tile (left
# padding); heads and S for 64-query and 128-query items and for attn_fwd.
MASKS = {"tail64": slice(64, None), "tail128": slice(128, None), "tail256": slice(256, None),
         "key64": slice(64, 65), "key128": slice(128, 129), "head64": slice(0, 64)}


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("t,fill", [(BF16, -np.inf), (BF16, -3.3895314e38), (BF16, -1e30), (F16, -np.inf),
                                    (F16, -65504.0)])
@pytest.mark.parametrize("D,H,S", [(64, 6, 500), (128, 6, 500), (64, 64, 300), (128, 64, 300), (64, 200, 300),
                                   (128, 200, 300)])
def test_attention_masked_keys(dnn, D, H, S, t, fill, causal):
    """Key groups (and a first tile) whose every score is -inf or hugely
    negative have weight 0; a row that sees only -inf scores is NaN."""
    r = np.random.default_rng(S + D)
    q = r.standard_normal((1, H, S, D)).astype(np.float32)
    k = r.standard_normal((1, H, S, D)).astype(np.float32)
    q[..., 0] = 1.0
    names = sorted(MASKS)
    for h, name in enumerate(names):
        k[0, h, MASKS[name]] = 0.0
        k[0, h, MASKS[name], 0] = fill
    o, qq, kq, v = run_attention(dnn, t, 1, H, S, D, causal, seed=3, q=q, k=k)
    for h, name in enumerate(names):
        ref = O.attention_head(qq[0, h], kq[0, h], v[0, h], causal, D ** -0.5)
        lo = 64 if causal and name == "head64" else 0     # rows before lo see masked keys only
        if np.isinf(fill):
            assert np.isnan(o[0, h, :lo]).all()
        assert np.isfinite(o[0, h, lo:]).all(), name
        assert normwise_rel_err(o[0, h, lo:], ref[lo:]) <= 1e-2, name


@pytest.mark.parametrize("causal", [False, True])
def test_attention_masked_group_maxima(dnn, causal):
    """Scores -1.5 * 2^35 and 4096 more (one ulp): scaled, both round to one
    float, which the first lies below and the second exceeds by 482 (the
    exponent of an overflowing weight). The group of the tiles 1 and 5, which
    hold them, must still add 0."""
    c = np.float32(0.125) * np.float32(1.4426950408889634)
    s = np.float32([-1.5 * 2.0 ** 35, -1.5 * 2.0 ** 35 + 4096])
    m, exact = (s * c).astype(np.float64), s.astype(np.float64) * np.float64(c)
    assert m[0] == m[1] and exact[0] < m[0] and exact[1] > m[1] + 140
    H, S, D = 6, 500, 64
    r = np.random.default_rng(8)
    q = r.standard_normal((1, H, S, D)).astype(np.float32)
    k = r.standard_normal((1, H, S, D)).astype(np.float32)
    q[..., :2] = 1.0
    for tile, low in ((1, 0.0), (5, 4096.0)):
        k[:, :, 64 * tile:64 * tile + 64] = 0.0
        k[:, :, 64 * tile:64 * tile + 64, 0] = -1.5 * 2.0 ** 35
        k[:, :, 64 * tile:64 * tile + 64, 1] = low
    o, qq, kq, v = run_attention(dnn, BF16, 1, H, S, D, causal, seed=8, q=q, k=k)
    assert np.isfinite(o).all()
    for h in range(H):
        assert normwise_rel_err(o[0, h], O.attention_head(qq[0, h], kq[0, h], v[0, h], causal, D ** -0.5)) <= 1e-2, h


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("t", [BF16, F16])
@pytest.mark.parametrize("H,S,D,kernel", [(24, 517, 64, "split2"), (24, 517, 128, "split2"), (40, 390, 64, "split4"),
                                          (40, 390, 128, "split4"), (200, 300, 64, "fwd"), (200, 300, 128, "fwd"),
                                          (90, 317, 64, "fwd")])   # 270 items of 128 queries on 256 CUs
def test_attention_kernel_choice(dnn, capfd, monkeypatch, H, S, D, kernel, t, causal):
    """Each kernel by its name in the log, on a packed [S, 3, H, D] buffer with
    partial key and query tiles. Heads are copies of five, which must agree."""
    r = np.random.default_rng(S + D)
    x = enc(r.standard_normal((S, 3, 5, D)).astype(np.float32), t).reshape(S, 3, 5, D)
    qkv = np.ascontiguousarray(x[:, :, np.arange(H) % 5])
    dx, do = to_dev(qkv), g.DeviceBuffer(2 * S * H * D)
    xd = g.TensorDesc(t, [1, H, S, D], [3 * S * H * D, D, 3 * H * D, 1])
    od = g.TensorDesc(t, [1, H, S, D], [S * H * D, D, H * D, 1])
    at = [ctypes.c_void_p(dx.p.value + 2 * H * D * i) for i in range(3)]
    say(f"attention t={t} H={H} S={S} D={D} causal={causal}, packed: {kernel}")
    capfd.readouterr()
    monkeypatch.setenv("GRXDNN_LOG", "1")
    s = dnn.attention(g.AttnDesc(causal, D ** -0.5), xd, at[0], xd, at[1], xd, at[2], od, do.p)
    monkeypatch.delenv("GRXDNN_LOG")
    assert s == g.SUCCESS, g.STATUS[s]
    g.synchronize()
    log = [l for l in capfd.readouterr().err.splitlines() if l.startswith("grxdnn: attention ")]
    assert len(log) == 1 and log[0].endswith(f"kernel={kernel}"), log
    o = dec(do.download(np.uint16, S * H * D), t).reshape(S, H, D)
    for h in range(5):
        q, k, v = (dec(np.ascontiguousarray(x[:, i, h]), t).reshape(S, D) for i in range(3))
        assert normwise_rel_err(o[:, h], O.attention_head(q, k, v, causal, D ** -0.5)) <= 1e-2, h
        assert np.array_equal(o[:, h::5], np.repeat(o[:, h:h + 1], len(range(h, H, 5)), 1)), h
