"""GemmEx and Sgemm into a C off 16-byte boundaries with beta = 0: the TN
kernels store it in place at element alignment (no workspace pass), on every
kernel and behind operand copies of odd pitches. Bit for bit on inputs whose
sums are exact, with guard bands, and the plan the library logs."""
import numpy as np
import pytest

import grxcp_amd as g
import oracle as O
from helpers import to_dev
from test_gpu_gemm import float_case, int8_case, logged_plans
from test_gpu_gemm_batched import batched_case

pytestmark = pytest.mark.gpu
BF16, F16, F32, I8, I32 = g.GRX_R_16BF, g.GRX_R_16F, g.GRX_R_32F, g.GRX_R_8I, g.GRX_R_32I


@pytest.mark.parametrize("it,ot,ta,tb,m,n,k,cpad,kernel", [
    (BF16, BF16, 1, 0, 1031, 300, 256, 0, "tn128"),     # every column at another alignment
    (F16, F32, 1, 0, 1030, 300, 520, 3, "tn128"),
    (BF16, BF16, 1, 0, 2305, 2302, 64, 0, "tn128"),     # two-stage ring
    (F16, F16, 1, 0, 4099, 2900, 136, 2, "tn256"),      # 256x256 tiles, partial ones too
    (BF16, F32, 1, 0, 4097, 2900, 64, 0, "tn256"),
    (BF16, BF16, 1, 0, 257, 255, 8192, 0, "tn128"),     # K slices, summed into C
    (F16, F32, 0, 0, 1999, 1037, 301, 0, "tn128"),      # both operands copied, K padded
    (BF16, BF16, 1, 1, 1027, 1025, 129, 5, "tn128"),
    (BF16, BF16, 0, 1, 333, 1029, 333, 0, "general64"),
])
def test_c_off_16_bytes(blas, capfd, it, ot, ta, tb, m, n, k, cpad, kernel):
    res = []
    plans = logged_plans(capfd, lambda: res.append(
        float_case(blas, it, ot, ta, tb, m, n, k, 1.5, 0.0, 0, cpad, seed=m + k, guard=True)))
    assert res == [(0, 0)]
    assert len(plans) == 1 and plans[0]["kernel"] == kernel and plans[0]["staged"] == "0", plans


@pytest.mark.parametrize("ta,tb,m,n,k", [(1, 0, 1030, 300, 256), (0, 0, 1999, 517, 301), (0, 1, 301, 1003, 157)])
def test_c_off_16_bytes_int8(blas, ta, tb, m, n, k):
    assert int8_case(blas, ta, tb, m, n, k, 2.0, 0.0, 0, fill="rand", seed=k, cpad=1, guard=True) == 0


@pytest.mark.parametrize("it,ot,ta,tb,m,n,k,cmode", [
    (BF16, BF16, 1, 0, 203, 203, 64, "gap"), (F16, F32, 1, 0, 101, 130, 128, "neg"),
    (BF16, BF16, 0, 0, 64, 203, 203, "gap"), (F16, F16, 0, 1, 131, 97, 87, "gap"),
    (I8, I32, 0, 0, 99, 131, 150, "gap")])
def test_batched_c_off_16_bytes(blas, it, ot, ta, tb, m, n, k, cmode):
    """Strided batches with odd leading dimensions, A broadcast in one."""
    assert batched_case(blas, it, ot, ta, tb, m, n, k, 1.0, 0.0, 40, "gap", "gap", cmode) == 0
    assert batched_case(blas, it, ot, ta, tb, m, n, k, 1.0, 0.0, 40, "zero", "neg", cmode) == 0


def test_sgemm_large_c_off_16_bytes(blas):
    """fp32 on 256x256 tiles (aligned operands, ldc odd)."""
    m, n, k, ldc = 4100, 4096, 64, 4101
    A, B = O.fill_quarters(m * k, 1), O.fill_quarters(k * n, 7)
    C = O.fill_quarters(ldc * n, 3)
    want = O.sgemm(1, 0, m, n, k, 1.0, A, k, B, k, 0.0, C.copy(), ldc)
    dA, dB, dC = to_dev(A), to_dev(B), to_dev(C)
    assert blas.sgemm(1, 0, m, n, k, 1.0, dA.p, k, dB.p, k, 0.0, dC.p, ldc) == g.SUCCESS
    g.synchronize()
    assert np.max(np.abs(dC.download(np.float32, C.size) - want)) <= 1e-5 * (k + 1)
