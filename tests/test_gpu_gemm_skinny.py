"""GemmEx of few columns (gemm_skinny): 16-bit and int8 TN problems of up to
64 columns, bit for bit on inputs whose sums are exact in any order, with guard
bands around C and the plan the library logs."""
import numpy as np
import pytest

import grxcp_amd as g
from test_gpu_gemm import dequant_case, float_case, int8_case, logged_plans

pytestmark = pytest.mark.gpu
BF16, F16, F32 = g.GRX_R_16BF, g.GRX_R_16F, g.GRX_R_32F

# rows and columns at the edges of 16 (32 from 8192 rows on), K of 4 stages,
# ending inside a stage and inside a 64-byte step, fewer stages than waves
SHAPES = [(1, 1, 256), (15, 16, 264), (17, 15, 1032), (130, 17, 512), (33, 32, 2056), (64, 33, 328),
          (250, 64, 1024), (8200, 3, 256), (8209, 40, 264), (8192, 64, 256)]


@pytest.mark.parametrize("in_t,out_t", [(BF16, BF16), (BF16, F32), (F16, F16)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_skinny_exact(blas, capfd, in_t, out_t, m, n, k):
    res = []
    plans = logged_plans(capfd, lambda: res.append(
        float_case(blas, in_t, out_t, 1, 0, m, n, k, 1.0, 0.0, 8, cpad=0, guard=True)))
    assert res == [(0, 0)]
    assert [p["kernel"] for p in plans] == ["skinny"], plans


@pytest.mark.parametrize("m,n,k,cpad", [(130, 17, 512, 1), (48, 5, 256, 8), (8209, 33, 256, 3)])
@pytest.mark.parametrize("out_t", [BF16, F32])
def test_skinny_alpha_beta_and_c_alignment(blas, out_t, m, n, k, cpad):
    """C's columns on and off 16-byte boundaries, alpha and beta."""
    assert float_case(blas, BF16, out_t, 1, 0, m, n, k, 0.5, 2.0, 0, cpad=cpad, guard=True) == (0, 0)


@pytest.mark.parametrize("m,n,k", [(31, 1, 512), (100, 16, 528), (130, 40, 1040), (8200, 32, 512)])
def test_skinny_int8_exact(blas, m, n, k):
    assert int8_case(blas, 1, 0, m, n, k, 1.0, 0.0, 0, guard=True) == 0
    assert int8_case(blas, 1, 0, m, n, k, 3.0, -2.0, 16, cpad=1, guard=True) == 0
    assert dequant_case(blas, 1, 0, m, n, k, 0, 0, 3, guard=True) == (0, 0)


def test_skinny_limits(blas, capfd):
    """Past 64 columns, below 4 stages of K, with an operand off 16 bytes or
    with many rows of long K the other kernels run."""
    for m, n, k, pad in [(128, 65, 512, 0), (128, 16, 248, 0), (128, 16, 512, 4), (4104, 9, 4104, 0),
                         (8200, 17, 2056, 0)]:
        res = []
        plans = logged_plans(capfd, lambda: res.append(
            float_case(blas, BF16, F32, 1, 0, m, n, k, 1.0, 0.0, pad, cpad=0)))
        assert res == [(0, 0)]
        assert [p["kernel"] for p in plans] != ["skinny"], (m, n, k, pad)


@pytest.mark.parametrize("m,n,kmax", [(16, 8, 14336), (2576, 3, 0), (128, 16, 12288), (3088, 32, 11264),
                                      (128, 17, 8192), (64, 33, 5120), (4096, 64, 5120),
                                      (2576, 8, 24576), (3088, 9, 20480), (8208, 17, 2048), (12304, 16, 4096)])
def test_skinny_k_bound(blas, capfd, m, n, kmax):
    """K of the longest that one workgroup takes runs on gemm_skinny, K one
    16-byte chunk longer on the 128x128 tiles and their K slices (kmax 0: no
    bound); both exact."""
    for k in (kmax, kmax + 8) if kmax else (40000,):
        res = []
        plans = logged_plans(capfd, lambda: res.append(
            float_case(blas, BF16, F32, 1, 0, m, n, k, 1.0, 0.0, 0, cpad=0)))
        assert res == [(0, 0)]
        assert [p["kernel"] == "skinny" for p in plans] == [k <= kmax or not kmax], (k, plans)
