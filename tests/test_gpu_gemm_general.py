"""GemmEx's general kernel: every layout at the edges of its 64x64 tiles, of its
128-byte K stages and of its 16-byte loads, with 1, 2 and 4 K groups, bit for
bit on inputs whose sums are exact in any order, with guard bands around C."""
import pytest

import grxcp_amd as g
from test_gpu_gemm import dequant_case, float_case, int8_case, logged_plans
from test_gpu_gemm_batched import batched_case

pytestmark = pytest.mark.gpu
BF16, F16, F32 = g.GRX_R_16BF, g.GRX_R_16F, g.GRX_R_32F
LAYOUTS = [(0, 0), (0, 1), (1, 1), (1, 0)]

# rows shorter than one load; exactly one; a stage and one element more; 2, 3,
# 5 and 10 stages (2 and 4 K groups, groups without a stage); a partial last one
SHAPES = [(1, 1, 1), (7, 9, 5), (8, 8, 8), (9, 8, 15), (64, 64, 64), (65, 63, 65), (63, 130, 127),
          (64, 128, 192), (70, 9, 193), (129, 67, 321), (257, 62, 639), (100, 3, 200)]


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("in_t,out_t", [(BF16, BF16), (F16, F32)])
def test_general_exact(blas, in_t, out_t, ta, tb):
    bad = []
    for m, n, k in SHAPES:
        for alpha, beta, pad, cpad in [(1.0, 0.0, 0, 1), (2.5, -1.5, 3, 0)]:
            res = float_case(blas, in_t, out_t, ta, tb, m, n, k, alpha, beta, pad, cpad, seed=m + k, guard=True)
            if res != (0, 0):
                bad.append((m, n, k, alpha, res))
    assert not bad, bad


@pytest.mark.parametrize("ta,tb", LAYOUTS)
def test_general_int8_exact(blas, ta, tb):
    for m, n, k in [(15, 17, 13), (16, 16, 16), (65, 31, 129), (70, 130, 385), (64, 64, 256)]:
        assert int8_case(blas, ta, tb, m, n, k, 1.0, 0.0, 1, cpad=0, guard=True) == 0, (m, n, k)
        assert int8_case(blas, ta, tb, m, n, k, 3.0, -2.0, 0, cpad=1, guard=True) == 0, (m, n, k)
        assert dequant_case(blas, ta, tb, m, n, k, 1, 3, seed=k, guard=True) == (0, 0), (m, n, k)


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("m,n,k,batch", [(130, 70, 330, 43), (130, 70, 330, 90)])
def test_general_group_counts_by_workgroups(blas, ta, tb, m, n, k, batch):
    """258 workgroups run 2 K groups, 540 run one."""
    assert batched_case(blas, BF16, BF16, ta, tb, m, n, k, 1.0, 0.0, batch, "packed", "packed", "gap") == 0


@pytest.mark.parametrize("m,n,k,kernel", [(301, 300, 1529, "general64"), (301, 300, 1536, "general64"),
                                          (301, 300, 1544, "tn128"), (1027, 1030, 300, "tn128")])
def test_general_or_copies(blas, capfd, m, n, k, kernel):
    """Past the copy threshold: the general kernel up to one workgroup per CU
    and 3072 bytes of K, operand copies beyond."""
    res = []
    plans = logged_plans(capfd, lambda: res.append(
        float_case(blas, F16, F16, 0, 0, m, n, k, 1.0, 0.0, 0, 0, seed=k, guard=True)))
    assert res == [(0, 0)]
    assert [p["kernel"] for p in plans] == [kernel], plans
