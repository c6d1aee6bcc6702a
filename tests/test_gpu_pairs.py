"""GPU parity of the matrix-core kernel that gathers group pairs (viper_amd/csrc/qgemm_mfma.hip): K of an even number of
groups, not a multiple of four, at the edges of its shapes: one pair, pairs a wave short of or past a wave's slots, four
and eight waves, one and two 16-row tiles per workgroup, a ragged last tile, staged and gathered activations, 2 to 16
rows.  Group dots bit-exact against the oracle, outputs to the usual bar."""
import numpy as np
import pytest

import oracle as O
import viper_amd as va
from test_gpu_folded import dev, u16, weights
from test_gpu_parity import REL_TOL, run_case, torch_dev  # noqa: F401

pytestmark = pytest.mark.gpu
FORMATS = [O.Q4_G64, O.Q5_G64, O.Q6_G64, O.W8_G32]
PAIRS = 7


def route(qtype, rows, N, K, M, matrices=1):
    return va.lib().viper_hip_qlinear_route(qtype, rows, N, K, M, matrices)


@pytest.mark.parametrize("qtype", FORMATS)
@pytest.mark.parametrize("N,ng,M,senc", [(1, 2, 9, 1), (300, 2, 16, 0), (17, 6, 10, 0), (2561, 6, 12, 1), (4100, 10, 16, 1),
                                         (16385, 6, 9, 0), (255, 22, 11, 1), (1031, 38, 16, 0), (129, 66, 9, 1),
                                         (2049, 78, 13, 0)])
def test_pairs_edges(torch_dev, qtype, N, ng, M, senc):  # noqa: F811
    K, seed = ng * O.group_size(qtype), 0x9A1000 + 13 * N + ng
    assert route(qtype, 0, N, K, M) == PAIRS
    a = run_case(torch_dev, qtype, N, K, M, seed, scale_enc=senc, residual=(N % 2 == 1), outlier=0.05)
    b = run_case(torch_dev, qtype, N, K, M, seed, scale_enc=senc, residual=(N % 2 == 1), outlier=0.05,
                 check_partials=False)
    np.testing.assert_array_equal(a, b)


# int8 rows gathered in their natural layout and the fused pair, a matrix's workgroups ending raggedly; 130 groups: Q4's
# second load segment, from the natural layout
@pytest.mark.parametrize("qtype,N,ng,M", [(O.Q4_G64, 515, 6, 2), (O.Q4_G64, 2100, 22, 16), (O.Q4_G64, 1030, 130, 16),
                                          (O.Q5_G64, 700, 6, 5), (O.Q6_G64, 2050, 70, 8), (O.W8_G32, 1025, 38, 3),
                                          (O.W8_G32, 10000, 10, 9)])
def test_pairs_int8_rows_and_fused(torch_dev, qtype, N, ng, M):  # noqa: F811
    torch = torch_dev
    G = O.group_size(qtype)
    K = ng * G
    assert route(qtype, 1, N, K, M) == PAIRS
    (w0, p0, s0), (w1, p1, s1) = (weights(torch, qtype, N, K, 0x9A3000 + i, O.SCALE_FP16)[:3] for i in (0, 1))
    x, res = O.gen_act(M, K, 0x9A3010, outlier_frac=0.02), O.gen_act(M, N, 4)
    xq, xs = O.quantize_act(x, G)
    xqd, xsd, rd = dev(torch, xq), dev(torch, xs), dev(torch, res)
    a, b, c, d, e = (torch.zeros((M, N), dtype=torch.int16, device="cuda") for _ in range(5))
    wk = torch.zeros(max(16, va.workspace_bytes(qtype, N, K, M)), dtype=torch.uint8, device="cuda")
    assert va.linear_prequantized(w0, xqd, xsd, a, residual=rd).ok()
    assert va.linear_fused2_prequantized(w0, w1, xqd, xsd, b, c).ok()
    assert va.linear_fused2(w0, w1, dev(torch, x), d, e, workspace=wk).ok()
    torch.cuda.synchronize()
    for packed, scales, r, ys in ((p0, s0, res, (a,)), (p0, s0, None, (b, d)), (p1, s1, None, (c, e))):
        y_ref, _, absterm = O.qlinear_prequant(qtype, packed, scales, O.SCALE_FP16, N, K, xq, xs, residual=r)
        for y in ys:
            O.assert_bf16_close(u16(y), y_ref, absterm, rel=REL_TOL)
