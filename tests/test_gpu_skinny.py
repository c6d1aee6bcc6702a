"""GPU parity of the streaming skinny GEMM (viper_amd/csrc/qgemm_stream.h): K that is no multiple of four groups, and
rows past what the row-contiguous kernel holds.

Group dots bit-exact against the oracle and outputs to the usual bar (1 bf16 ulp or 1e-5 * sum |group terms|) at the
edges of its shapes: one group, the group counts where the loads per lane or the waves' shares change (8 waves, 2 groups
per load and wave: 16, 32, 48, 64, 96), waves without a group, a second phase over K, 1..16 rows with 8 / 9 as the line
between two groups and one per accumulator, row counts around one 16-row tile and around one tile per workgroup, and an
odd number of scales (their array ends within a dword).
"""
import numpy as np
import pytest

import oracle as O
import viper_amd as va
from test_gpu_folded import dev, u16, weights
from test_gpu_frag import to_frag
from test_gpu_parity import REL_TOL, run_case, torch_dev  # noqa: F401

pytestmark = pytest.mark.gpu
FORMATS = [O.Q4_G64, O.Q5_G64, O.Q6_G64, O.W8_G32]


# K in groups (64 weights, W8 32)
@pytest.mark.parametrize("qtype", FORMATS)
@pytest.mark.parametrize("N,ng,M,senc", [
    (1, 1, 2, 1), (16, 2, 16, 0), (17, 3, 3, 1), (255, 7, 8, 0), (257, 9, 9, 1), (63, 17, 4, 1), (4355, 31, 2, 0),
    (31, 33, 16, 1), (513, 47, 7, 0), (129, 49, 5, 1), (2561, 55, 8, 1), (33, 63, 12, 0), (1025, 65, 6, 1),
    (77, 95, 8, 1), (77, 94, 16, 1), (65, 97, 8, 0), (40, 114, 10, 1), (21, 193, 2, 1), (8197, 5, 8, 1)])
def test_skinny_edges(torch_dev, qtype, N, ng, M, senc):  # noqa: F811
    K, seed = ng * O.group_size(qtype), 0x5C1000 + 11 * N + ng
    a = run_case(torch_dev, qtype, N, K, M, seed, scale_enc=senc, residual=(N % 2 == 1), outlier=0.05)
    b = run_case(torch_dev, qtype, N, K, M, seed, scale_enc=senc, residual=(N % 2 == 1), outlier=0.05,
                 check_partials=False)
    # the int32 dots' launch holds one group per accumulator, the other two for up to 8 rows: another fp32 order
    if M > 8:
        np.testing.assert_array_equal(a, b)


# one row whose quantized form is too long for the GEMV's LDS
def test_skinny_one_long_row(torch_dev):  # noqa: F811
    run_case(torch_dev, O.Q4_G64, 19, 50048, 1, 0x5C2000, scale_enc=1, residual=True)


# every layout of the activation and the fused pair, bit for bit: bf16 rows (quantized by the workgroups, or by a launch
# of their own), int8 rows, fragments; a pair's rows per workgroup differ from a single matrix's
@pytest.mark.parametrize("qtype,N,ng,M", [
    (O.Q4_G64, 2561, 55, 8), (O.Q5_G64, 515, 35, 16), (O.Q6_G64, 300, 130, 5), (O.W8_G32, 1031, 54, 11),
    (O.Q4_G64, 9217, 64, 4), (O.Q4_G64, 8200, 96, 16), (O.Q5_G64, 8193, 68, 8), (O.Q6_G64, 6200, 56, 13),
    (O.W8_G32, 12300, 92, 6)])
def test_skinny_layouts_agree(torch_dev, qtype, N, ng, M):  # noqa: F811
    torch = torch_dev
    G = O.group_size(qtype)
    K = ng * G
    w0, w1 = (weights(torch, qtype, N, K, 0x5C3000 + i, O.SCALE_FP16)[0] for i in (0, 1))
    x = O.gen_act(M, K, 0x5C3010, outlier_frac=0.02)
    xq, xs = O.quantize_act(x, G)
    xd, xqd, xsd, res = dev(torch, x), dev(torch, xq), dev(torch, xs), dev(torch, O.gen_act(M, N, 4))
    wk = torch.zeros(max(16, va.workspace_bytes(qtype, N, K, M)), dtype=torch.uint8, device="cuda")
    new = lambda: torch.zeros((M, N), dtype=torch.int16, device="cuda")
    a0, a1, b0, b1, c0, c1, d0, e0, f0 = (new() for _ in range(9))
    assert va.linear(w0, xd, a0, residual=res, workspace=wk).ok() and va.linear(w1, xd, a1, workspace=wk).ok()
    assert va.linear_prequantized(w0, xqd, xsd, b0, residual=res).ok()
    assert va.linear_prequantized(w1, xqd, xsd, b1).ok()
    assert va.linear_fused2(w0, w1, xd, c0, c1, workspace=wk).ok()
    assert va.linear_fused2_prequantized(w0, w1, xqd, xsd, d0, e0).ok()
    f0.copy_(res)
    assert va.linear(w0, xd, f0, residual=f0, workspace=wk).ok()  # the residual in place
    torch.cuda.synchronize()
    for a, b in ((a0, b0), (a1, b1), (a1, c1), (a1, e0), (c0, d0), (a0, f0)):
        np.testing.assert_array_equal(u16(a), u16(b))
    if ng % 4 == 0:
        xf, xsf = to_frag(xq, xs, G)
        g0, h0, h1 = new(), new(), new()
        xfd, xsfd = dev(torch, xf), dev(torch, xsf)
        assert va.linear_prequantized_frag(w0, xfd, xsfd, g0, residual=res).ok()
        assert va.linear_fused2_prequantized_frag(w0, w1, xfd, xsfd, h0, h1).ok()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(u16(g0), u16(a0))
        np.testing.assert_array_equal(u16(h1), u16(a1))


# a weight scale of infinity or a NaN activation stays in its own outputs
@pytest.mark.parametrize("M", [3, 16])
def test_skinny_nonfinite_stays(torch_dev, M):  # noqa: F811
    torch = torch_dev
    N, K = 70, 64 * 21
    w, packed, scales = weights(torch, O.Q4_G64, N, K, 0x5C4000, O.SCALE_BF16)[:3]
    x = O.gen_act(M, K, 0x5C4001)
    y = torch.zeros((M, N), dtype=torch.int16, device="cuda")
    ref = torch.zeros_like(y)
    wk = torch.zeros(max(16, va.workspace_bytes(O.Q4_G64, N, K, M)), dtype=torch.uint8, device="cuda")
    assert va.linear(w, dev(torch, x), ref, workspace=wk).ok()
    w.scales.view(torch.int16).view(-1)[33 * 21 + 4] = 0x7F80  # row 33
    x2 = x.copy()
    x2[1, 7 * 64 + 5] = 0x7FC0  # row 1
    assert va.linear(w, dev(torch, x2), y, workspace=wk).ok()
    torch.cuda.synchronize()
    a, b = u16(y), u16(ref)
    keep = np.ones((M, N), bool)
    keep[:, 33] = False
    keep[1, :] = False
    np.testing.assert_array_equal(a[keep], b[keep])


# The residual's values are requested by the wave that sums a tile: one to many tiles per workgroup, a ragged last one,
# rows short of 16, one and several phases, in place and apart, against the oracle.
@pytest.mark.parametrize("qtype,N,ng,M", [(O.Q4_G64, 15, 5, 3), (O.Q4_G64, 23260, 5, 10), (O.Q4_G64, 11000, 96, 16),
                                          (O.Q5_G64, 12289, 3, 9), (O.Q6_G64, 517, 101, 5), (O.W8_G32, 9001, 61, 7),
                                          (O.W8_G32, 300, 121, 12)])
def test_skinny_residual(torch_dev, qtype, N, ng, M):  # noqa: F811
    torch = torch_dev
    G = O.group_size(qtype)
    K = ng * G
    w, packed, scales = weights(torch, qtype, N, K, 0x5C5000 + N, O.SCALE_BF16)[:3]
    x, res = O.gen_act(M, K, 0x5C5010, outlier_frac=0.02), O.gen_act(M, N, 0x5C5011)
    rd, y = dev(torch, res), torch.zeros((M, N), dtype=torch.int16, device="cuda")
    wk = torch.zeros(max(16, va.workspace_bytes(qtype, N, K, M)), dtype=torch.uint8, device="cuda")
    z = rd.clone()
    assert va.linear(w, dev(torch, x), y, residual=rd, workspace=wk).ok()
    assert va.linear(w, dev(torch, x), z, residual=z, workspace=wk).ok()
    torch.cuda.synchronize()
    y_ref, _, absterm = O.qlinear(qtype, packed, scales, O.SCALE_BF16, N, K, x, residual=res)
    O.assert_bf16_close(u16(y), y_ref, absterm, rel=REL_TOL)
    np.testing.assert_array_equal(u16(y), u16(z))
