"""GPU parity of the streaming M = 1 GEMV (viper_amd/csrc/qgemv_stream.h): rows that no exact tiling covers.

Group dots bit-exact against the oracle and outputs to the usual bar, at the edges of its shapes: one chunk pair, the
widths where the team or the slot count changes, odd group counts (a unit's scales then start anywhere in a 16-byte
word, and an odd N ends the scale array within a dword), rows of more than one segment up to the longest K the entry
point takes, row counts around one unit, one wave turn and the two-rows-per-unit rule, and launches of several matrices.
"""
import numpy as np
import pytest

import oracle as O
import viper_amd as va
from test_gpu_folded import P, bf16, dev, u16, weights
from test_gpu_parity import run_case, torch_dev  # noqa: F401

pytestmark = pytest.mark.gpu


# Q4/Q5/Q6 chunks per row: K / 32; W8: K / 16
@pytest.mark.parametrize("qtype", [O.Q4_G64, O.Q5_G64, O.Q6_G64, O.W8_G32])
@pytest.mark.parametrize("N,K,senc", [
    (1, 64, 1), (9, 256, 0), (5, 320, 1), (37, 512, 1), (33, 576, 0), (129, 1024, 1), (67, 1088, 0), (61, 2048, 1),
    (65, 2112, 1), (2561, 3520, 0), (3001, 4096, 1), (257, 4160, 0), (100, 6144, 1), (43, 8128, 0), (19, 11008, 1),
    (13, 14400, 0), (11, 16448, 1), (7, 18432, 0), (5, 20480, 1), (3, 20544, 1), (9, 30016, 0), (5, 38976, 1)])
def test_stream_edges(torch_dev, qtype, N, K, senc):  # noqa: F811
    seed = 0x57A000 + 7 * N + K
    a = run_case(torch_dev, qtype, N, K, 1, seed, scale_enc=senc, residual=(N % 2 == 1), outlier=0.05)
    b = run_case(torch_dev, qtype, N, K, 1, seed, scale_enc=senc, residual=(N % 2 == 1), outlier=0.05,
                 check_partials=False)
    np.testing.assert_array_equal(a, b)


# several matrices in one launch equal single calls bit for bit: units and workgroups of each matrix end raggedly
@pytest.mark.parametrize("qtype,K,ns", [(O.Q4_G64, 4096, (3000, 77, 513)), (O.Q6_G64, 1984, (65, 1, 300)),
                                        (O.Q5_G64, 8896, (517, 2049)), (O.W8_G32, 1056, (1000, 31, 5))])
@pytest.mark.parametrize("pro", [P.BF16, P.INT8, P.RMSNORM, P.SWIGLU])
def test_stream_matrices_equal_single_calls(torch_dev, qtype, K, ns, pro):  # noqa: F811
    torch = torch_dev
    G = O.group_size(qtype)
    ws = [weights(torch, qtype, n, K, 0x57B00 + n, O.SCALE_BF16)[0] for n in ns]
    x = O.gen_act(1, K, 0x57C00, outlier_frac=0.02)
    second = {P.BF16: None, P.RMSNORM: dev(torch, bf16(1.0 + 0.1 * np.random.default_rng(1).standard_normal(K))),
              P.SWIGLU: dev(torch, O.gen_act(1, K, 0x57C01))}
    if pro == P.INT8:
        a, b = (dev(torch, t) for t in O.quantize_act(x, G))
    else:
        a, b = dev(torch, x), second[pro]
    new = lambda w: torch.zeros((1, w.rows), dtype=torch.int16, device="cuda")
    ys, refs, res = [new(w) for w in ws], [new(w) for w in ws], dev(torch, O.gen_act(1, ns[0], 3))
    assert va.linear_m1(ws, pro, a, b, ys, eps=1e-6, residual=res).ok()
    for i, (w, r) in enumerate(zip(ws, refs)):
        assert va.linear_m1([w], pro, a, b, [r], eps=1e-6, residual=res if i == 0 else None).ok()
    # the residual in place: its rows are read before the same wave stores them
    y0 = res.clone()
    assert va.linear_m1([ws[0]], pro, a, b, [y0], eps=1e-6, residual=y0).ok()
    torch.cuda.synchronize()
    for y, r in zip(ys + [y0], refs + [refs[0]]):
        np.testing.assert_array_equal(u16(y), u16(r))


# the gate/up pair equals the two outputs followed by the swiglu kernel, also over segments and two rows per unit
@pytest.mark.parametrize("qtype,N,K,pro", [(O.Q4_G64, 3072, 4096, P.RMSNORM), (O.Q4_G64, 64, 23040, P.BF16),
                                           (O.Q6_G64, 4096, 1984, P.BF16), (O.W8_G32, 96, 11200, P.RMSNORM),
                                           (O.Q5_G64, 2560, 3520, P.BF16)])
def test_stream_pair_equals_chain(torch_dev, qtype, N, K, pro):  # noqa: F811
    torch = torch_dev
    wg, wu = (weights(torch, qtype, N, K, 0x57D00 + i, O.SCALE_BF16)[0] for i in (0, 1))
    x = dev(torch, O.gen_act(1, K, 0x57D10, outlier_frac=0.02))
    gamma = dev(torch, bf16(1.0 + 0.1 * np.random.default_rng(2).standard_normal(K))) if pro == P.RMSNORM else None
    z = lambda: torch.zeros((1, N), dtype=torch.int16, device="cuda")
    h, g1, u1, h1, g, u, h2 = z(), z(), z(), z(), z(), z(), z()
    assert va.linear_m1_swiglu(wg, wu, pro, x, gamma, h, eps=1e-6).ok()
    assert va.linear_m1_swiglu(wg, wu, pro, x, gamma, h1, eps=1e-6, gate_out=g1, up_out=u1).ok()
    assert va.linear_m1([wg, wu], pro, x, gamma, [g, u], eps=1e-6).ok()
    G = O.group_size(qtype)
    xq = torch.zeros((1, N), dtype=torch.int8, device="cuda")
    xs = torch.zeros((1, N // G), dtype=torch.float32, device="cuda")
    assert va.swiglu_quantize(g, u, G, xq, xs, out=h2).ok()
    torch.cuda.synchronize()
    for a, b in ((g1, g), (u1, u), (h, h2), (h1, h2)):
        np.testing.assert_array_equal(u16(a), u16(b))


# Most slots per lane, one to three segments and staging rounds, and waves with no unit (few rows): the folded
# prologues equal the producer's kernel followed by the int8 row.
@pytest.mark.parametrize("qtype,N,K", [(O.Q6_G64, 1024, 10752), (O.Q6_G64, 3, 8256), (O.Q5_G64, 300, 12288),
                                       (O.Q4_G64, 5, 20480), (O.Q4_G64, 2048, 12288), (O.W8_G32, 77, 8192)])
@pytest.mark.parametrize("pro", [P.RMSNORM, P.SWIGLU])
def test_stream_idle_waves_every_prologue(torch_dev, qtype, N, K, pro):  # noqa: F811
    torch = torch_dev
    G = O.group_size(qtype)
    w = weights(torch, qtype, N, K, 0x57E00 + N, O.SCALE_BF16)[0]
    a = dev(torch, O.gen_act(1, K, 0x57E10, outlier_frac=0.02))
    b = dev(torch, bf16(1.0 + 0.1 * np.random.default_rng(3).standard_normal((1, K))))
    res = dev(torch, O.gen_act(1, N, 5))
    y, r = (torch.zeros((1, N), dtype=torch.int16, device="cuda") for _ in range(2))
    xq = torch.zeros((1, K), dtype=torch.int8, device="cuda")
    xs = torch.zeros((1, K // G), dtype=torch.float32, device="cuda")
    assert va.linear_m1([w], pro, a, b.view(-1) if pro == P.RMSNORM else b, [y], eps=1e-6, residual=res).ok()
    if pro == P.RMSNORM:
        assert va.rmsnorm_quantize(a, b.view(-1), 1e-6, G, xq, xs).ok()
    else:
        assert va.swiglu_quantize(a, b, G, xq, xs).ok()
    assert va.linear_m1([w], P.INT8, xq, xs, [r], residual=res).ok()
    torch.cuda.synchronize()
    np.testing.assert_array_equal(u16(y), u16(r))


# The pair equals the launch of both matrices also where single rows of the K take an exact tiling for some N.
@pytest.mark.parametrize("qtype,N,K", [(O.Q4_G64, 2560, 5120), (O.Q4_G64, 4608, 5120), (O.Q4_G64, 1536, 6144),
                                       (O.Q4_G64, 1280, 10240), (O.W8_G32, 2560, 5120), (O.Q5_G64, 1536, 20480)])
@pytest.mark.parametrize("pro", [P.BF16, P.RMSNORM])
def test_pair_equals_chain_over_tilings(torch_dev, qtype, N, K, pro):  # noqa: F811
    torch = torch_dev
    wg, wu = (weights(torch, qtype, N, K, 0x57F00 + i, O.SCALE_BF16)[0] for i in (0, 1))
    x = dev(torch, O.gen_act(1, K, 0x57F10, outlier_frac=0.02))
    gamma = dev(torch, bf16(1.0 + 0.1 * np.random.default_rng(4).standard_normal(K))) if pro == P.RMSNORM else None
    h, g, u, g1, u1, g2, u2 = (torch.zeros((1, N), dtype=torch.int16, device="cuda") for _ in range(7))
    assert va.linear_m1_swiglu(wg, wu, pro, x, gamma, h, eps=1e-6, gate_out=g, up_out=u).ok()
    assert va.linear_m1([wg, wu], pro, x, gamma, [g1, u1], eps=1e-6).ok()
    assert va.linear_m1([wg], pro, x, gamma, [g2], eps=1e-6).ok() and va.linear_m1([wu], pro, x, gamma, [u2], eps=1e-6).ok()
    torch.cuda.synchronize()
    for a, b in ((g, g1), (u, u1), (g, g2), (u, u2)):
        np.testing.assert_array_equal(u16(a), u16(b))
