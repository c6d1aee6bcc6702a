"""GPU parity of the LM head's matrix-core kernel (several activation rows) at the edges of its tiles: rows of the last
tile, one to many tiles per wave, row lengths around a 512-byte segment and a 16-byte chunk, every row count that picks
it, non-finite weights and activations staying in their own row and column."""
import numpy as np
import pytest

import oracle as O
import viper_amd as va
from test_gpu_lm_head import bf16, dev, host_u16, torch_dev  # noqa: F401

pytestmark = pytest.mark.gpu


def run(torch, w, x):
    M, N = x.shape[0], w.shape[0]
    y = torch.full((M, N), 7, dtype=torch.int16, device="cuda")
    assert va.linear_bf16(dev(torch, w), dev(torch, x), y).ok()
    torch.cuda.synchronize()
    return host_u16(y)


@pytest.mark.parametrize("M,N,K", [(5, 1, 8), (16, 15, 64), (7, 16, 248), (8, 17, 256), (6, 129, 264), (12, 1000, 2560),
                                   (16, 4097, 2048), (3, 700, 4096), (4, 333, 2568), (2, 65, 16384), (9, 40000, 72),
                                   (5, 12345, 512)])
def test_head_rows(torch_dev, M, N, K):  # noqa: F811
    rng = np.random.default_rng(7 * N + K + M)
    w = bf16(0.05 * rng.standard_normal((N, K)))
    x = O.gen_act(M, K, 0x4EAD + K)
    y_ref, _, absterm = O.linear_bf16(w, x)
    # fp32 sums in another order: 1e-5 of the sum of magnitudes covers K * 2^-24 for K up to 16384 (9.8e-4 * 1e-2)
    O.assert_bf16_close(run(torch_dev, w, x), y_ref, absterm, rel=1e-5)


def test_head_rows_nonfinite(torch_dev):  # noqa: F811
    M, N, K = 8, 100, 1000
    rng = np.random.default_rng(3)
    w, x = bf16(0.05 * rng.standard_normal((N, K))), O.gen_act(M, K, 0x4EAE)
    clean = run(torch_dev, w, x)
    w[41, 999], x[3, 0] = 0x7F80, 0x7FC0  # +inf in one weight row, NaN in one activation row
    y = O.bf16_to_f32(run(torch_dev, w, x))
    assert np.isnan(y[3]).all()
    assert not np.isfinite(y[:, 41]).any()
    keep = np.ones((M, N), dtype=bool)
    keep[3], keep[:, 41] = False, False
    np.testing.assert_array_equal(y[keep], O.bf16_to_f32(clean)[keep])


# Up to 8 tiles per workgroup, whose waves split the row segments of each: 256-element segments by one, two, four and
# eight waves (fewer than waves, uneven, a short last one), a last workgroup with fewer tiles; the last shapes of one
# round of workgroups (256 CUs) and the first of several.
@pytest.mark.parametrize("M,N,K", [(5, 16, 264), (6, 33, 520), (16, 1000, 776), (16, 4096, 2048), (5, 4097, 2312),
                                   (8, 8193, 1032), (3, 8500, 4104), (7, 12289, 520), (5, 16385, 264), (6, 32769, 264),
                                   (5, 65520, 72), (5, 65521, 72)])
def test_head_rows_shared_tiles(torch_dev, M, N, K):  # noqa: F811
    test_head_rows(torch_dev, M, N, K)


def test_head_few_weight_rows_spread(torch_dev):  # noqa: F811
    # A sixteenth of the weight rows spreads over the CUs and takes well under the whole's time (measured 0.41; nine
    # tiles to a workgroup's eight waves, whatever N, 0.79).
    torch = torch_dev
    M, K, reps = 8, 2560, 20
    x = dev(torch, O.gen_act(M, K, 0x4EAF))
    w = torch.full((reps, 16384, K), 0.01, dtype=torch.bfloat16, device="cuda").view(torch.int16)
    y = torch.zeros((M, 16384), dtype=torch.int16, device="cuda")
    us = {}
    for N in (16384, 1024):
        yn = y.view(-1)[:M * N].view(M, N)
        best = 1e9
        for _ in range(5):
            torch.cuda.synchronize()
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                for i in range(reps):
                    assert va.linear_bf16(w[i, :N], x, yn).ok()
            g.replay()
            a.record()
            g.replay()
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b) * 1e3 / reps)
        us[N] = best
    assert us[1024] < 0.6 * us[16384], us
