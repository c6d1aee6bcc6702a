"""The split greedy pick of many rows (more logits per workgroup from 49 workgroups on) against the CPU oracle's argmax:
exact, at the edges of its workgroups (16384 logits) and of the row count where it begins."""
import numpy as np
import pytest

import oracle as O
import viper_amd as va
from test_gpu_lm_head import bf16, dev, torch_dev, ws  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,V", [(48, 8), (49, 8), (6, 32768), (7, 32768), (16, 16376), (16, 16384), (16, 16392),
                                 (13, 49152 - 8), (2, 166144), (16, 166144)])
def test_greedy_rows(torch_dev, B, V):  # noqa: F811
    torch = torch_dev
    print(f"greedy B={B} V={V}", flush=True)
    rng = np.random.default_rng(B * V)
    lg = bf16(rng.standard_normal((B, V)))
    top = bf16([9.0])[0]
    lg[0, V - 1] = top                                            # the last element
    lg[1 % B, min(V - 1, 16383)] = lg[1 % B, min(V - 2, 16384)] = top  # equal maxima on both sides of an edge
    if B > 5:
        lg[2] = bf16([np.nan])[0]                                 # nothing above -inf: 0
        lg[3] = bf16([-np.inf])[0]
        lg[4] = bf16([-np.inf])[0]
        lg[4, V - 3] = bf16([-65504.0])[0]                        # the only finite value
        lg[5] = bf16([-3.0])[0]
        lg[5, V // 2] = bf16([-0.0])[0]
        lg[5, V - 1] = bf16([0.0])[0]                             # -0 and +0 are equal: the first
    x, w, expect = dev(torch, lg), ws(torch, B, True), O.argmax_bf16(lg)
    for _ in range(2):
        out = torch.full((B,), -1, dtype=torch.int32, device="cuda")
        assert va.sampling_greedy(x, out, workspace=w).ok()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.cpu().numpy(), expect)
        assert int(w.count_nonzero()) == 0
