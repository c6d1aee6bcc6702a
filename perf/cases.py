"""The work whose speed is measured: calls of the quantized linear path as a decode / speculative-verify program makes them.

A program that uses this library keeps a model's matrices on the GPU and runs, per generated token (M = 1) or per
verified draft (M = 2..16 rows), the same launches over all layers.  One pass of a case is one sweep over `layers` layers,
each with weights, input rows and outputs of its own, so a pass streams its weights from memory as a decode step does.
The launches are captured once into a HIP graph over fixed buffers (a serving loop's own form); a case with `graph` false
makes the Python calls themselves.

Kinds of work (`op`):
  linear  y = linear(w, x [+ residual]) from bf16 rows, any M, the general entry point
  pre     quantize_act, then linear_prequantized on its int8 rows (the reference engine's pair)
  attn    M = 1 attention projections: rmsnorm + q/k/v in one launch, the o projection + residual
  mlp     M = 1 MLP: rmsnorm + gate/up with the swiglu epilogue, the down projection + residual
  verify  M = 2..16 MLP of the verify step: rmsnorm fragments, gate/up, swiglu fragments, down + residual
  head    rows through the bf16 LM head, and the greedy pick of each
  step    one whole decode step of the looped stack (layers x passes slots), final norm, LM head, greedy pick

Codes are uniform over a format's range, scales log-uniform in [1e-3, 1e-2], activations N(0, 1) (with `outliers`, 5% of
the channels x20), the distributions of the repository's own benchmark.
"""
import math

import torch

import viper_amd as va
from viper_amd.stack import Stack

Q4, Q5, Q6, W8 = 4, 5, 6, 8
EPS = 1e-6
DEV = "cuda"


def listed():
    return [
        # the smallest work a program asks for: one attention-sized linear with its residual, called from Python
        dict(name="linear_call", op="linear", qtype=Q4, enc=1, M=1, N=2560, K=2560, layers=1, residual=True,
             outliers=False, graph=False),
        # a decode step's attention projections (20 query and 4 key/value heads of 128), 22 layers
        dict(name="decode_attn", op="attn", qtype=Q4, enc=1, hidden=2560, q=2560, kv=512, layers=22, graph=True),
        # a decode step's MLPs, the larger part of its bytes
        dict(name="decode_mlp", op="mlp", qtype=Q4, enc=1, hidden=2560, inter=10240, layers=8, graph=True),
        # a decode linear of a model whose hidden size is a power of two
        dict(name="decode_q4_4096", op="linear", qtype=Q4, enc=1, M=1, N=12288, K=4096, layers=10, residual=False,
             outliers=False, graph=True),
        # a down projection of a width that is no round number, in a wider format
        dict(name="decode_q6_ragged", op="linear", qtype=Q6, enc=1, M=1, N=3885, K=8896, layers=10, residual=True,
             outliers=True, graph=True),
        # the 8-bit format, fp16 scales, activations with outlier channels
        dict(name="decode_w8", op="linear", qtype=W8, enc=0, M=1, N=10240, K=2560, layers=10, residual=False,
             outliers=True, graph=True),
        # a small draft verified: 4 rows through a down projection
        dict(name="verify_q4_m4_down", op="linear", qtype=Q4, enc=1, M=4, N=2560, K=10240, layers=16, residual=True,
             outliers=False, graph=True),
        # a full draft verified: 16 rows
        dict(name="verify_q4_m16", op="linear", qtype=Q4, enc=1, M=16, N=10240, K=2560, layers=16, residual=False,
             outliers=False, graph=True),
        # 8 rows of a 5-bit model whose hidden size is a multiple of 64 only
        dict(name="verify_q5_m8_ragged", op="linear", qtype=Q5, enc=1, M=8, N=5001, K=3520, layers=16, residual=False,
             outliers=False, graph=True),
        # the verify step's MLP at the reference engine's sizes, producers writing fragments
        dict(name="verify_mlp", op="verify", qtype=Q4, enc=1, M=16, hidden=3072, inter=10752, layers=6, graph=True),
        # the head and the greedy pick for a verified draft
        dict(name="verify_head", op="head", M=8, N=166144, K=2560, layers=1, graph=True),
        # a whole decode step, 22 weight sets applied twice, its logits
        dict(name="decode_step", op="step", hidden=2560, inter=10240, heads=20, kv_heads=4, layers=22, passes=2,
             vocab=166144, graph=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _k(rng, lo=512, hi=16384):
    """A row length: half of them multiples of 256, a quarter of 128, the rest of 64 only."""
    unit = rng.choice((256, 256, 128, 64))
    return max(lo, int(round(_log(rng, lo, hi) / unit)) * unit)


def _layers(per_layer_bytes, most=44):
    """Layers whose weights come to about 250 MB (a few hundred launches at most)."""
    return max(2, min(most, int(250e6 / per_layer_bytes)))


def draw(rng):
    op = rng.choice(("linear",) * 9 + ("pre", "pre", "attn", "mlp", "verify", "head"))
    qtype = rng.choice((Q4, Q4, Q4, Q5, Q6, W8))
    c = dict(op=op, qtype=qtype, enc=rng.choice((0, 1, 1)), graph=True)
    if op in ("linear", "pre"):
        M = 1 if rng.random() < 0.45 else rng.choice((2, 3, 4, 5, 6, 7, 8, 10, 12, 16, 16))
        K = _k(rng)
        while M > 1 and K % (2 * va.GROUP[qtype]) and M * K > 55000:  # an odd number of groups: rows that fit a workgroup
            M //= 2
        N = _log(rng, 512, 28672)
        if rng.random() < 0.5:
            N = max(512, N // 256 * 256)
        while N * K > 16384 * 12288:
            N //= 2
        c.update(M=M, N=N, K=K, residual=rng.random() < 0.4, outliers=rng.random() < 0.25)
        c["layers"] = _layers(va.packed_bytes(qtype, N, K))
    elif op == "attn":
        hidden = _k(rng, 512, 8192)
        q = 128 * max(4, _log(rng, 4, 64))
        kv = 128 * max(1, _log(rng, 1, 16))
        c.update(hidden=hidden, q=q, kv=kv, layers=_layers(va.packed_bytes(qtype, 2 * q + 2 * kv, hidden)))
    elif op in ("mlp", "verify"):
        hidden = _k(rng, 512, 5120)
        inter = _k(rng, 1024, 16384)
        if op == "verify":  # the fragment entry points take rows of whole quads of groups
            hidden, inter = max(512, hidden // 256 * 256), max(1024, inter // 256 * 256)
            c["M"] = rng.choice((2, 3, 4, 5, 6, 8, 12, 16))
        c.update(hidden=hidden, inter=inter, layers=_layers(va.packed_bytes(qtype, 3 * inter, hidden)))
    else:
        K = _k(rng, 512, 5120)
        M = rng.choice((1, 1, 2, 3, 4, 8, 12, 16))
        while M * K * 2 > 65536:
            M //= 2
        V = _log(rng, 32000, 166144)
        c = dict(op="head", M=M, N=V, K=K, layers=1, graph=True)
    return c


# ----------------------------------------------------------------- inputs


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _weight(g, qtype, enc, N, K):
    nbytes = va.packed_bytes(qtype, N, K)
    G = va.GROUP[qtype]
    if qtype == W8:
        data = torch.randint(-127, 128, (nbytes,), dtype=torch.int8, device=DEV, generator=g).view(torch.uint8)
    else:
        data = torch.randint(0, 256, (nbytes,), dtype=torch.uint8, device=DEV, generator=g)
    u = torch.rand((N * (K // G),), device=DEV, generator=g)
    s = torch.exp(math.log(1e-3) + u * math.log(10.0)).to(torch.bfloat16 if enc else torch.float16)
    return va.QuantizedWeight(va.QType(qtype), data, s, N, K, group_size=G, scale_enc=va.ScaleEnc(enc))


def _rows(g, M, K, outliers=False):
    x = torch.randn((M, K), device=DEV, generator=g)
    if outliers:
        x = x * torch.where(torch.rand((K,), device=DEV, generator=g) < 0.05, 20.0, 1.0)
    return x.to(torch.bfloat16)


def _gamma(g, K):
    return (1.0 + 0.05 * torch.randn((K,), device=DEV, generator=g)).to(torch.bfloat16)


def _empty(*shape, dtype=torch.bfloat16):
    return torch.empty(shape, dtype=dtype, device=DEV)


def _inputs(case, seed):
    """Weights and input rows of every layer, from the seed alone."""
    g, op, L = _gen(seed), case["op"], case["layers"]
    if op == "head":
        K, N = case["K"], case["N"]
        return [dict(w=(0.02 * torch.randn((N, K), device=DEV, generator=g)).to(torch.bfloat16), x=_rows(g, case["M"], K))]
    qtype, enc, out = case["qtype"], case["enc"], []
    for _ in range(L):
        if op in ("linear", "pre"):
            M, N, K = case["M"], case["N"], case["K"]
            out.append(dict(w=_weight(g, qtype, enc, N, K), x=_rows(g, M, K, case["outliers"]),
                            res=_rows(g, M, N) if case["residual"] else None))
        elif op == "attn":
            H, q, kv = case["hidden"], case["q"], case["kv"]
            out.append(dict(q=_weight(g, qtype, enc, q, H), k=_weight(g, qtype, enc, kv, H),
                            v=_weight(g, qtype, enc, kv, H), o=_weight(g, qtype, enc, H, q), x=_rows(g, 1, H),
                            gamma=_gamma(g, H), a=_rows(g, 1, q)))
        else:
            H, I = case["hidden"], case["inter"]
            out.append(dict(gate=_weight(g, qtype, enc, I, H), up=_weight(g, qtype, enc, I, H),
                            down=_weight(g, qtype, enc, H, I), x=_rows(g, case.get("M", 1), H), gamma=_gamma(g, H)))
    return out


def _stack(case, seed):
    return Stack(torch, hidden=case["hidden"], inter=case["inter"], n_heads=case["heads"], n_kv_heads=case["kv_heads"],
                 layers=case["layers"], passes=case["passes"], vocab=case["vocab"], seed=int(seed), eps=EPS)


# ------------------------------------------------------------------- calls


def _ok(st):
    if not st.ok():
        raise RuntimeError(str(st))


def _calls(case, layers, buf):
    """The launches of one pass, as a program writes them."""
    op = case["op"]
    for i, d in enumerate(layers):
        if op == "linear":
            _ok(va.linear(d["w"], d["x"], buf["y"][i], residual=d["res"], workspace=buf["ws"]))
        elif op == "pre":
            _ok(va.quantize_act(d["x"], d["w"].group_size, buf["xq"], buf["xs"]))
            _ok(va.linear_prequantized(d["w"], buf["xq"], buf["xs"], buf["y"][i], residual=d["res"]))
        elif op == "attn":
            _ok(va.linear_m1([d["q"], d["k"], d["v"]], va.Prologue.RMSNORM, d["x"], d["gamma"],
                             [buf["q"][i], buf["k"][i], buf["v"][i]], eps=EPS))
            _ok(va.linear_m1([d["o"]], va.Prologue.BF16, d["a"], None, [buf["y"][i]], residual=d["x"]))
        elif op == "mlp":
            _ok(va.linear_m1_swiglu(d["gate"], d["up"], va.Prologue.RMSNORM, d["x"], d["gamma"], buf["h"][i], eps=EPS))
            _ok(va.linear_m1([d["down"]], va.Prologue.BF16, buf["h"][i], None, [buf["y"][i]], residual=d["x"]))
        elif op == "verify":
            G = d["down"].group_size
            _ok(va.rmsnorm_quantize_frag(d["x"], d["gamma"], EPS, G, buf["xq"], buf["xs"]))
            _ok(va.linear_fused2_prequantized_frag(d["gate"], d["up"], buf["xq"], buf["xs"], buf["gt"], buf["ut"]))
            _ok(va.swiglu_quantize_frag(buf["gt"], buf["ut"], G, buf["xq"], buf["xs"], out=buf["h"][i]))
            _ok(va.linear_prequantized_frag(d["down"], buf["xq"], buf["xs"], buf["y"][i], residual=d["x"],
                                            workspace=buf["ws"]))
        else:
            _ok(va.linear_bf16(d["w"], d["x"], buf["y"]))
            _ok(va.sampling_greedy(buf["y"], buf["token"], workspace=buf["ws"]))


def _buffers(case):
    """Output buffers and workspaces, as the program allocates them once."""
    op, L = case["op"], case["layers"]
    ws = lambda n: torch.zeros((n,), dtype=torch.uint8, device=DEV) if n else None
    if op == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return dict(y=_empty(L, M, N), ws=ws(va.workspace_bytes(case["qtype"], N, K, M)))
    if op == "pre":
        M, N, K = case["M"], case["N"], case["K"]
        return dict(y=_empty(L, M, N), xq=_empty(M, K, dtype=torch.int8),
                    xs=_empty(M, K // va.GROUP[case["qtype"]], dtype=torch.float32))
    if op == "attn":
        H, q, kv = case["hidden"], case["q"], case["kv"]
        return dict(q=_empty(L, q), k=_empty(L, kv), v=_empty(L, kv), y=_empty(L, H))
    if op == "mlp":
        return dict(h=_empty(L, case["inter"]), y=_empty(L, case["hidden"]))
    if op == "verify":
        M, H, I, q = case["M"], case["hidden"], case["inter"], case["qtype"]
        xq, xs = va.frag_bytes(max(H, I), va.GROUP[q])
        return dict(xq=_empty(xq, dtype=torch.int8), xs=_empty(xs // 4, dtype=torch.float32), gt=_empty(M, I),
                    ut=_empty(M, I), h=_empty(L, M, I), y=_empty(L, M, H), ws=ws(va.frag_workspace_bytes(q, H, I, M)))
    M = case["M"]
    return dict(y=_empty(M, case["N"]), token=_empty(M, dtype=torch.int32), ws=ws(va.greedy_workspace_bytes(M)))


OUTPUTS = dict(linear=("y",), pre=("y",), attn=("q", "k", "v", "y"), mlp=("h", "y"), verify=("h", "y"),
               head=("y", "token"))


def prepare(case, seed):
    if case["op"] == "step":
        st = _stack(case, seed)
        body, out, keep = st.step_fused, {"logits": st.logits, "x": st.x}, st
    else:
        layers, buf = _inputs(case, seed), _buffers(case)
        body, out = (lambda: _calls(case, layers, buf)), {k: buf[k] for k in OUTPUTS[case["op"]]}
        keep = (layers, buf)
    state = dict(body=body, out=out, keep=keep, graph=None)
    if case["graph"]:
        body()  # every kernel loaded before the capture
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            body()
        state["graph"] = graph
    return state


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
    else:
        state["body"]()
    return state["out"]


# ------------------------------------------------------------ what it needs


def _matrix(qtype, M, N, K, x=True, y=True):
    """Bytes and operations of one quantized matrix on M rows: weights, scales, and the bf16 rows in and out."""
    G = va.GROUP[qtype]
    b = va.packed_bytes(qtype, N, K) + 2 * N * (K // G) + (2 * M * K if x else 0) + (2 * M * N if y else 0)
    return b, 2 * M * N * K


def work(case):
    op = case["op"]
    if op == "head":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 2 * (N * K + M * K + M * N) + 4 * M, "flops": 2 * M * N * K}
    if op in ("linear", "pre"):
        M, N, K = case["M"], case["N"], case["K"]
        b, f = _matrix(case["qtype"], M, N, K)
        b += 2 * M * N if case["residual"] else 0
    elif op == "attn":
        H, q, kv = case["hidden"], case["q"], case["kv"]
        b0, f0 = _matrix(case["qtype"], 1, q + 2 * kv, H)
        b1, f1 = _matrix(case["qtype"], 1, H, q)
        b, f = b0 + b1 + 4 * H, f0 + f1  # and gamma, the residual
    elif op in ("mlp", "verify"):
        M, H, I = case.get("M", 1), case["hidden"], case["inter"]
        b0, f0 = _matrix(case["qtype"], M, 2 * I, H, y=False)
        b1, f1 = _matrix(case["qtype"], M, H, I, x=False)
        b, f = b0 + b1 + 2 * H + 2 * M * I + 2 * M * H, f0 + f1  # and gamma, h, the residual
    else:
        H, I, V = case["hidden"], case["inter"], case["vocab"]
        q, kv = case["heads"] * 128, case["kv_heads"] * 128
        b = f = 0
        for N, K in ((q + 2 * kv, H), (H, q), (2 * I, H), (H, I)):
            bb, ff = _matrix(Q4, 1, N, K, x=False, y=False)
            b, f = b + bb, f + ff
        slots = case["layers"] * case["passes"]
        return {"bytes": b * slots + 2 * V * H + 2 * V, "flops": f * slots + 2 * V * H}
    return {"bytes": b * case["layers"], "flops": f * case["layers"]}


def tolerance(case):
    """Outputs are bf16 (half an ulp is 2^-9 of a value; rms error about 1.7e-3 of the result), from exact int32 group
    dots and fp32 sums, so another order of the sums moves a value by one ulp now and then.  Where a bf16 value is
    quantized to int8 again (the MLP's h), one ulp there moves an int8 code now and then.  The whole step passes 88 such
    roundings, which travel through the residual stream to the logits (2.3e-3 from 64 bits on its own)."""
    if case["op"] == "step":
        return {"rel": 0.01, "max": 0.06}
    if case["op"] in ("mlp", "verify", "attn"):
        return {"rel": 0.01, "max": 0.04}
    if case["op"] == "head":
        return {"rel": 0.007, "max": 0.016, "differ": 0.01}
    return {"rel": 0.007, "max": 0.016}


# ------------------------------------------------- the same in 64 bits


def _codes(w, r0, r1):
    """Weight codes of rows r0..r1 as float64 [rows, K], from the packed planes."""
    N, K = w.rows, w.cols
    if w.qtype == W8:
        return w.data.view(torch.int8).view(N, K)[r0:r1].double()
    low = w.data[: N * K // 2].view(N, K // 2)[r0:r1]
    u = torch.stack((low & 15, low >> 4), dim=2).view(r1 - r0, K).to(torch.int32)
    off = {Q4: 8, Q5: 16, Q6: 32}[int(w.qtype)]
    if w.qtype != Q4:
        j = torch.arange(32, device=DEV)
        i, b, p = j // 8, (j % 8) // 2, j % 2
        wide = w.qtype == Q6
        byte = (4 * (i // 2) + b) if wide else b
        shift = (4 * (i % 2) + 2 * p) if wide else 2 * i + p
        high = w.data[N * K // 2:].view(N, K // 32, 8 if wide else 4)[r0:r1].to(torch.int32)
        bits = (high[:, :, byte] >> shift) & (3 if wide else 1)
        u = u | (bits << 4).view(r1 - r0, K)
    return (u - off).double()


def _product(xd, w):
    """float64 x [M, K] times the dequantized matrix, rows in pieces that fit."""
    K, G, out = w.cols, w.group_size, []
    step = max(64, (1 << 27) // K)
    for r0 in range(0, w.rows, step):
        r1 = min(w.rows, r0 + step)
        s = w.scales.view(w.rows, K // G)[r0:r1].double()
        wd = (_codes(w, r0, r1).view(r1 - r0, K // G, G) * s[:, :, None]).view(r1 - r0, K)
        out.append(xd @ wd.T)
    return torch.cat(out, dim=1)


def _quantized(x, G):
    """What the int8 quantize of bf16 rows holds, as float64 (the scale is the format's fp32 amax / 127)."""
    M, K = x.shape
    v = x.float().view(M, K // G, G)
    s = (v.abs().amax(dim=2) / 127.0).clamp_min(1e-8)
    q = torch.round(v / s[:, :, None]).clamp(-127, 127)
    return (q.double() * s.double()[:, :, None]).view(M, K)


def _norm(x, gamma):
    v = x.double()
    return (v * torch.rsqrt((v * v).mean(dim=1, keepdim=True) + EPS) * gamma.double()).to(torch.bfloat16)


def _swiglu(g, u):
    g, u = g.to(torch.bfloat16).double(), u.to(torch.bfloat16).double()
    return g / (1.0 + torch.exp(-g)) * u


def _lin(x, w):
    return _product(_quantized(x, w.group_size), w)


def exact(case, seed):
    op = case["op"]
    if op == "step":
        return _exact_step(case, seed)
    res = {k: [] for k in OUTPUTS[op]}
    for d in _inputs(case, seed):
        if op in ("linear", "pre"):
            y = _lin(d["x"], d["w"])
            res["y"].append(y if d["res"] is None else y + d["res"].double())
        elif op == "attn":
            v = _norm(d["x"], d["gamma"])
            for k in ("q", "k", "v"):
                res[k].append(_lin(v, d[k])[0])
            res["y"].append((_lin(d["a"], d["o"]) + d["x"].double())[0])
        elif op in ("mlp", "verify"):
            v = _norm(d["x"], d["gamma"])
            h = _swiglu(_lin(v, d["gate"]), _lin(v, d["up"]))
            y = _lin(h.to(torch.bfloat16), d["down"]) + d["x"].double()
            res["h"].append(h[0] if op == "mlp" else h)
            res["y"].append(y[0] if op == "mlp" else y)
        else:
            x, step = d["x"].double(), 1 << 14
            y = torch.cat([x @ d["w"][r:r + step].double().T for r in range(0, case["N"], step)], dim=1)
            return {"y": y, "token": None}
    return {k: torch.stack(v) for k, v in res.items()}


def _exact_step(case, seed):
    """The stack's slots with every stored value (bf16 rows, int8 activations) as the formats hold it and every sum and
    function in 64 bits."""
    st = _stack(case, seed)
    x = st.x0

    def weight(l, i):
        p, s, n, k = st.w[l][i]
        return va.QuantizedWeight(va.QType.Q4_G64, p, s, n, k, scale_enc=va.ScaleEnc.FP16)

    for slot in range(case["layers"] * case["passes"]):
        l = slot % case["layers"]
        x = (_lin(st.attn, weight(l, 3)) + x.double()).to(torch.bfloat16)
        v = _norm(x, st.ln[2 * l + 1])
        h = _swiglu(_lin(v, weight(l, 4)), _lin(v, weight(l, 5))).to(torch.bfloat16)
        x = (_lin(h, weight(l, 6)) + x.double()).to(torch.bfloat16)
    v = _norm(x, st.final_ln).double()
    step = 1 << 14
    logits = torch.cat([v @ st.head[r:r + step].double().T for r in range(0, case["vocab"], step)], dim=1)
    return {"logits": logits, "x": x.double()}
