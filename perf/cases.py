"""The calls that a program built on this library makes, as measurable cases.

Shapes are those of a 27B-class dense transformer layer, as in bench.py:
hidden 5120, q 8192, k and v 1024 each, feed-forward 17408.  The cases run from
one token (decode) over a few columns (speculative verification), tens of
columns (a batch of sequences being decoded together, short prompts) to prefill
chunks of 512 and 2048 tokens.

op        what one pass calls
mul_mat   one projection on fp32 activations in ggml's layout (quantise + multiply)
km        the same through the reference-named entry in the [K][M] -> [N][M] layout
qkv       residual add + RMS norm, then q, k and v against the same activations
mlp       residual add + RMS norm, gate and up, SwiGLU, down
decode    whole layers at one token, captured once into a HIP graph and replayed
dequant   a weight matrix expanded to fp32
"""
import importlib.util
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NAME = "qwen_3_8_27b_optimizations_amd"
HIDDEN, Q_ROWS, KV_ROWS, FFN = 5120, 8192, 1024, 17408
EPS = 1e-6


def package():
    """The library's Python side (its directory's name holds a dot)."""
    if NAME not in sys.modules:
        d = os.path.join(ROOT, "qwen_3.8_27b_optimizations_amd")
        spec = importlib.util.spec_from_file_location(NAME, os.path.join(d, "__init__.py"),
                                                      submodule_search_locations=[d])
        sys.modules[NAME] = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(sys.modules[NAME])
    return sys.modules[NAME]


def listed():
    return [
        # the smallest projection of a decode step: launch latency counts
        {"name": "k_proj_m1", "op": "mul_mat", "K": HIDDEN, "N": KV_ROWS, "M": 1},
        # single-stream decode: two layers with weights past every cache, replayed as a graph
        {"name": "decode_m1", "op": "decode", "layers": 2, "K": HIDDEN, "N": FFN, "M": 1},
        # attention projections of two sequences, or of a draft of two tokens
        {"name": "qkv_m2", "op": "qkv", "K": HIDDEN, "N": Q_ROWS, "M": 2},
        # feed-forward block while verifying drafts of four and of eight tokens
        {"name": "mlp_m4", "op": "mlp", "K": HIDDEN, "N": FFN, "M": 4},
        {"name": "mlp_m8", "op": "mlp", "K": HIDDEN, "N": FFN, "M": 8},
        # feed-forward block of a batch of sixteen sequences being decoded
        {"name": "mlp_m16", "op": "mlp", "K": HIDDEN, "N": FFN, "M": 16},
        # output projection of a short prompt of odd length
        {"name": "o_proj_m33", "op": "mul_mat", "K": Q_ROWS, "N": HIDDEN, "M": 33},
        # attention projections of a batch of 64
        {"name": "qkv_m64", "op": "qkv", "K": HIDDEN, "N": Q_ROWS, "M": 64},
        # a caller of the standalone kernel API, column-strided activations, ragged width
        {"name": "down_km_m130", "op": "km", "K": FFN, "N": HIDDEN, "M": 130},
        # feed-forward block of a prefill chunk of the usual 512 tokens
        {"name": "mlp_m512", "op": "mlp", "K": HIDDEN, "N": FFN, "M": 512},
        # the widest projection of a large prefill chunk
        {"name": "gate_m2048", "op": "mul_mat", "K": HIDDEN, "N": FFN, "M": 2048},
        # a matrix expanded once for a path that needs fp32 weights
        {"name": "dequant_up", "op": "dequant", "K": HIDDEN, "N": FFN, "M": 0},
    ]


def draw(rng):
    """A case of the same kinds over the whole range of widths, rows and row lengths."""
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(["mul_mat", "mul_mat", "qkv", "mlp", "mlp", "km", "dequant"])
    K = 256 * spread(3, 68)
    M = 1 if rng.random() < 0.1 else spread(1, 2048)
    N = spread(512, FFN)
    if op == "mlp":  # the rows of gate and up are down's row length
        N, M = 256 * spread(6, 68), min(M, 512)
        K = min(K, 8192)
    elif op == "qkv":
        M = min(M, 1024)
        K, N = min(K, 8192), min(N, Q_ROWS)
    elif op == "dequant":
        M = 0
        K = min(K, 256 * (HIDDEN * FFN // (256 * N)))
    # no more work than the largest listed case
    top = HIDDEN * FFN * 2048
    while op != "dequant" and K * N * M * (3 if op == "mlp" else 1) > top:
        M //= 2
    return {"op": op, "K": K, "N": N, "M": M}


# ------------------------------------------------------------------ inputs
def device():
    return torch.device("cuda:0")


def weights(gen, K, N):
    """Random IQ4_XS super-blocks: fp16 d ~ U(0.005, 0.02), uniform 6-bit scales and codes."""
    n = N * (K // 256)
    raw = torch.randint(0, 256, (n, 136), dtype=torch.uint8, device=device(), generator=gen)
    d = 0.005 + 0.015 * torch.rand(n, 1, device=device(), generator=gen)
    raw[:, :2] = d.to(torch.float16).view(torch.uint8)
    return raw.reshape(-1)


def normal(gen, *shape):
    return torch.randn(*shape, device=device(), generator=gen)


def activations(gen, M, K):
    """N(0, 1) with 1 % of the values twenty times larger, as transformer activations have."""
    x = normal(gen, M, K)
    return torch.where(torch.rand(M, K, device=device(), generator=gen) < 0.01, 20 * x, x)


def gain(gen, K):
    """RMS-norm gain that keeps projections of synthetic weights near unit size."""
    return (1 + 0.1 * normal(gen, K)) / (16 * math.sqrt(K))


def inputs(case, seed):
    """Everything random in a case, from the seed alone."""
    gen = torch.Generator(device=device()).manual_seed(1000003 * seed + 17)
    op, K, N, M = case["op"], case["K"], case["N"], case["M"]
    if op == "dequant":
        return {"W": weights(gen, K, N)}
    if op == "mul_mat":
        return {"W": weights(gen, K, N), "x": activations(gen, M, K)}
    if op == "km":
        return {"W": weights(gen, K, N), "x": activations(gen, M, K).t().contiguous()}
    s = {"x": activations(gen, M, K), "r": normal(gen, M, K)}
    if op == "qkv":
        s.update(gamma=gain(gen, K), Ns=qkv_rows(N), Ws=[weights(gen, K, n) for n in qkv_rows(N)])
    elif op == "mlp":
        s.update(gamma=gain(gen, K), gate=weights(gen, K, N), up=weights(gen, K, N), down=weights(gen, N, K))
    else:
        s["layers"] = [{"g1": gain(gen, K), "g2": gain(gen, K),
                        "qkv": [weights(gen, K, n) for n in qkv_rows(Q_ROWS)], "o": weights(gen, Q_ROWS, K),
                        "gate": weights(gen, K, N), "up": weights(gen, K, N), "down": weights(gen, N, K)}
                       for _ in range(case["layers"])]
    return s


def qkv_rows(N):
    """q's rows and the eighth of them that k and v have each."""
    return [N, max(1, N // 8), max(1, N // 8)]


# ------------------------------------------------------------------ one pass
def prepare(case, seed):
    pkg = package()
    op, K, N, M = case["op"], case["K"], case["N"], case["M"]
    s = inputs(case, seed)
    s.update(pkg=pkg, op=op, K=K, N=N, M=M)
    new = lambda *shape: torch.empty(*shape, dtype=torch.float32, device=device())  # noqa: E731
    if op == "dequant":
        s["y"] = new(N * K)
        return s
    if op == "mul_mat":
        s.update(ws=pkg.workspace(K, M), y=new(M, N))
    elif op == "km":
        s["y"] = new(N, M)
    elif op == "qkv":
        s.update(ws=pkg.workspace(K, M), h=new(M, K), ys=[new(M, n) for n in s["Ns"]])
        # the fused single-token launch where the library takes the shape, as its interface states
        s["fused"] = M == 1 and 2048 <= K <= 8192
    elif op == "mlp":
        s.update(ws=pkg.workspace(K, M), ws2=pkg.workspace(N, M), h=new(M, K), s=new(M, N), g=new(M, N),
                 u=new(M, N), y=new(M, K))
        s["fused"] = M == 1 and 2048 <= K <= 8192
        if s["fused"]:
            try:
                run_mlp(s)
            except pkg.Iq4xsError as e:
                if e.code != pkg.ERROR_NOT_SUPPORTED:
                    raise
                s["fused"] = False
    else:
        for l in s["layers"]:
            l.update(h1=new(K), h2=new(K), q=new(Q_ROWS), k=new(KV_ROWS), v=new(KV_ROWS), a=new(K), s=new(N),
                     y=new(K))
        s.update(ws_q=pkg.workspace(Q_ROWS, 1), ws_n=pkg.workspace(N, 1))
        run_layers(s)  # the library's first calls on a device are not captured
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            run_layers(s)
    return s


def run_qkv(s):
    pkg, K, M = s["pkg"], s["K"], s["M"]
    if s["fused"]:
        pkg.rms_norm_mul_mat_group(s["Ws"], s["x"], K, s["Ns"], residual=s["r"], out_h=s["h"], gamma=s["gamma"],
                                   eps=EPS, outs=s["ys"])
    else:
        pkg.rms_norm_q8_1(s["x"], K, M, residual=s["r"], out_h=s["h"], gamma=s["gamma"], eps=EPS, ws=s["ws"])
        pkg.mul_mat_q8_1_group(s["Ws"], s["ws"], K, s["Ns"], M, outs=s["ys"])
    return [s["h"], *s["ys"]]


def run_mlp(s):
    pkg, K, N, M = s["pkg"], s["K"], s["N"], s["M"]
    if s["fused"]:
        pkg.rms_norm_mul_mat_swiglu(s["gate"], s["up"], s["x"], K, N, residual=s["r"], out_h=s["h"],
                                    gamma=s["gamma"], eps=EPS, gate_out=s["g"], up_out=s["u"], out=s["s"])
        pkg.mul_mat(s["down"], s["s"], N, K, M, ws=s["ws2"], out=s["y"])
    else:
        pkg.rms_norm_q8_1(s["x"], K, M, residual=s["r"], out_h=s["h"], gamma=s["gamma"], eps=EPS, ws=s["ws"])
        pkg.mul_mat_q8_1_group([s["gate"], s["up"]], s["ws"], K, [N, N], M, outs=[s["g"], s["u"]])
        pkg.swiglu_q8_1(s["g"], s["u"], N, M, ws=s["ws2"])
        pkg.mul_mat_q8_1(s["down"], s["ws2"], N, K, M, out=s["y"])
    return [s["h"], s["g"], s["u"], s["y"]]


def run_layers(s):
    """The projections of whole layers at one token; q stands for the attention's output, which has its shape."""
    pkg, K, N = s["pkg"], s["K"], s["N"]
    x, r = s["x"], s["r"]
    for l in s["layers"]:
        pkg.rms_norm_mul_mat_group(l["qkv"], x, K, qkv_rows(Q_ROWS), residual=r, out_h=l["h1"], gamma=l["g1"],
                                   eps=EPS, outs=[l["q"], l["k"], l["v"]])
        pkg.mul_mat(l["o"], l["q"], Q_ROWS, K, 1, ws=s["ws_q"], out=l["a"])
        pkg.rms_norm_mul_mat_swiglu(l["gate"], l["up"], l["h1"], K, N, residual=l["a"], out_h=l["h2"],
                                    gamma=l["g2"], eps=EPS, keep_gate_up=False, out=l["s"])
        pkg.mul_mat(l["down"], l["s"], N, K, 1, ws=s["ws_n"], out=l["y"])
        x, r = l["h2"], l["y"]


def run(state):
    s, op = state, state["op"]
    if op == "dequant":
        return s["pkg"].dequant(s["W"], s["N"] * s["K"] // 256, out=s["y"])
    if op == "mul_mat":
        return s["pkg"].mul_mat(s["W"], s["x"], s["K"], s["N"], s["M"], ws=s["ws"], out=s["y"])
    if op == "km":
        s["pkg"].lib().check("gemm_iq4xs_stock_dp4a_gpu", s["W"].data_ptr(), s["x"].data_ptr(), s["y"].data_ptr(),
                             s["K"], s["N"], s["M"], torch.cuda.current_stream().cuda_stream)
        return s["y"]
    if op == "qkv":
        return run_qkv(s)
    if op == "mlp":
        return run_mlp(s)
    s["graph"].replay()
    return [[l[n].view(1, -1) for n in ("h1", "q", "k", "v", "a", "h2", "s", "y")] for l in s["layers"]]


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    op, K, N, M = case["op"], case["K"], case["N"], case["M"]
    w = lambda k, n: n * k // 256 * 136  # noqa: E731
    if op == "dequant":
        return {"bytes": w(K, N) + 4 * N * K, "flops": 0}
    if op in ("mul_mat", "km"):
        return {"bytes": w(K, N) + 4 * M * (K + N), "flops": 2 * M * N * K}
    if op == "qkv":
        rows = sum(qkv_rows(N))
        return {"bytes": w(K, rows) + 4 * M * (3 * K + rows), "flops": 2 * M * rows * K}
    if op == "mlp":
        return {"bytes": w(K, 2 * N) + w(N, K) + 4 * M * (4 * K + 2 * N), "flops": 6 * M * N * K}
    rows = sum(qkv_rows(Q_ROWS))
    per = w(K, rows) + w(Q_ROWS, K) + w(K, 2 * N) + w(N, K) + 4 * (8 * K + rows + N)
    return {"bytes": case["layers"] * per, "flops": case["layers"] * 2 * (K * rows + Q_ROWS * K + 3 * K * N)}


def tolerance(case):
    # dequantising is two products of exact factors; everything else sums in
    # fp32.  Where a norm or a SwiGLU lies before the Q8_1 quantiser, a last-bit
    # difference can move a code to its neighbour, and layer by layer that adds up.
    if case["op"] == "dequant":
        return "exact"
    if case["op"] in ("mul_mat", "km"):
        return {"rel": 2e-6, "max": 2e-5}
    return {"rel": 1e-3}


# ------------------------------------------------------------------ the same in 64 bits
KVALUES = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def dequantised(W, K, N):
    """fp64 [N][K] of IQ4_XS super-blocks {fp16 d, u16 scales_h, u8 scales_l[4], u8 qs[128]}."""
    b = W.view(-1, 136)
    d = b[:, :2].contiguous().view(torch.float16).double()
    scales_h = b[:, 2].int() | (b[:, 3].int() << 8)
    kv = torch.tensor(KVALUES, dtype=torch.float64, device=W.device)
    out = torch.empty(b.shape[0], 256, dtype=torch.float64, device=W.device)
    for i in range(8):
        lo = (b[:, 4 + i // 2].int() >> (4 * (i % 2))) & 15
        ls = lo | (((scales_h >> (2 * i)) & 3) << 4)
        q = b[:, 8 + 16 * i:24 + 16 * i].long()
        out[:, 32 * i:32 * i + 32] = kv[torch.cat([q & 15, q >> 4], 1)] * (d * (ls - 32).double()[:, None])
    return out.view(N, K)


def q8_1(x):
    """fp64 values of fp32 rows after Q8_1: per 32 values an fp32 d = amax / 127, codes round(x / d), half away
    from zero, and the scale kept as fp16 cut toward zero."""
    x = x.float()
    v = x.reshape(*x.shape[:-1], -1, 32)
    amax = v.abs().amax(-1, keepdim=True)
    d = amax / torch.full_like(amax, 127)  # a tensor: division by a number may be done by its reciprocal
    t = torch.where(d > 0, v / d, torch.zeros_like(v)).double()
    codes = torch.sign(t) * torch.floor(t.abs() + 0.5)
    near = d.half()
    cut = torch.where(near.float() > d, (near.view(torch.int16) - 1).view(torch.float16), near)
    return (codes * cut.double()).reshape(x.shape)


def rms_norm(h, gamma):
    return h * torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS) * gamma.double()


def product(W, x, K, N):
    return q8_1(x) @ dequantised(W, K, N).t().contiguous()


def exact(case, seed):
    op, K, N, M = case["op"], case["K"], case["N"], case["M"]
    s = inputs(case, seed)
    if op == "dequant":
        return dequantised(s["W"], K, N).reshape(-1)
    if op == "mul_mat":
        return product(s["W"], s["x"], K, N)
    if op == "km":
        return product(s["W"], s["x"].t().contiguous(), K, N).t().contiguous()
    if op == "decode":
        x, r, out = s["x"].double(), s["r"].double(), []
        for l in s["layers"]:
            h1 = x + r
            y = rms_norm(h1, l["g1"])
            q, k, v = (product(w, y, K, n) for w, n in zip(l["qkv"], qkv_rows(Q_ROWS)))
            a = product(l["o"], q, Q_ROWS, K)
            h2 = h1 + a
            y = rms_norm(h2, l["g2"])
            g, u = (product(l[n], y, K, N) for n in ("gate", "up"))
            sw = torch.nn.functional.silu(g) * u
            x, r = h2, product(l["down"], sw, N, K)
            out.append([h1, q, k, v, a, h2, sw, r])
        return out
    h = s["x"].double() + s["r"].double()
    y = rms_norm(h, s["gamma"])
    if op == "qkv":
        return [h, *(product(w, y, K, n) for w, n in zip(s["Ws"], s["Ns"]))]
    g, u = product(s["gate"], y, K, N), product(s["up"], y, K, N)
    return [h, g, u, product(s["down"], torch.nn.functional.silu(g) * u, N, K)]
