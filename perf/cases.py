"""The workloads that this library's speed is judged by, as a PyTorch program states them through the `neoGEMM` module.

A case is a dict of plain values; `kind` names what the program does with its sizes:
  gemm       C = gemm(A, B); layout "kn": B [K,N] as stored, "nk": B = W.t() of a stored W [N,K]
  v1         neoGemmV1(A, B, C): B [N,K], C preallocated and written column-major
  layer      one transformer layer's output, up and down projection on `rows` activations, weights stored [out, in]
  train      a linear layer's training step: forward, input gradient, weight gradient added to what has accumulated
  attention  scores q k^T and output p v of `heads` heads as batched products
"""
import math

import torch

import neoGEMM


def listed():
    return [
        # smallest square product of the benchmark set: the price of one call
        {"name": "square 512", "kind": "gemm", "layout": "kn", "M": 512, "N": 512, "K": 512},
        # the driver script's own shape and call
        {"name": "v1 1024", "kind": "v1", "M": 1024, "N": 1024, "K": 1024},
        # one token through a layer: weights are read once, nothing is reused
        {"name": "layer 1 row", "kind": "layer", "rows": 1, "hidden": 4096, "ffn": 14336},
        # decoding a batch of sixteen, weights stored [K,N]
        {"name": "decode 16 rows", "kind": "gemm", "layout": "kn", "M": 16, "N": 14336, "K": 4096},
        # a short prompt, or decoding a large batch
        {"name": "layer 128 rows", "kind": "layer", "rows": 128, "hidden": 4096, "ffn": 14336},
        # few outputs, deep sum: a projection onto few features, or a weight gradient over many tokens
        {"name": "tall K", "kind": "gemm", "layout": "kn", "M": 1024, "N": 1024, "K": 32768},
        # a prompt whose length is no multiple of any tile
        {"name": "irregular", "kind": "gemm", "layout": "nk", "M": 3000, "N": 5120, "K": 3584},
        # the headline: large, square, bound by arithmetic
        {"name": "square 8192", "kind": "gemm", "layout": "kn", "M": 8192, "N": 8192, "K": 8192},
        # nothing is a multiple of eight: rows of A, B and C begin at any two-byte address
        {"name": "odd", "kind": "gemm", "layout": "kn", "M": 1023, "N": 2047, "K": 1535},
        # forward and backward of a square layer, gradients accumulated over micro-batches
        {"name": "train 4096", "kind": "train", "tokens": 4096, "n_in": 4096, "n_out": 4096},
        # forward and backward of an output head whose number of classes is odd
        {"name": "train odd head", "kind": "train", "tokens": 512, "n_in": 1024, "n_out": 10001},
        # attention of 32 heads of 128 over 1024 positions
        {"name": "attention 32x1024", "kind": "attention", "heads": 32, "seq": 1024, "dim": 128},
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` from lo to hi, spread evenly over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, step * round(v / step)))


def draw(rng):
    kind = rng.choice(["square", "decode", "ragged", "v1", "layer", "tall", "odd", "train", "head", "attention"])
    while True:
        if kind in ("square", "decode", "ragged", "tall"):
            c = {"kind": "gemm", "layout": rng.choice(["kn", "nk"])}
            if kind == "square":
                n = _log(rng, 512, 8192, 64)
                c.update(M=n, N=n, K=n)
            elif kind == "decode":
                c.update(M=_log(rng, 1, 256), N=_log(rng, 2048, 28672, 64), K=_log(rng, 2048, 14336, 64))
            elif kind == "ragged":
                c.update(M=_log(rng, 257, 6000), N=_log(rng, 512, 8192, 8), K=_log(rng, 512, 8192, 8))
            else:
                c.update(M=_log(rng, 128, 2048, 8), N=_log(rng, 128, 2048, 8), K=_log(rng, 8192, 65536, 64))
        elif kind == "v1":
            c = {"kind": "v1", "M": _log(rng, 384, 8192, 8), "N": _log(rng, 384, 8192, 8), "K": _log(rng, 384, 8192, 8)}
        elif kind == "layer":
            h = _log(rng, 2048, 8192, 128)
            c = {"kind": "layer", "rows": _log(rng, 1, 512), "hidden": h, "ffn": 128 * round(h * rng.uniform(2.5, 4.0) / 128)}
        elif kind == "odd":
            c = {"kind": "gemm", "layout": rng.choice(["kn", "nk"]), "M": _log(rng, 65, 3000), "N": _log(rng, 65, 3000) | 1,
                 "K": _log(rng, 257, 3000) | 1}
        elif kind == "train":
            c = {"kind": "train", "tokens": _log(rng, 256, 8192, 8), "n_in": _log(rng, 512, 8192, 64), "n_out": _log(rng, 512, 8192, 64)}
        elif kind == "head":
            c = {"kind": "train", "tokens": _log(rng, 64, 1024), "n_in": _log(rng, 256, 2048, 8), "n_out": _log(rng, 501, 20001) | 1}
        else:
            c = {"kind": "attention", "heads": _log(rng, 4, 64), "seq": _log(rng, 64, 2048), "dim": rng.choice([64, 96, 128])}
        # no dearer than the listed case that stands for its range
        w = work(c)
        most = {"odd": 6.5e9, "head": 3.2e10, "attention": 1.8e10}.get(kind, 1.1e12)
        if w["flops"] <= most and w["bytes"] <= 6e8:
            return c


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, scale=1.0):
        return (torch.randn(*shape, generator=g, device="cuda") * scale).to(torch.bfloat16)

    k = case["kind"]
    if k in ("gemm", "v1"):
        M, N, K = case["M"], case["N"], case["K"]
        s = {"kind": k, "A": normal(M, K, scale=K ** -0.5)}
        if k == "v1":
            s.update(B=normal(N, K, scale=K ** -0.5), C=torch.zeros(M, N, dtype=torch.bfloat16, device="cuda"))
        elif case["layout"] == "nk":
            s["B"] = normal(N, K, scale=K ** -0.5).t()
        else:
            s["B"] = normal(K, N, scale=K ** -0.5)
        return s
    if k == "layer":
        m, h, f = case["rows"], case["hidden"], case["ffn"]
        return {"kind": k, "x": normal(m, h), "y": normal(m, f), "out": normal(h, h, scale=h ** -0.5), "up": normal(f, h, scale=h ** -0.5),
                "down": normal(h, f, scale=f ** -0.5)}
    if k == "train":
        t, i, o = case["tokens"], case["n_in"], case["n_out"]
        return {"kind": k, "x": normal(t, i), "dy": normal(t, o, scale=o ** -0.5), "W": normal(o, i, scale=i ** -0.5),
                "dW": normal(o, i, scale=t ** 0.5 * o ** -0.5)}
    b, n, d = case["heads"], case["seq"], case["dim"]
    return {"kind": k, "q": normal(b, n, d, scale=d ** -0.5), "k": normal(b, n, d), "v": normal(b, n, d),
            "p": torch.softmax(torch.randn(b, n, n, generator=g, device="cuda"), -1).to(torch.bfloat16)}


def run(s):
    k = s["kind"]
    if k == "gemm":
        return neoGEMM.gemm(s["A"], s["B"])
    if k == "v1":
        neoGEMM.neoGemmV1(s["A"], s["B"], s["C"])
        return s["C"]
    if k == "layer":
        return neoGEMM.gemm(s["x"], s["out"].t()), neoGEMM.gemm(s["x"], s["up"].t()), neoGEMM.gemm(s["y"], s["down"].t())
    if k == "train":
        y = neoGEMM.gemm(s["x"], s["W"].t())
        dx = neoGEMM.gemm(s["dy"], s["W"])
        neoGEMM.gemm_scaled(s["dy"].t(), s["x"], s["dW"], 1.0, 1.0)
        return y, dx, s["dW"]
    return neoGEMM.bmm(s["q"], s["k"].transpose(1, 2)), neoGEMM.bmm(s["p"], s["v"])


def work(case):
    k = case["kind"]
    if k in ("gemm", "v1"):
        products = [(1, case["M"], case["N"], case["K"], 1)]
    elif k == "layer":
        m, h, f = case["rows"], case["hidden"], case["ffn"]
        products = [(1, m, h, h, 1), (1, m, f, h, 1), (1, m, h, f, 1)]
    elif k == "train":
        t, i, o = case["tokens"], case["n_in"], case["n_out"]
        # the gradient is read and written
        products = [(1, t, o, i, 1), (1, t, i, o, 1), (1, o, i, t, 2)]
    else:
        b, n, d = case["heads"], case["seq"], case["dim"]
        products = [(b, n, n, d, 1), (b, n, d, n, 1)]
    return {"bytes": sum(2.0 * b * (m * kk + kk * n + c * m * n) for b, m, n, kk, c in products),
            "flops": sum(2.0 * b * m * n * kk for b, m, n, kk, c in products)}


def tolerance(case):
    # fp32 sums rounded once to bf16: another order of summation moves a few elements by one bf16 step, 2^-7 of the value at most
    # (against sums in fp64, rounded once, the cases show up to 6e-5 in the 2-norm and one step)
    return {"rel": 3e-4, "max": 0.016}
