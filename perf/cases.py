"""The work whose speed is measured: layers of a transformer training step, and one decoding step's
logits, each through the public entry points of hyperkernels_amd as a training program calls them.

The listed cases take the sizes of this repository's benchmark and configurations (a 124M-parameter
model of width 768 with a vocabulary of 50257, an 8192 x 1280 -> 5120 linear layer, a 4096^3 fp32
product) plus one small and one ragged or wide relative of the ones whose kernels choose their path
by size. `draw` spreads sizes over the same ranges.
"""
from __future__ import annotations

import math

import torch

from hyperkernels_amd import kernels as hk
from hyperkernels_amd import workloads

DEV = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
ONE_BF16, ZERO_BF16 = 0x3F80, 0x0000


def listed():
    return [
        # The smallest call of a training step: LayerNorm forward and backward of a short batch,
        # where the time is launches and latency.
        {"name": "norm_small", "kind": "norm", "dtype": "f32", "rows": 64, "cols": 768},
        # LayerNorm forward and backward of the benchmark's fp32 configuration.
        {"name": "norm_f32", "kind": "norm", "dtype": "f32", "rows": 4096, "cols": 768},
        # The same layer of a wider model in mixed precision.
        {"name": "norm_wide_bf16", "kind": "norm", "dtype": "bf16", "rows": 4096, "cols": 2560},
        # The loss of one batch of 8 x 1024 tokens: cross-entropy forward and backward.
        {"name": "loss", "kind": "loss", "rows": 8192, "vocab": 50257, "index": "i64"},
        # One optimizer step over the 148 parameter tensors of the 124M-parameter model.
        {"name": "adamw", "kind": "adamw", "tensors": 148, "scale": 1.0},
        # Causal self-attention forward and backward of the benchmark's batch.
        {"name": "attn_causal", "kind": "attn", "B": 8, "H": 12, "T": 1024, "causal": True,
         "heads_inner": False},
        # Attention over a small batch of a ragged length without a mask (an encoder, or the last
        # batch of an epoch).
        {"name": "attn_ragged", "kind": "attn", "B": 2, "H": 12, "T": 333, "causal": False,
         "heads_inner": False},
        # The first half of a feed-forward block in bf16, forward and backward: linear layer with
        # bias, GELU, and the gradients of the activation, the input and the weight.
        {"name": "mlp_bf16", "kind": "mlp", "tokens": 8192, "n_in": 1280, "n_out": 5120},
        # A query/key/value projection of a small batch, forward and backward.
        {"name": "proj_small", "kind": "linear", "tokens": 512, "n_in": 768, "n_out": 2304},
        # The language-model head with the tied embedding matrix, forward and backward: the
        # vocabulary is odd, so the logits' rows have every alignment.
        {"name": "lm_head", "kind": "head", "tokens": 2048, "width": 768, "vocab": 50257},
        # A linear layer in fp32, forward and backward, bias gradient included.
        {"name": "linear_f32", "kind": "linear_f32", "tokens": 4096, "n_in": 4096, "n_out": 4096},
        # Decoding: the logits of one token per sequence.
        {"name": "decode_logits", "kind": "decode", "batch": 1, "width": 768, "vocab": 50257},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi, odd=0.25):
    """A feature size: a multiple of 64 usually, any number sometimes."""
    n = _log_int(rng, lo, hi)
    return n if rng.random() < odd else max(64, n // 64 * 64)


def draw(rng):
    kind = rng.choice(["norm", "norm", "loss", "adamw", "attn", "attn", "mlp", "linear", "linear",
                       "head", "linear_f32", "decode"])
    if kind == "norm":
        return {"kind": kind, "dtype": rng.choice(["f32", "bf16", "f16"]),
                "rows": _log_int(rng, 16, 8192), "cols": _width(rng, 128, 4096)}
    if kind == "loss":
        return {"kind": kind, "rows": _log_int(rng, 64, 8192),
                "vocab": rng.choice([50257, 50304, 50272, _log_int(rng, 1000, 50000)]),
                "index": rng.choice(["i32", "i64"])}
    if kind == "adamw":
        return {"kind": kind, "tensors": rng.randint(2, 148), "scale": rng.uniform(0.1, 1.0)}
    if kind == "attn":
        # bounded to the work of 8 x 12 heads of 1024 x 1024 scores
        T = _log_int(rng, 64, 2048)
        H = rng.choice([4, 12, 16])
        most = 8 * 12 * 1024 * 1024 // (H * T * T)
        B = max(1, min(16, _log_int(rng, 1, max(1.01, most))))
        return {"kind": kind, "B": B, "H": H, "T": T, "causal": rng.random() < 0.6,
                "heads_inner": rng.random() < 0.5}
    if kind == "mlp":
        n_in = _width(rng, 256, 1280)
        return {"kind": kind, "tokens": _log_int(rng, 128, 4096), "n_in": n_in, "n_out": 4 * n_in}
    if kind == "linear":
        return {"kind": kind, "tokens": _log_int(rng, 64, 4096), "n_in": _width(rng, 256, 2048),
                "n_out": _width(rng, 256, 4096)}
    if kind == "head":
        return {"kind": kind, "tokens": _log_int(rng, 64, 2048),
                "width": 64 * rng.randint(4, 12),
                "vocab": rng.choice([50257, 50304, _log_int(rng, 1000, 50000)])}
    if kind == "linear_f32":
        return {"kind": kind, "tokens": _log_int(rng, 64, 4096), "n_in": _width(rng, 128, 4096),
                "n_out": _width(rng, 128, 4096)}
    return {"kind": "decode", "batch": rng.randint(1, 4), "width": _width(rng, 256, 2048),
            "vocab": rng.choice([50257, 50304, _log_int(rng, 1000, 50000)])}


# ---- inputs --------------------------------------------------------------------------------------
class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=self.g, device=DEV) * std).to(dtype)

    def uniform(self, *shape, lo=0.0, hi=1.0, dtype=torch.float32):
        return (torch.rand(*shape, generator=self.g, device=DEV) * (hi - lo) + lo).to(dtype)


def _adam_shapes(case):
    shapes = workloads.gpt2_param_shapes()
    if case["tensors"] == len(shapes) and case["scale"] == 1.0:
        return shapes
    # a smaller model: evenly chosen tensors, each a fraction of its size (odd lengths among them)
    n = case["tensors"]
    picked = [shapes[i * len(shapes) // n] for i in range(n)]
    return [(max(1, int(workloads.numel(s) * case["scale"])),) for s in picked]


def _inputs(case, seed):
    r = _Rand(seed)
    k = case["kind"]
    bf = torch.bfloat16
    if k == "norm":
        dt, rows, cols = DTYPES[case["dtype"]], case["rows"], case["cols"]
        return {"x": r.normal(rows, cols, dtype=dt), "dy": r.normal(rows, cols, dtype=dt),
                "gamma": r.uniform(cols, lo=0.5, hi=1.5, dtype=dt),
                "beta": r.normal(cols, std=0.1, dtype=dt)}
    if k == "loss":
        rows, V = case["rows"], case["vocab"]
        t = torch.randint(0, V, (rows,), generator=r.g, device=DEV, dtype=torch.int64)
        return {"logits": r.normal(rows, V, std=2.0),
                "targets": t if case["index"] == "i64" else t.to(torch.int32)}
    if k == "adamw":
        # every tensor is a view of one flat buffer, each from a 256-byte boundary on
        sizes = [workloads.numel(s) for s in _adam_shapes(case)]
        starts, total = [], 0
        for n in sizes:
            starts.append(total)
            total += -(-n // 64) * 64
        flat = {"p": r.normal(total, std=0.02), "g": r.normal(total, std=1e-2),
                "m": r.normal(total, std=1e-3), "v": r.uniform(total, lo=1e-6, hi=1e-4)}
        return {"flat": flat, "spans": list(zip(starts, sizes))}
    if k == "attn":
        B, H, T = case["B"], case["H"], case["T"]

        def t():
            if case["heads_inner"]:  # [B, T, H, 64] as a projection leaves it, viewed by head
                return r.normal(B, T, H, 64).transpose(1, 2)
            return r.normal(B, H, T, 64)
        return {"q": t(), "k": t(), "v": t(), "do": t()}
    if k in ("mlp", "linear"):
        M, I, O = case["tokens"], case["n_in"], case["n_out"]
        return {"x": r.normal(M, I, dtype=bf), "w": r.normal(I, O, std=I ** -0.5, dtype=bf),
                "b": r.normal(O, std=0.1, dtype=bf), "dy": r.normal(M, O, dtype=bf)}
    if k == "head":
        M, C, V = case["tokens"], case["width"], case["vocab"]
        return {"x": r.normal(M, C, dtype=bf), "wte": r.normal(V, C, std=0.05, dtype=bf),
                "dlogits": r.normal(M, V, std=1e-2, dtype=bf)}
    if k == "linear_f32":
        M, I, O = case["tokens"], case["n_in"], case["n_out"]
        return {"x": r.normal(M, I), "w": r.normal(I, O, std=I ** -0.5), "b": r.normal(O, std=0.1),
                "dy": r.normal(M, O)}
    C, V = case["width"], case["vocab"]
    return {"x": r.normal(case["batch"], C, dtype=bf), "wte": r.normal(V, C, std=0.05, dtype=bf)}


ADAM_BIAS = (1 - workloads.ADAMW["beta1"] ** 10, 1 - workloads.ADAMW["beta2"] ** 10)  # step 10


def prepare(case, seed):
    s = {"case": case, **_inputs(case, seed)}
    if case["kind"] == "norm":
        # the parameters' gradient buffers, which a program keeps and clears for each step
        s["grads"] = torch.zeros(2, case["cols"], device=DEV)
    elif case["kind"] == "adamw":
        s["plan"] = hk.AdamPlan(*([s["flat"][n][a:a + size] for a, size in s["spans"]]
                                  for n in ("p", "g", "m", "v")))
    return s


# ---- one pass ------------------------------------------------------------------------------------
def _stream():
    return torch.cuda.current_stream().cuda_stream


def _addmm(x, w, b):
    """x w + b, w [n_in, n_out]."""
    (M, K), N = x.shape, w.shape[1]
    y = torch.empty(M, N, device=x.device, dtype=x.dtype)
    hk.call("hk_bgemm_addmm", M, N, K, ONE_BF16, x.data_ptr(), K, 0, w.data_ptr(), N, 0, ONE_BF16,
            b.data_ptr(), N, y.data_ptr(), N, 0, 1, _stream())
    return y


def _linear_grads(dy, x, w):
    """(dy w^T, x^T dy)."""
    (M, N), K = dy.shape, x.shape[1]
    dx, dw = torch.empty_like(x), torch.empty_like(w)
    hk.call("hk_bgemm_nt_backward", M, K, N, ONE_BF16, dy.data_ptr(), N, 0, w.data_ptr(), N, 0,
            ZERO_BF16, dx.data_ptr(), K, 0, 1, _stream())
    hk.call("hk_bgemm_tn_backward", K, N, M, ONE_BF16, x.data_ptr(), K, 0, dy.data_ptr(), N, 0,
            ZERO_BF16, dw.data_ptr(), N, 0, 1, _stream())
    return dx, dw


def _bgemm(ta, tb, a, b, M, N, K):
    c = torch.empty(M, N, device=a.device, dtype=a.dtype)
    hk.call("hk_bgemm", ta, tb, M, N, K, ONE_BF16, a.data_ptr(), a.shape[1], 0, b.data_ptr(),
            b.shape[1], 0, ZERO_BF16, c.data_ptr(), N, 0, 1, _stream())
    return c


def _sgemm(layout, a, b, M, N, K, bias=None):
    c = torch.empty(M, N, device=a.device)
    hk.call("hk_sgemm", layout, M, N, K, 1.0, a.data_ptr(), a.shape[1], 0, b.data_ptr(),
            b.shape[1], 0, 0.0, c.data_ptr(), N, 0, None if bias is None else bias.data_ptr(),
            0 if bias is None else N, 1, 0, _stream())
    return c


NT, TN, NN = 0, 1, 2


def run(s):
    case = s["case"]
    k = case["kind"]
    if k == "norm":
        y, mean, rstd = hk.layer_norm_forward(s["x"], s["gamma"], s["beta"], 1e-5)
        grads = s["grads"].zero_()
        dx = hk.layer_norm_backward(s["dy"], s["x"], mean, rstd, s["gamma"], grads[0], grads[1])
        return {"y": y, "mean": mean, "rstd": rstd, "dx": dx, "grads": grads}
    if k == "loss":
        loss, mx, sm = hk.sparse_ce_forward(s["logits"], s["targets"])
        grad = hk.sparse_ce_backward(s["logits"], s["targets"], mx, sm,
                                     host_scale=1.0 / case["rows"])
        return {"loss": loss, "max": mx, "sum": sm, "grad": grad}
    if k == "adamw":
        c = workloads.ADAMW
        s["plan"].step(c["lr"], c["beta1"], c["beta2"], c["eps"], c["weight_decay"], *ADAM_BIAS)
        return {n: s["flat"][n] for n in ("p", "m", "v")}
    if k == "attn":
        o, lse = hk.fused_attn_forward(s["q"], s["k"], s["v"], case["causal"])
        D = hk.attn_bwd_precompute_D(s["do"], o)
        dq, dk, dv = hk.attn_backward(s["q"], s["k"], s["v"], s["do"], lse, D, case["causal"])
        return {"o": o, "lse": lse, "dq": dq, "dk": dk, "dv": dv}
    if k == "mlp":
        h = _addmm(s["x"], s["w"], s["b"])
        a = hk.gelu_forward(h)
        dh = hk.gelu_backward(s["dy"], h)
        dx, dw = _linear_grads(dh, s["x"], s["w"])
        return {"h": h, "a": a, "dh": dh, "dx": dx, "dw": dw}
    if k == "linear":
        y = _addmm(s["x"], s["w"], s["b"])
        dx, dw = _linear_grads(s["dy"], s["x"], s["w"])
        return {"y": y, "dx": dx, "dw": dw}
    if k == "head":
        M, C, V = case["tokens"], case["width"], case["vocab"]
        logits = _bgemm(0, 1, s["x"], s["wte"], M, V, C)
        dx = _bgemm(0, 0, s["dlogits"], s["wte"], M, C, V)
        dw = _bgemm(1, 0, s["dlogits"], s["x"], V, C, M)
        return {"logits": logits, "dx": dx, "dw": dw}
    if k == "linear_f32":
        M, I, O = case["tokens"], case["n_in"], case["n_out"]
        y = _sgemm(NN, s["x"], s["w"], M, O, I, s["b"])
        dx = _sgemm(NT, s["dy"], s["w"], M, I, O)
        dw = _sgemm(TN, s["x"], s["dy"], I, O, M)
        db = hk.unified_reduce_sum(s["dy"], hk.ReductionLayout(hk.REDUCE_OUTER, O, M, 0, O, O))
        return {"y": y, "dx": dx, "dw": dw, "db": db}
    B, C, V = case["batch"], case["width"], case["vocab"]
    y = torch.empty(B, V, device=DEV, dtype=torch.bfloat16)
    hk.call("hk_bgemv_nt_row", V, C, ONE_BF16, s["x"].data_ptr(), s["wte"].data_ptr(), C,
            ZERO_BF16, y.data_ptr(), B, C, 0, V, _stream())
    return y


# ---- what a pass cannot do without ---------------------------------------------------------------
def work(case):
    k = case["kind"]
    if k == "norm":
        e = 4 if case["dtype"] == "f32" else 2
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * n * e + 4 * case["rows"] * 4 + case["cols"] * (4 * e + 8),
                "flops": 20 * n}
    if k == "loss":
        n = case["rows"] * case["vocab"]
        return {"bytes": 8 * n + 24 * case["rows"], "flops": 8 * n}
    if k == "adamw":
        n = sum(workloads.numel(s) for s in _adam_shapes(case))
        return {"bytes": 28 * n, "flops": 16 * n}
    if k == "attn":
        B, H, T = case["B"], case["H"], case["T"]
        f = workloads.attn_fwd_flop(B, H, T, 64, case["causal"])
        return {"bytes": (8 * 64 + 2) * 4 * B * H * T, "flops": f + 5 * f // 2}
    if k == "decode":
        B, C, V = case["batch"], case["width"], case["vocab"]
        return {"bytes": 2 * (C * V + B * (C + V)), "flops": 2 * B * C * V}
    if k == "head":
        M, I, O, e = case["tokens"], case["width"], case["vocab"], 2
    else:
        M, I, O, e = case["tokens"], case["n_in"], case["n_out"], 4 if k == "linear_f32" else 2
    # x, w, dy read; y, dx, dw written
    b = 2 * e * (M * I + I * O + M * O)
    return {"bytes": b + (2 * e * M * O if k == "mlp" else 0), "flops": 6 * M * I * O}


def tolerance(case):
    """About four times the error of each path against `exact`, whose measured figures are beside."""
    k = case["kind"]
    if k == "norm":
        # 1.5e-7 (largest 5e-7) with fp32 outputs, one rounding of the outputs with 16-bit ones
        # (bf16 1.7e-3 and 3.9e-3, f16 2.1e-4 and 4.9e-4)
        return {"f32": {"rel": 1e-6, "max": 1e-5}, "bf16": {"rel": 7e-3, "max": 1.6e-2},
                "f16": {"rel": 1e-3, "max": 2e-3}}[case["dtype"]]
    if k in ("loss", "adamw"):
        return {"rel": 1e-6, "max": 4e-6}  # 1.8e-7 and 1e-6
    if k == "attn":
        return {"rel": 3.5e-5, "max": 1.6e-3}  # 8.5e-6 and 3.8e-4 (fp32 products as bf16x3)
    if k == "linear_f32":
        return {"rel": 1.8e-5, "max": 1e-4}  # 4.5e-6 and 2.5e-5 (the same)
    if k == "mlp":
        return {"rel": 1e-2, "max": 4.5e-2}  # 2.6e-3 and 1.1e-2: bf16 activations between
    return {"rel": 7e-3, "max": 1.6e-2}  # one bf16 rounding: 1.7e-3 and 3.9e-3


# ---- the same in 64 bits -------------------------------------------------------------------------
def exact(case, seed):
    s = _inputs(case, seed)
    k = case["kind"]
    if k == "norm":
        x, dy, g, b = (s[n].double() for n in ("x", "dy", "gamma", "beta"))
        mean = x.mean(1, keepdim=True)
        rstd = (((x - mean) ** 2).mean(1, keepdim=True) + 1e-5) ** -0.5
        xh = (x - mean) * rstd
        a = dy * g
        dx = rstd * (a - a.mean(1, keepdim=True) - xh * (a * xh).mean(1, keepdim=True))
        return {"y": xh * g + b, "mean": mean.flatten(), "rstd": rstd.flatten(), "dx": dx,
                "grads": torch.stack([(dy * xh).sum(0), dy.sum(0)])}
    if k == "loss":
        L, t = s["logits"].double(), s["targets"].long()
        mx = L.amax(1)
        at = L.gather(1, t[:, None])[:, 0]
        e = L.sub_(mx[:, None]).exp_()
        sm = e.sum(1)
        grad = e.div_(sm[:, None])
        grad.scatter_add_(1, t[:, None], torch.full_like(t, -1, dtype=torch.float64)[:, None])
        return {"loss": sm.log() + mx - at, "max": mx, "sum": sm, "grad": grad.div_(case["rows"])}
    if k == "adamw":
        c = workloads.ADAMW
        out = {n: s["flat"][n].double() for n in ("p", "g", "m", "v")}
        for a, size in s["spans"]:  # the padding between the tensors stays as it is
            p, g, m, v = (out[n][a:a + size] for n in ("p", "g", "m", "v"))
            m.mul_(c["beta1"]).add_(g, alpha=1 - c["beta1"])
            v.mul_(c["beta2"]).add_(g * g, alpha=1 - c["beta2"])
            u = (m / ADAM_BIAS[0]) / ((v / ADAM_BIAS[1]).sqrt() + c["eps"])
            p.sub_(c["lr"] * (u + c["weight_decay"] * p))
        del out["g"]
        return out
    if k == "attn":
        B, H, T = case["B"], case["H"], case["T"]
        out = {n: torch.empty(B, H, T, 64, device=DEV, dtype=torch.float64)
               for n in ("o", "dq", "dk", "dv")}
        out["lse"] = torch.empty(B, H, T, device=DEV, dtype=torch.float64)
        mask = torch.ones(T, T, device=DEV, dtype=torch.bool).triu(1) if case["causal"] else None
        for b in range(B):
            for h in range(H):
                q, kk, v, do = (s[n][b, h].double().contiguous() for n in ("q", "k", "v", "do"))
                sc = torch.mm(q, kk.t().contiguous()) / 8.0
                if mask is not None:
                    sc.masked_fill_(mask, float("-inf"))
                lse = torch.logsumexp(sc, 1)
                P = (sc - lse[:, None]).exp()
                o = torch.mm(P, v)
                dP = torch.mm(do, v.t().contiguous())
                dS = P * (dP - (do * o).sum(1, keepdim=True)) / 8.0
                out["o"][b, h], out["lse"][b, h] = o, lse
                out["dq"][b, h] = torch.mm(dS, kk)
                out["dk"][b, h] = torch.mm(dS.t().contiguous(), q)
                out["dv"][b, h] = torch.mm(P.t().contiguous(), do)
        return out
    if k in ("mlp", "linear", "linear_f32"):
        x, w, b, dy = (s[n].double() for n in ("x", "w", "b", "dy"))
        y = torch.addmm(b, x, w)
        if k != "mlp":
            out = {"y": y, "dx": torch.mm(dy, w.t()), "dw": torch.mm(x.t(), dy)}
            return {**out, "db": dy.sum(0)} if k == "linear_f32" else out
        c0, c1 = math.sqrt(2 / math.pi), 0.044715
        th = torch.tanh(c0 * (y + c1 * y ** 3))
        dh = dy * (0.5 * (1 + th) + 0.5 * y * (1 - th * th) * c0 * (1 + 3 * c1 * y * y))
        return {"h": y, "a": 0.5 * y * (1 + th), "dh": dh, "dx": torch.mm(dh, w.t()),
                "dw": torch.mm(x.t(), dh)}
    if k == "head":
        x, w, dl = (s[n].double() for n in ("x", "wte", "dlogits"))
        return {"logits": torch.mm(x, w.t()), "dx": torch.mm(dl, w), "dw": torch.mm(dl.t(), x)}
    return torch.mm(s["x"].double(), s["wte"].double().t())
