"""Performance cases of the library: what a program that trains or samples a GPT, or calls its
pieces, has it do, through the public binding (bmb) and the C entry points behind it.

A case is a dict of plain values whose "op" names the call (or the few calls that always go
together); listed() gives the ones quoted, draw() more of the same ranges. Everything is fp32 in
device memory and row-major. "math" picks the arithmetic of gemm(): "bf16x3" (the default) or
"fp32" (include/gemm.h).
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "bare-metal-bard_amd"))
import bmb  # noqa: E402

F32, F64 = torch.float32, torch.float64
LN_EPS = 1e-5
ADAMW = dict(lr=3e-4, beta1=0.9, beta2=0.999, eps=1e-8, wd=0.1)
OPT_STEP = 100  # optimizer steps already taken in the "optimizer" cases


def listed():
    return [
        # One layer of sampling: the QKV projection of one 256-token sequence of the
        # character-level model (C = 384). Two short launches: latency.
        dict(name="linear_sample", op="linear", rows=256, cin=384, cout=1152, train=False,
             math="bf16x3"),
        # The kernel table's headline: C = A B + 0.5 C at N = 4096 in fp32 products.
        dict(name="sgemm_4096_fp32", op="gemm", M=4096, N=4096, K=4096, ta=False, tb=False,
             beta=0.5, math="fp32"),
        # The widest layer of a GPT-2-small block over a batch of 8 x 1024 tokens, forward and
        # backward: Y = X W^T + b, dX, dW, db.
        dict(name="linear_gpt2_fc", op="linear", rows=8192, cin=768, cout=3072, train=True,
             math="bf16x3"),
        # The LM head and the loss over the unpadded 50257-word vocabulary (every row odd and
        # unaligned): logits, softmax and cross-entropy, dlogits, dX, dW.
        dict(name="head_v50257", op="head", rows=2048, C=768, V=50257, Vp=50257),
        # Fused causal attention, forward and backward, at GPT-2-small's training shape.
        dict(name="flash_gpt2", op="flash", B=8, T=1024, NH=12, hs=64),
        # The same for the character-level model: many short sequences.
        dict(name="flash_char", op="flash", B=16, T=256, NH=6, hs=64),
        # Long sequences, wide heads, a length that is no whole number of tiles.
        dict(name="flash_long_hs128", op="flash", B=2, T=4000, NH=8, hs=128),
        # The unfused attention (materialised scores), which keeps the probabilities.
        dict(name="attention_unfused", op="attention", B=16, T=256, NH=6, hs=64),
        # The elementwise part of a GPT-2-small block: residual, layernorm and GELU, both ways.
        dict(name="norm_gelu_gpt2", op="norm_gelu", rows=8192, C=768),
        # Gradient norm, clipping and AdamW over GPT-2-small's parameters.
        dict(name="optimizer_gpt2", op="optimizer", n=124475904),
        # Forward and backward of the character-level model (10.8 M parameters, 16 x 256
        # tokens): small layers, many launches.
        dict(name="gpt_char", op="gpt", B=16, T=256, L=6, NH=6, C=384, V=65, Vp=128, train=True),
        # Forward and backward of GPT-2 small over 8 x 1024 tokens.
        dict(name="gpt2_small", op="gpt", B=8, T=1024, L=12, NH=12, C=768, V=50257, Vp=50304,
             train=True),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    """A layer width: usually a multiple of 32 as models have it, sometimes any number."""
    n = _log(rng, lo, hi)
    return n if rng.random() < 0.25 else max(32, (n + 16) // 32 * 32)


def draw(rng):
    op = rng.choice(["gemm", "linear", "linear", "head", "flash", "flash", "attention",
                     "norm_gelu", "optimizer", "gpt"])
    if op == "gemm":
        n = [_log(rng, 192, 4608) for _ in range(3)]
        if rng.random() < 0.4:
            n = [n[0]] * 3
        return dict(op=op, M=n[0], N=n[1], K=n[2], ta=rng.random() < 0.3, tb=rng.random() < 0.3,
                    beta=rng.choice([0.0, 0.5]), math=rng.choice(["bf16x3", "fp32"]))
    if op == "linear":
        return dict(op=op, rows=_log(rng, 64, 8192), cin=_width(rng, 128, 3072),
                    cout=_width(rng, 128, 3072), train=rng.random() < 0.7,
                    math=rng.choice(["bf16x3", "bf16x3", "fp32"]))
    if op == "head":
        V = _log(rng, 65, 50257)
        return dict(op=op, rows=_log(rng, 128, 4096), C=_width(rng, 128, 1024), V=V,
                    Vp=V if rng.random() < 0.4 else (V + 63) // 64 * 64)
    if op in ("flash", "attention"):
        hs = rng.choice([32, 64, 64, 128])
        NH = rng.randint(2, 16)
        T = _log(rng, 32, 4096 if op == "flash" else 1024)
        B = _log(rng, 1, 32)
        while B > 1 and B * NH * T * T * hs > 16.5e9:
            B -= 1
        return dict(op=op, B=B, T=T, NH=NH, hs=hs)
    if op == "norm_gelu":
        return dict(op=op, rows=_log(rng, 128, 16384), C=_width(rng, 128, 1600))
    if op == "optimizer":
        return dict(op=op, n=_log(rng, 800000, 124475904))
    hs = rng.choice([32, 64, 64])
    NH = rng.randint(2, 12)
    V = rng.choice([65, 256, 4096, 50257])
    train = rng.random() < 0.7
    return dict(op="gpt", B=_log(rng, 1, 16) if train else 1, T=_log(rng, 32, 512),
                L=rng.randint(2, 8), NH=NH, C=NH * hs, V=V, Vp=(V + 127) // 128 * 128, train=train)


# ------------------------------------------------------------------- inputs
class _Rng:
    """Inputs of one seed, in the order they are asked for, made on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0):
        t = torch.empty(shape, device="cuda", dtype=F32)
        return t.normal_(mean, std, generator=self.g)

    def ids(self, n, below):
        return torch.randint(0, below, (n,), device="cuda", dtype=torch.int32, generator=self.g)


def _empty(*shape):
    return torch.empty(shape, device="cuda", dtype=F32)


class _View:
    """n floats at a device address of the library's, as torch sees them; keeps the owner."""

    def __init__(self, owner, ptr, n):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f4", "data": (ptr, False),
                                         "version": 2, "strides": None}


def _view(owner, ptr, n):
    return torch.as_tensor(_View(owner, ptr, n), device="cuda")


def _inputs(c, seed):
    """The case's inputs by name."""
    r, op = _Rng(seed), c["op"]
    if op == "gemm":
        M, N, K = c["M"], c["N"], c["K"]
        return dict(A=r.normal(*((K, M) if c["ta"] else (M, K))),
                    B=r.normal(*((N, K) if c["tb"] else (K, N))), C=r.normal(M, N))
    if op == "linear":
        rows, cin, cout = c["rows"], c["cin"], c["cout"]
        return dict(X=r.normal(rows, cin), W=r.normal(cout, cin, std=0.02),
                    b=r.normal(cout, std=0.02), dY=r.normal(rows, cout, std=1e-3))
    if op == "head":
        return dict(X=r.normal(c["rows"], c["C"]), W=r.normal(c["Vp"], c["C"], std=0.06),
                    y=r.ids(c["rows"], c["V"]))
    if op in ("flash", "attention"):
        B, T, C = c["B"], c["T"], c["NH"] * c["hs"]
        return dict(qkv=r.normal(B, T, 3 * C), dout=r.normal(B, T, C, std=1e-2))
    if op == "norm_gelu":
        rows, C = c["rows"], c["C"]
        return dict(a=r.normal(rows, C, mean=0.1), b=r.normal(rows, C, std=0.5),
                    w=r.normal(C, std=0.1, mean=1.0), bias=r.normal(C, std=0.1),
                    dln=r.normal(rows, C, std=1e-3), h=r.normal(rows, 4 * C),
                    dg=r.normal(rows, 4 * C, std=1e-3))
    if op == "optimizer":
        n = c["n"]
        return dict(p=r.normal(n, std=0.02), g=r.normal(n, std=3e-4), m=r.normal(n, std=1e-4),
                    v=r.normal(n, std=3e-4).square_())
    n = c["B"] * c["T"]
    return dict(p=torch.cat([_param(r, c, k, s) for k, s in _param_sizes(c)]),
                x=r.ids(n, c["V"]), y=r.ids(n, c["V"]))


def _param_sizes(c):
    cfg = (c["T"], c["V"], c["Vp"], c["L"], c["NH"], c["C"])
    return list(zip(bmb.PARAM_NAMES, bmb.param_sizes(cfg)))


def _param(r, c, name, n):
    """GPT-2's initial weights, with biases that a few steps have moved off zero."""
    if name in ("ln1w", "ln2w", "lnfw"):
        return r.normal(n, mean=1.0, std=0.02)
    std = 0.02 / math.sqrt(2 * c["L"]) if name in ("attprojw", "fcprojw") else 0.02
    return r.normal(n, std=std)


def prepare(case, seed):
    """Inputs, the output buffers a program keeps, and (gpt) the model handle."""
    c = dict(case)
    i, op = _inputs(c, seed), c["op"]
    s = dict(c=c, **i)
    if op == "linear":
        s["Y"] = _empty(c["rows"], c["cout"])
        if c["train"]:
            s["dX"] = _empty(c["rows"], c["cin"])
            s["dWb"] = _empty(c["cout"] * (c["cin"] + 1))  # dW, then db
    elif op == "head":
        s.update(logits=_empty(c["rows"], c["Vp"]), probs=_empty(c["rows"], c["Vp"]),
                 dlogits=_empty(c["rows"], c["Vp"]), losses=_empty(c["rows"]),
                 dX=_empty(c["rows"], c["C"]), dW=_empty(c["Vp"], c["C"]))
    elif op == "flash":
        B, T, NH, C = c["B"], c["T"], c["NH"], c["NH"] * c["hs"]
        s.update(out=_empty(B, T, C), lse=_empty(B, NH, T), dsum=_empty(B, NH, T),
                 dqkv=_empty(B, T, 3 * C))
    elif op == "attention":
        B, T, NH, C = c["B"], c["T"], c["NH"], c["NH"] * c["hs"]
        s.update(out=_empty(B, T, C), qkvr=_empty(4, B, NH, T, c["hs"]), att=_empty(B, NH, T, T),
                 dqkv=_empty(B, T, 3 * C), dqkvr=_empty(4, B, NH, T, c["hs"]),
                 datt=_empty(B, NH, T, T))
    elif op == "norm_gelu":
        rows, C = c["rows"], c["C"]
        s.update(res=_empty(rows, C), ln=_empty(rows, C), mean=_empty(rows), rstd=_empty(rows),
                 gelu=_empty(rows, 4 * C), dh=_empty(rows, 4 * C),
                 dres=_empty(rows * C + 2 * C))  # dinp, then dweight and dbias
    elif op == "optimizer":
        s["step"] = OPT_STEP
    elif op == "gpt":
        n = c["B"] * c["T"]
        m = bmb.Model((c["T"], c["V"], c["Vp"], c["L"], c["NH"], c["C"]), c["B"], c["T"])
        np_ = int(m.g.num_params)
        _view(m, m.g.params_mem, np_).copy_(s.pop("p"))
        torch.cuda.synchronize()
        s.update(model=m, x=s["x"].cpu().numpy(), y=s["y"].cpu().numpy(),
                 logits=_view(m, m.g.acts.logits, n * c["Vp"]).view(n, c["Vp"]),
                 grads=_view(m, m.g.grads_mem, np_))
    return s


# --------------------------------------------------------------------- runs
def run(s):
    return _RUN[s["c"]["op"]](s, s["c"])


def _math(c):
    return bmb.gemm_math(bmb.GEMM_MATH_FP32 if c["math"] == "fp32" else bmb.GEMM_MATH_BF16X3)


def _run_gemm(s, c):
    with _math(c):
        bmb.gemm(c["ta"], c["tb"], c["M"], c["N"], c["K"], 1.0, s["A"].data_ptr(),
                 s["B"].data_ptr(), c["beta"], s["C"].data_ptr())
    return s["C"]


def _run_linear(s, c):
    rows, cin, cout = c["rows"], c["cin"], c["cout"]
    X, W, Y, dY = (s[k].data_ptr() for k in ("X", "W", "Y", "dY"))
    with _math(c):
        bmb.gemm(False, True, rows, cout, cin, 1.0, X, W, 0.0, Y)
        bmb.call("bias_forward", Y, s["b"].data_ptr(), rows, cout)
        if not c["train"]:
            return s["Y"]
        dX, dW = s["dX"].data_ptr(), s["dWb"].data_ptr()
        bmb.call("zero_buffer", dW, cout * (cin + 1))
        bmb.gemm(False, False, rows, cin, cout, 1.0, dY, W, 0.0, dX)
        bmb.gemm(True, False, cout, cin, rows, 1.0, dY, X, 1.0, dW)
        bmb.call("bias_backward", dW + 4 * cout * cin, dY, rows, cout)
    return s["Y"], s["dX"], s["dWb"][:cout * cin], s["dWb"][cout * cin:]


def _run_head(s, c):
    rows, C, V, Vp = c["rows"], c["C"], c["V"], c["Vp"]
    X, W, y, logits, probs, losses, dlogits, dX, dW = (
        s[k].data_ptr() for k in ("X", "W", "y", "logits", "probs", "losses", "dlogits", "dX",
                                  "dW"))
    bmb.gemm(False, True, rows, Vp, C, 1.0, X, W, 0.0, logits)
    bmb.call("softmax_crossentropy_forward", probs, losses, logits, y, rows, V, Vp)
    bmb.call("crossentropy_softmax_backward", dlogits, probs, y, rows, V, Vp, 1.0 / rows)
    bmb.gemm(False, False, rows, C, Vp, 1.0, dlogits, W, 0.0, dX)
    bmb.gemm(True, False, Vp, C, rows, 1.0, dlogits, X, 0.0, dW)
    return s["logits"], s["probs"], s["losses"], s["dlogits"], s["dX"], s["dW"]


def _run_flash(s, c):
    dims = (c["B"], c["T"], c["NH"] * c["hs"], c["NH"])
    qkv, out, lse = (s[k].data_ptr() for k in ("qkv", "out", "lse"))
    bmb.flash_forward(out, lse, qkv, *dims)
    bmb.flash_backward(s["dqkv"].data_ptr(), s["dsum"].data_ptr(), s["dout"].data_ptr(), qkv, out,
                       lse, *dims)
    return s["out"], s["lse"], s["dqkv"]


def _run_attention(s, c):
    dims = (c["B"], c["T"], c["NH"] * c["hs"], c["NH"])
    qkvr, att, datt = (s[k].data_ptr() for k in ("qkvr", "att", "datt"))
    bmb.call("attention_forward", s["out"].data_ptr(), qkvr, att, s["qkv"].data_ptr(), *dims)
    bmb.call("attention_backward", s["dqkv"].data_ptr(), s["dqkvr"].data_ptr(), datt, datt,
             s["dout"].data_ptr(), qkvr, att, *dims)
    return s["out"], s["att"], s["dqkv"]


def _run_norm_gelu(s, c):
    rows, C = c["rows"], c["C"]
    p = {k: s[k].data_ptr() for k in ("a", "b", "w", "bias", "dln", "h", "dg", "res", "ln", "mean",
                                      "rstd", "gelu", "dh", "dres")}
    bmb.call("residual_forward", p["res"], p["a"], p["b"], rows * C)
    bmb.call("layernorm_forward", p["ln"], p["mean"], p["rstd"], p["res"], p["w"], p["bias"], rows,
             C)
    bmb.call("gelu_forward", p["gelu"], p["h"], rows * 4 * C)
    bmb.call("gelu_backward", p["dh"], p["h"], p["dg"], rows * 4 * C)
    dw = p["dres"] + 4 * rows * C
    bmb.call("zero_buffer", p["dres"], rows * C + 2 * C)
    bmb.call("layernorm_backward", p["dres"], dw, dw + 4 * C, p["dln"], p["res"], p["w"],
             p["mean"], p["rstd"], rows, C)
    n = rows * C
    return (s["res"], s["ln"], s["mean"], s["rstd"], s["gelu"], s["dh"], s["dres"][:n],
            s["dres"][n:n + C], s["dres"][n + C:])


def _run_optimizer(s, c):
    n = c["n"]
    p, g, m, v = (s[k].data_ptr() for k in "pgmv")
    norm = bmb.call("grad_global_norm", g, n)
    scale = 1.0 / norm if norm > 1.0 else 1.0
    s["step"] += 1
    bmb.call("adamw_update", p, g, m, v, n, ADAMW["lr"], ADAMW["beta1"], ADAMW["beta2"],
             ADAMW["eps"], ADAMW["wd"], s["step"], scale)
    return norm, s["p"], s["m"], s["v"]


def _run_gpt(s, c):
    if not c["train"]:
        s["model"].forward(s["x"])
        return s["logits"]
    loss = s["model"].forward(s["x"], s["y"])
    s["model"].backward()
    return loss, s["logits"], s["grads"]


_RUN = dict(gemm=_run_gemm, linear=_run_linear, head=_run_head, flash=_run_flash,
            attention=_run_attention, norm_gelu=_run_norm_gelu, optimizer=_run_optimizer,
            gpt=_run_gpt)


# --------------------------------------------------------------------- work
def work(case):
    """Bytes and flops of one pass: every input of a call read once, every output written once
    (what one call of the pass leaves for the next counts as both)."""
    c, op = case, case["op"]
    if op == "gemm":
        M, N, K = c["M"], c["N"], c["K"]
        return dict(bytes=4 * (M * K + K * N + M * N * (2 if c["beta"] else 1)),
                    flops=2 * M * N * K)
    if op == "linear":
        x, w, y = c["rows"] * c["cin"], c["cin"] * c["cout"], c["rows"] * c["cout"]
        t = 2 * c["rows"] * w
        if not c["train"]:
            return dict(bytes=4 * (x + w + y), flops=t)
        return dict(bytes=4 * (2 * x + 2 * w + 2 * y), flops=3 * t)
    if op == "head":
        x, w, y = c["rows"] * c["C"], c["Vp"] * c["C"], c["rows"] * c["Vp"]
        return dict(bytes=4 * (2 * x + 2 * w + 3 * y), flops=6 * c["rows"] * w)
    if op == "flash":
        n, P = c["B"] * c["T"] * c["NH"] * c["hs"], c["B"] * c["NH"] * c["T"] * (c["T"] + 1) / 2
        return dict(bytes=4 * (12 * n + 2 * c["B"] * c["NH"] * c["T"]), flops=14 * c["hs"] * P)
    if op == "attention":
        n, P = c["B"] * c["T"] * c["NH"] * c["hs"], c["B"] * c["NH"] * c["T"] * (c["T"] + 1) / 2
        return dict(bytes=4 * (12 * n + 2 * c["B"] * c["NH"] * c["T"] ** 2),
                    flops=12 * c["hs"] * P)
    if op == "norm_gelu":
        return dict(bytes=4 * c["rows"] * c["C"] * (3 + 1 + 2 + 12 + 8), flops=0)
    if op == "optimizer":
        return dict(bytes=4 * 8 * c["n"], flops=0)
    N, C, L = c["B"] * c["T"], c["C"], c["L"]
    params = sum(s for _, s in _param_sizes(c))
    lin = 2 * N * (12 * C * C * L + c["Vp"] * C)
    att = 4 * (c["T"] + 1) / 2 * C * N * L
    if not c["train"]:
        return dict(bytes=4 * (params + N * c["Vp"]), flops=lin + att)
    return dict(bytes=4 * (3 * params + 3 * N * c["Vp"]), flops=3 * lin + 3.5 * att)


# ---------------------------------------------------------------- tolerance
def tolerance(case):
    """About four times the relative error (2-norm) against 64 bits that the path shows."""
    op = case["op"]
    if op in ("gemm", "linear"):
        return dict(rel=2e-5 if case["math"] == "bf16x3" else 4e-6)
    return dict(rel=dict(head=3e-5, flash=4e-6, attention=1.5e-6, norm_gelu=6e-7, optimizer=6e-7,
                         gpt=5e-5)[op])


# -------------------------------------------------------------------- exact
def exact(case, seed):
    c = dict(case)
    i = {k: v.to(F64) if v.dtype == F32 else v for k, v in _inputs(c, seed).items()}
    with torch.no_grad():
        return _EXACT[c["op"]](i, c)


def _exact_gemm(i, c):
    A = i["A"].t().contiguous() if c["ta"] else i["A"]
    B = i["B"].t().contiguous() if c["tb"] else i["B"]
    return A @ B + c["beta"] * i["C"]


def _exact_linear(i, c):
    Y = i["X"] @ i["W"].t().contiguous() + i["b"]
    if not c["train"]:
        return Y
    dW = i["dY"].t().contiguous() @ i["X"]
    return Y, i["dY"] @ i["W"], dW.reshape(-1), i["dY"].sum(0)


def _softmax_loss(logits, y, V):
    """Probabilities (0 in the padding columns) and per-row losses."""
    probs = torch.zeros_like(logits)
    probs[:, :V] = torch.softmax(logits[:, :V], 1)
    losses = torch.logsumexp(logits[:, :V], 1) - logits.gather(1, y.long()[:, None])[:, 0]
    return probs, losses


def _exact_head(i, c):
    logits = i["X"] @ i["W"].t().contiguous()
    probs, losses = _softmax_loss(logits, i["y"], c["V"])
    d = probs.clone()
    d[torch.arange(c["rows"], device=d.device), i["y"].long()] -= 1.0
    d /= c["rows"]
    return logits, probs, losses, d, d @ i["W"], d.t().contiguous() @ i["X"]


def _heads(x, NH):
    """(B, T, C) as (B, NH, T, hs)."""
    B, T, C = x.shape
    return x.reshape(B, T, NH, C // NH).transpose(1, 2).contiguous()


def _rows(x):
    """(B, NH, T, hs) as (B, T, C)."""
    B, NH, T, hs = x.shape
    return x.transpose(1, 2).reshape(B, T, NH * hs)


def _causal(q, k):
    """Scaled causal scores (B, NH, T, T), -inf past the diagonal."""
    T = q.shape[2]
    s = (q @ k.transpose(2, 3).contiguous()) / math.sqrt(q.shape[3])
    return s.masked_fill_(torch.ones(T, T, dtype=torch.bool, device=s.device).triu(1),
                          float("-inf"))


def _attention_fwd(qkv, NH):
    q, k, v = (_heads(t, NH) for t in qkv.chunk(3, 2))
    s = _causal(q, k)
    lse = torch.logsumexp(s, 3)
    p = (s - lse[..., None]).exp_()
    return q, k, v, p, lse, p @ v


def _attention_bwd(q, k, v, p, o, do):
    dv = p.transpose(2, 3).contiguous() @ do
    ds = do @ v.transpose(2, 3).contiguous()
    ds.sub_((do * o).sum(3, keepdim=True)).mul_(p).div_(math.sqrt(q.shape[3]))
    return torch.cat([_rows(t) for t in (ds @ k, ds.transpose(2, 3).contiguous() @ q, dv)], 2)


def _exact_flash(i, c):
    q, k, v, p, lse, o = _attention_fwd(i["qkv"], c["NH"])
    return _rows(o), lse, _attention_bwd(q, k, v, p, o, _heads(i["dout"], c["NH"]))


def _exact_attention(i, c):
    q, k, v, p, _, o = _attention_fwd(i["qkv"], c["NH"])
    return _rows(o), p, _attention_bwd(q, k, v, p, o, _heads(i["dout"], c["NH"]))


GELU_K = math.sqrt(2.0 / math.pi)


def _gelu(x):
    t = torch.tanh(GELU_K * (x + 0.044715 * x ** 3))
    d = 0.5 * (1 + t) + 0.5 * x * (1 - t * t) * GELU_K * (1 + 3 * 0.044715 * x * x)
    return 0.5 * x * (1 + t), d


def _layernorm(x, w, b):
    """Output, mean, 1 / std and the normalised input."""
    mean = x.mean(1)
    rstd = (x.var(1, unbiased=False) + LN_EPS).rsqrt()
    xh = (x - mean[:, None]) * rstd[:, None]
    return xh * w + b, mean, rstd, xh


def _layernorm_bwd(d, w, rstd, xh):
    dx = d * w
    dx = rstd[:, None] * (dx - dx.mean(1, keepdim=True) - xh * (dx * xh).mean(1, keepdim=True))
    return dx, (d * xh).sum(0), d.sum(0)


def _exact_norm_gelu(i, c):
    # The layernorm's input is the fp32 residual stream that the first call writes.
    res = (i["a"] + i["b"]).to(F32).to(F64)
    ln, mean, rstd, xh = _layernorm(res, i["w"], i["bias"])
    dx, dw, db = _layernorm_bwd(i["dln"], i["w"], rstd, xh)
    g, dg = _gelu(i["h"])
    return res, ln, mean, rstd, g, i["dg"] * dg, dx.reshape(-1), dw, db


def _exact_optimizer(i, c):
    a, t = ADAMW, OPT_STEP + 1
    norm = float(i["g"].square().sum().sqrt())
    g = i["g"] / norm if norm > 1.0 else i["g"]
    m = a["beta1"] * i["m"] + (1 - a["beta1"]) * g
    v = a["beta2"] * i["v"] + (1 - a["beta2"]) * g * g
    u = (m / (1 - a["beta1"] ** t)) / ((v / (1 - a["beta2"] ** t)).sqrt() + a["eps"])
    return torch.tensor(norm, dtype=F64), i["p"] - a["lr"] * (u + a["wd"] * i["p"]), m, v


def _exact_gpt(i, c):
    B, T, L, NH, C = (c[k] for k in ("B", "T", "L", "NH", "C"))
    sizes, P, at = _param_sizes(c), {}, 0
    shapes = dict(wte=(-1, C), wpe=(-1, C), qkvw=(L, 3 * C, C), qkvb=(L, 3 * C),
                  attprojw=(L, C, C), fcw=(L, 4 * C, C), fcb=(L, 4 * C), fcprojw=(L, C, 4 * C),
                  lnfw=(C,), lnfb=(C,))
    for name, n in sizes:
        P[name] = i["p"][at:at + n].view(shapes.get(name, (L, C)))
        at += n
    x = (P["wte"][i["x"].long()].view(B, T, C) + P["wpe"][:T]).view(B * T, C)
    keep = []
    for l in range(L):
        W = {k: P[k][l] for k in ("ln1w", "ln1b", "qkvw", "qkvb", "attprojw", "attprojb", "ln2w",
                                  "ln2b", "fcw", "fcb", "fcprojw", "fcprojb")}
        h1, _, r1, xh1 = _layernorm(x, W["ln1w"], W["ln1b"])
        qkv = (h1 @ W["qkvw"].t().contiguous() + W["qkvb"]).view(B, T, 3 * C)
        q, k, v, p, _, o = _attention_fwd(qkv, NH)
        att = _rows(o).reshape(B * T, C)
        x2 = x + att @ W["attprojw"].t().contiguous() + W["attprojb"]
        h2, _, r2, xh2 = _layernorm(x2, W["ln2w"], W["ln2b"])
        f = h2 @ W["fcw"].t().contiguous() + W["fcb"]
        g, dg = _gelu(f)
        x = x2 + g @ W["fcprojw"].t().contiguous() + W["fcprojb"]
        if c["train"]:
            keep.append((W, h1, r1, xh1, q, k, v, p, o, att, h2, r2, xh2, g, dg))
    xf, _, rf, xhf = _layernorm(x, P["lnfw"], P["lnfb"])
    logits = xf @ P["wte"].t().contiguous()
    if not c["train"]:
        return logits
    probs, losses = _softmax_loss(logits, i["y"], c["V"])
    d = probs
    d[torch.arange(B * T, device=d.device), i["y"].long()] -= 1.0
    d /= B * T
    G = {name: torch.zeros(P[name].shape, device=d.device, dtype=F64) for name, _ in sizes}
    G["wte"] += d.t().contiguous() @ xf
    dx, G["lnfw"], G["lnfb"] = _layernorm_bwd(d @ P["wte"], P["lnfw"], rf, xhf)
    for l in range(L - 1, -1, -1):
        W, h1, r1, xh1, q, k, v, p, o, att, h2, r2, xh2, g, dg = keep.pop()
        G["fcprojw"][l], G["fcprojb"][l] = dx.t().contiguous() @ g, dx.sum(0)
        df = (dx @ W["fcprojw"]) * dg
        G["fcw"][l], G["fcb"][l] = df.t().contiguous() @ h2, df.sum(0)
        d2, G["ln2w"][l], G["ln2b"][l] = _layernorm_bwd(df @ W["fcw"], W["ln2w"], r2, xh2)
        dx = dx + d2
        G["attprojw"][l], G["attprojb"][l] = dx.t().contiguous() @ att, dx.sum(0)
        datt = _heads((dx @ W["attprojw"]).view(B, T, C), NH)
        dqkv = _attention_bwd(q, k, v, p, o, datt).reshape(B * T, 3 * C)
        G["qkvw"][l], G["qkvb"][l] = dqkv.t().contiguous() @ h1, dqkv.sum(0)
        d1, G["ln1w"][l], G["ln1b"][l] = _layernorm_bwd(dqkv @ W["qkvw"], W["ln1w"], r1, xh1)
        dx = dx + d1
    G["wpe"][:T] = dx.view(B, T, C).sum(0)
    G["wte"].index_add_(0, i["x"].long(), dx)
    grads = torch.cat([G[name].reshape(-1) for name, _ in sizes])
    return torch.tensor(float(losses.mean()), dtype=F64), logits, grads


_EXACT = dict(gemm=_exact_gemm, linear=_exact_linear, head=_exact_head, flash=_exact_flash,
              attention=_exact_attention, norm_gelu=_exact_norm_gelu, optimizer=_exact_optimizer,
              gpt=_exact_gpt)
