"""The GPT model (gpt.h) on the GPU against the fp64 CPU oracle.

Config of tools/test_grad.cu:57 -- B=4, T=64, C=128, L=2, NH=4, V=65 (Vp=128)
-- with both attention paths (fused flash and the unfused attention.h):
  * forward loss, per-position losses and logits against the oracle's fp64
    GPT (oracle/oracle_gpt.c, itself pinned to torch autograd), and every
    parameter gradient, tensor by tensor;
  * tools/test_grad.cu's directional-derivative check run on the GPU model
    itself (eps 1e-2, relative error < 2e-2 per tensor and for ALL);
  * a short AdamW training run (global-norm clipping at 1.0) whose loss
    trajectory follows the oracle's (fp64 model, fp32 AdamW restatement);
  * invariants: wte = 0 gives loss = ln V exactly; repeated steps are
    bit-identical; gpt_init statistics; the GPT1 checkpoint round trip.
Tolerances: fp32 arithmetic through two layers against fp64 -- loss 1e-5
relative, logits and each gradient tensor 1e-4 normwise (the measured errors
are printed; they sit near 1e-6).
"""
import math

import numpy as np
import pytest

import bmb
import oracle as O
from gpu_util import d2h, h2d, sync

pytestmark = pytest.mark.gpu

CFG = (64, 65, 128, 2, 4, 128)  # max_seq_len, V, Vp, L, NH, C
B, T = 4, 64


def _batch(seed, V=CFG[1], n=B * T):
    r = np.random.default_rng(seed)
    return r.integers(0, V, n).astype(np.int32), r.integers(0, V, n).astype(np.int32)


def _model(use_flash, seed=1337, cfg=CFG, b=B, t=T):
    m = bmb.Model(cfg, b, t, use_flash=use_flash)
    m.init(seed)
    sync("gpt_init")
    return m


def _params(m):
    return d2h(m.g.params_mem, m.g.num_params)


def _grads(m):
    return d2h(m.g.grads_mem, m.g.num_params)


def _offsets(cfg=CFG):
    return np.cumsum([0] + O.gpt_param_sizes(cfg))


@pytest.mark.parametrize("use_flash", [True, False], ids=["flash", "unfused"])
def test_forward_backward_vs_oracle(gpu, use_flash):
    m = _model(use_flash)
    x, y = _batch(4242)
    print("gpt fwd/bwd use_flash=%s" % use_flash, flush=True)
    loss = m.forward(x, y)
    m.backward()
    sync("gpt forward/backward")
    p = _params(m)
    ref_loss, ref_losses, ref_g, ref_logits = O.gpt_forward_backward(CFG, B, T, p, x, y,
                                                                     logits=True)
    losses = d2h(m.g.acts.losses, B * T)
    logits = d2h(m.g.acts.logits, B * T * CFG[2]).reshape(B * T, CFG[2])
    print("loss gpu %.8f oracle %.8f" % (loss, ref_loss))
    assert abs(loss - ref_loss) <= 1e-5 * ref_loss
    assert np.abs(losses - ref_losses).max() <= 1e-5 * ref_loss
    el = O.normwise(logits, ref_logits)[0]
    assert el < 1e-4, el
    g = _grads(m)
    off = _offsets()
    worst = 0.0
    for t, name in enumerate(O.PARAM_NAMES):
        e, bad = O.normwise(g[off[t]:off[t + 1]], ref_g[off[t]:off[t + 1]])
        print("  %-9s normwise %.2e" % (name, e))
        assert bad == 0 and e < 1e-4, name
        worst = max(worst, e)
    print("logits %.2e, worst gradient %.2e" % (el, worst))


# The backward's column sums come from the kernels that make the gradients:
# rows that are no whole tile or wave of rows, a ragged width of the MLP, and a
# width whose layernorm sums do not fit the fused kernel.
@pytest.mark.parametrize("cfg,b", [((50, 65, 128, 2, 3, 96), 3), ((33, 65, 66, 1, 1, 32), 1),
                                   ((8, 65, 128, 1, 16, 2048), 1),
                                   # one and three token rows through every layer
                                   ((1, 65, 128, 2, 2, 64), 1), ((3, 65, 66, 2, 1, 32), 1)],
                         ids=["C96", "C32", "C2048", "1row", "3rows"])
def test_gradients_at_other_widths(gpu, cfg, b):
    n = b * cfg[0]
    m = _model(True, cfg=cfg, b=b, t=cfg[0])
    x, y = _batch(99, cfg[1], n)
    print("gpt gradients", cfg, b, flush=True)
    loss = m.forward(x, y)
    m.backward()
    sync("gpt backward")
    ref_loss, _, ref_g, _ = O.gpt_forward_backward(cfg, b, cfg[0], _params(m), x, y)
    assert abs(loss - ref_loss) <= 1e-5 * ref_loss
    g, off = _grads(m), _offsets(cfg)
    for t, name in enumerate(O.PARAM_NAMES):
        e, bad = O.normwise(g[off[t]:off[t + 1]], ref_g[off[t]:off[t + 1]])
        assert bad == 0 and e < 1e-4, (name, e)


def test_column_sums_of_a_banded_gelu_gradient(gpu, capfd, monkeypatch):
    """The FC layer's bias gradient comes from partial sums that the GELU-grad
    GEMM leaves, one row per wave tile row: here of two bands (256 x 256 tiles,
    then 64 x 64 with a ragged last one), whose second writes behind the first.
    Against the column sums of the stored gradient in fp64: chains of fewer
    than 128 fp32 additions (64 rows of a lane, the lane's other half, up to
    32 partials of a slice, 32 slices) of at most 2^-24 of the sum of
    magnitudes each."""
    cfg, b, t = (1101, 65, 128, 1, 12, 768), 5, 1101
    n, width = b * t, 4 * 768
    m = _model(True, cfg=cfg, b=b, t=t)
    x, y = _batch(77, cfg[1], n)
    monkeypatch.setenv("BMB_GEMM_PLAN_TRACE", "1")
    print("gpt banded gelu gradient", cfg, b, flush=True)
    m.forward(x, y)
    capfd.readouterr()
    m.backward()
    sync("gpt backward")
    trace = capfd.readouterr().err
    plans = [l for l in trace.splitlines() if "gemm plan %dx%dx768:" % (n, width) in l]
    assert plans and "m1 5376" in plans[0] and "parts (0,1,768) (2,1,768)" in plans[0], trace
    dfch = d2h(m.g.gr.dfch, n * width).reshape(n, width).astype(np.float64)
    off = _offsets(cfg)
    i = O.PARAM_NAMES.index("fcb")
    got = _grads(m)[off[i]:off[i + 1]]
    bound = 128 * 2.0 ** -24 * np.abs(dfch).sum(axis=0)
    assert np.all(np.abs(got - dfch.sum(axis=0)) <= bound)
    assert np.abs(got).max() > 0


def _loss_double(m, x, y):
    """Mean loss with the per-position losses summed in fp64 on the host
    (tools/test_grad.cu:44-52)."""
    m.forward(x, y)
    return float(d2h(m.g.acts.losses, B * T).astype(np.float64).mean())


@pytest.mark.parametrize("use_flash", [True, False], ids=["flash", "unfused"])
def test_directional_derivative_gradcheck(gpu, use_flash):
    """tools/test_grad.cu:77-176 on the GPU model: for each tensor step along
    u = g/||g||; (L(p + eps u) - L(p - eps u)) / 2 eps must match ||g||."""
    eps = 1e-2
    m = _model(use_flash)
    x, y = _batch(4242)
    L0 = _loss_double(m, x, y)
    m.backward()
    g = _grads(m).astype(np.float64)
    p = _params(m)
    off = _offsets()
    print("loss at theta %.6f (ln V = %.6f)" % (L0, math.log(CFG[1])))
    failures, checked = [], 0
    dirs = [(name, off[t], off[t + 1]) for t, name in enumerate(O.PARAM_NAMES)]
    dirs.append(("ALL", 0, p.size))
    for name, a, b in dirs:
        gt = g[a:b]
        gn = float(np.sqrt((gt * gt).sum()))
        if gn < 1e-9:
            print("  %-9s skipped (zero grad)" % name)
            continue
        pp = p.copy()
        pp[a:b] = (p[a:b] + eps * (gt / gn)).astype(np.float32)
        h2d(m.g.params_mem, pp)
        lp = _loss_double(m, x, y)
        pp[a:b] = (p[a:b] - eps * (gt / gn)).astype(np.float32)
        h2d(m.g.params_mem, pp)
        lm = _loss_double(m, x, y)
        num = (lp - lm) / (2 * eps)
        rel = abs(num - gn) / max(gn, 1e-12)
        print("  %-9s analytic %.6e numeric %.6e rel %.2e" % (name, gn, num, rel))
        checked += 1
        if not rel < 2e-2:
            failures.append(name)
        h2d(m.g.params_mem, p)
    assert checked >= 15 and not failures, failures


def test_steps_are_deterministic(gpu):
    m = _model(True)
    x, y = _batch(7)
    l1 = m.forward(x, y)
    m.backward()
    g1 = _grads(m)
    l2 = m.forward(x, y)
    m.backward()
    g2 = _grads(m)
    assert l1 == l2 and np.array_equal(g1, g2)


def test_zero_embedding_gives_ln_v(gpu):
    """wte = 0 makes every logit 0: loss = ln V for every position."""
    m = _model(True)
    h2d(m.g.params_mem, np.zeros(m.g.psize[0], np.float32))
    x, y = _batch(9)
    loss = m.forward(x, y)
    losses = d2h(m.g.acts.losses, B * T)
    assert abs(loss - math.log(CFG[1])) < 1e-6
    assert np.abs(losses - math.log(CFG[1])).max() < 1e-6
    assert not np.any(d2h(m.g.acts.logits, B * T * CFG[2]))


def _train(use_gpu_model, steps, lr=1e-3, wd=0.1, clip=1.0):
    """Losses of `steps` AdamW steps on one fixed batch: the GPU model, or
    the oracle's fp64 model with the fp32 AdamW restatement."""
    m = _model(True)
    x, y = _batch(11)
    losses = []
    if use_gpu_model:
        for step in range(1, steps + 1):
            losses.append(m.forward(x, y))
            m.backward()
            gn = bmb.call("grad_global_norm", m.g.grads_mem, m.g.num_params)
            gs = clip / gn if gn > clip else 1.0
            bmb.call("adamw_update", m.g.params_mem, m.g.grads_mem, m.g.m_mem, m.g.v_mem,
                     m.g.num_params, lr, 0.9, 0.999, 1e-8, wd, step, gs)
        sync("train")
        return losses
    p = _params(m)
    mm = np.zeros_like(p)
    vv = np.zeros_like(p)
    for step in range(1, steps + 1):
        loss, _, g, _ = O.gpt_forward_backward(CFG, B, T, p, x, y)
        losses.append(loss)
        g32 = g.astype(np.float32)
        gn = float(np.sqrt((g32.astype(np.float64) ** 2).sum()))
        gs = clip / gn if gn > clip else 1.0
        p, mm, vv = O.adamw_f32(p, g32, mm, vv, lr, 0.9, 0.999, 1e-8, wd, step, gs)
    return losses


def test_training_trajectory_tracks_oracle(gpu):
    steps = 8
    gpu_l = _train(True, steps)
    ref_l = _train(False, steps)
    print("gpu   ", " ".join("%.6f" % v for v in gpu_l))
    print("oracle", " ".join("%.6f" % v for v in ref_l))
    assert gpu_l[-1] < gpu_l[0] - 0.05  # it learns the batch
    for a, b in zip(gpu_l, ref_l):
        assert abs(a - b) <= 2e-4 * b, (a, b)


def test_init_statistics_and_seed(gpu):
    cfg = (64, 65, 128, 4, 4, 128)
    m = _model(True, seed=1337, cfg=cfg)
    p = _params(m)
    off = _offsets(cfg)
    sl = {n: p[off[t]:off[t + 1]] for t, n in enumerate(O.PARAM_NAMES)}
    for n in ("ln1w", "ln2w", "lnfw"):
        assert np.all(sl[n] == 1.0)
    for n in ("ln1b", "ln2b", "lnfb", "qkvb", "attprojb", "fcb", "fcprojb"):
        assert not np.any(sl[n])
    for n in ("wte", "wpe", "qkvw", "fcw"):
        assert abs(sl[n].std() / 0.02 - 1) < 0.02 and abs(sl[n].mean()) < 1e-3, n
    rs = 0.02 / math.sqrt(2 * cfg[3])
    for n in ("attprojw", "fcprojw"):
        assert abs(sl[n].std() / rs - 1) < 0.02, n
    m2 = _model(True, seed=1337, cfg=cfg)
    assert np.array_equal(_params(m2), p)
    m3 = _model(True, seed=1338, cfg=cfg)
    assert not np.array_equal(_params(m3), p)


def test_checkpoint_roundtrip(gpu, tmp_path):
    import ctypes
    m = _model(True)
    path = str(tmp_path / "gpt.bin").encode()
    itos = bytes(range(32, 32 + CFG[1]))
    assert bmb.call("gpt_save_checkpoint", ctypes.byref(m.g), path, itos, len(itos)) == 0
    raw = np.fromfile(tmp_path / "gpt.bin", dtype=np.uint8)
    assert raw[:4].view(np.int32)[0] == 0x47505431
    assert list(raw[4:28].view(np.int32)) == list(CFG)
    g2 = bmb.GPT()
    g2.B, g2.use_flash = B, True
    buf = ctypes.create_string_buffer(256)
    nv = ctypes.c_int(0)
    assert bmb.call("gpt_load_checkpoint", ctypes.byref(g2), path, buf, 256, ctypes.byref(nv)) == 0
    assert nv.value == len(itos) and buf.raw[:len(itos)] == itos
    assert g2.T == CFG[0] and tuple(getattr(g2.config, f) for f, _ in bmb.GPTConfig._fields_) == CFG
    assert np.array_equal(d2h(g2.params_mem, g2.num_params), _params(m))
    bmb.call("gpt_free", ctypes.byref(g2))
    bad = tmp_path / "bad.bin"
    bad.write_bytes(b"XXXX" + bytes(64))
    g3 = bmb.GPT()
    g3.B = B
    assert bmb.call("gpt_load_checkpoint", ctypes.byref(g3), str(bad).encode(), None, 0, None) == -1


GPT2_SMALL = (1024, 50257, 50304, 12, 12, 768)


def test_gpt2_small_b8_step(gpu):
    """The benchmarked config-5 step at its own size: GPT-2 small
    (12L/768/12H, T=1024, V=50257 -> 50304), B=8, gpt_init(1337), i.i.d.
    uniform token ids. The fp64 oracle cannot run a 7-TFLOP step, so the
    checks are the properties the model fixes at any size:
      * the first loss sits near ln V (logits start small) and every
        gradient is finite; two forward+backward calls give the same bits;
      * batch decomposition: each sequence's per-position losses, and the
        mean-loss gradient, depend only on that sequence. The B=8 losses
        must match four B=2 models on the same weights, sequence by sequence,
        and the B=8 gradient must equal the mean of the four B=2 gradients
        (only fp32 summation orders differ: 1e-5 relative on losses, 1e-3
        normwise per gradient tensor through 12 layers);
      * three clipped AdamW steps on that batch (src/train_gpt.cu:430-446)
        lower its loss each time."""
    cfg = GPT2_SMALL
    Bb, Tt = 8, 1024
    r = np.random.default_rng(5)
    x = r.integers(0, cfg[1], Bb * Tt).astype(np.int32)
    y = r.integers(0, cfg[1], Bb * Tt).astype(np.int32)
    m = _model(True, cfg=cfg, b=Bb, t=Tt)
    n = m.g.num_params
    print("GPT-2 small B=8 step", flush=True)
    l1 = m.forward(x, y)
    m.backward()
    gn1 = bmb.call("grad_global_norm", m.g.grads_mem, n)
    losses8 = d2h(m.g.acts.losses, Bb * Tt)
    g8 = _grads(m)
    l2 = m.forward(x, y)
    m.backward()
    gn2 = bmb.call("grad_global_norm", m.g.grads_mem, n)
    sync("B=8 step")
    print("loss %.6f (ln V %.6f), |g| %.6f" % (l1, math.log(cfg[1]), gn1), flush=True)
    assert abs(l1 - math.log(cfg[1])) < 0.5
    assert np.isfinite(g8).all() and np.isfinite(gn1) and gn1 > 0
    assert l1 == l2 and gn1 == gn2
    assert np.array_equal(g8.view(np.uint32), _grads(m).view(np.uint32))

    m2 = _model(True, cfg=cfg, b=2, t=Tt)
    assert np.array_equal(_params(m2), _params(m))
    gsum = np.zeros(n, np.float64)
    for j in range(4):
        sl = slice(j * 2 * Tt, (j + 1) * 2 * Tt)
        m2.forward(x[sl], y[sl])
        m2.backward()
        l2j = d2h(m2.g.acts.losses, 2 * Tt)
        e = np.abs(l2j - losses8[sl]).max()
        print("  sequences %d-%d: max |loss diff| %.2e" % (2 * j, 2 * j + 1, e), flush=True)
        assert e <= 1e-5 * math.log(cfg[1])
        gsum += _grads(m2)
    m2.free()
    gmean = gsum / 4
    off = np.cumsum([0] + O.gpt_param_sizes(cfg))
    worst = 0.0
    for t, name in enumerate(O.PARAM_NAMES):
        e, bad = O.normwise(g8[off[t]:off[t + 1]], gmean[off[t]:off[t + 1]])
        worst = max(worst, e)
        assert bad == 0 and e < 1e-3, (name, e)
    print("  gradient vs mean of four B=2 gradients: worst tensor normwise %.2e" % worst)

    L = bmb.lib()
    hist = []
    for step in range(1, 4):
        loss = m.forward(x, y)
        m.backward()
        gn = L.grad_global_norm(m.g.grads_mem, n)
        L.adamw_update(m.g.params_mem, m.g.grads_mem, m.g.m_mem, m.g.v_mem, n, 1e-4, 0.9,
                       0.999, 1e-8, 0.1, step, 1.0 / gn if gn > 1.0 else 1.0)
        hist.append(loss)
    hist.append(m.forward(x, y))
    sync("AdamW steps")
    print("  loss over three AdamW steps: %s" % ", ".join("%.5f" % v for v in hist))
    assert all(b < a for a, b in zip(hist, hist[1:]))
    m.free()


def test_flash_gpt_odd_sizes(gpu):
    """B*T*L odd (B=1, T=33, L=1): every activation still starts on a 16-byte
    boundary, which the flash kernels require; forward and gradients match
    the oracle."""
    cfg = (33, 65, 128, 1, 4, 128)
    b, t = 1, 33
    m = _model(True, cfg=cfg, b=b, t=t)
    for name in ("qkv", "atty", "lse", "ln1", "fch"):
        assert getattr(m.g.acts, name) % 16 == 0, name
    r = np.random.default_rng(33)
    x = r.integers(0, cfg[1], b * t).astype(np.int32)
    y = r.integers(0, cfg[1], b * t).astype(np.int32)
    loss = m.forward(x, y)
    m.backward()
    sync("odd-size GPT")
    ref_loss, _, ref_g, _ = O.gpt_forward_backward(cfg, b, t, _params(m), x, y)
    assert abs(loss - ref_loss) <= 1e-5 * ref_loss
    e, bad = O.normwise(_grads(m), ref_g)
    print("odd sizes: loss %.6f oracle %.6f, gradient normwise %.2e" % (loss, ref_loss, e))
    assert bad == 0 and e < 1e-4


def test_fused_forward_matches_separate_ops(gpu):
    """gpt_forward fuses bias (and GELU) into the GEMM epilogue and each
    residual add into the following layernorm. Recompute layer 0 and the start
    of layer 1 from the stored activations with the reference's separate
    launches (gemm, bias_forward, gelu_forward, residual_forward,
    layernorm_forward, src/gpt.cu:254-283): every tensor must be bit-identical."""
    import torch
    m = _model(True)
    x, y = _batch(31)
    m.forward(x, y)
    sync("forward")
    C, N = CFG[5], B * T
    off = _offsets()
    p = _params(m)
    P = {n: p[off[t]:off[t + 1]] for t, n in enumerate(O.PARAM_NAMES)}
    a = m.g.acts
    get = lambda ptr, n, o=0: d2h(ptr + 4 * o, n)
    ln1, qkv = get(a.ln1, N * C), get(a.qkv, N * 3 * C)
    atty, attproj = get(a.atty, N * C), get(a.attproj, N * C)
    res2, ln2 = get(a.residual2, N * C), get(a.ln2, N * C)
    fch, fchg = get(a.fch, N * 4 * C), get(a.fch_gelu, N * 4 * C)
    fcproj, res3 = get(a.fcproj, N * C), get(a.residual3, N * C)
    ln1_next = get(a.ln1, N * C, N * C)

    def dv(h):
        return torch.from_numpy(np.ascontiguousarray(h, np.float32)).cuda()

    def linear(inp, w, bias, cout, cin):
        out = torch.empty(N * cout, device="cuda", dtype=torch.float32)
        d_in, d_w, d_b = dv(inp), dv(w), dv(bias)
        bmb.gemm(False, True, N, cout, cin, 1.0, d_in.data_ptr(), d_w.data_ptr(), 0.0,
                 out.data_ptr())
        bmb.call("bias_forward", out.data_ptr(), d_b.data_ptr(), N, cout)
        sync("linear")
        return out.cpu().numpy()

    def layernorm(inp, w, b):
        d_in, d_w, d_b = dv(inp), dv(w), dv(b)
        out = torch.empty(N * C, device="cuda", dtype=torch.float32)
        mean = torch.empty(N, device="cuda", dtype=torch.float32)
        rstd = torch.empty(N, device="cuda", dtype=torch.float32)
        bmb.call("layernorm_forward", out.data_ptr(), mean.data_ptr(), rstd.data_ptr(),
                 d_in.data_ptr(), d_w.data_ptr(), d_b.data_ptr(), N, C)
        sync("layernorm")
        return out.cpu().numpy()

    assert np.array_equal(linear(ln1, P["qkvw"][:3 * C * C], P["qkvb"][:3 * C], 3 * C, C), qkv)
    assert np.array_equal(linear(atty, P["attprojw"][:C * C], P["attprojb"][:C], C, C), attproj)
    assert np.array_equal(res2, get(a.encoded, N * C) + attproj)
    assert np.array_equal(layernorm(res2, P["ln2w"][:C], P["ln2b"][:C]), ln2)
    assert np.array_equal(linear(ln2, P["fcw"][:4 * C * C], P["fcb"][:4 * C], 4 * C, C), fch)
    d_fch = dv(fch)
    g_out = torch.empty(N * 4 * C, device="cuda", dtype=torch.float32)
    bmb.call("gelu_forward", g_out.data_ptr(), d_fch.data_ptr(), N * 4 * C)
    sync("gelu")
    assert np.array_equal(g_out.cpu().numpy(), fchg)
    assert np.array_equal(linear(fchg, P["fcprojw"][:4 * C * C], P["fcprojb"][:C], C, 4 * C), fcproj)
    assert np.array_equal(res3, res2 + fcproj)
    assert np.array_equal(layernorm(res3, P["ln1w"][C:2 * C], P["ln1b"][C:2 * C]), ln1_next)


def test_bad_token_rejected_before_launch(gpu):
    """A token id outside [0, Vp) would index past wte on the device: gpt_forward
    checks the host ids first, reports and returns NaN without launching."""
    m = _model(True)
    x, y = _batch(3)
    ref = m.forward(x, y)
    x_bad = x.copy()
    x_bad[17] = CFG[2]
    assert math.isnan(m.forward(x_bad, y))
    x_bad[17] = -1
    assert math.isnan(m.forward(x_bad, y))
    assert m.forward(x, y) == ref  # the model is untouched
