"""The work a user has this framework do, as measured cases.

A case is one pass through the public API on one GPU: a training step of a
packed layer (forward, backward with the optimizer inside it, rebalance), a
forward alone, the Muon drive, or the export of deploy weights.  Layer states
are those of a checkpoint in mid-training, made from the seed without the
library's own kernels; activations are N(0, 1) and output gradients
N(0, 1e-3), as the SDXL and char-GPT configurations use them.

`captured` steps are replayed from one HIP graph, the way a training program
that captures its step runs them; the others are called eagerly.
"""
import math

import torch
import torch.nn.functional as F

import concord_amd as ca

DEV = "cuda"
BETA2 = 0.999
LARGEST = 6.0 * 4096 * 10240 * 1280   # flops of the largest listed step


def _step(name, n, k, m, flags="winner", captured=False, cache=False, bias=True, dtype="bf16"):
    return {"name": name, "kind": "step", "n": n, "k": k, "m": m, "flags": flags, "captured": captured,
            "cache": cache, "bias": bias, "dtype": dtype}


def _conv(name, cin, cout, hw, batch, kernel=3, stride=1, input_grad=True, flags="default", captured=False):
    return {"name": name, "kind": "conv", "cin": cin, "cout": cout, "hw": hw, "batch": batch, "kernel": kernel,
            "stride": stride, "input_grad": input_grad, "flags": flags, "captured": captured}


def listed():
    return [
        # the smallest call: SDXL's time embedding at batch 4 (four rows), the
        # default optimizer flags, called eagerly; latency and launches only
        _step("time_embed", 1280, 320, 4, flags="default"),
        # SDXL cross-attention k/v on 77 x 4 text tokens: a few hundred tokens
        # against 2.6 M weights, so the update and the weight reads dominate
        _step("cross_attn_kv", 1280, 2048, 308, captured=True),
        # SDXL attention q/k/v/out, the most frequent layer of the UNet
        _step("attn_proj", 1280, 1280, 4096, captured=True),
        # SDXL GEGLU in, the largest product of the UNet, called eagerly
        _step("geglu_in", 10240, 1280, 4096),
        # SDXL GEGLU out in the cached-weight mode (the update emits the bf16
        # weight that forward and dgrad read)
        _step("geglu_out_cached", 1280, 5120, 2048, captured=True, cache=True),
        # SDXL attention at the 64 x 64 level: many tokens, a small weight
        _step("attn_proj_hires", 640, 640, 16384, captured=True),
        # char GPT's head: vocabulary 65 (no multiple of anything), fp32
        # activations, no bias, default flags, called eagerly
        _step("char_head", 65, 384, 16384, flags="default", bias=False, dtype="fp32"),
        # SDXL resnet 3 x 3 convolution, implicit GEMM, called eagerly
        _conv("conv_res", 640, 640, 64, 2),
        # SDXL conv_in: 4 latent channels (patch rows of 36), whose input
        # takes no gradient, called eagerly
        _conv("conv_in", 4, 320, 128, 2, input_grad=False),
        # forward alone (sampling, evaluation): GEGLU in at the 64 x 64 level
        {"name": "forward_hires", "kind": "forward", "n": 5120, "k": 640, "m": 8192},
        # the Muon drive of a 1280 x 5120 gradient
        {"name": "muon_drive", "kind": "muon", "n": 1280, "k": 5120},
        # deploy export of one transformer block's linears
        {"name": "export_block", "kind": "export", "n": 1280, "k": 1280, "layers": 8, "ff": 10240},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, ragged, lo=64, hi=10240):
    v = _log_int(rng, lo, hi)
    if ragged:
        return v
    unit = 64 if v >= 512 else 8
    return max(unit, (v + unit // 2) // unit * unit)


def draw(rng):
    kind = rng.choice(["step"] * 6 + ["conv"] * 2 + ["forward", "muon", "export"])
    ragged = rng.random() < 0.25
    if kind in ("step", "forward"):
        cap = LARGEST / 8 if ragged else LARGEST
        while True:
            n, k = _width(rng, ragged), _width(rng, ragged)
            m = _log_int(rng, 4, 16384)
            if n * k <= 10240 * 1280 and 6.0 * m * n * k <= cap:
                break
        if kind == "forward":
            return {"kind": "forward", "n": n, "k": k, "m": m}
        c = _step("", n, k, m, flags=rng.choice(["winner", "default"]), cache=rng.random() < 0.2,
                  bias=rng.random() < 0.8, dtype=rng.choice(["bf16", "bf16", "fp32"]))
        c["captured"] = c["flags"] == "winner" and rng.random() < 0.6
    elif kind == "conv":
        while True:
            cin, cout = (rng.choice([4, 64, 128, 192, 320, 640, 960, 1280] if not ragged else [3, 4, 9, 100, 330])
                         for _ in range(2))
            hw, batch, kernel = _log_int(rng, 8, 128), rng.choice([1, 2, 3, 4]), rng.choice([1, 3, 3, 3])
            # at most the listed resnet convolution's work
            if 6.0 * batch * hw * hw * cout * cin * kernel * kernel <= 6.0 * 8192 * 640 * 5760:
                break
        c = _conv("", cin, cout, hw, batch, kernel=kernel, stride=rng.choice([1, 1, 2]),
                  input_grad=rng.random() < 0.8, flags=rng.choice(["winner", "default"]))
        c["captured"] = c["flags"] == "winner" and rng.random() < 0.5
    elif kind == "muon":
        while True:
            n, k = _width(rng, ragged, 64, 5120), _width(rng, ragged, 64, 5120)
            if n * k * min(n, k) <= (1280 * 1280 * 5120) // (8 if ragged else 1):
                break
        return {"kind": "muon", "n": n, "k": k}
    else:
        n = _width(rng, ragged, 64, 1536)
        return {"kind": "export", "n": n, "k": _width(rng, ragged, 64, 1536), "layers": rng.randint(1, 8),
                "ff": _width(rng, ragged, 64, 10240)}
    del c["name"]
    return c


# ---- states -----------------------------------------------------------------
def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device=DEV)


def _packed_state(gen, n, k):
    """Packed words of a weight of variance 2 / (n + k) in mid-training: half
    of each mantissa in either slow field, the fields a few units apart and a
    residual in the fast field; row exponents from the row maxima."""
    w = _randn(gen, n, k) * math.sqrt(2.0 / (n + k))
    re = torch.ceil(torch.log2(w.abs().amax(1).clamp_min(1e-30)) + 1.0).clamp(-8, 7)
    m = torch.round(w * torch.exp2(15.0 - re)[:, None])
    vs = torch.round(m / 256.0).clamp(-120, 120)
    ss = (torch.round((m - 128.0 * vs) / 128.0) + torch.round(_randn(gen, n, k))).clamp(-120, 120)
    sf = (m - 128.0 * (ss + vs) + torch.round(30.0 * _randn(gen, n, k))).clamp(-20000, 20000)
    sf, ss, vs = (t.to(torch.int32) for t in (sf, ss, vs))
    words = (sf << 16) | ((ss & 255) << 8) | (vs & 255)
    return words, re.to(torch.int8), torch.zeros(k, dtype=torch.int8, device=DEV)


def _checkpoint(gen, n, k, m, bias):
    """The buffers a checkpoint of the layer holds; v-hat at the level that
    gradients of m rows of N(0, 1e-3) x N(0, 1) keep it."""
    words, re, ce = _packed_state(gen, n, k)
    g2 = 1e-6 * m
    sd = {"packed_w": words, "row_exp": re, "col_exp": ce,
          "v_row": g2 * k * (1.0 + 0.1 * torch.rand(n, generator=gen, device=DEV)),
          "v_col": g2 * n * (1.0 + 0.1 * torch.rand(k, generator=gen, device=DEV))}
    if bias:
        sd["bias"] = (0.02 * _randn(gen, n)).to(torch.bfloat16)
    return sd


def _resume(layer, sd, seed):
    """Load `sd` into the layer as a resumed run does, the salt of its
    rounding streams included."""
    full = layer.state_dict()
    full.update(sd)
    full["_reb_seed"] = torch.full_like(full["_reb_seed"], seed % 1000)
    full["_row_max_hwm"] = torch.zeros_like(full["_row_max_hwm"])
    full["_col_max_hwm"] = torch.zeros_like(full["_col_max_hwm"])
    extra = dict(full["_extra_state"])
    extra["salt_counter"] = 1000 + seed % 100000
    full["_extra_state"] = extra
    layer.load_state_dict(full)


def _set_flags(layer, flags):
    winner = flags == "winner"
    ca.set_ratio_coh(winner)
    if winner:
        ca.set_ratio_coh_floors(0.9, 0.999)
        layer.disable_cohpre()
        layer.gf_consol = 50.0


def _conv_out(case):
    pad = case["kernel"] // 2
    return (case["hw"] + 2 * pad - case["kernel"]) // case["stride"] + 1


def _inputs(case, seed):
    """(checkpoint, x, dy) of a step or forward case."""
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    if case["kind"] == "conv":
        n, k = case["cout"], case["cin"] * case["kernel"] ** 2
        out = _conv_out(case)
        m = case["batch"] * out * out
        sd = _checkpoint(gen, n, k, m, True)
        x = _randn(gen, case["batch"], case["cin"], case["hw"], case["hw"]).to(torch.bfloat16)
        dy = (1e-3 * _randn(gen, case["batch"], n, out, out)).to(torch.bfloat16)
        x, dy = (t.contiguous(memory_format=torch.channels_last) for t in (x, dy))
        return sd, x, dy
    n, k, m = case["n"], case["k"], case["m"]
    sd = _checkpoint(gen, n, k, m, case.get("bias", True))
    dt = torch.float32 if case.get("dtype") == "fp32" else torch.bfloat16
    return sd, _randn(gen, m, k).to(dt), (1e-3 * _randn(gen, m, n)).to(dt)


def _train_step(s):
    layer, x = s["layer"], s["x"]
    x.grad = None
    layer.zero_grad(set_to_none=True)
    y = layer(x)
    y.backward(s["dy"])
    layer.rebalance()
    return y


def prepare(case, seed):
    kind = case["kind"]
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    if kind == "muon":
        return {"kind": kind, "g": (1e-3 * _randn(gen, case["n"], case["k"])).to(torch.bfloat16)}
    if kind == "export":
        shapes = [(case["n"], case["k"])] * case["layers"] + [(case["ff"], case["k"])]
        layers = []
        for n, k in shapes:
            layer = ca.ConcordLinearPackedB(k, n, bias=True, device=DEV, lr=5e-4)
            layer.disable_cohpre()
            _resume(layer, _checkpoint(gen, n, k, 4096, True), seed)
            layers.append(layer)
        return {"kind": kind, "layers": layers, "names": ["l%d" % i for i in range(len(layers))]}
    sd, x, dy = _inputs(case, seed)
    if kind == "conv":
        layer = ca.ConcordConv2dPackedB(case["cin"], case["cout"], case["kernel"], stride=case["stride"],
                                        padding=case["kernel"] // 2, device=DEV, lr=5e-4)
    else:
        layer = ca.ConcordLinearPackedB(case["k"], case["n"], bias=case.get("bias", True), device=DEV, lr=5e-4,
                                        weight_cache=case.get("cache", False))
    _set_flags(layer, case.get("flags", "winner"))
    _resume(layer, sd, seed)
    if kind == "forward":
        return {"kind": kind, "layer": layer, "x": x}
    if case.get("input_grad", True):
        x.requires_grad_(True)
    s = {"kind": kind, "layer": layer, "x": x, "dy": dy, "graph": None}
    if case["captured"]:
        # the usual capture recipe: warm up on a side stream, capture one
        # step, then load the state the warm-up has stepped past
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(2):
                _train_step(s)
        torch.cuda.current_stream().wait_stream(side)
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["y"] = _train_step(s)
        _resume(layer, sd, seed)
    return s


def run(state):
    if state["kind"] == "muon":
        return ca.muon_ns5(state["g"])
    if state["kind"] == "export":
        return ca.consolidated_state_dict(state["layers"], state["names"])
    layer, x = state["layer"], state["x"]
    if state["kind"] == "forward":
        with torch.no_grad():
            return layer(x)
    if state["graph"] is not None:
        state["graph"].replay()
        y = state["y"]
    else:
        y = _train_step(state)
    return {"y": y.detach(), "dx": x.grad, "db": None if layer.bias is None else layer.bias.grad,
            "words": layer.packed_w, "row_exp": layer.row_exp, "col_exp": layer.col_exp,
            "v_row": layer.v_row, "v_col": layer.v_col}


# ---- work, tolerance, 64-bit results -----------------------------------------
def _mnk(case):
    if case["kind"] == "conv":
        out = _conv_out(case)
        return case["batch"] * out * out, case["cout"], case["cin"] * case["kernel"] ** 2
    return case.get("m", 0), case["n"], case["k"]


def work(case):
    kind = case["kind"]
    m, n, k = _mnk(case)
    if kind == "muon":
        a, b = min(n, k), max(n, k)
        # five iterations of X X^T and A A (symmetric: half the products) and B X
        return {"bytes": 4.0 * n * k, "flops": 5.0 * (a * a * b + a * a * a + 2.0 * a * a * b)}
    if kind == "export":
        words = case["layers"] * n * k + case["ff"] * k
        return {"bytes": 6.0 * words, "flops": 0.0}
    es = 4 if case.get("dtype") == "fp32" else 2
    if kind == "forward":
        return {"bytes": 2.0 * m * (n + k) + 4.0 * n * k, "flops": 2.0 * m * n * k}
    # words read and written; default flags: the coherence EMA too; the cached
    # mode writes the bf16 weight and reads it in place of the words
    per_word = 8.0 + (8.0 if case["flags"] == "default" else 0.0) + (4.0 if case.get("cache") else 0.0)
    if kind == "conv":
        pixels = case["batch"] * case["hw"] ** 2 * case["cin"]
        acts = 2.0 * (pixels * (2 if case["input_grad"] else 1) + 2 * m * n)
        flops = (6.0 if case["input_grad"] else 4.0) * m * n * k
    else:
        acts = 2.0 * es * m * (n + k)
        flops = 6.0 * m * n * k
    return {"bytes": acts + per_word * n * k, "flops": flops}


def tolerance(case):
    if case["kind"] == "export":
        return "exact"
    if case["kind"] == "muon":
        # fifteen bf16 products in a chain: about 2e-2 from the 64-bit result
        return {"rel": 0.03, "max": 0.2}
    # bf16 outputs round by 1.7e-3 against the 64-bit result; another order of
    # the fp32 sums moves a value by one bf16 step at most (2^-7 of it), and
    # the words it steps with it (up to 1.2e-4 of them, seen against gradients
    # rounded from their 64-bit sums)
    return {"rel": 7e-3, "max": 0.02, "differ": 1e-3}


def _fields(words):
    return words >> 16, (words << 16) >> 24, (words << 24) >> 24


def _dense(sd, consolidated=False):
    sf, ss, vs = (t.double() for t in _fields(sd["packed_w"]))
    m = 128.0 * (ss + vs) + (0.0 if consolidated else sf)
    e = sd["row_exp"].double()[:, None] + sd["col_exp"].double()[None, :] - 15.0
    return m * torch.exp2(e)


def exact(case, seed):
    kind = case["kind"]
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    if kind == "muon":
        g = (1e-3 * _randn(gen, case["n"], case["k"])).to(torch.bfloat16).double()
        x = g.T if case["n"] > case["k"] else g
        x = x / x.norm()
        for _ in range(5):
            a = x @ x.T
            x = 3.4445 * x + (-4.7750 * a + 2.0315 * (a @ a)) @ x
        x = x * math.sqrt(max(case["n"], case["k"]))
        return x.T if case["n"] > case["k"] else x
    if kind == "export":
        shapes = [(case["n"], case["k"])] * case["layers"] + [(case["ff"], case["k"])]
        out = {}
        for i, (n, k) in enumerate(shapes):
            sd = _checkpoint(gen, n, k, 4096, True)
            out["l%d.weight" % i] = _dense(sd, consolidated=True)
            out["l%d.bias" % i] = sd["bias"].double()
        return out
    sd, x, dy = _inputs(case, seed)
    # the layer computes with bf16 activations and the bf16 decoded weight
    w = _dense(sd).to(torch.bfloat16).double()
    x, dy = x.to(torch.bfloat16).double(), dy.to(torch.bfloat16).double()
    bias = sd["bias"].double() if "bias" in sd else None
    if kind == "conv":
        geom = dict(kernel_size=case["kernel"], padding=case["kernel"] // 2, stride=case["stride"])
        out = _conv_out(case)
        cols = F.unfold(x, **geom).transpose(1, 2).reshape(-1, w.shape[1])
        rows = dy.permute(0, 2, 3, 1).reshape(-1, w.shape[0])
        y = (cols @ w.T + bias).view(case["batch"], out, out, -1).permute(0, 3, 1, 2)
        dx = None
        if case["input_grad"]:
            dcols = (rows @ w).view(case["batch"], out * out, -1).transpose(1, 2)
            dx = F.fold(dcols, (case["hw"], case["hw"]), **geom)
    else:
        cols, rows = x, dy
        y = cols @ w.T if bias is None else cols @ w.T + bias
        dx = None if kind == "forward" else rows @ w
    if kind == "forward":
        return y
    g2 = (rows.T @ cols) ** 2
    return {"y": y, "dx": dx, "db": None if bias is None else rows.sum(0), "words": None, "row_exp": None,
            "col_exp": None, "v_row": BETA2 * sd["v_row"].double() + (1 - BETA2) * g2.sum(1),
            "v_col": BETA2 * sd["v_col"].double() + (1 - BETA2) * g2.sum(0)}
