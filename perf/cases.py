"""The calls this framework is timed and compared on: sizes, inputs, the call, its work, its tolerance, its float64 value.

Six groups of public entry points: attention (forward, forward + backward), the attention prologue, cross-entropy, the
token embedding, AdamW and Muon.  ``listed`` holds the sizes of the workloads and training defaults this repository is
written for; ``draw`` takes further sizes from the same ranges.
"""
import math

import numpy as np
import torch

import femtochat_amd as F
from femtochat_amd import workloads as W
from femtochat_amd.optim import polar_express_grouped_, polar_workspace_bytes

DEV = "cuda"


def listed():
    return [
        # The smallest call: the README's toy GPT (fp32, 2 x 4 tokens), one training step of its attention through autograd.
        # Only launches and host work count.
        dict(name="toy_step", kind="attention", mode="exact", entry="autograd", inputs="fp32",
             B=2, T=4, H=2, Hkv=1, D=16, left=-1, positions="linear"),
        # One layer of the training script's default model (n_embed 512, 8 heads of 64, 4 x 2048 tokens), through autograd.
        dict(name="small_model_step", kind="attention", mode="fast", entry="autograd", inputs="bf16",
             B=4, T=2048, H=8, Hkv=8, D=64, left=-1, positions="none"),
        # The headline layer: n_embed 1280, GQA 2:1, 16 x 2048 tokens, into buffers and workspaces the caller keeps.
        dict(name="gqa_step", kind="attention", mode="fast", entry="buffers", inputs="bf16",
             B=16, T=2048, H=10, Hkv=5, D=128, left=-1, positions="none"),
        # A sliding-window layer ('S' of 'SSSL': 512 keys) of the 10-head model, through autograd.
        dict(name="window_step", kind="attention", mode="fast", entry="autograd", inputs="bf16",
             B=16, T=2048, H=10, Hkv=10, D=128, left=512, positions="none"),
        # Long context with packed documents (lognormal lengths, mean 400): the document mask.
        dict(name="documents_step", kind="attention", mode="fast", entry="buffers", inputs="bf16",
             B=4, T=8192, H=16, Hkv=8, D=128, left=8192, positions="packed"),
        # fp32 exact mode at a 12-layer model's size, through autograd.
        dict(name="exact_step", kind="attention", mode="exact", entry="autograd", inputs="fp32",
             B=8, T=2048, H=6, Hkv=6, D=128, left=2048, positions="linear"),
        # Evaluation of one sequence of odd length: forward only, fp32 tensors into the default (bf16) path, 96-wide heads
        # (n_embed 768, 8 heads).
        dict(name="eval_ragged", kind="attention", mode="fast", entry="forward", inputs="fp32",
             B=1, T=777, H=8, Hkv=4, D=96, left=-1, positions="none"),
        # The headline layer's rotary embedding + RMS norm on Q and K, forward and backward, positions as a loader of
        # packed documents gives them.
        dict(name="prologue_step", kind="prologue", dtype="bf16", B=16, T=2048, H=10, Hkv=5, D=128, positions="packed"),
        # Loss of a training step: 4 x 2048 tokens over a vocabulary of 2^15, mean, forward and gradient.
        dict(name="loss_step", kind="loss", N=8192, V=32768, ignored=0.0, reduction="mean", index="int64"),
        # Token embedding of the same step (512 wide, bf16 out) and its gradient; token ids as frequent as words of a text.
        dict(name="embedding_step", kind="embedding", N=8192, V=32768, D=512, out="bf16", index="int64"),
        # One AdamW step over 2^26 parameters.
        dict(name="adamw_step", kind="adamw", n=1 << 26),
        # One Muon step over the training model's matrices (8 layers, n_embed 512): gather, Polar Express in bf16, write.
        dict(name="muon_step", kind="muon", n=512, layers=8, ratio=4, compute="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["attention", "prologue", "loss", "embedding", "adamw", "muon"], [50, 10, 10, 10, 8, 12])[0]
    if kind == "attention":
        mode = rng.choices(["fast", "exact"], [3, 1])[0]
        D = rng.choices([16, 32, 48, 64, 80, 96, 112, 128], [2, 2, 1, 8, 2, 2, 1, 10])[0]
        H = rng.choice([1, 2, 4, 6, 8, 10, 12, 16])
        Hkv = H // rng.choice([r for r in (1, 1, 2, 4, 5) if H % r == 0])
        T, B = _log(rng, 4, 8192), _log(rng, 1, 16)
        left = rng.choice([-1, -1, T, min(T, -(-T // 512) * 128), rng.randint(0, T)])
        most = 1.0e11 if mode == "exact" else 3.0e11  # algorithmic FLOPs, so that no draw costs more than the largest above
        while B > 1 and 7.0 * D * H * B * T * T > most:
            B -= 1
        while 7.0 * D * H * B * T * T > most:
            T = T * 3 // 4
        left = min(left, T)
        return dict(kind=kind, mode=mode, entry=rng.choices(["autograd", "buffers", "forward"], [5, 2, 3])[0],
                    inputs="fp32" if mode == "exact" else rng.choices(["bf16", "fp32"], [4, 1])[0],
                    B=B, T=T, H=H, Hkv=Hkv, D=D, left=left, positions=rng.choice(["none", "none", "none", "packed"]))
    if kind == "prologue":
        H = rng.choice([1, 2, 4, 6, 8, 10, 12])
        return dict(kind=kind, dtype=rng.choices(["bf16", "fp32"], [3, 1])[0], B=_log(rng, 1, 16), T=_log(rng, 4, 2048), H=H,
                    Hkv=H // rng.choice([r for r in (1, 2) if H % r == 0]), D=rng.choice([16, 32, 64, 64, 128, 128]),
                    positions=rng.choice(["none", "packed"]))
    if kind == "loss":
        V = rng.choice([8192, 32768, _log(rng, 50, 50257), 50257, 50304])
        return dict(kind=kind, N=_log(rng, 8, min(8192, (1 << 28) // V)), V=V, ignored=rng.choice([0.0, 0.0, 0.1, 0.5]),
                    reduction=rng.choices(["mean", "sum", "none"], [4, 1, 1])[0], index=rng.choice(["int32", "int64"]))
    if kind == "embedding":
        return dict(kind=kind, N=_log(rng, 8, 16384), V=rng.choice([8192, 32768, 50257, _log(rng, 50, 32768)]),
                    D=rng.choice([32, 256, 512, 768, 1000, 1280]), out=rng.choice(["bf16", "fp32"]),
                    index=rng.choice(["int32", "int64"]))
    if kind == "adamw":
        return dict(kind=kind, n=_log(rng, 1000, 1 << 26))
    n, compute = rng.choice([64, 128, 192, 256, 320, 384, 512, 640]), rng.choices(["bf16", "fp32"], [3, 1])[0]
    layers = rng.randint(1, 12)
    while layers > 1 and 300.0 * layers * n ** 3 > (1.2e11 if compute == "fp32" else 3.2e11):
        layers -= 1
    return dict(kind=kind, n=n, layers=layers, ratio=4, compute=compute)


# ---- inputs ---------------------------------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(*shape, device=DEV, generator=g)


def _positions(case, seed):
    """Linear positions, or packed documents of the lengths the long-context workload has."""
    B, T = case["B"], case["T"]
    if case["positions"] == "none":
        return None
    if case["positions"] == "linear":
        p = np.tile(np.arange(T, dtype=np.int32), (B, 1))
    else:
        p = W.document_positions(T, B, seed, mean=400, sigma=1.0, cap=4096)
    return torch.from_numpy(p).to(DEV)


def _window(case):
    return (case["left"], 0)


def _unit_rms(x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True))


def _attention_inputs(case, seed):
    g = _gen(seed)
    B, T, H, Hkv, D = (case[k] for k in ("B", "T", "H", "Hkv", "D"))
    dt = torch.bfloat16 if case["inputs"] == "bf16" else torch.float32
    Q, K = _unit_rms(_randn(g, B, T, H, D)).to(dt), _unit_rms(_randn(g, B, T, Hkv, D)).to(dt)  # as the prologue leaves them
    V, dO = _randn(g, B, T, Hkv, D).to(dt), (0.1 * _randn(g, B, T, H, D)).to(dt)
    return Q, K, V, dO


def _prepare_attention(case, seed):
    Q, K, V, dO = _attention_inputs(case, seed)
    s = dict(window=_window(case), positions=_positions(case, seed), A=F.MFMAExact() if case["mode"] == "exact" else F.MFMAFast())
    if case["entry"] == "buffers":
        # a program with buffers of its own converts its tensors once and keeps outputs and workspaces
        Q, K, V = F.attention_inputs(s["A"], Q, K, V)
        s.update(O=torch.empty_like(dO), l=torch.empty(case["B"], case["H"], case["T"], device=DEV),
                 m=torch.empty(case["B"], case["H"], case["T"], device=DEV),
                 dQ=torch.empty(Q.shape, device=DEV, dtype=dO.dtype), dK=torch.empty(K.shape, device=DEV, dtype=dO.dtype),
                 dV=torch.empty(V.shape, device=DEV, dtype=dO.dtype))
        n = F.forward_workspace_bytes(s["A"], Q, K, positions=s["positions"])
        s["fwd_ws"] = torch.empty(n, dtype=torch.uint8, device=DEV) if n else None
        n = F.backward_workspace_bytes(s["A"], Q, K, positions=s["positions"], dout_dtype=dO.dtype)
        s["bwd_ws"] = torch.empty(n, dtype=torch.uint8, device=DEV)
    if case["entry"] == "autograd":
        Q, K, V = (x.requires_grad_(True) for x in (Q, K, V))
    s.update(Q=Q, K=K, V=V, dO=dO)
    return s


def _run_attention(case, s):
    if case["entry"] == "forward":
        return {"O": F.attention(s["A"], s["Q"], s["K"], s["V"], s["window"], positions=s["positions"])}
    if case["entry"] == "autograd":
        leaves = (s["Q"], s["K"], s["V"])
        O = F.AttentionFunction.apply(*leaves, s["window"], s["A"], s["positions"])
        dQ, dK, dV = torch.autograd.grad(O, leaves, s["dO"])
        return {"O": O, "dQ": dQ, "dK": dK, "dV": dV}
    F.attention_(s["A"], s["O"], s["l"], s["m"], s["Q"], s["K"], s["V"], s["window"], positions=s["positions"], workspace=s["fwd_ws"])
    F.delta_attention_(s["A"], s["dQ"], s["dK"], s["dV"], s["dO"], s["Q"], s["K"], s["V"], s["O"], s["l"], s["m"], s["window"],
                       positions=s["positions"], accumulate=False, workspace=s["bwd_ws"])
    return {"O": s["O"], "dQ": s["dQ"], "dK": s["dK"], "dV": s["dV"]}


def _rope(case, seed):
    g = _gen(seed)
    dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    B, T, D = case["B"], case["T"], case["D"]
    X = [_randn(g, B, T, h, D).to(dt) for h in (case["H"], case["Hkv"])]
    dY = [(0.1 * _randn(g, B, T, h, D)).to(dt) for h in (case["H"], case["Hkv"])]
    return X, dY, F.rotary_embeddings(max(T, 4096), D, device=DEV), _positions(case, seed)


def _logits(case, seed):
    g = _gen(seed)
    logits = 2.5 * _randn(g, case["N"], case["V"])
    targets = torch.randint(0, case["V"], (case["N"],), device=DEV, generator=g)
    targets[torch.rand(case["N"], device=DEV, generator=g) < case["ignored"]] = -1
    targets[0] = 0  # a batch with no target at all has no mean
    return logits, targets.to(getattr(torch, case["index"])), 1.0 + torch.rand(case["N"], device=DEV, generator=g)


def _tokens(case, seed):
    """Weights, token ids drawn with word frequencies (1 / (rank + 2.7)), and the output's gradient."""
    g = _gen(seed)
    weights = _randn(g, case["V"], case["D"])
    p = 1.0 / (torch.arange(case["V"], device=DEV, dtype=torch.float64) + 2.7)
    tokens = torch.multinomial(p, case["N"], replacement=True, generator=g).to(getattr(torch, case["index"]))
    dy = (0.01 * _randn(g, case["N"], case["D"])).to(torch.bfloat16 if case["out"] == "bf16" else torch.float32)
    return weights, tokens, dy


_ADAMW = dict(alpha=0.02, beta1=0.8, beta2=0.95, eps=1e-10, lam=0.01)


def _adamw(case, seed):
    g = _gen(seed)
    return _randn(g, case["n"]), 0.01 * _randn(g, case["n"]), 0.01 * _randn(g, case["n"]), (0.01 * _randn(g, case["n"])).square()


def _stack_shapes(case):
    """(count, n, m) torch shapes of the model's matrix groups: attention projections, MLP up, MLP down."""
    n, w, k = case["n"], case["ratio"] * case["n"], case["layers"]
    return [(4 * k, n, n), (k, w, n), (k, n, w)]


def _muon(case, seed):
    g = _gen(seed)
    total = sum(math.prod(s) for s in _stack_shapes(case))
    return 0.05 * _randn(g, total), 1e-3 * _randn(g, total)  # parameters, momentum


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "attention":
        s.update(_prepare_attention(case, seed))
    elif kind == "prologue":
        X, dY, sin_cos, positions = _rope(case, seed)
        s.update(X=[x.requires_grad_(True) for x in X], dY=dY, sin_cos=sin_cos, positions=positions)
    elif kind == "loss":
        logits, targets, dy = _logits(case, seed)
        s.update(logits=logits.requires_grad_(True), targets=targets, dy=dy if case["reduction"] == "none" else None)
    elif kind == "embedding":
        weights, tokens, dy = _tokens(case, seed)
        s.update(weights=weights.requires_grad_(True), tokens=tokens, dy=dy)
    elif kind == "adamw":
        theta, grad, m, v = _adamw(case, seed)
        opt = F.AdamW(theta, t=9, **_ADAMW)
        opt.m.copy_(m)
        opt.v.copy_(v)
        s.update(theta=theta, grad=grad, opt=opt)
    else:
        s["theta"], s["momentum"] = _muon(case, seed)
        shapes = _stack_shapes(case)
        s["stacks"] = [torch.empty(sh, device=DEV) for sh in shapes]
        s["compute"] = torch.bfloat16 if case["compute"] == "bf16" else torch.float32
        s["ws"] = [torch.empty(polar_workspace_bytes(G, 5, s["compute"]), dtype=torch.uint8, device=DEV) for G in s["stacks"]]
        s["offsets"], at = [], 0
        for k, a, b in shapes:
            s["offsets"].append(at + a * b * torch.arange(k, device=DEV, dtype=torch.int64))
            at += k * a * b
        s["eta"], s["lam"] = torch.full((1,), 0.02, device=DEV), torch.full((1,), 0.1, device=DEV)
    return s


# ---- the calls ------------------------------------------------------------------------------------------------------


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "attention":
        return _run_attention(case, s)
    if kind == "prologue":
        Y = [F.AttentionPrologueFunction.apply(x, *s["sin_cos"], s["positions"]) for x in s["X"]]
        dX = torch.autograd.grad(Y, s["X"], s["dY"])
        return {"Y": Y, "dX": dX}
    if kind == "loss":
        loss = F.CrossEntropyFunction.apply(s["logits"], s["targets"], -1, case["reduction"])
        (grad,) = torch.autograd.grad(loss, (s["logits"],), s["dy"])
        return {"loss": loss, "grad": grad}
    if kind == "embedding":
        y = F.EmbeddingFunction.apply(s["weights"], s["tokens"], s["dy"].dtype)
        (grad,) = torch.autograd.grad(y, (s["weights"],), s["dy"])
        return {"y": y, "grad": grad}
    if kind == "adamw":
        s["opt"](s["theta"], s["grad"])
        return {"theta": s["theta"], "m": s["opt"].m, "v": s["opt"].v}
    for G, offsets in zip(s["stacks"], s["offsets"]):
        F.gather_(G, s["momentum"], offsets, validate=False)
    polar_express_grouped_(s["stacks"], 5, s["ws"], s["compute"])
    for G, offsets in zip(s["stacks"], s["offsets"]):
        F.muon_update_(s["theta"], G, s["eta"], s["lam"], offsets, validate=False)
    return {"X": s["stacks"], "theta": s["theta"]}


# ---- work and tolerance ---------------------------------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "attention":
        B, T, H, Hkv, D = (case[k] for k in ("B", "T", "H", "Hkv", "D"))
        size = 2 if case["inputs"] == "bf16" else 4
        p = None if case["positions"] != "packed" else W.document_positions(T, B, 1, mean=400, sigma=1.0, cap=4096)
        pairs = W.visible_pairs(T, B, H, _window(case), p)
        qo, kv = B * T * H * D * size, B * T * Hkv * D * size
        if case["entry"] == "forward":
            return {"bytes": 2 * qo + 2 * kv, "flops": 4 * D * pairs}
        return {"bytes": 4 * qo + 4 * kv, "flops": 14 * D * pairs}
    if kind == "prologue":
        n = case["B"] * case["T"] * (case["H"] + case["Hkv"]) * case["D"]
        return {"bytes": n * (2 if case["dtype"] == "bf16" else 4) * 4, "flops": 30 * n}
    if kind == "loss":
        n = case["N"] * case["V"]
        return {"bytes": 8 * n, "flops": 6 * n}
    if kind == "embedding":
        size = 2 if case["out"] == "bf16" else 4
        n = case["N"] * case["D"]
        return {"bytes": n * (4 + 2 * size) + 4 * case["V"] * case["D"], "flops": n}
    if kind == "adamw":
        return {"bytes": 28 * case["n"], "flops": 15 * case["n"]}
    flops, total = 0.0, 0
    for k, a, b in _stack_shapes(case):
        lo, hi = min(a, b), max(a, b)
        flops += 5.0 * k * (4.0 * lo * lo * hi + 2.0 * lo ** 3)
        total += k * a * b
    return {"bytes": 16 * total, "flops": flops}


def tolerance(case):
    """About four times the difference from the float64 value (2-norm), or from the same sums in another order."""
    kind = case["kind"]
    if kind == "attention":
        return {"rel": 1.2e-2} if case["mode"] == "fast" else {"rel": 4e-6}
    if kind == "prologue":
        return {"rel": 1.5e-2} if case["dtype"] == "bf16" else {"rel": 2e-6}
    if kind == "loss":
        return {"rel": 2e-6}
    if kind == "embedding":
        return {"rel": 2e-6}
    if kind == "adamw":
        return {"rel": 1e-6}
    return {"rel": 3e-2} if case["compute"] == "bf16" else {"rel": 4e-5}


# ---- float64 --------------------------------------------------------------------------------------------------------


def _exact_attention(case, seed):
    Q, K, V, dO = (x.double() for x in _attention_inputs(case, seed))
    pos = _positions(case, seed)
    B, T, H, Hkv, D = (case[k] for k in ("B", "T", "H", "Hkv", "D"))
    q = torch.arange(T, device=DEV)[:, None]
    k = torch.arange(T, device=DEV)[None, :]
    hidden0 = (k > q) if case["left"] < 0 else (k > q) | (k < q - case["left"])
    O, dQ, dK, dV = torch.zeros_like(Q), torch.zeros_like(Q), torch.zeros_like(K), torch.zeros_like(V)
    for b in range(B):
        hidden = hidden0 if pos is None else hidden0 | (k < q - pos[b].long()[:, None])
        for h in range(H):
            j = h // (H // Hkv)
            Qh, Kh, Vh, dOh = (x.contiguous() for x in (Q[b, :, h], K[b, :, j], V[b, :, j], dO[b, :, h]))
            P = (Qh @ Kh.t().contiguous()) / math.sqrt(D)
            P = torch.softmax(P.masked_fill_(hidden, -math.inf), -1)  # every row sees at least its own key
            O[b, :, h] = P @ Vh
            if case["entry"] == "forward":
                continue
            dV[b, :, j] += P.t().contiguous() @ dOh
            dP = dOh @ Vh.t().contiguous()
            dP -= (dOh * O[b, :, h]).sum(-1, keepdim=True)
            P *= dP
            P /= math.sqrt(D)
            dQ[b, :, h] = P @ Kh
            dK[b, :, j] += P.t().contiguous() @ Qh
    return {"O": O} if case["entry"] == "forward" else {"O": O, "dQ": dQ, "dK": dK, "dV": dV}


def _exact_prologue(case, seed):
    X, dY, (sin, cos), pos = _rope(case, seed)
    T, d = case["T"], case["D"] // 2
    at = torch.arange(T, device=DEV).expand(case["B"], T) if pos is None else pos.long()
    s, c = sin.double()[at][:, :, None, :], cos.double()[at][:, :, None, :]
    out = {"Y": [], "dX": []}
    eps = float(torch.finfo(torch.bfloat16 if case["dtype"] == "bf16" else torch.float32).eps)
    for x, g in zip(X, dY):
        x, g = x.detach().double(), 1.2 * g.double()
        u = torch.cat([x[..., :d] * c + x[..., d:] * s, x[..., d:] * c - x[..., :d] * s], -1)
        r = torch.sqrt(u.square().mean(-1, keepdim=True) + eps)
        y = u / r
        out["Y"].append(1.2 * y)
        g = (g - y * (g * y).mean(-1, keepdim=True)) / r
        out["dX"].append(torch.cat([g[..., :d] * c - g[..., d:] * s, g[..., :d] * s + g[..., d:] * c], -1))
    return out


def _exact_loss(case, seed):
    logits, targets, dy = _logits(case, seed)
    valid = targets != -1
    count = int(valid.sum())
    losses, grad = torch.zeros(case["N"], dtype=torch.float64, device=DEV), torch.empty_like(logits, dtype=torch.float64)
    for at in range(0, case["N"], 1024):
        x, t, ok = logits[at:at + 1024].double(), targets[at:at + 1024].long().clamp_min(0)[:, None], valid[at:at + 1024]
        lse = torch.logsumexp(x, -1, keepdim=True)
        losses[at:at + 1024] = (lse - x.gather(1, t))[:, 0] * ok
        p = torch.exp(x - lse)
        p.scatter_add_(1, t, -torch.ones_like(t, dtype=torch.float64))
        w = dy[at:at + 1024].double() if case["reduction"] == "none" else 1.0 / count if case["reduction"] == "mean" else 1.0
        grad[at:at + 1024] = p * (ok * w)[:, None]
    loss = losses if case["reduction"] == "none" else losses.sum() / (count if case["reduction"] == "mean" else 1)
    return {"loss": loss, "grad": grad}


def _exact_muon(case, seed):
    theta, momentum = (x.double() for x in _muon(case, seed))
    X, at = [], 0
    # the published Polar Express coefficients, one (a, b, c) per step
    steps = [(8.156554524902461, -22.48329292557795, 15.878769915207462), (4.042929935166739, -2.808917465908714, 0.5000178451051316),
             (3.8916678022926607, -2.772484153217685, 0.5060648178503393), (3.285753657755655, -2.3681294933425376, 0.46449024233003106),
             (2.3465413258596377, -1.7097828382687081, 0.42323551169305323)]
    for k, n, m in _stack_shapes(case):
        G = momentum[at:at + k * n * m].reshape(k, n, m)
        at += k * n * m
        out = torch.empty_like(G)
        for j in range(k):
            g = G[j] if n <= m else G[j].t().contiguous()
            x = g / (1.01 * g.norm() + 1e-6)
            for a, b, c in steps:
                A = x @ x.t().contiguous()
                x = a * x + (b * A + c * (A @ A)) @ x
            out[j] = x if n <= m else x.t()
        X.append(out)
    flat = torch.cat([x.reshape(-1) for x in X])
    decay = torch.where(flat * theta >= 0, 0.02 * 0.1 * theta, torch.zeros_like(theta))
    return {"X": X, "theta": theta - 0.02 * flat - decay}


def exact(case, seed):
    kind = case["kind"]
    if kind == "attention":
        return _exact_attention(case, seed)
    if kind == "prologue":
        return _exact_prologue(case, seed)
    if kind == "loss":
        return _exact_loss(case, seed)
    if kind == "embedding":
        weights, tokens, dy = _tokens(case, seed)
        tokens = tokens.long()
        return {"y": weights.double()[tokens], "grad": torch.zeros_like(weights, dtype=torch.float64).index_add_(0, tokens, dy.double())}
    if kind == "adamw":
        theta, g, m, v = (x.double() for x in _adamw(case, seed))
        a, b1, b2, eps, lam = _ADAMW.values()
        m = b1 * m + (1 - b1) * g
        v = b2 * v + (1 - b2) * g.square()
        theta = theta * (1 - a * lam) - a * (m / (1 - b1 ** 10)) / ((v / (1 - b2 ** 10)).sqrt() + eps)
        return {"theta": theta, "m": m, "v": v}
    return _exact_muon(case, seed)
