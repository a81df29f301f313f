"""The work that a training program has this framework do, as timed cases: the GRPO loss
head on logits, log-probs alone, the fused LM head, the rollout sampler, the optimizer
step around them and the weight payload, each through its public entry point.

Inputs are made on the GPU from the seed alone, with torch; `exact` restates each path in
64 bits with torch alone. Calls use the entry points' defaults, so a pass ends as a user's
call does. A training loop keeps its output buffers, so `prepare` makes them.
"""
from __future__ import annotations

import math

import torch

from pcp_amd import formats, grpo, step

DEV = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
QWEN_VOCAB = 151936      # the vocabulary of configurations 2 to 5
GPT_VOCAB = 50257        # odd: its 16-bit rows start off 16 bytes
QWEN05_PARAMS = 494032768


def listed() -> list[dict]:
    return [
        # Configuration 1: the toy model's step, where launches and latency are the time.
        dict(name="loss_toy", kind="loss", mode="clip_kl", dtype="f32", S=8, T=128, V=1024, group=4,
             lengths="uniform", shifted=False, zero_fill=True),
        # A micro-batch: one group of short answers over the real vocabulary, fewer rows than the GPU has CUs.
        dict(name="loss_micro", kind="loss", mode="clip_kl", dtype="bf16", S=4, T=16, V=QWEN_VOCAB, group=4,
             lengths="uniform", shifted=False, zero_fill=True),
        # Two prompts of configuration 2's batch: the ordinary step over the real vocabulary.
        dict(name="loss_vocab152k", kind="loss", mode="clip_kl", dtype="bf16", S=16, T=512, V=QWEN_VOCAB, group=8,
             lengths="uniform", shifted=False, zero_fill=True),
        # The reference graph itself: f32 logits, REINFORCE, logits[:, :-1] against ids[:, 1:].
        dict(name="loss_f32_shifted", kind="loss", mode="reinforce", dtype="f32", S=4, T=128, V=QWEN_VOCAB, group=4,
             lengths="uniform", shifted=True, zero_fill=True),
        # An odd vocabulary with long-tailed lengths, dead rows left alone.
        dict(name="loss_ragged", kind="loss", mode="clip_kl", dtype="bf16", S=16, T=512, V=GPT_VOCAB, group=8,
             lengths="lognormal", shifted=False, zero_fill=False),
        # Scoring a batch of rollouts under the policy and the reference model, forward only.
        dict(name="logprob", kind="logprob", dtype="bf16", S=8, T=64, V=QWEN_VOCAB, ref=True),
        # The fused LM head of a 0.5B model (H = 896) on one small group.
        dict(name="lmhead_small", kind="lmhead", mode="clip_kl", S=4, T=128, H=896, V=QWEN_VOCAB, group=4, norm=False,
             exact_bf16=False),
        # With the decoder's final norm fused, REINFORCE, an odd vocabulary, a middle-sized batch.
        dict(name="lmhead_norm", kind="lmhead", mode="reinforce", S=8, T=256, H=2048, V=GPT_VOCAB, group=8, norm=True,
             exact_bf16=False),
        # Configuration 5: 16,384 tokens at H = 4096, the largest call.
        dict(name="lmhead_large", kind="lmhead", mode="clip_kl", S=32, T=512, H=4096, V=QWEN_VOCAB, group=8,
             norm=False, exact_bf16=False),
        # One decode step of configuration 2's 64 rollouts.
        dict(name="sample", kind="sample", dtype="f32", R=64, V=QWEN_VOCAB, temperature=1.0),
        # What a step does with the model's gradients: their statistics tensor by tensor (a 0.5B model's 290
        # tensors), then the Nesterov update of the flat parameters with their bf16 copy.
        dict(name="optimizer", kind="optimizer", hidden=896, ff=4864, kv=128, layers=24, V=QWEN_VOCAB),
        # The updated weights as the base64 payload that workers get, and back.
        dict(name="wire", kind="wire", nbytes=4 * QWEN05_PARAMS),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _vocab(rng) -> int:
    return rng.choice([QWEN_VOCAB, GPT_VOCAB, _log_int(rng, 1000, 262144), 8 * _log_int(rng, 125, 32768)])


def draw(rng) -> dict:
    kind = rng.choice(["loss", "loss", "loss", "logprob", "lmhead", "lmhead", "sample", "optimizer", "wire"])
    if kind in ("loss", "logprob"):
        dtype = rng.choice(["bf16", "bf16", "f32", "f16" if kind == "logprob" else "bf16"])
        V = _vocab(rng)
        group = rng.choice([1, 2, 4, 8, 16]) if kind == "logprob" else rng.choice([2, 4, 8, 16])
        # Up to the largest listed logits (2.5 GB).
        tokens = _log_int(rng, 4 * group, max(4 * group, min(32768, 2489319424 // (V * DTYPES[dtype].itemsize))))
        S = group * _log_int(rng, 1, max(1, min(8, tokens // (4 * group))))
        T = max(2, tokens // S)
        if kind == "logprob":
            return dict(kind=kind, dtype=dtype, S=S, T=T, V=V, ref=rng.random() < 0.5)
        return dict(kind=kind, mode=rng.choice(["clip_kl", "clip_kl", "reinforce"]), dtype=dtype, S=S, T=T, V=V,
                    group=group, lengths=rng.choice(["uniform", "lognormal"]), shifted=rng.random() < 0.3,
                    zero_fill=rng.random() < 0.7)
    if kind == "lmhead":
        H = 64 * _log_int(rng, 4, 64)
        V = rng.choice([QWEN_VOCAB, GPT_VOCAB, _log_int(rng, 1000, QWEN_VOCAB)])
        group = rng.choice([2, 4, 8])
        # Up to the largest listed call's products.
        tokens = _log_int(rng, 8 * group, max(8 * group, min(16384, 16384 * 4096 * QWEN_VOCAB // (H * V))))
        S = group * _log_int(rng, 1, max(1, min(8, tokens // (8 * group))))
        return dict(kind=kind, mode=rng.choice(["clip_kl", "clip_kl", "reinforce"]), S=S, T=max(2, tokens // S), H=H,
                    V=V, group=group, norm=rng.random() < 0.5, exact_bf16=rng.random() < 0.2)
    if kind == "sample":
        return dict(kind=kind, dtype=rng.choice(["f32", "bf16"]), R=_log_int(rng, 1, 512), V=_vocab(rng),
                    temperature=rng.choice([0.0, 0.7, 1.0]))
    if kind == "optimizer":
        hidden = 2 * _log_int(rng, 32, 448)
        return dict(kind=kind, hidden=hidden, ff=_log_int(rng, 2 * hidden, 5 * hidden + 384), kv=max(8, hidden // 7),
                    layers=_log_int(rng, 2, 24), V=_log_int(rng, 1000, QWEN_VOCAB))
    return dict(kind=kind, nbytes=_log_int(rng, 1000, 4 * QWEN05_PARAMS))


# ---- inputs ---------------------------------------------------------------------------


def _gen(seed: int, salt: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed * 64 + salt)


def _lengths(kind: str, S: int, T: int, seed: int) -> torch.Tensor:
    g = torch.Generator().manual_seed(seed * 64 + 1)
    if kind == "lognormal":   # configuration 4's shape: median T / 8, sigma 1
        x = torch.exp(torch.randn(S, generator=g) + math.log(T / 8)).round().clamp(1, T)
    else:                     # configurations 2 and 3: from T / 8 to T
        lo = max(1, T // 8)
        x = torch.randint(lo, T + 1, (S,), generator=g)
    return x.to(torch.int64)


def _live_share(kind: str) -> float:
    return 0.21 if kind == "lognormal" else 0.5625


def _group_advantages(rewards: torch.Tensor, group: int) -> torch.Tensor:
    r = rewards.double()
    out = torch.empty_like(r)
    for i in range(0, r.numel(), group):
        b = r[i:i + group]
        out[i:i + group] = (b - b.mean()) / (((b - b.mean()) ** 2).mean().sqrt() + 1e-8)
    return out


def _draw_tokens(logits: torch.Tensor, g: torch.Generator) -> tuple[torch.Tensor, torch.Tensor]:
    """One token per row of logits [n, V] drawn from its softmax (Gumbel-max), and its log-prob."""
    ids, lps = [], []
    n = max(1, (1 << 27) // logits.shape[1])
    for i in range(0, logits.shape[0], n):
        x = logits[i:i + n].float()
        u = torch.rand(x.shape, device=DEV, generator=g).clamp_(1e-20, 1 - 1e-7)
        t = (x - torch.log(-torch.log(u))).argmax(-1)
        ids.append(t)
        lps.append(x.gather(1, t[:, None])[:, 0] - torch.logsumexp(x, -1))
    return torch.cat(ids), torch.cat(lps)


def _randn(shape, dtype, std: float, g: torch.Generator) -> torch.Tensor:
    return torch.randn(shape, dtype=dtype, device=DEV, generator=g).mul_(std)


def _token_inputs(case: dict, seed: int, logp: torch.Tensor) -> dict:
    """Mask, rewards or advantages and old log-probs of [S, T] tokens whose log-probs are logp: the policy has
    moved towards the better answers since the rollout."""
    S, T = logp.shape
    lengths = _lengths(case.get("lengths", "uniform"), S, T, seed).to(DEV)
    mask = (torch.arange(T, device=DEV)[None, :] < lengths[:, None]).float()
    rewards = torch.rand(S, device=DEV, generator=_gen(seed, 2))
    d = {"mask": mask}
    if case["mode"] == "clip_kl":
        adv = _group_advantages(rewards, case["group"]).float()
        noise = torch.randn(S, T, device=DEV, generator=_gen(seed, 3))
        d.update(rewards=rewards, old_logp=(logp - 0.1 * adv[:, None] + 0.1 * noise).contiguous())
    else:                     # REINFORCE on the rewards themselves
        d.update(advantages=rewards)
    return d


def _logit_inputs(case: dict, seed: int, want_ref: bool) -> tuple:
    S, T, V, dt = case["S"], case["T"], case["V"], DTYPES[case["dtype"]]
    std, std_r = (2.0, 0.05) if V <= 4096 else (3.0, 0.1)   # configuration 1, configurations 2 to 4
    g = _gen(seed, 0)
    logits = _randn((S, T, V), dt, std, g)
    ref = None
    if want_ref:
        ref = torch.empty_like(logits)
        for s in range(S):
            torch.add(logits[s], _randn((T, V), dt, std_r, g), out=ref[s])
    ids, logp = _draw_tokens(logits.view(S * T, V), g)
    return logits, ref, ids.view(S, T), logp.view(S, T)


def _prepare_loss(case: dict, seed: int) -> dict:
    clip = case["mode"] == "clip_kl"
    logits, ref, ids, logp = _logit_inputs(case, seed, clip)
    if case["shifted"]:       # row t scores token t + 1
        ids, logp = ids.roll(1, 1).contiguous(), logp.roll(1, 1).contiguous()
    S, T, V = logits.shape
    f32 = dict(dtype=torch.float32, device=DEV)
    out = grpo.GrpoOutputs(
        loss=torch.zeros((), **f32), dlogits=torch.zeros_like(logits), logp=torch.zeros((S, T), **f32),
        ref_logp=torch.zeros((S, T), **f32) if clip else None, token_loss=torch.zeros((S, T), **f32),
        advantages=torch.zeros(S, **f32))
    kw = dict(group_size=case["group"], loss_mode=grpo.LossMode.GRPO_CLIP_KL if clip else grpo.LossMode.REINFORCE,
              ref_logits=ref, zero_fill=case["zero_fill"], outputs=out)
    if case["shifted"]:
        kw.update(rows=T - 1, tok_offset=1)
    t = _token_inputs(case, seed, logp)
    return {"logits": logits, "ids": ids, "mask": t.pop("mask"), "kw": {**kw, **t}}


def _run_loss(s: dict) -> dict:
    o = grpo.grpo_loss_fwd_bwd(s["logits"], s["ids"], s["mask"], **s["kw"])
    return {"loss": o.loss, "dlogits": o.dlogits, "logp": o.logp, "ref_logp": o.ref_logp, "token_loss": o.token_loss,
            "advantages": o.advantages}


def _prepare_lmhead(case: dict, seed: int) -> dict:
    S, T, H, V = case["S"], case["T"], case["H"], case["V"]
    clip, norm = case["mode"] == "clip_kl", case["norm"]
    g = _gen(seed, 0)
    std_w = 0.02 * math.sqrt(4096 / H)   # logits of configuration 5's spread at any H
    weight = _randn((V, H), torch.bfloat16, std_w, g)
    ref = weight + _randn((V, H), torch.bfloat16, std_w / 10, g) if clip else None
    f32 = dict(dtype=torch.float32, device=DEV)
    gamma = None
    if norm:                  # a residual stream of its own scale per row
        gamma = 1.0 + 0.1 * torch.randn(H, generator=g, **f32)
        hidden = (_randn((S * T, H), torch.float32, 1.0, g) *
                  torch.exp(torch.randn(S * T, 1, generator=g, **f32))).to(torch.bfloat16)
        operand = _norm_rows(hidden, gamma)[0].to(torch.bfloat16)
    else:
        hidden = operand = _randn((S * T, H), torch.bfloat16, 1.0, g)
    ids, logp = zip(*(_draw_tokens(operand[i:i + 2048] @ weight.t(), g) for i in range(0, S * T, 2048)))
    ids, logp = torch.cat(ids).view(S, T), torch.cat(logp).view(S, T)
    out = grpo.LmheadOutputs(
        loss=torch.zeros((), **f32), logp=torch.zeros((S, T), **f32),
        ref_logp=torch.zeros((S, T), **f32) if clip else None, token_loss=torch.zeros((S, T), **f32),
        advantages=torch.zeros(S, **f32), dhidden=torch.zeros((S * T, H), **f32),
        dweight=torch.zeros((V, H), **f32), dnorm_weight=torch.zeros(H, **f32) if norm else None)
    t = _token_inputs(case, seed, logp)
    kw = dict(ref_weight=ref, group_size=case["group"], norm_weight=gamma, exact_bf16=case["exact_bf16"], outputs=out,
              loss_mode=grpo.LossMode.GRPO_CLIP_KL if clip else grpo.LossMode.REINFORCE)
    return {"hidden": hidden, "weight": weight, "ids": ids, "mask": t.pop("mask"), "kw": {**kw, **t}}


def _run_lmhead(s: dict) -> dict:
    o = grpo.lmhead_fwd_bwd(s["hidden"], s["weight"], s["ids"], s["mask"], **s["kw"])
    return {"loss": o.loss, "logp": o.logp, "ref_logp": o.ref_logp, "token_loss": o.token_loss,
            "advantages": o.advantages, "dhidden": o.dhidden, "dweight": o.dweight, "dnorm": o.dnorm_weight}


def _tensor_counts(case: dict) -> list[int]:
    """The decoder's parameter tensors in named_parameters() order (tied head)."""
    h, ff, kv = case["hidden"], case["ff"], case["kv"]
    layer = [h * h, h, kv * h, kv, kv * h, kv, h * h, ff * h, ff * h, h * ff, h, h]
    return [case["V"] * h] + layer * case["layers"] + [h]


def _prepare_optimizer(case: dict, seed: int) -> dict:
    counts = _tensor_counts(case)
    n, g = sum(counts), _gen(seed, 0)
    params = _randn(n, torch.float32, 0.02, g)
    grads = _randn(n, torch.float32, 1e-3, g)
    opt = step.Nesterov(counts)
    velocity = _randn(n, torch.float32, 1e-3, g)
    opt.update_flat(params, velocity)   # the step before left its velocities
    return {"params": params, "grads": grads, "tensors": list(grads.split(counts)), "opt": opt,
            "shadow": torch.zeros(n, dtype=torch.bfloat16, device=DEV)}


def _run_optimizer(s: dict) -> dict:
    stats = step.grad_stats(s["tensors"])
    s["opt"].update_flat(s["params"], s["grads"], s["shadow"])
    return {"stats": stats, "params": s["params"], "shadow": s["shadow"]}


def prepare(case: dict, seed: int):
    kind = case["kind"]
    if kind == "loss":
        return kind, _prepare_loss(case, seed)
    if kind == "logprob":
        logits, ref, ids, _ = _logit_inputs(case, seed, case["ref"])
        S, T = ids.shape
        mask = (torch.arange(T, device=DEV)[None, :] < _lengths("uniform", S, T, seed).to(DEV)[:, None]).float()
        return kind, {"logits": logits, "ref": ref, "ids": ids, "mask": mask}
    if kind == "lmhead":
        return kind, _prepare_lmhead(case, seed)
    if kind == "sample":
        R, V, dt = case["R"], case["V"], DTYPES[case["dtype"]]
        g = _gen(seed, 0)
        rows = _randn((R, (V + 7) // 8 * 8), dt, 3.0, g)   # a row pitch of 16 bytes
        return kind, {"logits": rows[:, :V], "u": torch.rand(R, device=DEV, generator=g), "t": case["temperature"]}
    if kind == "optimizer":
        return kind, _prepare_optimizer(case, seed)
    n = case["nbytes"]
    m = (n + 3) // 4
    data = _randn(m, torch.float32, 0.02, _gen(seed, 0)).view(torch.uint8)[:n]   # f32 weights
    return kind, {"data": data, "text": torch.zeros((n + 2) // 3 * 4, dtype=torch.uint8, device=DEV),
                  "back": torch.zeros((n + 2) // 3 * 3, dtype=torch.uint8, device=DEV)}


def run(state):
    kind, s = state
    if kind == "loss":
        return _run_loss(s)
    if kind == "logprob":
        lp, lr = grpo.logprob_fwd(s["logits"], s["ids"], s["ref"], mask=s["mask"])
        return {"logp": lp, "ref_logp": lr}
    if kind == "lmhead":
        return _run_lmhead(s)
    if kind == "sample":
        return {"ids": step.sample_tokens(s["logits"], s["t"], s["u"])}
    if kind == "optimizer":
        return _run_optimizer(s)
    text = formats.b64encode(s["data"], out=s["text"])
    return {"text": text, "data": formats.b64decode(text, out=s["back"])}


# ---- what a pass cannot do without -------------------------------------------------------


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("loss", "logprob"):
        S, T, V, e = case["S"], case["T"], case["V"], DTYPES[case["dtype"]].itemsize
        if kind == "logprob":
            reads = 2 if case["ref"] else 1
            live = S * T * _live_share("uniform")
            return {"bytes": live * reads * V * e + S * T * (12 + 4 * reads), "flops": live * reads * V * 4}
        reads = 2 if case["mode"] == "clip_kl" else 1
        rows = S * (T - 1 if case["shifted"] else T)
        live = rows * _live_share(case["lengths"])
        written = S * T if case["zero_fill"] else live
        return {"bytes": (live * reads + written) * V * e + S * T * 28, "flops": live * V * (4 * reads + 4)}
    if kind == "lmhead":
        N, H, V = case["S"] * case["T"], case["H"], case["V"]
        models = 2 if case["mode"] == "clip_kl" else 1
        live = N * _live_share("uniform")
        return {"bytes": models * 2 * V * H + 4 * V * H + live * 2 * H + N * 4 * H + N * 28,
                "flops": (models + 2) * 2 * live * H * V}
    if kind == "sample":
        n = case["R"] * case["V"]
        return {"bytes": n * DTYPES[case["dtype"]].itemsize + case["R"] * 12, "flops": 4 * n}
    if kind == "optimizer":
        n = sum(_tensor_counts(case))
        return {"bytes": 26 * n, "flops": 8 * n}   # g for the statistics; p, v, g in and p, v, bf16 p out
    n = case["nbytes"]
    return {"bytes": 2 * (n + (n + 2) // 3 * 4), "flops": 0}


def tolerance(case: dict):
    kind = case["kind"]
    if kind in ("sample", "wire"):
        return "exact"
    if kind == "loss":
        # f32: an exponential and 32-bit sums over the vocabulary; 16-bit dlogits: their rounding.
        return {"rel": {"f32": 1e-5, "bf16": 1e-2}[case["dtype"]]}
    if kind == "logprob":
        return {"rel": 1e-6}
    if kind == "lmhead":
        return {"rel": 1e-2}   # bf16 dlogits and f16 softmax terms into the gradients
    return {"rel": 1e-7}       # elementwise f32 in a fixed order; statistics in 64 bits


# ---- 64 bits ---------------------------------------------------------------------------


def _norm_rows(h: torch.Tensor, gamma: torch.Tensor) -> tuple:
    """The final RMSNorm with its bf16 roundings: (operand, normalised rows, 1 / rms), in 64 bits."""
    x = h.double()
    r = torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6)
    n = (x * r).to(torch.bfloat16).double()
    return (gamma.double() * n).to(torch.bfloat16).double(), n, r


def _terms(case: dict, kw: dict, mask, adv, lp, lr) -> tuple:
    """(token loss, coefficient, loss) of [S, T] tokens in 64 bits (rows past the last one have mask 0)."""
    m = mask.double()
    L = m.sum(1).clamp(min=1.0)
    scale = m / (m.shape[0] * L)[:, None]
    A = adv[:, None]
    if case["mode"] != "clip_kl":
        tl = -lp * m
        return tl, -A * scale, (tl.sum(1) / L * adv).mean()
    rho = torch.exp(lp - kw["old_logp"].double())
    eps, beta = float(torch.tensor(0.2)), float(torch.tensor(0.04))
    surr = torch.minimum(rho * A, rho.clamp(1 - eps, 1 + eps) * A)
    d = lr - lp
    tl = (-surr + beta * (torch.expm1(d) - d)) * m
    free = torch.where(A >= 0, rho <= 1 + eps, rho >= 1 - eps)
    coef = scale * (torch.where(free, -A * rho, torch.zeros_like(rho)) - beta * torch.expm1(d))
    return tl, coef, (tl.sum(1) / L).mean()


def _exact_loss(case: dict, s: dict) -> dict:
    kw, logits, ids, mask = s["kw"], s["logits"], s["ids"], s["mask"]
    S, T, V = logits.shape
    off = 1 if case["shifted"] else 0
    m = mask.clone()
    m[:, :off] = 0
    adv = kw["advantages"].double() if "advantages" in kw else _group_advantages(kw["rewards"], case["group"])
    models = [logits] + ([kw["ref_logits"]] if kw["ref_logits"] is not None else [])
    lse = torch.zeros(len(models), S, T, dtype=torch.float64, device=DEV)
    lp = torch.zeros_like(lse)
    for k, x in enumerate(models):
        for q in range(S):
            z = x[q, :T - off].double()
            lse[k, q, off:] = torch.logsumexp(z, -1)
            lp[k, q, off:] = z.gather(1, ids[q, off:, None])[:, 0] - lse[k, q, off:]
    live = m > 0
    lp = torch.where(live, lp, torch.zeros_like(lp))
    tl, coef, loss = _terms(case, kw, m, adv, lp[0], lp[-1])
    d = torch.zeros((S, T, V), dtype=torch.float64, device=DEV)
    for q in range(S):
        z = d[q, :T - off]
        torch.exp(logits[q, :T - off].double() - lse[0, q, off:, None], out=z)
        z.mul_(-coef[q, off:, None])
        z.scatter_add_(1, ids[q, off:, None], coef[q, off:, None].contiguous())
    return {"loss": loss, "dlogits": d, "logp": lp[0], "ref_logp": lp[1] if len(models) > 1 else None,
            "token_loss": tl, "advantages": adv}


def _exact_lmhead(case: dict, s: dict) -> dict:
    kw, mask = s["kw"], s["mask"]
    S, T = mask.shape
    N, V = S * T, case["V"]
    adv = kw["advantages"].double() if "advantages" in kw else _group_advantages(kw["rewards"], case["group"])
    y = s["hidden"].double()
    if case["norm"]:
        y, normed, r = _norm_rows(s["hidden"], kw["norm_weight"])
    at = mask.reshape(-1).nonzero()[:, 0]
    ids = s["ids"].reshape(-1)[at]
    n = max(1, (1 << 28) // V)
    lp, lse = [], None
    for w in [s["weight"]] + ([kw["ref_weight"]] if kw["ref_weight"] is not None else []):
        w64 = w.double().t()
        sums, got = [], torch.zeros(N, dtype=torch.float64, device=DEV)
        for i in range(0, at.numel(), n):
            z = y[at[i:i + n]] @ w64
            sums.append(torch.logsumexp(z, -1))
            got[at[i:i + n]] = z.gather(1, ids[i:i + n, None])[:, 0] - sums[-1]
        lse = torch.cat(sums) if lse is None else lse
        lp.append(got.view(S, T))
    tl, coef, loss = _terms(case, kw, mask, adv, lp[0], lp[-1])
    c = coef.reshape(-1)[at]
    w64 = s["weight"].double()
    dy = torch.zeros_like(y)
    dw = torch.zeros_like(w64)
    for i in range(0, at.numel(), n):
        rows = y[at[i:i + n]]
        d = torch.exp(rows @ w64.t() - lse[i:i + n, None]).mul_(-c[i:i + n, None])
        d.scatter_add_(1, ids[i:i + n, None], c[i:i + n, None].contiguous())
        dy[at[i:i + n]] = d @ w64
        dw.addmm_(d.t(), rows)
    dgamma = None
    if case["norm"]:
        dgamma = (dy * normed).sum(0)
        g, h = dy * kw["norm_weight"].double(), s["hidden"].double()
        dy = r * g - h * (r ** 3 / case["H"]) * (g * h).sum(-1, keepdim=True)
    return {"loss": loss, "logp": lp[0], "ref_logp": lp[1] if len(lp) > 1 else None, "token_loss": tl,
            "advantages": adv, "dhidden": dy, "dweight": dw, "dnorm": dgamma}


def exact(case: dict, seed: int):
    kind, s = prepare(case, seed)
    if kind == "loss":
        return _exact_loss(case, s)
    if kind == "logprob":
        got = []
        for x in (s["logits"], s["ref"]):
            if x is None:
                got.append(None)
                continue
            lp = torch.stack([z.double().gather(1, t[:, None])[:, 0] - torch.logsumexp(z.double(), -1)
                              for z, t in zip(x, s["ids"])])
            got.append(torch.where(s["mask"] > 0, lp, torch.zeros_like(lp)))
        return {"logp": got[0], "ref_logp": got[1]}
    if kind == "lmhead":
        return _exact_lmhead(case, s)
    if kind == "optimizer":
        n = sum(_tensor_counts(case))
        g = _gen(seed, 0)
        p, grad, v0 = (_randn(n, torch.float32, std, g).double() for std in (0.02, 1e-3, 1e-3))
        lr, mu = float(torch.tensor(0.01)), float(torch.tensor(0.9))
        p -= lr * (v0 + mu * v0)
        v = mu * v0 + grad
        sumsq = float((grad * grad).sum())
        p -= lr * (grad + mu * v)
        stats = {"sumsq": sumsq, "l2_norm": math.sqrt(sumsq), "max_abs": float(grad.abs().max()), "nan_count": 0,
                 "inf_count": 0, "elements": n}
        return {"stats": stats, "params": p, "shadow": p}
    return None   # tokens and bytes
