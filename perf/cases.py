"""Performance cases of the cross-entropy entry points.

Each case is one call that a training or evaluation program makes: its sizes,
dtype and options are plain values, ``prepare`` makes the tensors that such a
program has in hand, ``run`` makes the call through the public entry points and
returns its outputs, and ``exact`` gives the same outputs in 64 bits with plain
torch.  Kinds:

  train    fused lm_head projection + loss, forward and backward; gradients of
           hidden and (unless the weight is frozen) of the weight and bias
  eval     the same projection + loss per row, without gradients
  logits   loss over logits that already exist, forward and backward
  grad     loss and gradient of existing logits from one call
"""
import math

import torch

from chronicals_amd.kernels.cut_cross_entropy import CutCrossEntropyLoss, cut_cross_entropy
from chronicals_amd.kernels.fused_linear_cross_entropy import fused_linear_cross_entropy
from chronicals_amd.kernels.logits_cross_entropy import chunked_cross_entropy_loss, fused_cross_entropy

IGNORE = -100
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _case(kind, N, V, d=0, dtype="bf16", ignored=0.05, labels="uniform", frozen=False, bias=False, eps=0.0, z=0.0):
    """ignored: share of rows labelled -100; eps: label smoothing; z: z-loss weight."""
    return {"kind": kind, "N": N, "d": d, "V": V, "dtype": dtype, "ignored": ignored, "labels": labels,
            "frozen": frozen, "bias": bias, "eps": eps, "z": z}


def listed():
    return [
        # one short chat turn on a small head: launches and host time count
        dict(_case("train", 64, 32000, 896), name="train_64"),
        # GPT-2-sized head in fp32, a micro-batch of 256 tokens
        dict(_case("train", 256, 50257, 768, "fp32", 0.10), name="train_256_fp32"),
        # one 2048-token sequence per micro-batch on a 152k vocabulary
        dict(_case("train", 2048, 151936, 896), name="train_2048"),
        # the headline training step: 16384 tokens, 0.5B-parameter model's head
        dict(_case("train", 16384, 151936, 896), name="train_16384"),
        # wide hidden, 128k vocabulary, word-frequency labels
        dict(_case("train", 8192, 128256, 4096, "bf16", 0.02, "zipf"), name="train_8192_wide"),
        # packed sequences, the largest batch
        dict(_case("train", 32768, 151936, 2048, "bf16", 0.001), name="train_32768"),
        # LoRA fine-tuning: frozen lm_head, prompt tokens (40%) without a label
        dict(_case("train", 4096, 151936, 2048, "bf16", 0.40, frozen=True), name="train_frozen"),
        # hidden size that is no multiple of 64, bias, smoothing and z-loss
        dict(_case("train", 1500, 50257, 1000, "bf16", 0.10, bias=True, eps=0.1, z=1e-4), name="train_ragged"),
        # perplexity of held-out text: per-row losses, no gradients
        dict(_case("eval", 3001, 128256, 2048, "bf16", 0.05, "zipf"), name="eval_rows"),
        # a model that returns logits: loss and backward over them
        dict(_case("logits", 4096, 151936), name="logits_4096"),
        # a few rows of logits, as a short continuation has them
        dict(_case("logits", 16, 151936, 0, "fp32", 0.0, eps=0.1), name="logits_16_fp32"),
        # loss and fp32 gradient in one call, rows that start off alignment
        dict(_case("grad", 2048, 50257, 0, "bf16", 0.05, eps=0.1, z=1e-4), name="grad_2048"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["train", "train", "train", "train", "eval", "logits", "grad"])
    ignored = rng.choice([0.0, 0.02, 0.05, 0.1, 0.4])
    labels = rng.choice(["uniform", "zipf"])
    eps, z = rng.choice([(0.0, 0.0), (0.0, 0.0), (0.1, 0.0), (0.1, 1e-4)])
    V = _log(rng, 5000, 152064)
    if kind in ("logits", "grad"):
        # at most the largest listed logits
        N = _log(rng, 8, min(16384, 4096 * 151936 // (2 * V)))
        return _case(kind, N, V, 0, rng.choice(["bf16", "bf16", "fp16", "fp32"]), ignored, labels, eps=eps, z=z)
    # hidden sizes of models are mostly multiples of 64
    d = _log(rng, 2, 64) * 64 if rng.random() < 0.7 else _log(rng, 16, 256) * 8 + 8
    # at most the work of the largest listed case
    N = _log(rng, 32, min(32768, 32768 * 2048 * 151936 // (d * V)))
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
    if kind == "eval":
        return _case(kind, N, V, d, dtype, ignored, labels, eps=eps, z=z)
    return _case(kind, N, V, d, dtype, ignored, labels, frozen=rng.random() < 0.3, bias=rng.random() < 0.2, eps=eps, z=z)


def _labels(case, g, dev):
    N, V = case["N"], case["V"]
    if case["labels"] == "zipf":  # p(k) ~ (k + 1)^-1.1, by the inverse of the cumulative sum
        cdf = torch.cumsum(torch.arange(1, V + 1, dtype=torch.float64, device=dev) ** -1.1, 0)
        u = torch.rand(N, generator=g, dtype=torch.float64, device=dev)
        lab = torch.searchsorted(cdf / cdf[-1], u).clamp_(max=V - 1)
    else:
        lab = torch.randint(0, V, (N,), generator=g, device=dev)
    lab[torch.rand(N, generator=g, device=dev) < case["ignored"]] = IGNORE
    return lab


def _inputs(case, seed):
    """Hidden ~ N(0, 1) and weight ~ N(0, 0.02) as after a final norm and a usual
    initialisation; logits ~ N(0, 2)."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(int(seed))
    dt = DTYPES[case["dtype"]]
    N, d, V = case["N"], case["d"], case["V"]
    if case["kind"] in ("logits", "grad"):
        return {"x": (torch.randn(N, V, generator=g, device=dev) * 2).to(dt), "labels": _labels(case, g, dev)}
    return {"h": torch.randn(N, d, generator=g, device=dev).to(dt),
            "w": (torch.randn(V, d, generator=g, device=dev) * 0.02).to(dt),
            "b": torch.randn(V, generator=g, device=dev) * 0.1 if case["bias"] else None,
            "labels": _labels(case, g, dev)}


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    if case["kind"] == "train":
        s["h"].requires_grad_(True)
        if not case["frozen"]:
            s["w"].requires_grad_(True)
            if s["b"] is not None:
                s["b"].requires_grad_(True)
        s["loss"] = CutCrossEntropyLoss(label_smoothing=case["eps"], z_loss_weight=case["z"])
    elif case["kind"] == "logits":
        s["x"].requires_grad_(True)
    return s


def run(s):
    case, lab = s["case"], s["labels"]
    eps, z = case["eps"], case["z"]
    if case["kind"] == "train":
        h, w, b = s["h"], s["w"], s["b"]
        h.grad = w.grad = None
        if b is not None:
            b.grad = None
            loss, zl = fused_linear_cross_entropy(h, w, lab, b, eps, z)
            loss.backward()
            return {"loss": loss.detach(), "z_loss": zl, "dh": h.grad, "dw": w.grad, "db": b.grad}
        loss = s["loss"](h, w, lab)
        loss.backward()
        return {"loss": loss.detach(), "dh": h.grad, "dw": w.grad}
    if case["kind"] == "eval":
        with torch.no_grad():
            return cut_cross_entropy(s["h"], s["w"], lab, label_smoothing=eps, z_loss_weight=z, reduction="none")
    if case["kind"] == "logits":
        x = s["x"]
        x.grad = None
        loss = chunked_cross_entropy_loss(x, lab, label_smoothing=eps, z_loss_weight=z)
        loss.backward()
        return {"loss": loss.detach(), "dx": x.grad}
    loss, dx = fused_cross_entropy(s["x"], lab, label_smoothing=eps, z_loss_weight=z)
    return {"loss": loss, "dx": dx}


def work(case):
    """Each input read once and each output written once; the products over the labelled rows."""
    N, d, V = case["N"], case["d"], case["V"]
    size = {"bf16": 2, "fp16": 2, "fp32": 4}[case["dtype"]]
    live = N * (1.0 - case["ignored"])
    if case["kind"] in ("logits", "grad"):
        read, written = live * V * size, N * V * (4 if case["kind"] == "grad" else size)
        return {"bytes": int(read + written + 8 * N), "flops": int(8 * live * V)}
    read = (live * d + V * d) * size + 8 * N + (4 * V if case["bias"] else 0)
    if case["kind"] == "eval":
        return {"bytes": int(read + 4 * N), "flops": int(2 * live * d * V)}
    written = N * d * size
    products = 2
    if not case["frozen"]:
        written += V * d * size + (4 * V if case["bias"] else 0)
        products = 3
    return {"bytes": int(read + written), "flops": int(2 * products * live * d * V)}


def tolerance(case):
    """About four times the error against ``exact`` measured over the listed and 24 drawn cases."""
    kind, dt = case["kind"], case["dtype"]
    if kind == "train":
        # bf16 operands and a bf16 gradient of the logits: 0.2 to 0.4%; gradients returned in fp16 are partly
        # subnormal there: up to 0.9%.  The weight rows of frequent labels are sums of many large terms, against
        # a root mean square that the other rows keep small: 0.1 of it with even labels, 0.5 with word frequencies.
        return {"rel": 3e-2 if dt == "fp16" else 1.5e-2, "max": 1.0 if case["labels"] == "zipf" else 0.4}
    if kind == "eval":
        # fp32 sums of bf16 products (fp16 and fp32 operands are rounded to bf16 first, alike in every pass)
        return {"rel": 1e-5}
    if kind == "grad" or dt == "fp32":
        # fp32 exponentials: 4e-8, single values to 2e-6
        return {"rel": 1e-6, "max": 1e-5}
    # a gradient rounded to 16 bits, in fp16 partly subnormal: 0.3%
    return {"rel": 1e-2, "max": 0.06}


def _row_loss(case, lse, target, mean, uniform):
    eps, V = case["eps"], case["V"]
    smooth = lse - mean if uniform else math.log(V)
    return (1 - eps) * (lse - target) + eps * smooth + case["z"] * lse * lse


def exact(case, seed):
    s = _inputs(case, seed)
    lab, N, V, eps, z = s["labels"], case["N"], case["V"], case["eps"], case["z"]
    valid = lab != IGNORE
    n_valid = max(int(valid.sum()), 1)
    kind = case["kind"]
    fused = "h" in s
    if fused:
        h, w = s["h"].double(), s["w"].double()
        dh = torch.zeros_like(h) if kind == "train" else None
        need_dw = kind == "train" and not case["frozen"]
        dw = torch.zeros_like(w) if need_dw else None
        db = torch.zeros(V, dtype=torch.float64, device=w.device) if need_dw and s["b"] is not None else None
    else:
        dx = torch.empty(N, V, dtype=torch.float64, device=lab.device)
    rows = torch.zeros(N, dtype=torch.float64, device=lab.device)
    zrows = torch.zeros_like(rows)
    for a in range(0, N, 2048):
        e = min(a + 2048, N)
        if fused:
            x = h[a:e] @ w.t()
            if s["b"] is not None:
                x += s["b"].double()
        else:
            x = s["x"][a:e].double()
        ok, at = valid[a:e], lab[a:e].clamp(min=0)
        lse = torch.logsumexp(x, 1)
        target = x.gather(1, at[:, None])[:, 0]
        r = _row_loss(case, lse, target, x.mean(1), kind == "grad")
        rows[a:e] = torch.where(ok, r, 0.0)
        zrows[a:e] = torch.where(ok, z * lse * lse, 0.0)
        if kind == "eval":
            continue
        g = x.sub_(lse[:, None]).exp_()  # softmax
        if kind == "logits":
            # the derivative of (1-eps)*(lse - target) + z*lse^2: the smoothing term eps*log(V) has none
            g *= (1 - eps + 2 * z * lse)[:, None]
        else:
            g *= (1 + 2 * z * lse)[:, None]
            g -= eps / V
        g.scatter_add_(1, at[:, None], torch.full_like(lse, -(1 - eps))[:, None])
        g *= (ok if kind == "grad" else ok / n_valid)[:, None]
        if not fused:
            dx[a:e] = g
            continue
        dh[a:e] = g @ w
        if dw is not None:
            dw.addmm_(g.t(), h[a:e])
        if db is not None:
            db += g.sum(0)
    if kind == "eval":
        return rows
    loss = rows.sum() / n_valid
    if not fused:
        return {"loss": loss, "dx": dx}
    out = {"loss": loss, "dh": dh, "dw": dw}
    if s["b"] is not None:
        out.update(z_loss=zrows.sum() / n_valid, db=db)
    return out
