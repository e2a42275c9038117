"""The work a training or scoring program has this package do, as cases that can be timed and compared.

A case is a dict of plain values; `prepare` makes what a program holds before the call (model outputs, batch, trainer),
`run` is one pass through the public entry points, `work` what that pass cannot do without.  The kinds:

  score       per-token log-probs and entropies of given tokens from model logits, no gradient: the old and the
              reference policy's pass of an on-policy trainer (`per_token_logps_and_entropies`)
  grpo        the loss part of a GRPO training step: `GRPOLossMixin._compute_loss` on the model's logits, and the gradient
              with respect to them.  Token-level importance weights, or one weight per sequence (GSPO)
  dpo         the loss part of a DPO training step: `DPOLossMixin._compute_loss` and the gradient of the logits
  head_score  per-token log-probs and entropies from the last hidden states and the lm_head weight, no gradient
              (`chunked_logprobs_from_hidden`)
  sft         chunked next-token cross-entropy from the hidden states, with both gradients
              (`_chunked_cross_entropy_loss`)
  head_grpo   GRPO loss from the hidden states with both gradients (`FusedLinearGRPOLoss`)
  head_dpo    DPO loss from the hidden states of policy and reference, with both gradients (`FusedLinearDPOLoss`)
"""
import math
from collections import defaultdict
from types import SimpleNamespace

import torch

import trl_amd
from trl_amd.trainer.sft_trainer import _chunked_cross_entropy_loss

DEVICE = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
VOCABS = (32000, 32001, 50257, 50264, 128256, 128257, 151665, 151936, 151937, 202048, 256000, 262144)
LARGEST_LOGITS = 32 * 1024 * 151936  # entries of the largest logits tensor of any case
LARGEST_HEAD = 8 * 2048 * 3584 * 151936  # positions x hidden size x vocabulary of the largest head case
VOCAB_CHUNK = 8192  # vocabulary rows per slab that callers of the fused head pass


def listed():
    return [
        # scoring one short completion: the smallest call, launches and latency only
        dict(name="score_one", kind="score", B=1, T=64, V=32000, dtype="bf16", temperature=1.0),
        # the fp32 forward-only benchmark configuration: one round of workgroups
        dict(name="score_fp32", kind="score", B=8, T=256, V=32000, dtype="fp32", temperature=1.0),
        # the reference policy's pass over a long batch
        dict(name="score_long", kind="score", B=8, T=2048, V=128256, dtype="bf16", temperature=0.9),
        # one micro-batch of a small run: a group of four completions, a 32000-entry vocabulary
        dict(name="grpo_small", kind="grpo", B=4, T=256, V=32000, dtype="bf16", temperature=1.0, loss_type="dapo",
             level="token", beta=0.0, old=True, sampler_ratio=False),
        # an ordinary micro-batch on a vocabulary that is no multiple of the vector width, with KL term
        dict(name="grpo_odd_vocab", kind="grpo", B=16, T=509, V=50257, dtype="bf16", temperature=0.9, loss_type="grpo",
             level="token", beta=0.04, old=True, sampler_ratio=False),
        # the headline benchmark's rows (1024 tokens, V = 151936), 32 sequences
        dict(name="grpo_large", kind="grpo", B=32, T=1024, V=151936, dtype="bf16", temperature=0.9, loss_type="dapo",
             level="token", beta=0.04, old=True, sampler_ratio=True),
        # sequence-level importance weights: the loss needs every token's log-prob before any gradient
        dict(name="gspo", kind="grpo", B=16, T=512, V=151936, dtype="bf16", temperature=1.0, loss_type="grpo",
             level="sequence", beta=0.0, old=True, sampler_ratio=False),
        # eight preference pairs with a tokenizer that gained a token
        dict(name="dpo", kind="dpo", B=16, T=1024, V=128257, dtype="bf16"),
        # scoring a few hundred tokens from hidden states
        dict(name="head_score", kind="head_score", B=2, T=300, H=3584, V=151936, dtype="bf16", temperature=1.0),
        # fine-tuning micro-batch
        dict(name="sft", kind="sft", B=4, T=513, H=2048, V=50257, dtype="bf16"),
        # the fused-head benchmark's head and sequence length, eight sequences
        dict(name="head_grpo", kind="head_grpo", B=8, T=2048, H=3584, V=151936, dtype="bf16", temperature=1.0,
             loss_type="dapo", beta=0.04),
        # two preference pairs through the fused-linear operator, reference model with its own head
        dict(name="head_dpo", kind="head_dpo", B=4, T=512, H=2048, V=128256, dtype="bf16"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("score", "grpo", "grpo", "dpo", "head_score", "sft", "head_grpo", "head_dpo"))
    V = rng.choice(VOCABS)
    dtype = rng.choice(("bf16", "bf16", "bf16", "bf16", "fp16", "fp32"))
    if kind in ("score", "grpo", "dpo"):
        B = {"score": _log_uniform(rng, 1, 32), "grpo": 4 * _log_uniform(rng, 1, 8), "dpo": 2 * _log_uniform(rng, 1, 16)}[kind]
        most = LARGEST_LOGITS // (B * V * (2 if dtype == "fp32" else 1))
        T = min(_log_uniform(rng, 24, 4096), most)
        case = dict(kind=kind, B=B, T=T, V=V, dtype=dtype)
        if kind != "dpo":
            case["temperature"] = rng.choice((1.0, 0.9, 0.7))
        if kind == "grpo":
            case.update(loss_type=rng.choice(("dapo", "dapo", "grpo", "dr_grpo", "bnpo", "cispo")),
                        level=rng.choice(("token", "token", "token", "sequence")), beta=rng.choice((0.0, 0.04)),
                        old=rng.random() < 0.8, sampler_ratio=rng.random() < 0.3)
        return case
    H = rng.choice((1024, 1536, 2048, 2560, 3072, 3584, 4096))
    B = {"head_score": 1, "sft": 1, "head_grpo": 4, "head_dpo": 2}[kind] * _log_uniform(rng, 1, 4)
    most = LARGEST_HEAD // (B * V * H * (2 if kind == "head_dpo" else 1))
    T = min(_log_uniform(rng, 48, 4096), most)
    case = dict(kind=kind, B=B, T=T, H=H, V=V, dtype="fp16" if dtype == "fp16" else "bf16")
    if kind in ("head_score", "head_grpo"):
        case["temperature"] = rng.choice((1.0, 0.9, 0.7))
    if kind == "head_grpo":
        case.update(loss_type=rng.choice(("dapo", "grpo", "dr_grpo")), beta=rng.choice((0.0, 0.04)))
    return case


# ---------------------------------------------------------------------------------------------- batch layout
def _completion_lengths(B, T):
    """Completion lengths of a batch, 1/16 of the longest to the longest; the seed only permutes them."""
    return [max(1, round(T / 16 + (T - T / 16) * (i + 1) / B)) for i in range(B)]


def _prompt_and_total(B, T):
    """Prompt and total lengths of prompt + completion sequences padded to T; the seed only permutes them."""
    prompts = [max(1, round(T / 16 + (T / 4 - T / 16) * i / B)) for i in range(B)]
    totals = [max(prompts[i] + 1, round(T / 2 + (T - T / 2) * (i + 1) / B)) for i in range(B)]
    return list(zip(prompts, totals))


def _active_tokens(case):
    B, T = case["B"], case["T"]
    if case["kind"] == "score":
        return B * T
    if case["kind"] in ("grpo", "head_grpo"):
        return sum(_completion_lengths(B, T))
    return sum(total - prompt for prompt, total in _prompt_and_total(B, T))


def _permuted(values, g):
    order = torch.randperm(len(values), generator=g).tolist()
    return [values[i] for i in order]


def _length_mask(B, T, g):
    lengths = torch.tensor(_permuted(_completion_lengths(B, T), g), device=DEVICE)
    return (torch.arange(T, device=DEVICE)[None] < lengths[:, None]).long()


def _pair_masks(B, T, g):
    """(attention mask, completion mask) of prompt + completion sequences, right-padded."""
    spans = torch.tensor(_permuted(_prompt_and_total(B, T), g), device=DEVICE)
    at = torch.arange(T, device=DEVICE)[None]
    attention = (at < spans[:, 1:]).long()
    return attention, attention * (at >= spans[:, :1]).long()


# ---------------------------------------------------------------------------------------------- inputs
def _generators(seed):
    return torch.Generator().manual_seed(seed), torch.Generator(device=DEVICE).manual_seed(seed)


def _logits(B, L, V, ids, first, dtype, gd):
    """Model logits [B, L, V]: a spread of 2 around 0, and at position first + t the logit of token ids[:, t] raised
    to where the model's own samples lie (probabilities from a few percent to nearly 1)."""
    logits = torch.empty((B, L, V), dtype=dtype, device=DEVICE)
    T = ids.shape[1]
    for b in range(B):
        logits[b].normal_(0.0, 2.0, generator=gd)
        top = math.log(V) + 3.5 + 2.0 * torch.randn(T, generator=gd, device=DEVICE)
        logits[b, first : first + T].scatter_(1, ids[b, :, None], top[:, None].to(dtype))
    return logits


def _token_logps(logits, ids, first, temperature):
    """fp32 log-probs of ids under softmax(logits / temperature), a few rows at a time, in plain torch."""
    B, T = ids.shape
    out = torch.empty((B, T), device=DEVICE)
    step = max(1, (1 << 28) // logits.shape[-1])
    for b in range(B):
        for t in range(0, T, step):
            x = logits[b, first + t : first + min(T, t + step)].float() / temperature
            out[b, t : t + step] = x.gather(1, ids[b, t : t + step, None]).squeeze(1) - x.logsumexp(1)
    return out


def _head(B, T, H, V, ids, dtype, gd):
    """Last hidden states [B, T, H] that point towards the rows of ids in an lm_head weight [V, H]."""
    weight = torch.empty((V, H), dtype=dtype, device=DEVICE).normal_(0.0, 0.02, generator=gd)
    hidden = torch.randn((B, T, H), generator=gd, device=DEVICE)
    rows = weight[ids.reshape(-1)].float().view(B, T, H)
    lift = (math.log(V) + 1.5 + 1.5 * torch.randn((B, T, 1), generator=gd, device=DEVICE)) / (0.02**2 * H)
    return (hidden + lift * rows).to(dtype), weight


def _head_token_logps(hidden, weight, ids, temperature):
    flat, target = hidden.reshape(-1, hidden.shape[-1]), ids.reshape(-1)
    out = torch.empty(flat.shape[0], device=DEVICE)
    for i in range(0, flat.shape[0], 1024):
        z = torch.mm(flat[i : i + 1024], weight.t()).float() / temperature
        out[i : i + 1024] = z.gather(1, target[i : i + 1024, None]).squeeze(1) - z.logsumexp(1)
    return out.view(ids.shape)


class _OneProcess:
    """The accelerator of a single-process run."""

    num_processes, sync_gradients, scaler, gradient_accumulation_steps = 1, True, None, 1
    gather = gather_for_metrics = staticmethod(lambda x: x)
    reduce = staticmethod(lambda x, reduction="sum": x)


class _GRPOTrainer(trl_amd.GRPOLossMixin):
    pass


class _DPOTrainer(trl_amd.DPOLossMixin):
    pass


def _trainer(cls):
    tr = cls()
    tr.accelerator, tr.model = _OneProcess(), SimpleNamespace(training=True)
    tr.aux_loss_enabled = False
    return tr


def _prepare_grpo(case, g, gd):
    B, T, V, P = case["B"], case["T"], case["V"], 16
    ids = torch.randint(0, V, (B, T), generator=gd, device=DEVICE)
    prompt = torch.randint(0, V, (B, P), generator=gd, device=DEVICE)
    mask = _length_mask(B, T, g)
    logits = _logits(B, T + 1, V, ids, 0, DTYPES[case["dtype"]], gd)  # (the model keeps the last T + 1 positions)
    logp = _token_logps(logits, ids, 0, case["temperature"])
    noise = lambda size: size * torch.randn((B, T), generator=gd, device=DEVICE)  # noqa: E731
    inputs = dict(prompt_ids=prompt, prompt_mask=torch.ones_like(prompt), completion_ids=ids, completion_mask=mask,
                  advantages=trl_amd.group_advantages(torch.randn((B,), generator=gd, device=DEVICE), 4),
                  num_items_in_batch=mask.sum().float())
    if case["old"]:
        inputs["old_per_token_logps"] = logp + noise(0.1)
    if case["beta"]:
        inputs["ref_per_token_logps"] = logp + noise(0.2)
    if case["sampler_ratio"]:
        inputs["importance_sampling_ratio"] = noise(0.05).exp().clamp(max=3.0)
    tr = _trainer(_GRPOTrainer)
    tr.temperature, tr.model_kwarg_keys = case["temperature"], {"logits_to_keep"}
    tr._entropy_bonus_enabled, tr.entropy_coef, tr.use_adaptive_entropy = False, 0.0, False
    tr.top_entropy_quantile, tr.off_policy_mask_threshold = 1.0, None
    tr.importance_sampling_level, tr.loss_type = case["level"], case["loss_type"]
    tr.beta, tr.epsilon_low, tr.epsilon_high = case["beta"], 0.2, 0.28
    tr.use_vllm = tr.vllm_importance_sampling_correction = case["sampler_ratio"]
    tr.max_completion_length, tr.current_gradient_accumulation_steps = T, 1
    tr.args = SimpleNamespace(delta=None, use_bias_correction_kl=False)
    return dict(trainer=tr, logits=logits.requires_grad_(True), inputs=inputs)


def _prepare_dpo(case, g, gd):
    B, T, V = case["B"], case["T"], case["V"]
    ids = torch.randint(0, V, (B, T), generator=gd, device=DEVICE)
    attention, completion = _pair_masks(B, T, g)
    logits = _logits(B, T, V, ids[:, 1:], 0, DTYPES[case["dtype"]], gd)
    seq = (_token_logps(logits, ids[:, 1:], 0, 1.0) * completion[:, 1:]).sum(1)
    ref = seq + 3.0 * torch.randn((B,), generator=gd, device=DEVICE)
    tr = _trainer(_DPOTrainer)
    tr.precompute_ref_logps, tr.beta, tr.loss_types, tr.loss_weights = True, 0.1, ["sigmoid"], [1.0]
    tr.label_smoothing, tr.ld_alpha, tr.use_weighting = 0.0, None, False
    tr.f_divergence_type, tr.f_alpha_divergence_coef = "reverse_kl", 1.0
    tr.args = SimpleNamespace(discopop_tau=0.05)
    tr._total_train_tokens = 0
    inputs = dict(input_ids=ids, attention_mask=attention, completion_mask=completion,
                  ref_chosen_logps=ref[: B // 2].clone(), ref_rejected_logps=ref[B // 2 :].clone())
    return dict(trainer=tr, logits=logits.requires_grad_(True), inputs=inputs)


def _prepare_head(case, g, gd):
    kind, B, T, H, V = (case[k] for k in ("kind", "B", "T", "H", "V"))
    dtype = DTYPES[case["dtype"]]
    ids = torch.randint(0, V, (B, T), generator=gd, device=DEVICE)
    if kind == "head_grpo":
        hidden, weight = _head(B, T, H, V, ids, dtype, gd)
        logp = _head_token_logps(hidden, weight, ids, case["temperature"])
        noise = lambda size: size * torch.randn((B, T), generator=gd, device=DEVICE)  # noqa: E731
        op = trl_amd.FusedLinearGRPOLoss(beta=case["beta"], epsilon_low=0.2, epsilon_high=0.2,
                                         temperature=case["temperature"], use_ref_model=case["beta"] != 0.0,
                                         loss_type=case["loss_type"], max_completion_length=T)
        return dict(op=op, hidden=hidden.requires_grad_(True), weight=weight.requires_grad_(True), ids=ids,
                    mask=_length_mask(B, T, g), old=logp + noise(0.1), ref=logp + noise(0.2) if case["beta"] else None,
                    advantages=trl_amd.group_advantages(torch.randn((B,), generator=gd, device=DEVICE), 4))
    attention, completion = _pair_masks(B, T, g)
    hidden, weight = _head(B, T, H, V, ids.roll(-1, 1), dtype, gd)  # (position t predicts token t + 1)
    if kind == "head_score":
        return dict(hidden=hidden, weight=weight, ids=ids, completion=completion, temperature=case["temperature"])
    if kind == "sft":
        labels = torch.where(completion.bool(), ids, torch.full_like(ids, -100))
        return dict(hidden=hidden.requires_grad_(True), weight=weight.requires_grad_(True), labels=labels)
    # head_dpo: labels are aligned with the hidden states; the reference is the policy before a few updates
    target = torch.where(completion.bool(), ids, torch.full_like(ids, -100)).roll(-1, 1)
    target[:, -1] = -100
    drift = lambda t, size: (t.float() + size * torch.randn(t.shape, generator=gd, device=DEVICE)).to(dtype)  # noqa: E731
    ref_hidden, ref_weight = drift(hidden, 0.02), drift(weight, 0.0002)
    return dict(op=trl_amd.FusedLinearDPOLoss(beta=0.1), hidden=hidden.requires_grad_(True),
                weight=weight.requires_grad_(True), target=target, ref_hidden=ref_hidden, ref_weight=ref_weight)


def prepare(case, seed):
    g, gd = _generators(seed)
    kind = case["kind"]
    if kind == "score":
        B, T, V = case["B"], case["T"], case["V"]
        ids = torch.randint(0, V, (B, T), generator=gd, device=DEVICE)
        state = dict(ids=ids, logits=_logits(B, T + 1, V, ids, 0, DTYPES[case["dtype"]], gd), temperature=case["temperature"])
    elif kind == "grpo":
        state = _prepare_grpo(case, g, gd)
    elif kind == "dpo":
        state = _prepare_dpo(case, g, gd)
    else:
        state = _prepare_head(case, g, gd)
    state["kind"] = kind
    return state


# ---------------------------------------------------------------------------------------------- one pass
def run(state):
    kind = state["kind"]
    if kind == "score":
        with torch.no_grad():
            return trl_amd.per_token_logps_and_entropies(state["logits"], state["ids"], state["ids"].shape[1],
                                                         state["temperature"])
    if kind in ("grpo", "dpo"):
        tr, logits = state["trainer"], state["logits"]
        tr._metrics = {"train": defaultdict(list), "eval": defaultdict(list)}
        args = (state["inputs"],) if kind == "grpo" else (state["inputs"], False)
        loss = tr._compute_loss(lambda **kw: SimpleNamespace(logits=logits, aux_loss=None), *args)
        (grad,) = torch.autograd.grad(loss, logits)
        log = tr._metrics["train"]
        metrics = torch.tensor([log[k][-1] for k in sorted(log) if k != "num_tokens"], dtype=torch.float64)
        return loss.detach(), metrics, grad
    hidden, weight = state["hidden"], state["weight"]
    if kind == "head_score":
        with torch.no_grad():
            return trl_amd.chunked_logprobs_from_hidden(hidden, weight, state["ids"], state["completion"],
                                                        state["temperature"], VOCAB_CHUNK)
    if kind == "sft":
        loss, correct, entropy, n_valid = _chunked_cross_entropy_loss(hidden, weight, VOCAB_CHUNK, labels=state["labels"])
        more = (correct, entropy, n_valid)
    elif kind == "head_grpo":
        loss, more = state["op"](hidden, weight, state["ids"], state["mask"], state["advantages"], None, state["old"],
                                 state["ref"])
    else:
        loss, more = state["op"](weight, hidden, state["target"], None, state["ref_hidden"], state["ref_weight"])
    return loss.detach(), more, torch.autograd.grad(loss, (hidden, weight))


def work(case):
    B, T, V, n = case["B"], case["T"], case["V"], _active_tokens(case)
    size = 4 if case["dtype"] == "fp32" else 2
    per_token = 40 * B * T  # token ids, masks, log-probs and the like
    kind = case["kind"]
    if kind == "score":
        return {"bytes": n * V * size + per_token, "flops": 0}
    if kind == "grpo":  # the completion's rows are read, the gradient of all T + 1 positions is written
        return {"bytes": (n + B * (T + 1)) * V * size + per_token, "flops": 0}
    if kind == "dpo":
        return {"bytes": (n + B * T) * V * size + per_token, "flops": 0}
    H = case["H"]
    product, operands = 2 * n * H * V, (B * T * H + V * H) * size
    if kind == "head_score":
        return {"bytes": operands + per_token, "flops": product}
    if kind == "head_dpo":
        return {"bytes": 3 * operands + per_token, "flops": 4 * product}
    return {"bytes": 2 * operands + per_token, "flops": 3 * product}


def tolerance(case):
    """About four times what another order of summation makes.  Log-probs and entropies against float64: relative L2
    1.3e-6, one value 7e-6.  One pass over the logits against two: gradient 2.5e-5 (16-bit, where single entries move by
    a rounding step, 7e-3) or 1.7e-6 (fp32, single entries 1e-3), a loss whose advantages cancel 4e-5.  The head's
    gradients come from 16-bit products: 1.2e-3 (one entry 3e-2) off the fp32 products rounded once."""
    kind = case["kind"]
    if kind in ("score", "head_score"):
        return {"rel": 5e-6, "max": 3e-5}
    if kind in ("grpo", "dpo"):
        return {"rel": 1.6e-4, "max": 4e-3 if case["dtype"] == "fp32" else 3e-2}
    return {"rel": 4e-3, "max": 0.11}
