"""Timed cases of the library's public entry points over the sizes it is used at.

A case names one kind of call and its shape:

  grpo    one GRPO update pass, forward and backward, over a batch of sequences
          (grpo_loss_value_and_grad; optionally adding into a gradient accumulator, leaving masked
          tokens out of the backward products, with a final-logit softcap)
  sft     one supervised pass through autograd with a bf16 lm_head parameter (sft_fused_loss)
  ppo     token-level GAE, then the actor-critic pass with entropy bonus and value head through
          autograd, with float32 master weights (compute_gae_advantages, PPOActorCriticModule)
  score   log-probs and entropies of given tokens, no gradient (grpo_fused_loss under no_grad)
  sample  one decode step: last-position logits, top-k and a draw (last_position_logits,
          top_k_sampling_batched)
  norm    the final RMSNorm, forward and backward (rms_norm)
  adv     group-relative, leave-one-out or DAPO advantages of a batch of rewards

Hidden sizes and vocabularies are those of the benchmark configurations (Qwen2.5 0.5B / 1.5B / 7B,
Llama-3-8B, Gemma-2-2B) in the listed cases and anything between them in the drawn ones.
"""
from __future__ import annotations

import math

import torch

import mllm_jax_amd as M

TOP_K = 50
LOGIT_STD = 0.9            # standard deviation of a logit before the sampled token's lift
LIFT = 14.0                # a sampled token's logit stands up to this far above the others

_LARGEST = 16384 * 3584 * 152064


def _loss(name, kind, seqs, length, hidden, vocab, **options):
    return dict({"name": name, "kind": kind, "seqs": seqs, "length": length, "hidden": hidden, "vocab": vocab}, **options)


def listed():
    return [
        # GRPO advantages of one rollout of 16 prompts x 8 samples: the smallest call of a training step
        {"name": "adv_128", "kind": "adv", "estimator": "grpo", "seqs": 128, "group": 8},
        # one interactive stream decoding on the smallest model
        {"name": "sample_1", "kind": "sample", "seqs": 1, "hidden": 896, "vocab": 151936},
        # a partly filled serving batch
        {"name": "sample_37", "kind": "sample", "seqs": 37, "hidden": 4096, "vocab": 128256},
        # a full rollout batch
        {"name": "sample_128", "kind": "sample", "seqs": 128, "hidden": 3584, "vocab": 152064},
        # the norm in front of the headline batch
        {"name": "norm_16384", "kind": "norm", "rows": 16384, "hidden": 3584},
        # the smallest benchmark configuration: two sequences of the 0.5B model
        _loss("grpo_512", "grpo", 2, 256, 896, 151936),
        # a ragged micro-batch of the softcapped model under gradient accumulation, masked tokens left out
        _loss("grpo_1113_accumulate", "grpo", 7, 159, 2304, 256000, softcap=30.0, accumulate=True, skip_masked=True),
        # fine-tuning on three packed sequences, bf16 parameters
        _loss("sft_2049", "sft", 3, 683, 4096, 128256),
        # an actor-critic micro-batch from float32 master weights
        _loss("ppo_2048", "ppo", 8, 256, 1536, 151936),
        # a GRPO batch of the 1.5B model
        _loss("grpo_4096", "grpo", 32, 128, 1536, 151936),
        # old log-probs of a rollout before the update, sequences of uneven number and length
        _loss("score_5005", "score", 13, 385, 3584, 152064),
        # the headline batch: 128 sequences of the 7B model
        _loss("grpo_16384", "grpo", 128, 128, 3584, 152064),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["grpo", "grpo", "grpo", "sft", "ppo", "score", "sample", "sample", "norm", "adv"])
    hidden = 8 * rng.randint(896 // 8, 4096 // 8)
    vocab = 8 * rng.randint(32000 // 8, 256000 // 8)
    if kind == "adv":
        group = rng.randint(2, 16)
        return {"kind": "adv", "estimator": rng.choice(["grpo", "rloo", "dapo"]), "seqs": group * _log_int(rng, 4, 64) + rng.randint(0, group - 1),
                "group": group}
    if kind == "norm":
        return {"kind": "norm", "rows": _log_int(rng, 64, 16384), "hidden": hidden}
    if kind == "sample":
        return {"kind": "sample", "seqs": _log_int(rng, 1, 256), "hidden": hidden, "vocab": vocab}
    most = min(16384, _LARGEST // (hidden * vocab))
    if kind == "ppo":
        most = min(most, 8192)
    tokens = _log_int(rng, 128, most)
    length = min(_log_int(rng, 32, 512), tokens)
    case = {"kind": kind, "seqs": max(1, tokens // length), "length": length, "hidden": hidden, "vocab": vocab}
    if kind == "grpo":
        case.update(softcap=rng.choice([0.0, 0.0, 30.0]), accumulate=rng.random() < 0.3, skip_masked=rng.random() < 0.3)
    return case


class _Inputs:
    """Seeded tensors of one batch on the GPU."""

    def __init__(self, seed):
        self.dev = torch.device("cuda")
        self.gen = torch.Generator(device=self.dev).manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.gen, device=self.dev)

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.gen, device=self.dev)

    def ids(self, hi, *shape):
        return torch.randint(0, hi, shape, generator=self.gen, device=self.dev)

    def weights(self, h, v):
        return (self.normal(h, v) * (LOGIT_STD / math.sqrt(h))).to(torch.bfloat16)

    def hidden(self, w, ids):
        """Final hidden states whose logit for `ids` is lifted above the others by 0..LIFT, as a language
        model's is for the tokens sampled from it; also the logit itself."""
        n = ids.numel()
        wy = w.index_select(1, ids.reshape(-1)).t().float()
        lift = (self.uniform(n) * LIFT / LOGIT_STD**2)[:, None]
        hid = (self.normal(n, w.shape[0]) + lift * wy).to(torch.bfloat16)
        return hid, (hid.float() * wy).sum(-1)

    def spans(self, b, t):
        """[b, t] mask of completions: each sequence's first tokens up to a length of its own."""
        lo = max(1, t // 2)
        lens = lo + self.ids(t - lo + 1, b)
        return (torch.arange(t, device=self.dev)[None, :] < lens[:, None]).float()


def prepare(case, seed):
    x = _Inputs(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "adv":
        b = case["seqs"]
        s["rewards"] = (x.uniform(b) < 0.5).float() + 0.1 * x.normal(b)
        s["group_ids"] = torch.arange(b, device=x.dev, dtype=torch.int32) // case["group"]
        return s
    if kind == "norm":
        n, h = case["rows"], case["hidden"]
        s["x"] = (2.0 * x.normal(n, h)).to(torch.bfloat16).requires_grad_()
        s["scale"] = (1.0 + 0.1 * x.normal(h)).requires_grad_()
        s["dy"] = x.normal(n, h).to(torch.bfloat16)
        return s
    h, v = case["hidden"], case["vocab"]
    w = x.weights(h, v)
    if kind == "sample":
        s["hidden"], _ = x.hidden(w, x.ids(v, case["seqs"]))
        s["w"] = w
        s["generator"] = torch.Generator(device=x.dev).manual_seed(seed + 1)
        return s
    b, t = case["seqs"], case["length"]
    y = x.ids(v, b, t)
    hid, zy = x.hidden(w, y)
    # the rollout's log-probs: those of the tokens under these weights (the sum over the other tokens in
    # closed form) with the drift of a few updates
    if case.get("softcap"):
        zy = case["softcap"] * torch.tanh(zy / case["softcap"])
    others = math.log(v) + 0.5 * (hid.float() ** 2).sum(-1) * LOGIT_STD**2 / h
    old = zy - torch.logaddexp(zy, others) + 0.08 * x.normal(b * t)
    mask = x.spans(b, t)
    s.update(hidden=hid, w=w, y=y.reshape(-1), old=old, mask=mask.reshape(-1), tokens=float(mask.sum().item()))
    reward = (x.uniform(b) < 0.5).float() + 0.1 * x.normal(b)
    if kind == "grpo":
        s["advantages"] = (reward - reward.mean()) / (reward.std(unbiased=False) + 1e-4) if b > 1 else reward
        if case.get("accumulate"):
            s["accumulator"] = torch.zeros(h, v, device=x.dev)
    elif kind == "score":
        s["advantages"] = torch.zeros(b, device=x.dev)
    elif kind == "sft":
        s["hidden"], s["w"] = hid.requires_grad_(), w.requires_grad_()
    else:
        # module form: states and tokens of one position more than the loss looks at
        s["hidden"] = torch.cat([hid.reshape(b, t, h), torch.zeros(b, 1, h, dtype=torch.bfloat16, device=x.dev)], 1).requires_grad_()
        s["w"] = w.float().requires_grad_()
        s["value_w"] = (x.normal(h) / math.sqrt(h)).requires_grad_()
        s["value_b"] = torch.zeros((), device=x.dev).requires_grad_()
        s["values"] = 0.3 * x.normal(b, t)
        s["rewards"] = reward
        first = torch.zeros(b, 1, device=x.dev)
        s["inputs"] = {"input_ids": torch.cat([first.long(), y], 1), "attention_mask": torch.ones(b, t + 1, device=x.dev),
                       "labels": torch.cat([first, mask], 1), "old_per_token_logps": old.reshape(b, t), "old_values": s["values"],
                       "total_valid_token_count": mask.sum()}
        s["mask"] = mask
        s["module"] = M.PPOActorCriticModule(model=lambda input_ids, attention_mask: s["hidden"], lm_head=s["w"],
                                             value_head=(s["value_w"], s["value_b"]), entropy_coef=0.01)
    return s


_ESTIMATORS = {"grpo": M.compute_grpo_advantages_by_group_id, "rloo": M.compute_rloo_advantages_by_group_id,
               "dapo": M.compute_dapo_advantages_by_group_id}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "adv":
        return _ESTIMATORS[case["estimator"]](rewards=s["rewards"], group_ids=s["group_ids"])
    if kind == "norm":
        y = M.rms_norm(s["x"], s["scale"])
        return (y, *torch.autograd.grad(y, [s["x"], s["scale"]], s["dy"]))
    if kind == "sample":
        logits = M.last_position_logits(s["hidden"], s["w"])
        return (logits, *M.top_k_sampling_batched(s["generator"], logits, k=TOP_K, t=0.9, return_top_k=True))
    if kind == "sft":
        out = M.sft_fused_loss(s["hidden"], s["w"], s["y"], s["mask"], total_valid_token_count=s["tokens"])
        return out["loss"], out["per_token_logps"], torch.autograd.grad(out["loss"], [s["hidden"], s["w"]])
    if kind == "ppo":
        adv, ret = M.compute_gae_advantages(rewards=s["rewards"], values=s["values"], completion_mask=s["mask"])
        out = s["module"](dict(s["inputs"], advantages=adv, returns=ret))
        grads = torch.autograd.grad(out["loss"], [s["hidden"], s["w"], s["value_w"], s["value_b"]])
        return {**out, "advantages": adv, "returns": ret, "grads": grads}
    options = dict(total_valid_token_count=s["tokens"], seq_shape=(case["seqs"], case["length"]), epsilon_high=0.28,
                   final_logit_softcap=case.get("softcap") or None)
    if kind == "score":
        with torch.no_grad():
            return M.grpo_fused_loss(s["hidden"], s["w"], s["y"], None, s["advantages"], s["mask"], return_token_entropy=True, **options)
    return M.grpo_loss_value_and_grad(s["hidden"], s["w"], s["y"], s["old"], s["advantages"], s["mask"], accumulate_into=s.get("accumulator"),
                                      skip_masked=case.get("skip_masked", False), **options)


def work(case):
    kind = case["kind"]
    if kind == "adv":
        return {"bytes": 12 * case["seqs"], "flops": 4 * case["seqs"]}
    if kind == "norm":
        n, h = case["rows"], case["hidden"]
        return {"bytes": 5 * 2 * n * h + 8 * h, "flops": 14 * n * h}      # x, y; dy, x again, dx
    h, v = case["hidden"], case["vocab"]
    if kind == "sample":
        b = case["seqs"]
        return {"bytes": 2 * h * v + 2 * b * h + 4 * b * v + b * (8 * TOP_K + 4), "flops": 2 * b * h * v}
    n = case["seqs"] * case["length"]
    if kind == "score":
        return {"bytes": 2 * h * v + 2 * n * h + 20 * n, "flops": 2 * n * h * v}
    bytes_ = 2 * 2 * n * h + 24 * n                                        # hidden, d_hidden, per-token rows
    bytes_ += {"sft": 2 + 2, "ppo": 4 + 4, "grpo": 2 + (8 if case.get("accumulate") else 4)}[kind] * h * v
    # with masked tokens left out (a quarter of them on average) the two backward products are that much smaller
    return {"bytes": bytes_, "flops": (5 if case.get("skip_masked") else 6) * n * h * v}


def tolerance(case):
    """About four times the error against the same formulas in 64 bits.  The largest error of a loss
    pass is over the root mean square of a gradient most of whose entries are nearly zero."""
    kind = case["kind"]
    if kind == "adv":
        return {"rel": 1e-6, "max": 1e-5}
    if kind == "score":
        return {"rel": 1e-5, "max": 3e-5}
    if kind == "sample":
        return {"rel": 1e-5, "max": 3e-5, "differ": 0.01}
    if kind == "norm":
        return {"rel": 7e-3, "max": 2e-2}
    return {"rel": 1e-2, "max": 0.8}
