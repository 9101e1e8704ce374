"""Workloads of the RL training hot path, as a trainer runs them through the public Python API.

A training step of a policy goes through these calls, and each is a ``path`` below:

* ``logp``    forward-only label log-probabilities of a packed batch (``engine.compute_logprobs``)
* ``adv``     advantages of a padded rollout batch (``ppo.actor.compute_advantages``)
* ``gae``     the same on a packed batch (``ppo.gae.compute_gae_packed_normalized``)
* ``pack``    padded batch -> packed -> padded to the micro-batch length, and a per-token result
              back to rows (``packing``)
* ``step``    fused lm_head forward, actor loss, backward to dHidden and dWeight
              (``fused_lm_head_logprobs_entropy`` + ``grpo_loss_fn``, or ``FusedLMHeadAdapter``
              with fp32 master weights)
* ``logits``  log-probabilities and entropy of logits the model already made, and their gradient
* ``loss``    the loss stage alone on per-token arrays, forward and backward

Hidden sizes and vocabularies are those of the shapes ``bench.py`` and the GPU tests use.
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

from areal_amd.config import NormConfig, RejectionSamplingConfig
from areal_amd.data import KLEstimator, Normalization
from areal_amd.engine import FusedLMHeadAdapter, compute_logprobs
from areal_amd.functional import (
    fused_lm_head_logprobs_entropy,
    gather_logprobs_entropy,
    ppo_critic_loss_fn,
)
from areal_amd.packing import pack_tensor_dict, pad_packed_tensor_dict, unpack_reorder_pad
from areal_amd.ppo.actor import compute_advantages, grpo_loss_fn
from areal_amd.ppo.gae import compute_gae_packed_normalized

# (hidden size, vocabulary) of the shapes in bench.py and tests/test_gpu_lmhead_shapes.py
MODELS = [
    (896, 151936), (1024, 151936), (1536, 151936), (2048, 151936), (2560, 151936), (3584, 152064),
    (4096, 128256), (4096, 151936), (5120, 151936), (8192, 128256),
]
MAX_STEP = 32768 * 4096 * 151936       # tokens x hidden x vocabulary of the largest training step
MAX_LOGITS = 4096 * 151936
MAX_SLOTS = 1024 * 8192


# -- the cases -------------------------------------------------------------------------------

def listed():
    return [
        # A short micro-batch (a few hundred tokens left over by the packer) of the smallest model:
        # the weight is read and written for few tokens, launches and host work count.
        dict(name="step small ragged", path="step", tokens=509, hidden=896, vocab=151936, seqs=3,
             loss="ppo", level="token", stats="reduced", defer=False, master=False, micro=1),
        # 0.5B-model micro-batch with the logged statistics, as a trainer runs it by default.
        dict(name="step 0.5b", path="step", tokens=4096, hidden=896, vocab=151936, seqs=16,
             loss="ppo", level="token", stats="reduced", defer=False, master=False, micro=1),
        # 1.5B model with fp32 master weights: two micro-batches, gradient added in fp32.
        dict(name="step 1.5b fp32 masters", path="step", tokens=16384, hidden=1536, vocab=151936, seqs=64,
             loss="cispo", level="token", stats="none", defer=False, master=True, micro=2),
        # 8B-model micro-batch, the step of bench.py's default workload.
        dict(name="step 8b", path="step", tokens=32768, hidden=4096, vocab=151936, seqs=32,
             loss="ppo", level="token", stats="none", defer=True, master=False, micro=1),
        # Recomputing the proximal log-probs of a ragged batch before training.
        dict(name="logp 1.5b ragged", path="logp", tokens=10007, hidden=1536, vocab=151936, pad=231),
        # A model that still makes its logits: log-probs, entropy, gradient, bf16.
        dict(name="logits bf16", path="logits", rows=4096, vocab=151936, dtype="bf16", grad=True),
        # The loss stage of an ordinary micro-batch, with the statistics a trainer logs.
        dict(name="loss 32k", path="loss", tokens=32768, seqs=32, loss="ppo", level="token", stats="reduced"),
        # The loss stage over a whole large batch, sequence-level rejection.
        dict(name="loss 4M", path="loss", tokens=4 << 20, seqs=2048, loss="ppo", level="sequence", stats="none"),
        # Advantages of a small rollout batch without a critic (GRPO).
        dict(name="adv small", path="adv", rows=64, length=1000, group=8, unit="token", critic=False),
        # Advantages of a large rollout batch with a critic and a KL penalty.
        dict(name="adv large", path="adv", rows=1024, length=8192, group=16, unit="token", critic=True),
        # The packed form: 1024 sequences with lognormal lengths, groups of 16.
        dict(name="gae packed", path="gae", seqs=1024, mean_len=1750, group=16),
        # A rollout batch on its way into micro-batches and a per-token result on its way back.
        dict(name="pack", path="pack", rows=256, length=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["step", "step", "step", "step", "logp", "logits", "loss", "loss", "adv", "adv", "gae", "pack"])
    if path in ("step", "logp"):
        hidden, vocab = rng.choice(MODELS)
        tokens = _log_int(rng, 256, min(32768, MAX_STEP // (hidden * vocab)))
        if path == "logp":
            return dict(path=path, tokens=tokens, hidden=hidden, vocab=vocab, pad=rng.randint(0, min(255, tokens // 2)))
        master = rng.random() < 0.4
        return dict(path=path, tokens=tokens, hidden=hidden, vocab=vocab, seqs=max(1, tokens // rng.randint(200, 1200)),
                    loss=rng.choice(["ppo", "ppo", "cispo"]), level=rng.choice(["token", "token", "sequence"]),
                    stats="none" if master else rng.choice(["none", "reduced"]), defer=rng.random() < 0.5,
                    master=master, micro=rng.randint(1, 2) if master and tokens >= 1024 else 1)
    if path == "logits":
        vocab = rng.choice([32000, 50257, 128256, 151936, 152064])
        rows = _log_int(rng, 16, MAX_LOGITS // 2 // vocab)
        return dict(path=path, rows=rows, vocab=vocab, dtype=rng.choice(["bf16", "bf16", "fp32"]), grad=rng.random() < 0.7)
    if path == "loss":
        tokens = _log_int(rng, 512, 4 << 20)
        return dict(path=path, tokens=tokens, seqs=max(1, tokens // rng.randint(200, 4000)),
                    loss=rng.choice(["ppo", "ppo", "cispo", "sapo", "critic"]), level=rng.choice(["token", "sequence"]),
                    stats=rng.choice(["none", "reduced", "tensors"]))
    if path == "adv":
        length = _log_int(rng, 200, 8192)
        group = rng.choice([4, 8, 16])
        rows = group * _log_int(rng, 1, max(1, min(1024, MAX_SLOTS // length) // group))
        return dict(path=path, rows=rows, length=length, group=group, unit=rng.choice(["token", "token", "turn"]),
                    critic=rng.random() < 0.5)
    if path == "gae":
        mean_len = _log_int(rng, 100, 8192)
        group = rng.choice([4, 8, 16])
        return dict(path=path, seqs=group * _log_int(rng, 1, max(1, min(4096, (4 << 20) // mean_len) // group)),
                    mean_len=mean_len, group=group)
    length = _log_int(rng, 200, 8192)
    return dict(path="pack", rows=_log_int(rng, 4, min(1024, (4 << 20) // length)), length=length)


# -- what a case cannot do without, and how exact it is ---------------------------------------

def work(case):
    path = case["path"]
    if path in ("step", "logp"):
        t, h, v = case["tokens"], case["hidden"], case["vocab"]
        if path == "logp":  # hidden, weight, labels in; log-probs out
            return dict(bytes=2 * t * h + 2 * v * h + 12 * t, flops=2 * t * h * v)
        # hidden and weight in, dHidden and dWeight out; labels, mask and four fp32 arrays in,
        # log-prob, entropy, vocabulary extremes out
        grad = 4 if case["master"] else 2
        return dict(bytes=4 * t * h + (2 + grad) * v * h + 41 * t, flops=6 * t * h * v)
    if path == "logits":
        t, v, e = case["rows"], case["vocab"], 2 if case["dtype"] == "bf16" else 4
        return dict(bytes=t * v * e * (2 if case["grad"] else 1) + 20 * t, flops=8 * t * v)
    if path == "loss":
        t = case["tokens"]
        if case["loss"] == "critic":  # value, old, target, mask in; gradient, loss, clip mask out
            return dict(bytes=22 * t, flops=20 * t)
        # log-probs (three), advantage, entropy, mask in; gradient out; statistics as tensors: 13 more
        stats = {"none": 0, "reduced": 4, "tensors": 4 + 40}[case["stats"]]
        return dict(bytes=(21 + stats) * t, flops=100 * t)
    if path == "adv":
        n = case["rows"] * case["length"]
        # masks, log-probs, reference log-probs (values, turn ids) in; loss mask, log-probs, KL and
        # total rewards, returns, advantages out
        per = 10 + (4 if case["critic"] else 0) + (4 if case["unit"] == "turn" else 0) + 24
        return dict(bytes=per * n, flops=60 * n)
    if path == "gae":
        n = case["seqs"] * case["mean_len"]
        return dict(bytes=24 * n, flops=40 * n)
    n = case["rows"] * case["length"]
    # 25 bytes a token of five tensors read and written packed, again padded, one fp32 array back to rows
    return dict(bytes=int(0.5 * n * (4 * 25 + 4) + 4 * n + n), flops=n)


def tolerance(case):
    path = case["path"]
    if path == "step":  # bf16 gradients of bf16 operands
        return {"rel": 1e-2, "max": 0.1}
    if path == "logp":  # fp32 sums over bf16 operands
        return {"rel": 1e-5}
    if path == "logits":
        return {"rel": 1e-2, "max": 0.05} if case["dtype"] == "bf16" and case["grad"] else {"rel": 1e-5}
    if path == "pack":
        return "exact"
    return {"rel": 1e-5}


# -- inputs -----------------------------------------------------------------------------------

def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _gens(seed):
    return torch.Generator().manual_seed(seed), torch.Generator(device=_device()).manual_seed(seed)


def _lengths(n_seqs, total, g):
    """Lognormal sequence lengths (at least 2) that add up to ``total``."""
    w = torch.exp(torch.randn(n_seqs, generator=g, dtype=torch.float64) * 0.8)
    lens = 2 + torch.floor((total - 2 * n_seqs) * w / w.sum()).long()
    lens[-1] += total - int(lens.sum())
    return lens


def _token_batch(tokens, n_seqs, g, gd):
    """Packed layout of a micro-batch: ``cu_seqlens``, the response mask (prompts and each
    sequence's last token left out) and one group-normalised advantage per sequence."""
    dev = _device()
    lens = _lengths(n_seqs, tokens, g)
    cu = torch.cat([torch.zeros(1, dtype=torch.long), lens.cumsum(0)]).to(dev)
    lens = lens.to(dev)
    pos = torch.arange(tokens, device=dev) - cu[:-1].repeat_interleave(lens, output_size=tokens)
    own = lens.repeat_interleave(lens, output_size=tokens)
    mask = (pos >= own // 4) & (pos < own - 1)
    adv = torch.randn(n_seqs, generator=gd, device=dev).repeat_interleave(lens, output_size=tokens)
    return cu.to(torch.int32), mask, adv


def _laplace(shape, scale, gd):
    u = torch.rand(shape, generator=gd, device=_device()) - 0.5
    return -scale * u.sign() * torch.log1p(-2 * u.abs() * (1 - 1e-6))


def _rejection(case):
    if case["level"] == "token":
        return RejectionSamplingConfig(level="token", action="mask", metric="ratio", lower=0.5, upper=2.0)
    return RejectionSamplingConfig(level="sequence", action="mask", metric="kl_k2", agg="mean", upper=0.012)


def _loss_fn(case):
    return functools.partial(
        grpo_loss_fn, eps_clip=0.2, eps_clip_higher=0.28 if case["loss"] == "cispo" else None, c_clip=None,
        rejection_sampling=None if case["loss"] == "sapo" else _rejection(case),
        use_cispo_loss=case["loss"] == "cispo", use_sapo_loss=case["loss"] == "sapo",
        defer_host_reads=case.get("defer", False),
    )


class _Trunk(torch.nn.Module):
    """Stands for the transformer in front of the lm_head: its output is the leaf it is given."""

    def forward(self, input_ids=None, inputs_embeds=None):
        return inputs_embeds[None]


class _CausalLM(torch.nn.Module):
    def __init__(self, weight):
        super().__init__()
        self.model = _Trunk()
        self.lm_head = torch.nn.Linear(weight.size(1), weight.size(0), bias=False, device="meta")
        self.lm_head.weight = torch.nn.Parameter(weight)


def _n_valid(mb):
    return mb["loss_mask"].count_nonzero()


def _prepare_step(case, g, gd):
    dev = _device()
    h, v = case["hidden"], case["vocab"]
    weight = torch.randn(v, h, generator=gd, device=dev, dtype=torch.bfloat16).mul_(0.02)
    parts = []
    for i in range(case["micro"]):
        t = case["tokens"] // case["micro"] + (case["tokens"] % case["micro"] if i == 0 else 0)
        hidden = torch.randn(t, h, generator=gd, device=dev, dtype=torch.bfloat16)
        ids = torch.randint(0, v, (t,), generator=gd, device=dev)
        labels = torch.roll(ids, -1)
        # The log-probs of the policy before the update: the label's logit minus the log-sum-exp of
        # normally distributed logits. The rollout engine's differ from them by Laplace noise.
        hf = hidden.float()
        own = torch.empty(t, device=dev)
        for a in range(0, t, 8192):
            own[a:a + 8192] = (hf[a:a + 8192] * weight[labels[a:a + 8192]].float()).sum(-1)
        prox = own - math.log(v) - 0.5 * (0.02 * hf.norm(dim=-1)) ** 2
        cu, mask, adv = _token_batch(t, max(1, case["seqs"] // case["micro"]), g, gd)
        data = dict(logprobs=prox + _laplace((t,), 0.1, gd), prox_logp=prox, advantages=adv, loss_mask=mask,
                    cu_seqlens=cu)
        parts.append(dict(hidden=hidden.requires_grad_(True), ids=ids, labels=labels, data=data))
    state = dict(case=case, parts=parts, loss_fn=_loss_fn(case))
    if case["master"]:
        state["lm"] = _CausalLM(weight.float())
        state["head"] = FusedLMHeadAdapter(state["lm"], temperature=1.0)
        state["micro_batches"] = [
            dict(model_inputs=dict(input_ids=p["ids"][None], inputs_embeds=p["hidden"]), mb_input=p["data"])
            for p in parts
        ]
    else:
        state["weight"] = weight.requires_grad_(True)
    return state


def _prepare_logp(case, g, gd):
    dev = _device()
    t, h, v = case["tokens"], case["hidden"], case["vocab"]
    return dict(case=case,
                weight=torch.randn(v, h, generator=gd, device=dev, dtype=torch.bfloat16).mul_(0.02),
                hidden=torch.randn(1, t, h, generator=gd, device=dev, dtype=torch.bfloat16),
                inputs=dict(input_ids=torch.randint(0, v, (1, t), generator=gd, device=dev)))


def _prepare_logits(case, g, gd):
    dev = _device()
    t, v = case["rows"], case["vocab"]
    dtype = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    return dict(case=case,
                logits=torch.randn(t, v, generator=gd, device=dev, dtype=dtype).mul_(2.0).requires_grad_(case["grad"]),
                labels=torch.randint(0, v, (t,), generator=gd, device=dev),
                grad=torch.randn(t, generator=gd, device=dev) / t)


def _prepare_loss(case, g, gd):
    dev = _device()
    t = case["tokens"]
    cu, mask, adv = _token_batch(t, case["seqs"], g, gd)
    normal = lambda: torch.randn(t, generator=gd, device=dev)  # noqa: E731
    if case["loss"] == "critic":
        value = normal().requires_grad_(True)
        return dict(case=case, value=value, old=value.detach() + 0.2 * normal(), target=value.detach() + normal(),
                    mask=mask)
    prox = 0.5 * normal() - 1.0
    logprobs = (prox + 0.1 * normal()).requires_grad_(True)
    data = dict(logprobs=prox + _laplace((t,), 0.1, gd), prox_logp=prox, advantages=adv, loss_mask=mask, cu_seqlens=cu)
    return dict(case=case, logprobs=logprobs, entropy=torch.rand(t, generator=gd, device=dev) * 3, data=data,
                loss_fn=_loss_fn(case))


def _prepare_adv(case, g, gd):
    dev = _device()
    bs, length = case["rows"], case["length"]
    lens = torch.clamp(torch.exp(torch.randn(bs, generator=gd, device=dev) * 0.8 + math.log(length * 0.3)).long(),
                       16, length)
    pos = torch.arange(length, device=dev)[None, :]
    attn = pos < lens[:, None]
    normal = lambda: torch.randn(bs, length, generator=gd, device=dev)  # noqa: E731
    data = dict(input_ids=torch.randint(0, 151936, (bs, length), generator=gd, device=dev), attention_mask=attn,
                loss_mask=attn & (pos >= lens[:, None] // 4), logprobs=0.1 * normal() - 1, ref_logp=0.1 * normal() - 1,
                rewards=(torch.rand(bs, generator=gd, device=dev) > 0.5).float())
    if case["critic"]:
        data["values"] = normal()
    if case["unit"] == "turn":  # turns of about 300 tokens
        data["turn_ids"] = torch.where(attn, (pos // 300).expand(bs, length), -1).to(torch.int32).contiguous()
    norm = Normalization(NormConfig(mean_level="group", std_level="group", group_size=case["group"]))
    options = dict(kl_ctl=0.01, kl_estimator=KLEstimator("k1"), reward_norm=norm, adv_norm=norm, discount=1.0,
                   gae_lambda=0.95 if case["critic"] else 1.0, gae_timestep_unit=case["unit"])
    return dict(case=case, data=data, options=options)


def _prepare_gae(case, g, gd):
    dev = _device()
    n, tokens = case["seqs"], case["seqs"] * case["mean_len"]
    cu, mask, _ = _token_batch(tokens, n, g, gd)
    rewards = torch.zeros(tokens, device=dev)
    rewards[cu[1:].long() - 2] = (torch.rand(n, generator=gd, device=dev) > 0.5).float()
    return dict(case=case, rewards=rewards, values=torch.randn(tokens, generator=gd, device=dev), mask=mask.float(),
                cu=cu, norm=Normalization(NormConfig(mean_level="group", std_level="group", group_size=case["group"])))


def _prepare_pack(case, g, gd):
    dev = _device()
    bs, length = case["rows"], case["length"]
    # evenly spread lengths up to the padded one, in the seed's order
    lens = torch.linspace(max(1, length // 16), length, bs).long()[torch.randperm(bs, generator=g)]
    attn = torch.arange(length, device=dev)[None, :] < lens.to(dev)[:, None]
    normal = lambda: torch.randn(bs, length, generator=gd, device=dev)  # noqa: E731
    data = dict(attention_mask=attn, input_ids=torch.randint(0, 151936, (bs, length), generator=gd, device=dev),
                logprobs=normal(), prox_logp=normal(), advantages=normal(), loss_mask=attn.clone(), position=normal())
    total = int(lens.sum())
    return dict(case=case, data=data, pad_to=(total + 256) // 256 * 256, lens=lens.tolist(),
                order=torch.randperm(bs, generator=g).tolist(), result=torch.randn(total, generator=gd, device=dev))


def prepare(case, seed):
    g, gd = _gens(seed)
    return globals()["_prepare_" + case["path"]](case, g, gd)


# -- one pass ---------------------------------------------------------------------------------

def _logged(stats):
    """The reduced statistics of a loss call as the table a trainer logs: one row per statistic."""
    rows = [stats[k] for k in sorted(stats) if isinstance(stats[k], dict)]
    return np.array([[r["avg"], r["min"], r["max"]] for r in rows], dtype=np.float64)


def _run_step(s):
    case, parts = s["case"], s["parts"]
    for p in parts:
        p["hidden"].grad = None
    if case["master"]:
        s["lm"].zero_grad()
        losses = s["head"].forward_backward_batch(s["micro_batches"], s["loss_fn"], _n_valid)
        return losses, [p["hidden"].grad for p in parts], s["lm"].lm_head.weight.grad
    s["weight"].grad = None
    (p,) = parts
    stats = {} if case["stats"] == "reduced" else None
    out = fused_lm_head_logprobs_entropy(p["hidden"], s["weight"], p["labels"], temperature=1.0)
    loss = s["loss_fn"](out.logprobs, out.entropy, p["data"], vocab_min_logits=out.vocab_min_logits,
                        vocab_max_logits=out.vocab_max_logits, stats=stats, stats_mode="reduced")
    loss.backward()
    table = None
    if stats is not None:
        table = _logged(stats["reduction"].results if case["defer"] else stats)
    return loss.detach(), p["hidden"].grad, s["weight"].grad, out.logprobs.detach(), out.entropy, table


def _run_logp(s):
    return compute_logprobs(s["hidden"], s["weight"], s["inputs"], temperature=1.0, pad_length=s["case"]["pad"])


def _run_logits(s):
    s["logits"].grad = None
    lp, ent = gather_logprobs_entropy(s["logits"], s["labels"], temperature=1.0)
    if s["case"]["grad"]:
        lp.backward(s["grad"])
    return lp.detach(), ent.detach(), s["logits"].grad


def _run_loss(s):
    case = s["case"]
    if case["loss"] == "critic":
        s["value"].grad = None
        loss, stat = ppo_critic_loss_fn(s["value"], s["old"], s["target"], 0.2, s["mask"])
        loss.backward()
        return loss.detach(), s["value"].grad, stat["clip_mask"], stat["loss"]
    s["logprobs"].grad = None
    stats = {} if case["stats"] != "none" else None
    loss = s["loss_fn"](s["logprobs"], s["entropy"], s["data"], stats=stats,
                        stats_mode="tensors" if case["stats"] == "tensors" else "reduced")
    loss.backward()
    if case["stats"] == "reduced":
        stats = _logged(stats)
    return loss.detach(), s["logprobs"].grad, stats


def _run_adv(s):
    out = compute_advantages(dict(s["data"]), **s["options"])
    return {k: out[k] for k in ("advantages", "returns", "kl_rewards", "tot_rewards", "loss_mask", "logprobs")}


def _run_gae(s):
    return compute_gae_packed_normalized(s["rewards"], s["values"], s["mask"], s["cu"], None, 1.0, 0.95, s["norm"])


def _run_pack(s):
    packed = pack_tensor_dict(s["data"])
    padded, pad_length, old_cu, _ = pad_packed_tensor_dict(packed, s["pad_to"])
    back = unpack_reorder_pad(s["result"], s["lens"], s["order"])
    return padded, pad_length, old_cu, back


def run(state):
    return globals()["_run_" + state["case"]["path"]](state)
