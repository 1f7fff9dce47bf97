"""The work that the users of this package have it do, as cases that can be timed and compared.

A case is a dict of plain values.  ``prepare`` makes, on the GPU and from the seed alone, what the user's program holds before
the call; ``run`` is one pass through the package's public entry points as a trainer or a scoring worker calls them, and
returns everything that the pass computes: log-probabilities, entropies, losses and gradients.

``path`` says which entry point a case goes through:

  score         from_parallel_hidden_to_logprobs without a gradient: the reference policy's log-probabilities
  score_tail    action_log_probs_from_hidden without a gradient, entropy included: the old policy's log-probabilities
  train_dense   from_parallel_hidden_to_logprobs, the actor loss, gradients
  train_packed  the same for sequences packed into one token stream (attention-mask layout)
  train_tail    action_log_probs_from_hidden with entropy, the actor loss with KL, entropy and off-policy terms, gradients
  head          linear_cross_entropy with upstream gradients on the log-probabilities and, optionally, the entropy
  fused         FusedLinearLogprobHip.apply and the gradient of the summed negative log-probabilities
  soft_ce       draft_soft_ce_from_hidden and the draft head's gradient
  soft_ce_topk  draft_soft_ce_topk_from_hidden and the draft head's gradient
  logits        action_log_probs_from_logits on materialised logits and their gradient

Sizes: ``batch`` x ``seq`` tokens (``seq`` is the longest sequence of a packed stream), ``hidden``, ``vocab``.  ``masked`` is the
share of a sequence that is prompt, which takes no gradient.
"""

from __future__ import annotations

from types import SimpleNamespace

import torch

from skyrl_amd.fused_linear_logprob_hip import FusedLinearLogprobHip, linear_cross_entropy
from skyrl_amd.model_utils import from_parallel_hidden_to_logprobs, from_parallel_hidden_to_logprobs_packed_sequences
from skyrl_amd.model_wrapper import action_log_probs_from_hidden, action_log_probs_from_logits
from skyrl_amd.mtp_soft_ce import draft_soft_ce_from_hidden, draft_soft_ce_topk_from_hidden, shift_mask_for_mtp
from skyrl_amd.policy_loss import actor_loss

DEFAULTS = {"batch": 1, "temperature": 1.0, "masked": 0.5, "entropy_grad": False, "frozen": False, "fp32_weight": False, "topk": 0}


def listed():
    return [
        # A worker scores one short answer as it arrives: the smallest call, bounded by launches and latency.
        dict(name="score one answer", path="score", seq=137, hidden=896, vocab=151936),
        # The smallest forward configuration of the benchmark: four sequences, log-probabilities and entropy.
        dict(name="score a group", path="score_tail", batch=4, seq=512, hidden=896, vocab=151936),
        # The largest forward configuration: sixteen long sequences under the reference policy.
        dict(name="score a long batch", path="score", batch=16, seq=2048, hidden=5120, vocab=151936),
        # A micro-batch of one sequence, the trainer's default, at a length that fits no tile.
        dict(name="train one sequence", path="train_dense", seq=611, hidden=1536, vocab=151936, masked=0.3),
        # The second benchmark configuration as the FSDP worker runs it: half of the tokens are prompt, KL, entropy and
        # off-policy terms in the loss.
        dict(name="train a group", path="train_tail", batch=8, seq=1024, hidden=1536, vocab=151936, entropy_grad=True),
        # The headline configuration: a packed stream of 16384 tokens, temperature 0.6, gradients on both outputs.
        dict(name="train a packed stream", path="head", seq=16384, hidden=3584, vocab=152064, temperature=0.6, masked=0.0,
             entropy_grad=True),
        # The long-context sweep on one vocabulary shard: more tokens than one block of the library takes.
        dict(name="train a long context", path="fused", seq=65536, hidden=2048, vocab=62080, masked=0.0),
        # Adapter training (the head is frozen) on a vocabulary with a few tokens added to it, sequences of unlike lengths
        # packed into one stream.
        dict(name="train an adapter", path="train_packed", batch=5, seq=1000, hidden=4096, vocab=128261, temperature=0.9,
             masked=0.4, frozen=True),
        # An output layer kept in fp32 next to bf16 hidden states.
        dict(name="train an fp32 head", path="head", batch=3, seq=700, hidden=1024, vocab=32000, masked=0.5, fp32_weight=True),
        # The draft head's loss against the policy, full vocabulary and top-k.
        dict(name="draft loss", path="soft_ce", batch=4, seq=1024, hidden=2048, vocab=151936, masked=0.3),
        dict(name="draft loss top-k", path="soft_ce_topk", batch=2, seq=900, hidden=2048, vocab=151936, masked=0.3, topk=32),
        # The worker that keeps its logits: the tail of the forward and its gradient, HBM-bound.
        dict(name="logits tail", path="logits", batch=3, seq=515, hidden=0, vocab=151936, masked=0.5, entropy_grad=True),
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    path = rng.choice(["score", "score_tail", "train_dense", "train_packed", "train_tail", "head", "head", "fused", "soft_ce",
                       "soft_ce_topk", "logits"])
    vocab = _log_uniform(rng, 32000, 248320)
    vocab = rng.choice([vocab // 128 * 128, vocab // 128 * 128, vocab // 64 * 64, vocab])  # most vocabularies are padded
    case = dict(path=path, batch=rng.choice([1, 1, 2, 3, 4, 8, 16]), hidden=64 * _log_uniform(rng, 8, 80), vocab=vocab,
                temperature=rng.choice([1.0, 1.0, 0.6, 0.9]), masked=rng.choice([0.0, 0.3, 0.5, 0.7]))
    if path in ("head", "train_tail", "logits"):
        case["entropy_grad"] = rng.random() < 0.5
    if path == "head":
        case["fp32_weight"] = rng.random() < 0.3
    if path.startswith("train"):
        case["frozen"] = rng.random() < 0.25
    if path == "soft_ce_topk":
        case["topk"] = rng.choice([8, 32, 64, 128])
    if path.startswith("soft_ce"):
        case["temperature"] = 1.0
    if path == "logits":
        case["hidden"] = 0
        tokens = min(_log_uniform(rng, 16, 16384), (1 << 31) // vocab)
    else:
        # the longest stream that costs no more than the headline configuration (6 T V H with every token active)
        cost = {"score": 2, "score_tail": 2, "soft_ce_topk": 2}.get(path, 6) * (3 if case.get("fp32_weight") else 1)
        limit = int(6 * 16384 * 3584 * 152064 / (cost * vocab * case["hidden"]))
        tokens = min(_log_uniform(rng, 16, 65536), limit)
    case["batch"] = min(case["batch"], max(1, tokens // 16))
    case["seq"] = max(4, tokens // case["batch"])
    return case


def _lengths(c):
    """Lengths of the sequences of a packed stream: from a sixteenth of the longest one up to it, in even steps."""
    n, longest = c["batch"], c["seq"]
    return [longest if n == 1 else max(2, longest * (n - 1 + 15 * i) // (16 * (n - 1))) for i in range(n)]


def _tokens(c):
    return sum(_lengths(c)) if c["path"] == "train_packed" else c["batch"] * c["seq"]


def _token_logprobs(hidden, weight, labels, temperature):
    """Log-probabilities of ``labels``, by plain torch in slabs: what an earlier scoring pass has left with the trainer."""
    out, w = [], weight.detach().to(torch.bfloat16)
    rows = max(1, (1 << 27) // w.shape[0])
    for h, y in zip(hidden.detach().split(rows), labels.split(rows)):
        z = torch.matmul(h, w.t()).float() / temperature
        out.append(z.gather(1, y.unsqueeze(1)).squeeze(1) - torch.logsumexp(z, dim=1))
    return torch.cat(out)


def _algorithm(c):
    """The trainer's algorithm section: the clipped surrogate, and for the FSDP path the other terms that it can carry."""
    tail = c["path"] == "train_tail"
    return SimpleNamespace(
        policy_loss_type="dual_clip" if c["path"] == "train_packed" else "regular", eps_clip_low=0.2, eps_clip_high=0.28,
        clip_ratio_c=3.0, use_kl_loss=tail, kl_loss_coef=0.001, kl_estimator_type="k3",
        use_entropy_loss=bool(c["entropy_grad"]), entropy_loss_coef=0.01,
        off_policy_correction=SimpleNamespace(tis_ratio_type="token", token_tis_ratio_clip_high=2.0) if tail else None)


def prepare(case, seed):
    c = {**DEFAULTS, **case}
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    rand = lambda *shape: torch.randn(*shape, generator=gen, device=dev)  # noqa: E731
    B, S, H, V, path, T = c["batch"], c["seq"], c["hidden"], c["vocab"], c["path"], _tokens(c)
    s = SimpleNamespace(case=c, path=path, vocab=V, temperature=float(c["temperature"]), topk=c["topk"], algorithm=_algorithm(c))
    trains = path not in ("score", "score_tail")
    prompt = min(S - 2, int(S * c["masked"]))
    s.actions = S - 1 - prompt

    def loss_inputs(logprobs, shape):
        """What the trainer holds per token: the two earlier policies' log-probabilities, the rollout engine's, advantages."""
        n = float(logprobs.numel())
        near = lambda spread: (logprobs + spread * rand(logprobs.numel())).reshape(shape)  # noqa: E731
        s.old, s.base, s.rollout = near(0.05), near(0.1), near(0.02)
        s.advantages = (rand(shape[0], 1) / n).expand(shape).contiguous()

    if path == "logits":
        s.logits = torch.empty(B, S, V, dtype=torch.bfloat16, device=dev)
        for b in range(B):
            s.logits[b] = 3.0 * rand(S, V)
        s.logits.requires_grad_(True)
        s.tokens = torch.randint(0, V, (B, S), generator=gen, device=dev)
        s.attention_mask = torch.ones(B, S, dtype=torch.int64, device=dev)
        s.upstream = rand(B, s.actions)
        s.upstream_entropy = 0.01 * rand(B, S) if c["entropy_grad"] else None
        return s

    weight = torch.empty(V, H, dtype=torch.float32 if c["fp32_weight"] else torch.bfloat16, device=dev)
    for rows in weight.split(max(1, (1 << 27) // H)):
        rows.copy_(rand(rows.shape[0], H) * (3.0 / H ** 0.5))
    s.weight = weight.requires_grad_(trains and not c["frozen"] and not path.startswith("soft_ce"))
    hidden = rand(T, H).to(torch.bfloat16)
    labels = torch.randint(0, V, (T,), generator=gen, device=dev)

    if path == "head":
        s.hidden, s.labels = hidden.requires_grad_(True), labels
        active = (torch.arange(S, device=dev) >= prompt).repeat(B)
        s.upstream = rand(T) * active
        s.upstream_entropy = 0.01 * rand(T) * active if c["entropy_grad"] else None
        return s
    if path.startswith("soft_ce"):
        s.teacher = (hidden + 0.5 * rand(T, H)).to(torch.bfloat16).reshape(B, S, H)
        s.hidden = hidden.reshape(B, S, H).requires_grad_(True)
        s.mask = (torch.arange(S, device=dev) >= prompt).float().repeat(B, 1)
        return s
    if path == "train_packed":
        lengths = _lengths(c)
        order = torch.randperm(B, generator=torch.Generator().manual_seed(int(seed))).tolist()
        lengths = [lengths[i] for i in order]
        s.seq = max(lengths)
        cu = [0]
        for n in lengths:
            cu.append(cu[-1] + n)
        s.cu = torch.tensor(cu, dtype=torch.int32, device=dev)
        s.hidden, s.tokens = hidden.reshape(1, T, H).requires_grad_(True), labels.reshape(1, T)
        at, length = torch.arange(s.seq, device=dev), torch.tensor(lengths, device=dev).unsqueeze(1)
        s.attention_mask = at.unsqueeze(0) < length
        s.loss_mask = ((at[:-1] >= (length * c["masked"]).long()) & (at[:-1] < length - 1)).float()
        nxt = labels.roll(-1)
        lp = torch.zeros(B, s.seq - 1, device=dev)
        lp[s.attention_mask[:, 1:]] = torch.cat([p[:-1] for p in _token_logprobs(hidden, weight, nxt, s.temperature).split(lengths)])
        loss_inputs(lp.reshape(-1), (B, s.seq - 1))
        return s
    s.hidden, s.tokens = hidden.reshape(B, S, H), labels.reshape(B, S)
    if not trains:
        s.attention_mask = torch.ones(B, S, dtype=torch.int64, device=dev)
        return s
    s.hidden.requires_grad_(True)
    if path == "fused":
        return s
    lp = _token_logprobs(hidden, weight, s.tokens.roll(-1, dims=1).reshape(-1), s.temperature).reshape(B, S)[:, :-1]
    if path == "train_tail":
        s.attention_mask = torch.ones(B, S, dtype=torch.int64, device=dev)
        s.loss_mask = torch.ones(B, s.actions, device=dev)
        loss_inputs(lp[:, prompt:].reshape(-1), (B, s.actions))
    else:
        s.loss_mask = (torch.arange(S - 1, device=dev) >= prompt).float().repeat(B, 1)
        loss_inputs(lp.reshape(-1), (B, S - 1))
    return s


def _gradients(loss, *leaves):
    return torch.autograd.grad(loss, [t for t in leaves if t.requires_grad])


def run(s):
    path, V = s.path, s.vocab
    if path == "score":
        return from_parallel_hidden_to_logprobs(s.hidden, s.weight, s.tokens, 0, V, None, inference_only=True,
                                                temperature=s.temperature)
    if path == "score_tail":
        with torch.no_grad():
            logprobs, extra = action_log_probs_from_hidden(s.hidden, s.weight, s.tokens, s.actions, s.attention_mask, s.temperature,
                                                           return_output=True, compute_entropy=True)
        return logprobs, extra["entropy"]
    if path == "head":
        logprobs, entropy = linear_cross_entropy(s.hidden, s.weight, s.labels, s.temperature, "none", None)
        loss = (logprobs * s.upstream).sum()
        if s.upstream_entropy is not None:
            loss = loss + (entropy * s.upstream_entropy).sum()
        return logprobs.detach(), entropy.detach(), _gradients(loss, s.hidden, s.weight)
    if path == "fused":
        logprobs = FusedLinearLogprobHip.apply(s.hidden, s.weight, s.tokens, 0, V, 1024, None, False)
        return logprobs.detach(), _gradients((-logprobs).sum(), s.hidden, s.weight)
    if path == "soft_ce":
        loss = draft_soft_ce_from_hidden(s.hidden, s.teacher, s.weight, shift_mask_for_mtp(s.mask), 0)
        return loss.detach(), _gradients(loss, s.hidden)
    if path == "soft_ce_topk":
        loss = draft_soft_ce_topk_from_hidden(s.hidden, s.teacher, s.weight, shift_mask_for_mtp(s.mask), s.topk, roll_shift=1)
        return loss.detach(), _gradients(loss, s.hidden)
    if path == "logits":
        logprobs, extra = action_log_probs_from_logits(s.logits, s.tokens, s.actions, s.attention_mask, s.temperature,
                                                       return_output=True, compute_entropy=True, inplace_backward=False)
        loss = (logprobs * s.upstream).sum()
        if s.upstream_entropy is not None:
            loss = loss + (extra["entropy"].float() * s.upstream_entropy).sum()
        return logprobs.detach(), extra["entropy"].detach(), _gradients(loss, s.logits)
    if path == "train_tail":
        logprobs, extra = action_log_probs_from_hidden(s.hidden, s.weight, s.tokens, s.actions, s.attention_mask, s.temperature,
                                                       return_output=True, compute_entropy=True,
                                                       entropy_requires_grad=s.algorithm.use_entropy_loss)
        loss, metrics = actor_loss(logprobs, s.old, s.advantages, s.algorithm, s.loss_mask, base_log_probs=s.base,
                                   entropy=extra["entropy"][:, -s.actions - 1:-1], rollout_logprobs=s.rollout)
        return logprobs.detach(), extra["entropy"].detach(), loss.detach(), _gradients(loss, s.hidden, s.weight)
    if path == "train_packed":
        logprobs = from_parallel_hidden_to_logprobs_packed_sequences(
            s.hidden, s.weight, s.tokens, s.cu, s.seq, 0, V, None, attention_mask=s.attention_mask, temperature=s.temperature)
    else:
        logprobs = from_parallel_hidden_to_logprobs(s.hidden, s.weight, s.tokens, 0, V, None, temperature=s.temperature)
    loss, metrics = actor_loss(logprobs, s.old, s.advantages, s.algorithm, s.loss_mask)
    return logprobs.detach(), loss.detach(), metrics["clip_ratio"].detach(), _gradients(loss, s.hidden, s.weight)


def work(case):
    """Multiplications and additions of the products that a pass needs, and every input read and output written once."""
    c = {**DEFAULTS, **case}
    T, H, V, path = _tokens(c), c["hidden"], c["vocab"], c["path"]
    if path == "logits":
        return {"bytes": 4.0 * T * V, "flops": 10.0 * T * V}
    product = 2.0 * T * H * V
    weight, hidden = (4.0 if c["fp32_weight"] else 2.0) * V * H, 2.0 * T * H
    if path.startswith("score"):
        return {"bytes": weight + hidden + 20.0 * T, "flops": product}
    active = 1.0 - c["masked"]
    if path == "soft_ce":
        return {"bytes": weight + 3 * hidden, "flops": (2.0 + active) * product}
    if path == "soft_ce_topk":
        return {"bytes": weight + 3 * hidden, "flops": product + 6.0 * T * c["topk"] * H}
    gradients = 1.0 if c["frozen"] else 2.0
    return {"bytes": weight * gradients + 2 * hidden + 40.0 * T, "flops": (1.0 + gradients * active) * product}


def tolerance(case):
    """About four times what each path showed against the same products and sums in 64 bits, over the listed and 28 drawn cases."""
    path = case["path"]
    if path.startswith("score"):  # fp32 sums: 1e-7 on log-probabilities, up to 1e-6 on a small entropy
        return {"rel": 5e-6, "max": 3e-5}
    if path == "logits":  # 2e-6, 7e-3: an element-wise bf16 result whose last bit may fall the other way
        return {"rel": 1e-4, "max": 3e-2}
    if path == "soft_ce_topk":  # 1e-4, 8e-3: fp32 sums of k rows, rounded to bf16 once
        return {"rel": 4e-4, "max": 3e-2}
    # gradients: dz is rounded to bf16 in front of the products and the result behind them; 3.3e-3, single elements 0.15
    return {"rel": 1.2e-2, "max": 0.6}
