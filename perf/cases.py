"""Performance cases: the work that a training program has this framework do, through its public entry points.

Six kinds of pass, each named by what a worker of an RL iteration calls:

* ``step``        an actor update's loss from the logits, forward and backward (loss object, dlogits)
* ``score``       a forward-only pass over the logits (old or reference log-probs)
* ``hidden_step`` the same update from the hidden states and the lm_head weight (dHidden, dWeight)
* ``hidden_score`` the forward-only pass from the hidden states and the lm_head weight
* ``value``       PPO's value side: KL-penalised rewards, GAE with whitening, critic loss and its backward
* ``experience``  the columns of an iteration: wire format, masks, group advantages, packing

A case is a dict of plain values; everything it measures follows from it and a seed.
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "mindspeed-rl_amd"))       # imported with the repository's root as working folder

import mindspeed_rl_amd as mrl  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32, "f16": torch.float16}
_BYTES = {"bf16": 2, "f32": 4, "f16": 2}
_GROUP = 8                  # responses per prompt
_DRIFT = 0.1                # spread of log(new policy / old policy) over the tokens of an update


# ------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest update: 4 x 4 short responses, a 32 k vocabulary in fp32; launches and host latency count
        dict(name="step_small_f32", kind="step", loss="grpo", layout="packed", dtype="f32", vocab=32000, seqs=16,
             prompt_lo=1, prompt_hi=1, resp_lo=64, resp_hi=256, lengths=1, micro=1),
        # the ordinary update: one micro-batch of a 32 k-token budget, prompts and responses packed, 152 k vocabulary
        dict(name="step_packed_bf16", kind="step", loss="grpo", layout="packed", dtype="bf16", vocab=152064, seqs=20,
             prompt_lo=64, prompt_hi=512, resp_lo=512, resp_hi=2048, lengths=2, micro=1),
        # the same rows as fp32 logits, which is what a model's last stage hands over without a cast
        dict(name="step_packed_f32", kind="step", loss="grpo", layout="packed", dtype="f32", vocab=152064, seqs=8,
             prompt_lo=64, prompt_hi=512, resp_lo=512, resp_hi=2048, lengths=3, micro=1),
        # padded [B, S, V] logits without remove-padding, DAPO with a mask of its own and sequence means
        dict(name="step_padded_bf16", kind="step", loss="dapo_seq", layout="padded", dtype="bf16", vocab=129280, seqs=16,
             prompt_lo=128, prompt_hi=512, resp_lo=256, resp_hi=1536, lengths=4, micro=1),
        # long responses: two of them fill the micro-batch, one of 32 whose loss is divided before the backward
        dict(name="step_long_bf16", kind="step", loss="dapo", layout="packed", dtype="bf16", vocab=129280, seqs=2,
             prompt_lo=512, prompt_hi=2048, resp_lo=12288, resp_hi=16384, lengths=5, micro=32),
        # a 32 k vocabulary with three added tokens and no padding: rows start at odd addresses; PPO, small model
        dict(name="step_odd_vocab", kind="step", loss="ppo", layout="packed", dtype="bf16", vocab=32003, seqs=16,
             prompt_lo=16, prompt_hi=200, resp_lo=128, resp_hi=1024, lengths=6, micro=1),
        # reference-policy log-probs at the forward budget of 64 k tokens
        dict(name="score_packed_bf16", kind="score", layout="packed", dtype="bf16", vocab=152064, seqs=40, prompt_lo=64,
             prompt_hi=512, resp_lo=512, resp_hi=2048, lengths=7, entropy=False),
        # old log-probs and entropies of a few short padded samples
        dict(name="score_small", kind="score", layout="padded", dtype="bf16", vocab=32000, seqs=8, prompt_lo=8,
             prompt_hi=64, resp_lo=16, resp_hi=128, lengths=8, entropy=True),
        # log-probs straight from the hidden states of a 7 B-sized model
        dict(name="hidden_score", kind="hidden_score", layout="packed", vocab=152064, hidden=3584, seqs=12, prompt_lo=64,
             prompt_hi=512, resp_lo=512, resp_hi=2048, lengths=9, entropy=False),
        # the update from the hidden states of the same model
        dict(name="hidden_step", kind="hidden_step", loss="grpo", layout="packed", vocab=152064, hidden=3584, seqs=10,
             prompt_lo=64, prompt_hi=512, resp_lo=512, resp_hi=2048, lengths=10, micro=1),
        # PPO's value side for a batch of 128 responses
        dict(name="value_side", kind="value", seqs=128, width=2048, prompt=256, lengths=11, penalty="low_var_kl"),
        # an iteration's columns for 256 samples
        dict(name="experience", kind="experience", seqs=256, prompt_lo=16, prompt_hi=512, resp_lo=32, resp_hi=2048,
             lengths=12, align=8),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _draw_vocab(rng, hi):
    v = int(_log_uniform(rng, 8000, hi))
    unit = rng.choice([1, 8, 64, 128])
    return max(v // unit * unit, unit)


def _draw_lengths(rng, tokens, longest):
    """Sequences whose prompts and responses add up to about `tokens`."""
    mean = min(_log_uniform(rng, 48, longest), tokens)
    hi = max(8, int(mean * 1.3))
    lo = max(4, int(hi * rng.uniform(0.1, 0.8)))
    p_hi = max(1, int(hi * rng.uniform(0.02, 0.5)))
    p_lo = rng.randint(1, p_hi)
    per_seq = (lo + hi) / 2 + (p_lo + p_hi) / 2
    return dict(seqs=max(1, int(tokens / per_seq)), prompt_lo=p_lo, prompt_hi=p_hi, resp_lo=lo, resp_hi=hi,
                lengths=rng.randrange(1 << 30))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "step", "score", "score", "hidden_score", "hidden_step", "value",
                       "experience"])
    if kind in ("step", "score"):
        dtype = rng.choice(["bf16", "bf16", "bf16", "f32", "f16"])
        vocab = _draw_vocab(rng, 152064)
        budget = _log_uniform(rng, 3e7, 5e9 if kind == "step" else 8e9)
        tokens = min(max(64, budget / (vocab * _BYTES[dtype])), 65536)
        c = dict(kind=kind, layout=rng.choice(["packed", "packed", "padded"]), dtype=dtype, vocab=vocab,
                 **_draw_lengths(rng, tokens, 12288))
        if c["layout"] == "padded":
            c["seqs"] = max(1, c["seqs"] * 2 // 3)          # padding rows count as well
        if kind == "step":
            c.update(loss=rng.choice(["grpo", "dapo", "dapo_seq", "ppo"]), micro=rng.choice([1, 1, 4, 32]))
        else:
            c.update(entropy=rng.choice([False, True]))
        return c
    if kind in ("hidden_score", "hidden_step"):
        hidden = max(512, int(_log_uniform(rng, 512, 5120)) // 64 * 64)
        vocab = int(_log_uniform(rng, 8000, 152064)) // 8 * 8
        flops = _log_uniform(rng, 2e11, 1.2e13)             # of one product
        tokens = min(max(64, flops / (2.0 * hidden * vocab)), 32768)
        c = dict(kind=kind, layout=rng.choice(["packed", "packed", "padded"]), vocab=vocab, hidden=hidden,
                 **_draw_lengths(rng, tokens, 4096))
        if c["layout"] == "padded":
            c["seqs"] = max(1, c["seqs"] * 2 // 3)
        if kind == "hidden_step":
            c.update(loss=rng.choice(["grpo", "dapo", "ppo"]), micro=rng.choice([1, 1, 4]))
        else:
            c.update(entropy=rng.choice([False, True]))
        return c
    if kind == "value":
        width = int(_log_uniform(rng, 100, 4096))
        return dict(kind=kind, seqs=max(2, min(int(_log_uniform(rng, 4, 512)), 500000 // width)), width=width,
                    prompt=rng.randint(1, 512), lengths=rng.randrange(1 << 30),
                    penalty=rng.choice(["low_var_kl", "kl", "abs", "mse"]))
    hi = int(_log_uniform(rng, 64, 4096))
    return dict(kind=kind, seqs=_GROUP * max(1, min(int(_log_uniform(rng, 1, 64)), 500000 // (hi * _GROUP))),
                prompt_lo=rng.randint(1, 16), prompt_hi=rng.randint(17, 512), resp_lo=rng.randint(1, hi // 2), resp_hi=hi,
                lengths=rng.randrange(1 << 30), align=rng.choice([1, 2, 8]))


# ------------------------------------------------------------------------------------------ shapes
def _lengths(case):
    """Prompt and response lengths of the case's samples (part of its shape, so not made from the seed)."""
    r = random.Random(case["lengths"])
    plen = [r.randint(case["prompt_lo"], case["prompt_hi"]) for _ in range(case["seqs"])]
    rlen = [r.randint(case["resp_lo"], case["resp_hi"]) for _ in range(case["seqs"])]
    return plen, rlen


def _rows(case):
    """(rows of the logits or hidden states, rows that lie in a response window)."""
    plen, rlen = _lengths(case)
    total = sum(plen) + sum(rlen) if case["layout"] == "packed" else case["seqs"] * max(p + r for p, r in zip(plen, rlen))
    return total, sum(rlen)


def work(case):
    kind = case["kind"]
    if kind in ("step", "score"):
        total, live = _rows(case)
        row = case["vocab"] * _BYTES[case["dtype"]]
        # rows of a response window are read; an update writes a gradient for every row
        return {"bytes": live * row + (total * row if kind == "step" else 0) + total * 64, "flops": 0}
    if kind in ("hidden_score", "hidden_step"):
        total, live = _rows(case)
        products = 3 if kind == "hidden_step" else 1
        tensors = 2 if kind == "hidden_step" else 1         # the gradients have the size of what they belong to
        return {"bytes": tensors * 2 * case["hidden"] * (total + case["vocab"]) + total * 64,
                "flops": 2.0 * products * live * case["hidden"] * case["vocab"]}
    if kind == "value":
        n = case["seqs"] * case["width"]
        # old, ref, values, mask in; rewards, advantages, returns out; value head output in, its gradient out
        return {"bytes": 4 * n * 3 + 8 * n + 4 * n * 3 + 2 * 4 * case["seqs"] * (case["prompt"] + case["width"]), "flops": 0}
    plen, rlen = _lengths(case)
    tokens, resp, n = sum(plen) + sum(rlen), sum(rlen), case["seqs"]
    seq, width = max(p + r for p, r in zip(plen, rlen)), max(rlen)
    flat = 8 * tokens + 8 * resp + 4 * resp                 # token ids, responses, old log-probs on the wire
    padded = n * (8 * seq + 8 * width + 4 * width)
    masks = n * 8 * (seq + width)
    return {"bytes": flat + padded + masks + 2 * 4 * n * width + (8 + 8 + 4) * tokens + 2 * 4 * resp, "flops": 0}


# Four times what the path (or, for the value side, the same arithmetic in fp32) differs by from a 64-bit restatement.
_TOLERANCE = {
    # bf16 / fp16 gradients: one rounding of the result
    "step": {"rel": 7e-3, "max": 1.6e-2},
    # fp32 gradients themselves are within 7e-7; the mean of log(old / new), nearly zero, sets the bound
    "step_f32": {"rel": 4e-4, "max": 4e-4},
    "score": {"rel": 2e-6, "max": 1e-5},
    "hidden_score": {"rel": 2e-6, "max": 1e-5},
    # bf16 logits and dlogits between the products; a token whose ratio crosses the clip changes its row as a whole
    "hidden_step": {"rel": 1.6e-2, "max": 0.5},
    "value": {"rel": 3e-6, "max": 1.5e-5},
    "experience": {"rel": 1e-6, "max": 5e-6},
}


def tolerance(case):
    kind = case["kind"]
    return _TOLERANCE["step_f32" if kind == "step" and case["dtype"] == "f32" else kind]


# ------------------------------------------------------------------------------------------ inputs
def _int_column(values, dev):
    return torch.tensor(values, dtype=torch.int32, device=dev).view(-1, 1)


def _scored_rows(total, vocab, make_rows, gen, dev):
    """Calls make_rows(lo, hi) -> fp32 logits for chunks of rows; returns labels sampled from their softmax and the
    log-probabilities of these labels."""
    labels = torch.empty(total, dtype=torch.int64, device=dev)
    logp = torch.empty(total, dtype=torch.float32, device=dev)
    chunk = max(1, min(total, (1 << 27) // vocab))
    for lo in range(0, total, chunk):
        hi = min(total, lo + chunk)
        z = make_rows(lo, hi)
        noise = torch.empty_like(z).exponential_(generator=gen).log_()
        y = torch.argmax(z - noise, dim=-1)
        labels[lo:hi] = y
        logp[lo:hi] = z.gather(1, y[:, None]).squeeze(1) - torch.logsumexp(z, -1)
        del z, noise
    return labels, logp


def _batch(case, labels, row_logp, gen, dev):
    """The batch dict and the keyword arguments that a training engine hands to a loss object."""
    plen, rlen = _lengths(case)
    n, width = case["seqs"], max(rlen)
    p, r = _int_column(plen, dev), _int_column(rlen, dev)
    seqlens = (p + r).flatten()
    cols = torch.arange(width, device=dev)[None, :]
    live = cols < r
    kw = {}
    if case["layout"] == "packed":
        cu = torch.zeros(n + 1, dtype=torch.int32, device=dev)
        cu[1:] = torch.cumsum(seqlens, 0)
        first = cu[:-1].view(-1, 1) + p - 1
        kw = dict(use_remove_padding=True, seqlens_in_batch=seqlens, cu_seqlens_padded=cu,
                  seq_len=max(a + b for a, b in zip(plen, rlen)))
        labels = labels.view(1, -1)
    else:
        padded = row_logp.numel() // n
        first = torch.arange(n, device=dev).view(-1, 1) * padded + p - 1
        labels = labels.view(n, padded)
    rows = (first.to(torch.int64) + cols).clamp(max=row_logp.numel() - 1)
    current = torch.where(live, row_logp[rows], torch.zeros((), device=dev))
    responses = torch.where(live, labels.reshape(-1)[rows], torch.zeros((), dtype=torch.int64, device=dev))

    def drifted():
        # tokens were sampled from the old policy: log(new / old) has mean -spread^2 / 2
        noise = torch.randn(n, width, generator=gen, device=dev) * _DRIFT + 0.5 * _DRIFT * _DRIFT
        return torch.where(live, current + noise, torch.zeros((), device=dev))

    rewards = (torch.rand(n, _GROUP, generator=gen, device=dev) < torch.rand(n, 1, generator=gen, device=dev)).float()
    adv = ((rewards - rewards.mean(1, keepdim=True)) / (rewards.std(1, keepdim=True) + 1e-6))[:, :1]
    batch = {"labels": labels, "responses": responses, "prompt_length": p, "response_length": r,
             "advantages": adv * live, "old_log_prob": drifted()}
    if case.get("loss") == "grpo":
        batch["ref_log_prob"] = drifted()
    if case.get("loss") in ("dapo", "dapo_seq"):
        batch["response_mask"] = live.to(torch.int64)
    return batch, kw


def _actor(loss):
    if loss == "grpo":
        fn = mrl.LossFuncFactory.get_instance("ray_grpo", "actor")
        fn.add_loss_meta_info({"clip_ratio": 0.2, "kl_ctrl": mrl.FixedKLController(0.001), "kl_penalty": "low_var_kl",
                               "entropy_coeff": 0.001})
    elif loss == "ppo":
        fn = mrl.LossFuncFactory.get_instance("ray_ppo", "actor")
        fn.add_loss_meta_info({"clip_ratio": 0.2, "kl_ctrl": mrl.FixedKLController(0.001), "entropy_coeff": 0.0})
    else:
        fn = mrl.LossFuncFactory.get_instance("ray_dapo", "actor")
        fn.add_loss_meta_info({"clip_ratio": 0.2, "kl_ctrl": mrl.FixedKLController(0.0), "entropy_coeff": 0.0,
                               "token_level_loss": loss == "dapo", "clip_higher_enable": True, "clip_ratio_low": 0.2,
                               "clip_ratio_high": 0.28})
    return fn


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev).manual_seed(seed)
    kind = case["kind"]
    if kind == "value":
        return _prepare_value(case, gen, dev)
    if kind == "experience":
        return _prepare_experience(case, gen, dev)
    total, _ = _rows(case)
    plen, rlen = _lengths(case)
    vocab = case["vocab"]
    lead = (1, total) if case["layout"] == "packed" else (case["seqs"], total // case["seqs"])
    state = {"kind": kind, "micro": case.get("micro", 1)}
    if kind in ("step", "score"):
        sigma = 2.0 if case["dtype"] == "f32" else 3.0
        logits = torch.empty(total, vocab, dtype=_DTYPES[case["dtype"]], device=dev)

        def make_rows(lo, hi):
            logits[lo:hi] = torch.randn(hi - lo, vocab, generator=gen, device=dev) * sigma
            return logits[lo:hi].float()

        labels, logp = _scored_rows(total, vocab, make_rows, gen, dev)
        state["output"] = logits.view(*lead, vocab)
    else:
        hidden = torch.randn(total, case["hidden"], generator=gen, device=dev).to(torch.bfloat16)
        weight = (torch.randn(vocab, case["hidden"], generator=gen, device=dev) * 0.02).to(torch.bfloat16)
        labels, logp = _scored_rows(total, vocab, lambda lo, hi: (hidden[lo:hi] @ weight.t()).float(), gen, dev)
        state["output"] = hidden.view(*lead, case["hidden"])
        state["weight"] = weight
    state["batch"], state["kw"] = _batch(case, labels, logp, gen, dev)
    if kind in ("step", "hidden_step"):
        state["output"].requires_grad_()
        if kind == "hidden_step":
            state["weight"].requires_grad_()
        state["fn"] = _actor(case["loss"])
        if state["micro"] != 1:         # the schedule divides the loss by the number of micro-batches and says so
            state["kw"]["expected_grad_scale"] = 1.0 / state["micro"]
    else:
        state["entropy"] = case["entropy"]
        state["fn"] = (_actor("grpo") if case["entropy"] else mrl.LossFuncFactory.get_instance("ray_grpo", "reference"))
    if kind.startswith("hidden"):
        state["kw"]["lm_head_weight"] = state["weight"]
    return state


def _prepare_value(case, gen, dev):
    n, width, prompt = case["seqs"], case["width"], case["prompt"]
    r = random.Random(case["lengths"])
    rlen = _int_column([r.randint(max(1, width // 8), width) for _ in range(n)], dev)
    mask = (torch.arange(width, device=dev)[None, :] < rlen).to(torch.int64)
    old = -torch.empty(n, width, device=dev).exponential_(0.7, generator=gen)
    ref = old + torch.randn(n, width, generator=gen, device=dev) * _DRIFT
    values = torch.randn(n, width, generator=gen, device=dev) * 0.3
    # the value head's output over the whole sequences, moved a little since `values` were taken
    head = torch.zeros(n, prompt + width, 1, device=dev)
    head[:, prompt - 1:prompt - 1 + width, 0] = values + torch.randn(n, width, generator=gen, device=dev) * 0.3
    fn = mrl.LossFuncFactory.get_instance("ray_ppo", "critic")
    fn.add_loss_meta_info({"cliprange_value": 0.5})
    return {"kind": "value", "old": old, "ref": ref, "mask": mask, "values": values, "head": head.requires_grad_(),
            "scores": torch.randn(n, generator=gen, device=dev), "penalty": case["penalty"], "fn": fn,
            "batch": {"responses": torch.zeros(n, width, dtype=torch.int64, device=dev), "response_length": rlen,
                      "prompt_length": torch.full_like(rlen, prompt), "values": values}}


def _prepare_experience(case, gen, dev):
    plen, rlen = _lengths(case)
    p, r = _int_column(plen, dev), _int_column(rlen, dev)
    tokens, resp = sum(plen) + sum(rlen), sum(rlen)
    data = {"input_ids": torch.randint(1, 152064, (tokens,), generator=gen, device=dev),
            "responses": torch.randint(1, 152064, (resp,), generator=gen, device=dev),
            "old_log_prob": -torch.empty(resp, device=dev).exponential_(0.7, generator=gen),
            "prompt_length": p.flatten(), "response_length": r.flatten()}
    ones = torch.ones(case["seqs"], dtype=torch.int32, device=dev)
    lengths = {"input_ids": (p + r).flatten(), "responses": r.flatten(), "old_log_prob": r.flatten(),
               "prompt_length": ones, "response_length": ones}
    chance = torch.rand(case["seqs"] // _GROUP, 1, generator=gen, device=dev).expand(-1, _GROUP).reshape(-1, 1)
    rewards = (torch.rand(case["seqs"], 1, generator=gen, device=dev) < chance).float()
    return {"kind": "experience", "data": data, "lengths": lengths, "rewards": rewards, "align": case["align"]}


# ------------------------------------------------------------------------------------------ one pass
def run(state):
    return _RUN[state["kind"]](state)


def _run_step(state):
    loss, stats = state["fn"].compute_loss(state["output"], state["batch"], **state["kw"])
    inputs = [state["output"]] + ([state["weight"]] if state["kind"] == "hidden_step" else [])
    grads = torch.autograd.grad(loss / state["micro"], inputs)
    return {"loss": loss.detach(), "stats": dict(stats), "grads": grads}


def _run_score(state):
    with torch.no_grad():
        if state["entropy"]:
            return state["fn"].compute_log_probs(state["output"], state["batch"], skip_entropy=False, **state["kw"])
        return state["fn"].compute_loss(state["output"], state["batch"], forward_only=True, **state["kw"])


def _run_value(state):
    batch = dict(state["batch"])
    rewards, kl = mrl.kl_token_level_rewards(state["old"], state["ref"], batch["response_length"], state["scores"], 0.05,
                                             state["penalty"])
    advantages, batch["returns"] = mrl.compute_gae_advantage_return(rewards, state["values"], state["mask"], 1.0, 0.95)
    loss, stats = state["fn"].compute_loss(state["head"], batch)
    (grad,) = torch.autograd.grad(loss, state["head"])
    return {"rewards": rewards, "kl": kl, "advantages": advantages, "returns": batch["returns"], "loss": loss.detach(),
            "stats": stats, "grad": grad}


def _run_experience(state):
    batch = mrl.unpack_pad_experience(state["data"], state["lengths"], 0, 1)
    mask = mrl.generate_mask(batch["responses"], batch["response_length"])
    advantages, returns = mrl.compute_group_norm_advantage_return(state["rewards"], mask, batch["response_length"], _GROUP)
    keep = mrl.dynamic_sampling_keep_mask(state["rewards"], _GROUP)
    ids = batch["input_ids"]
    attention = mrl.generate_mask(ids, batch["prompt_length"] + batch["response_length"])
    packed = mrl.preprocess_packed_seqs(ids, torch.roll(ids, -1, 1), attention, state["align"])
    length = batch["response_length"]
    flat = mrl.pack_padded_columns({"advantages": advantages, "returns": returns},
                                   {"advantages": length, "returns": length})
    return {"batch": batch, "mask": mask, "keep": keep, "packed": packed, "flat": flat}


_RUN = {"step": _run_step, "hidden_step": _run_step, "score": _run_score, "hidden_score": _run_score,
        "value": _run_value, "experience": _run_experience}
