"""What a user of this package has it do, as cases that can be timed and compared.

A case is a dict of plain values; ``listed()`` gives the ones that are followed and
``draw()`` more of the same ranges.  Each goes through the public entry points only, with
inputs shaped as in GRPO training: logits spread like a language model's, a prompt and a
padding that carry no gradient, responses of uneven length.

Kinds (the ``kind`` of a case):

* ``logprob``    next-token logprobs of logits, forward only or with the backward
* ``grpo``       one whole policy step: advantages, logprobs, clipped loss, backward
* ``packed``     the same over sequences packed into one row, with the k3 KL penalty
* ``filter``     logprobs under the sampler's temperature, top-k and top-p, with the backward
* ``distill``    a divergence of student and teacher over the whole vocabulary, with the backward
* ``topk``       the teacher's top-k export
* ``advantage``  group-normalised advantages from prompt token rows
* ``hidden``     logprobs straight from hidden states and the output weight

``work()`` counts each operand of the forward once and each operand of the backward once:
the upstream gradient exists only after the forward has ended, so the rows that carry one
are needed a second time, by any program.
"""

import math

import torch

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
DEVICE = "cuda"


def listed():
    return [
        # scoring a small batch (an evaluation, a reference policy's logprobs): launch and
        # latency count
        dict(name="logprob_small", kind="logprob", B=2, S=256, V=32000, dtype="fp32", train=False),
        # a supervised step of an ordinary size over an odd vocabulary: no row but the first
        # starts on a 16-byte boundary
        dict(name="logprob_odd", kind="logprob", B=3, S=1021, V=100003, dtype="bf16", train=True),
        # the training step the package is for: one prompt, eight generations, whole vocabulary
        dict(name="grpo", kind="grpo", B=8, S=2048, V=151936, dtype="bf16"),
        # sequence packing with a reference policy; the widest vocabulary in use
        dict(name="packed_kl", kind="packed", n=16, len_min=64, len_max=1024, V=256000),
        # a policy step whose sampler ran with temperature, top-k and top-p
        dict(name="filter_k50_p09", kind="filter", B=4, S=4096, V=151936, dtype="bf16",
             top_k=50, top_p=0.9, T=0.7),
        # top-p alone keeps a large part of the vocabulary
        dict(name="filter_p09", kind="filter", B=2, S=2048, V=151936, dtype="bf16",
             top_k=0, top_p=0.9, T=0.7),
        # the same on logits that the model returns in fp32
        dict(name="filter_p09_f32", kind="filter", B=1, S=2048, V=151936, dtype="fp32",
             top_k=0, top_p=0.9, T=0.7),
        # distillation on the student's own samples
        dict(name="distill_rkl", kind="distill", B=4, S=2048, V=151936, dtype="bf16", what="reverse_kl"),
        # a teacher that hands on its top tokens instead of its logits
        dict(name="teacher_topk", kind="topk", B=4, S=2048, V=151936, dtype="bf16", k=64),
        # a large rollout batch's advantages; the prompts are the group keys
        dict(name="advantage", kind="advantage", groups=128, n=16, K=512, loo=True),
        # the fused LM head: logits are never held; forward and both gradients
        dict(name="hidden_bf16", kind="hidden", S=2048, B=8, H=4096, V=151936, dtype="bf16",
             chunk=256, train=True),
        # the same on fp32 master weights and activations, a microbatch of two
        dict(name="hidden_f32", kind="hidden", S=1024, B=2, H=4096, V=151936, dtype="fp32",
             chunk=256, train=True),
    ]


def _between(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm where that spans more than tenfold."""
    if hi > 10 * lo:
        return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))
    return rng.randint(lo, hi)


def _vocab(rng):
    return rng.choice([_between(rng, 1000, 256000), _between(rng, 1000, 256000), 32000, 131072, 151936])


def _rows(rng, V, esz, most=2.5e9):
    """(B, S) whose logits stay below `most` bytes."""
    B = rng.choice([1, 2, 3, 4, 8])
    return B, _between(rng, 16, max(17, min(4096, int(most / (V * esz * B)))))


def draw(rng):
    kind = rng.choice(["logprob", "grpo", "packed", "filter", "filter", "distill", "topk",
                       "advantage", "hidden", "hidden"])
    V = _vocab(rng)
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    esz = 4 if dtype == "fp32" else 2
    if kind == "packed":
        n = 8 * rng.randint(1, 3)
        top = min(1024, max(40, int(2.5e9 / (V * 2 * n))))
        return dict(kind=kind, n=n, len_min=rng.randint(8, 32), len_max=_between(rng, 33, top), V=V)
    if kind == "advantage":
        return dict(kind=kind, groups=_between(rng, 1, 256), n=rng.choice([2, 4, 8, 16, 32]),
                    K=rng.choice([1, _between(rng, 2, 1024)]), loo=rng.random() < 0.5)
    if kind == "hidden":
        H = rng.choice([8 * _between(rng, 8, 512), 1024, 2048, 4096])
        B = rng.choice([1, 2, 4])
        flops = 2e12 if dtype == "fp32" else 1.5e13
        S = _between(rng, 32, max(33, min(2048, int(flops / (2.0 * B * H * V)))))
        return dict(kind=kind, S=S, B=B, H=H, V=V, dtype=dtype, chunk=rng.choice([0, 64, 256]),
                    train=rng.random() < 0.75)
    B, S = _rows(rng, V, esz, 1.25e9 if kind == "distill" else 2.5e9)
    if kind == "logprob":
        return dict(kind=kind, B=B, S=S, V=V, dtype=dtype, train=rng.random() < 0.5)
    if kind == "grpo":
        return dict(kind=kind, B=B, S=max(64, S), V=V, dtype=dtype)
    if kind == "filter":
        top_k = rng.choice([0, 0, 20, 50, _between(rng, 1, 512), 2000])
        return dict(kind=kind, B=B, S=S, V=max(V, 4000), dtype=dtype, top_k=top_k,
                    top_p=rng.choice([0.8, 0.9, 0.95, round(rng.uniform(0.5, 0.99), 3)]),
                    T=rng.choice([1.0, 0.7, 0.6, 1.2]))
    if kind == "distill":
        return dict(kind=kind, B=B, S=S, V=V, dtype=dtype,
                    what=rng.choice(["reverse_kl", "reverse_kl", "cross_entropy", "entropy"]))
    return dict(kind="topk", B=B, S=S, V=max(V, 2000), dtype=dtype, k=rng.choice([8, 64, 256, _between(rng, 1, 1024)]))


# ---------------------------------------------------------------------------------------
# Inputs


class _Random:
    def __init__(self, seed):
        self.cpu = torch.Generator().manual_seed(int(seed))
        self.gpu = torch.Generator(device=DEVICE).manual_seed(int(seed) ^ 0x5DEECE66D)

    def ints(self, lo, hi, shape):
        return torch.randint(lo, hi, shape, generator=self.cpu)

    def normal(self, shape):
        return torch.randn(shape, generator=self.gpu, device=DEVICE)

    def uniform(self, shape):
        return torch.rand(shape, generator=self.gpu, device=DEVICE)

    def logits(self, B, S, V, std, dtype):
        """N(0, std^2) in `dtype`, made in blocks of rows."""
        out = torch.empty((B * S, V), dtype=dtype, device=DEVICE)
        step = max(1, (1 << 27) // V)
        for a in range(0, B * S, step):
            n = min(step, B * S - a)
            out[a : a + n].copy_(torch.randn((n, V), generator=self.gpu, device=DEVICE).mul_(std))
        return out.view(B, S, V)

    def responses(self, B, S):
        """[B, S] mask: a prompt of a quarter of the row, a response of uneven length, padding."""
        prompt = S // 4
        length = self.ints(max(1, S // 8), max(2, S - prompt + 1), (B, 1))
        pos = torch.arange(S).unsqueeze(0)
        return ((pos >= prompt) & (pos < prompt + length)).float().to(DEVICE)


def _blocks(n, V, most=1 << 26):
    step = max(1, most // V)
    return [(a, min(n, a + step)) for a in range(0, n, step)]


def _row_logprobs(logits, targets, wide):
    """[n] logprobs of flat rows [n, V] in the float type `wide`, in blocks of rows."""
    out = torch.empty(targets.shape, dtype=wide, device=logits.device)
    for a, b in _blocks(logits.shape[0], logits.shape[1]):
        x = logits[a:b].to(wide)
        out[a:b] = x.gather(1, targets[a:b, None])[:, 0] - torch.logsumexp(x, -1)
    return out


def _inputs_logprob(case, r):
    B, S, V = case["B"], case["S"], case["V"]
    s = {"logits": r.logits(B, S, V, 1.5, DTYPES[case["dtype"]]), "ids": r.ints(0, V, (B, S)).to(DEVICE)}
    s["grad"] = r.normal((B, S - 1)) * r.responses(B, S)[:, 1:]
    return s


def _inputs_grpo(case, r):
    B, S, V = case["B"], case["S"], case["V"]
    s = {"logits": r.logits(B, S, V, 1.5, DTYPES[case["dtype"]]), "ids": r.ints(0, V, (B, S)).to(DEVICE)}
    s["mask"] = r.responses(B, S)
    s["rewards"] = r.ints(0, 2, (B,)).float().to(DEVICE)
    s["prompts"] = torch.zeros((B, 1), dtype=torch.int64, device=DEVICE)
    # one row of logits predicts the next token, so the last row of each sample is not scored
    now = torch.empty((B, S - 1), dtype=torch.float32, device=DEVICE)
    for b in range(B):
        now[b] = _row_logprobs(s["logits"][b, :-1], s["ids"][b, 1:], torch.float32)
    s["old"] = torch.zeros((B, S), device=DEVICE)
    s["old"][:, 1:] = now + 0.05 * r.normal((B, S - 1))
    return s


def _inputs_packed(case, r):
    n, V = case["n"], case["V"]
    # the lengths are sizes, not values: the case's own
    lens = _Random(n).ints(case["len_min"], case["len_max"] + 1, (n,))
    cu = [0]
    for x in lens.tolist():
        cu.append(cu[-1] + x)
    S = int(lens.max())
    s = {"logits": r.logits(1, cu[-1], V, 1.5, torch.bfloat16), "cu": tuple(cu)}
    pos = torch.arange(S).unsqueeze(0)
    live = pos < lens.unsqueeze(1)
    s["ids"] = (r.ints(0, V, (n, S)) * live).to(DEVICE)
    s["lengths"] = lens.to(DEVICE)
    s["mask"] = (live & (pos > 0)).float().to(DEVICE)
    s["rewards"] = r.ints(0, 2, (n,)).float().to(DEVICE)
    s["prompts"] = (torch.arange(n) // 8).unsqueeze(1).to(DEVICE)
    s["old"] = torch.zeros((n, S), device=DEVICE)
    for i in range(n):
        a, b = cu[i], cu[i + 1]
        s["old"][i, 1 : b - a] = _row_logprobs(s["logits"][0, a : b - 1], s["ids"][i, 1 : b - a], torch.float32)
    s["old"] += 0.05 * r.normal(s["old"].shape) * s["mask"]
    s["reference"] = s["old"] + 0.1 * r.normal(s["old"].shape) * s["mask"]
    return s


def _scaled(x, T):
    """``x.div_(T)`` as the GPU computes it, in the logits' own type."""
    return x if T == 1.0 else (x.float() * torch.tensor(1.0 / T, device=x.device)).to(x.dtype)


def _kept(y, case):
    """(kept mask in descending order, the order) of rows y in 64 bits: the k largest, then the
    shortest head of them whose tail weighs no more than 1 - top_p; ties by position."""
    vals, order = torch.sort(y.flip(-1), dim=-1, descending=True, stable=True)
    order = y.shape[-1] - 1 - order  # of equal values the later position comes first
    keep = torch.ones_like(vals, dtype=torch.bool)
    k = case["top_k"]
    if 0 < k < vals.shape[-1]:
        keep = vals >= vals[:, k - 1 : k]
    p = torch.softmax(vals.masked_fill(~keep, -math.inf), -1)
    at_and_below = p.flip(-1).cumsum(-1).flip(-1)
    keep &= at_and_below > 1.0 - case["top_p"]
    keep[:, 0] = True
    return keep, order


def _inputs_filter(case, r):
    B, S, V = case["B"], case["S"], case["V"]
    s = {"logits": r.logits(B, S, V, 1.0, DTYPES[case["dtype"]])}
    flat = s["logits"].view(B * S, V)
    # a confident model: one token of each row stands out, by an uneven amount
    best = r.ints(0, V, (B * S, 1)).to(DEVICE)
    lift = (4.0 + 8.0 * r.uniform((B * S, 1))).to(flat.dtype)
    flat.scatter_add_(1, best, lift)
    # the sampled tokens: from the heavier 60% of the filtered mass
    choice = torch.empty(B * S, dtype=torch.int64, device=DEVICE)
    u = r.uniform((B * S, 1)) * 0.6
    k = case["top_k"]
    for a, b in _blocks(B * S, V):
        y = _scaled(flat[a:b], case["T"]).float()
        # what top-p alone keeps has no bound: its 60% is looked up among the whole row
        vals, order = torch.topk(y, k, dim=-1) if 0 < k <= 512 else torch.sort(y, dim=-1, descending=True)
        p = torch.softmax(vals[:, :k] if k > 0 else vals, -1)
        at = (p.cumsum(-1) < u[a:b]).sum(-1, keepdim=True)
        choice[a:b] = order.gather(1, at)[:, 0]
    s["ids"] = choice.view(B, S).roll(1, dims=1)  # row s predicts ids[s + 1]
    s["grad"] = r.normal((B, S - 1)) * (r.uniform((B, S - 1)) < 0.9)
    return s


def _inputs_distill(case, r):
    B, S, V = case["B"], case["S"], case["V"]
    t = DTYPES[case["dtype"]]
    s = {"logits": r.logits(B, S, V, 1.5, t)}
    s["teacher"] = r.logits(B, S, V, 1.5, t) if case["what"] != "entropy" else None
    s["grad"] = r.responses(B, S) / (B * S)
    return s


def _inputs_topk(case, r):
    return {"logits": r.logits(case["B"], case["S"], case["V"], 1.5, DTYPES[case["dtype"]])}


def _inputs_advantage(case, r):
    B, K = case["groups"] * case["n"], case["K"]
    group = torch.arange(case["groups"]).repeat_interleave(case["n"])
    tokens = group.unsqueeze(1) if K == 1 else r.ints(0, 32000, (case["groups"], K))[group]
    if K > 1:
        tokens[:, 0] = 1  # every prompt starts with the same token
    return {"prompts": tokens.to(DEVICE), "group": group, "rewards": r.uniform((B,)).round(decimals=2),
            "mask": torch.ones((B, 64), device=DEVICE)}


def _inputs_hidden(case, r):
    S, B, H, V = case["S"], case["B"], case["H"], case["V"]
    t = DTYPES[case["dtype"]]
    s = {"hidden": r.logits(S, B, H, 1.0, t), "weight": r.logits(1, V, H, 1.5 / math.sqrt(H), t)[0],
         "ids": r.ints(0, V, (B, S)).to(DEVICE)}
    s["grad"] = r.normal((B, S - 1)) * r.responses(B, S)[:, 1:]
    return s


_INPUTS = {"logprob": _inputs_logprob, "grpo": _inputs_grpo, "packed": _inputs_packed, "filter": _inputs_filter,
           "distill": _inputs_distill, "topk": _inputs_topk, "advantage": _inputs_advantage, "hidden": _inputs_hidden}


def _inputs(case, seed):
    return _INPUTS[case["kind"]](case, _Random(seed))


def _loss(kl):
    from rl_amd.algorithms.advantage_estimator import AdvEstimatorConfig, GRPOAdvantageEstimator
    from rl_amd.algorithms.loss import ClippedPGLossConfig, ClippedPGLossFn

    config = ClippedPGLossConfig(reference_policy_kl_penalty=kl)
    return ClippedPGLossFn(config), GRPOAdvantageEstimator(AdvEstimatorConfig(use_leave_one_out_baseline=False), config)


def _group():
    """The tensor-parallel group of a program on one GPU."""
    import torch.distributed as dist

    if not dist.is_initialized():
        dist.init_process_group("gloo", store=dist.HashStore(), rank=0, world_size=1)
    return dist.group.WORLD


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    for name in ("logits", "hidden", "weight"):
        if name in s and case["kind"] != "topk" and case.get("train", True):
            s[name].requires_grad_(True)
    if case["kind"] in ("grpo", "packed"):
        B = s["ids"].shape[0]
        s["batch"] = {"input_ids": s["ids"], "token_mask": s["mask"], "sample_mask": torch.ones(B, device=DEVICE),
                      "prev_logprobs": s["old"], "generation_logprobs": s["old"],
                      "reference_policy_logprobs": s.get("reference", s["old"])}
        if case["kind"] == "packed":
            s["batch"]["input_lengths"] = s["lengths"]
        s["seqs"] = torch.tensor(float(B), device=DEVICE)
        s["toks"] = s["mask"][:, 1:].sum()
        s["loss"], s["estimator"] = _loss(0.01 if case["kind"] == "packed" else 0.0)
        if case["kind"] == "packed":
            from rl_amd.algorithms.loss import SequencePackingFusionLossWrapper, prepare_packed_loss_input

            s["wrapper"] = SequencePackingFusionLossWrapper(s["loss"], prepare_packed_loss_input, s["cu"], s["cu"],
                                                            vocab_parallel_rank=0, vocab_parallel_group=_group())
    if case["kind"] == "advantage":
        from rl_amd.algorithms.advantage_estimator import AdvEstimatorConfig, GRPOAdvantageEstimator

        s["estimator"] = GRPOAdvantageEstimator(AdvEstimatorConfig(use_leave_one_out_baseline=case["loo"]))
    return s


# ---------------------------------------------------------------------------------------
# One pass


def _run_logprob(s, case):
    from rl_amd.distributed.model_utils import from_parallel_logits_to_logprobs

    lp = from_parallel_logits_to_logprobs(s["logits"], s["ids"], 0, case["V"], None,
                                          inference_only=not case["train"])
    if not case["train"]:
        return {"logprobs": lp}
    (grad,) = torch.autograd.grad(lp, [s["logits"]], s["grad"])
    return {"logprobs": lp, "grad": grad}


def _run_grpo(s, case):
    from rl_amd.distributed.model_utils import from_parallel_logits_to_logprobs

    batch = dict(s["batch"])
    batch["advantages"] = s["estimator"].compute_advantage(s["prompts"], s["rewards"], s["mask"])
    lp = from_parallel_logits_to_logprobs(s["logits"], s["ids"], 0, case["V"], None)
    loss, _ = s["loss"](lp, batch, s["seqs"], s["toks"])
    (grad,) = torch.autograd.grad(loss, [s["logits"]])
    return {"advantages": batch["advantages"], "logprobs": lp, "loss": loss, "grad": grad}


def _run_packed(s, case):
    batch = dict(s["batch"])
    batch["advantages"] = s["estimator"].compute_advantage(s["prompts"], s["rewards"], s["mask"])
    loss, _ = s["wrapper"](s["logits"], batch, s["seqs"], s["toks"])
    (grad,) = torch.autograd.grad(loss, [s["logits"]])
    return {"advantages": batch["advantages"], "loss": loss, "grad": grad}


def _run_filter(s, case):
    from rl_amd.distributed.sampling import filtered_next_token_logprobs

    lp = filtered_next_token_logprobs(s["logits"], s["ids"], case["top_k"], case["top_p"], temperature=case["T"],
                                      decision_dtype=torch.float32)
    (grad,) = torch.autograd.grad(lp, [s["logits"]], s["grad"])
    return {"logprobs": lp, "grad": grad}


def _run_distill(s, case):
    from rl_amd.distributed import model_utils

    S = case["S"]
    if case["what"] == "entropy":
        out = model_utils.ChunkedDistributedEntropy.apply(s["logits"], S, None, False)
    elif case["what"] == "cross_entropy":
        out = model_utils.ChunkedDistributedCrossEntropyToFixedLogits.apply(s["logits"], s["teacher"], S, None, False)
    else:
        out = model_utils.ChunkedDistributedReverseKLToFixedLogits.apply(s["logits"], s["teacher"], S, None, False)
    (grad,) = torch.autograd.grad(out, [s["logits"]], s["grad"])
    return {"divergence": out, "grad": grad}


def _run_topk(s, case):
    from rl_amd.distributed.model_utils import distributed_vocab_topk

    values, ids = distributed_vocab_topk(s["logits"], case["k"], None, vocab_start_index=0,
                                         vocab_end_index=case["V"])
    return {"values": values, "ids": ids}


def _run_advantage(s, case):
    return s["estimator"].compute_advantage(s["prompts"], s["rewards"], s["mask"])


def _run_hidden(s, case):
    from rl_amd.distributed.model_utils import from_parallel_hidden_states_to_logprobs

    lp = from_parallel_hidden_states_to_logprobs(s["hidden"], s["weight"], False, s["ids"], 0, case["V"], None,
                                                 inference_only=not case["train"], chunk_size=case["chunk"] or None)
    if not case["train"]:
        return {"logprobs": lp}
    gh, gw = torch.autograd.grad(lp, [s["hidden"], s["weight"]], s["grad"])
    return {"logprobs": lp, "grad_hidden": gh, "grad_weight": gw}


_RUN = {"logprob": _run_logprob, "grpo": _run_grpo, "packed": _run_packed, "filter": _run_filter,
        "distill": _run_distill, "topk": _run_topk, "advantage": _run_advantage, "hidden": _run_hidden}


def run(state):
    case = state["case"]
    return _RUN[case["kind"]](state, case)


# ---------------------------------------------------------------------------------------
# What a pass needs, how far results may be off, and the results in 64 bits

_ACTIVE = 7 / 16  # the responses' share of a row, on average: half way from an eighth to three quarters


def work(case):
    kind = case["kind"]
    if kind == "advantage":
        B = case["groups"] * case["n"]
        return {"bytes": B * (8 * case["K"] + 4 + 4), "flops": 0}
    if kind == "packed":
        T = case["n"] * (case["len_min"] + case["len_max"]) / 2
        return {"bytes": 3 * T * case["V"] * 2, "flops": 0}
    V, rows, esz = case["V"], case["B"] * case["S"], 4 if case["dtype"] == "fp32" else 2
    if kind == "hidden":
        H = case["H"]
        tensors = (rows + V) * H * esz
        if not case["train"]:
            return {"bytes": tensors, "flops": 2 * rows * H * V}
        return {"bytes": 3 * tensors, "flops": (1 + 3 * _ACTIVE) * 2 * rows * H * V}
    if kind == "topk":
        return {"bytes": rows * (V * esz + 12 * case["k"]), "flops": 0}
    if kind == "filter":
        # at most 1024 kept entries are worth keeping from the forward: beyond, the backward
        # needs the rows again
        again = 0.0 if 0 < case["top_k"] <= 1024 else 0.9
        return {"bytes": (2 + again) * rows * V * esz, "flops": 0}
    if kind == "distill":
        read = 1 if case["what"] == "entropy" else 2
        return {"bytes": (read * (1 + _ACTIVE) + 1) * rows * V * esz, "flops": 0}
    if not case.get("train", True):
        return {"bytes": rows * (V * esz + 12), "flops": 0}
    return {"bytes": (2 + _ACTIVE) * rows * V * esz, "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind == "topk":
        return "exact"
    if kind == "advantage":
        return {"rel": 1e-5}  # fp32 sums of a group, a square root and a quotient
    t = case.get("dtype", "bf16")
    if kind == "hidden":
        # 16 bits: the logits are rounded to the type (2^-9 or 2^-12 of values up to 7), then
        # the logits gradient to bf16; fp32: sums of 4096 products and of 151936
        return {"rel": 1e-5 if t == "fp32" else 1e-2}
    if kind == "grpo" and t == "fp32":
        return {"rel": 4e-5}  # the loss is a difference of sums
    if kind == "filter" and t == "fp32":
        return {"rel": 5e-6}  # the last token kept may be another of nearly the same weight
    if not case.get("train", True):
        return {"rel": 5e-7}  # fp32 sums over the vocabulary, whatever the logits' type
    # the gradient is rounded to the logits' type: half a unit in the last place
    return {"rel": {"fp32": 2e-6, "fp16": 2e-3, "bf16": 8e-3}[t]}


def _exact_rows(logits, targets, g):
    """(logprobs, gradient) of rows [n, V] in 64 bits for an upstream gradient g [n] or None."""
    n, V = logits.shape
    lp = _row_logprobs(logits, targets, torch.float64)
    if g is None:
        return lp, None
    grad = torch.zeros((n, V), dtype=torch.float64, device=logits.device)
    for a, b in _blocks(n, V):
        x = torch.softmax(logits[a:b].double(), -1).mul_(-g[a:b, None])
        x.scatter_add_(1, targets[a:b, None], g[a:b, None])
        grad[a:b] = x
    return lp, grad


def _exact_batch(s, g):
    """Next-token logprobs [B, S - 1] of s["logits"], and their gradient [B, S, V]."""
    B, S, V = s["logits"].shape
    lp = torch.empty((B, S - 1), dtype=torch.float64, device=DEVICE)
    grad = None if g is None else torch.zeros((B, S, V), dtype=torch.float64, device=DEVICE)
    for b in range(B):
        lp[b], gr = _exact_rows(s["logits"][b, :-1], s["ids"][b, 1:], None if g is None else g[b])
        if g is not None:
            grad[b, :-1] = gr
    return lp, grad


def _exact_advantages(rewards, group, loo):
    r = rewards.double()
    out = torch.empty_like(r)
    for k in group.unique().tolist():
        at = (group == k).nonzero()[:, 0].to(r.device)
        x = r[at]
        n = x.numel()
        if n < 2:
            out[at] = 0.0
            continue
        rest = n - 1 if loo else n
        part = (1.0 - torch.eye(n, device=x.device, dtype=x.dtype)) if loo else torch.ones((n, n), device=x.device, dtype=x.dtype)
        base = part @ x / rest
        # of a single remaining sample the spread is 0 * (1 / 0), taken as none
        var = (part @ x.square() / rest - base.square()).clamp(min=0.0) * (rest / (rest - 1)) if rest > 1 else torch.zeros_like(x)
        held = x.expand(n, n)
        low = held.masked_fill(part == 0, math.inf).amin(1)
        high = held.masked_fill(part == 0, -math.inf).amax(1)
        std = torch.where(low == high, torch.zeros_like(var), var.sqrt())
        out[at] = torch.where(std > 0, (x - base) / (std + 1e-6), x - base)
    return out


def _exact_policy(now, s, advantages, kl):
    """(loss, gradient of the logprobs) of the clipped objective, and of the k3 penalty."""
    now = now.detach().requires_grad_(True)
    mask, old = s["mask"][:, 1:].double(), s["old"][:, 1:].double()
    A = advantages.unsqueeze(1)
    ratio = (now - old).exp()
    per = torch.maximum(-A * ratio, -A * ratio.clamp(0.8, 1.2))
    if kl:
        d = s["reference"][:, 1:].double() - now
        per = per + kl * (torch.exp(d) - 1 - d)
    loss = (per * mask).sum() / (mask.sum() + 1e-8)
    (g,) = torch.autograd.grad(loss, [now])
    return loss.detach(), g


def _exact_logprob(case, s):
    lp, grad = _exact_batch(s, s["grad"].double() if case["train"] else None)
    return {"logprobs": lp, "grad": grad} if case["train"] else {"logprobs": lp}


def _exact_grpo(case, s):
    adv = _exact_advantages(s["rewards"], s["prompts"][:, 0].cpu(), False)
    lp, _ = _exact_batch(s, None)
    loss, g = _exact_policy(lp, s, adv, 0.0)
    return {"advantages": adv.unsqueeze(1).expand(case["B"], case["S"]), "logprobs": lp, "loss": loss,
            "grad": _exact_batch(s, g)[1]}


def _exact_packed(case, s):
    adv = _exact_advantages(s["rewards"], s["prompts"][:, 0].cpu(), False)
    n, S = s["ids"].shape
    cu = s["cu"]
    lp = torch.zeros((n, S - 1), dtype=torch.float64, device=DEVICE)
    for i in range(n):
        a, b = cu[i], cu[i + 1]
        lp[i, : b - a - 1] = _row_logprobs(s["logits"][0, a : b - 1], s["ids"][i, 1 : b - a], torch.float64)
    loss, g = _exact_policy(lp, s, adv, 0.01)
    grad = torch.zeros(s["logits"].shape, dtype=torch.float64, device=DEVICE)
    for i in range(n):
        a, b = cu[i], cu[i + 1]
        grad[0, a : b - 1] = _exact_rows(s["logits"][0, a : b - 1], s["ids"][i, 1 : b - a], g[i, : b - a - 1])[1]
    return {"advantages": adv.unsqueeze(1).expand(n, S), "loss": loss, "grad": grad}


def _exact_filter(case, s):
    B, S, V = s["logits"].shape
    lp = torch.empty((B, S - 1), dtype=torch.float64, device=DEVICE)
    grad = torch.zeros((B, S, V), dtype=torch.float64, device=DEVICE)
    for b in range(B):
        x, t, g = s["logits"][b, :-1], s["ids"][b, 1:], s["grad"][b].double()
        for a, z in _blocks(S - 1, V):
            y = _scaled(x[a:z], case["T"]).double()
            keep, order = _kept(y, case)
            kept = torch.zeros_like(keep).scatter_(1, order, keep)
            y.masked_fill_(~kept, -math.inf)
            at = t[a:z, None]
            lp[b, a:z] = y.gather(1, at)[:, 0] - torch.logsumexp(y, -1)
            d = torch.softmax(y, -1).mul_(-g[a:z, None])
            d.scatter_add_(1, at, g[a:z, None])
            grad[b, a:z] = d.mul_(1.0 / case["T"])
    return {"logprobs": lp, "grad": grad}


def _exact_distill(case, s):
    B, S, V = s["logits"].shape
    out = torch.empty((B, S), dtype=torch.float64, device=DEVICE)
    grad = torch.zeros((B, S, V), dtype=torch.float64, device=DEVICE)
    for b in range(B):
        for a, z in _blocks(S, V):
            logp = torch.log_softmax(s["logits"][b, a:z].double(), -1)
            w = torch.zeros_like(logp) if case["what"] == "cross_entropy" else logp.clone()
            if case["what"] != "entropy":
                w -= torch.log_softmax(s["teacher"][b, a:z].double(), -1)
            p = logp.exp_()
            out[b, a:z] = (p * w).sum(-1)
            grad[b, a:z] = p * (w - out[b, a:z, None]) * s["grad"][b, a:z, None]
    return {"divergence": out, "grad": grad}


def _exact_topk(case, s):
    return None  # copies of inputs and whole numbers


def _exact_advantage(case, s):
    return _exact_advantages(s["rewards"], s["group"], case["loo"]).unsqueeze(1).expand(s["mask"].shape)


def _exact_hidden(case, s):
    S, B, H, V = case["S"], case["B"], case["H"], case["V"]
    W = s["weight"].double()
    gh, gw = torch.zeros((S * B, H), dtype=torch.float64, device=DEVICE), torch.zeros((V, H), dtype=torch.float64, device=DEVICE)
    x = s["hidden"].view(S * B, H)
    # row (s, b) predicts position s + 1 of sample b; the last position's rows are not scored
    t = s["ids"].roll(-1, dims=1).t().reshape(-1)
    g = torch.cat([s["grad"].double(), torch.zeros((B, 1), dtype=torch.float64, device=DEVICE)], 1).t().reshape(-1)
    lp = torch.empty(S * B, dtype=torch.float64, device=DEVICE)
    for a, b in _blocks(S * B, V, 1 << 28):
        h = x[a:b].double()
        y = h @ W.t()
        at = t[a:b, None]
        lp[a:b] = y.gather(1, at)[:, 0] - torch.logsumexp(y, -1)
        if case["train"]:
            d = torch.softmax(y, -1).mul_(-g[a:b, None])
            del y
            d.scatter_add_(1, at, g[a:b, None])
            gh[a:b] = d @ W
            gw.addmm_(d.t(), h)
    lp = lp.view(S, B).t()[:, :-1]
    return {"logprobs": lp, "grad_hidden": gh.view(S, B, H), "grad_weight": gw} if case["train"] else {"logprobs": lp}


_EXACT = {"logprob": _exact_logprob, "grpo": _exact_grpo, "packed": _exact_packed, "filter": _exact_filter,
          "distill": _exact_distill, "topk": _exact_topk, "advantage": _exact_advantage, "hidden": _exact_hidden}


def exact(case, seed):
    return _EXACT[case["kind"]](case, _inputs(case, seed))
