"""The work a user of nanoep_amd has it do, as cases that can be timed: one MoE layer's data movement on
one GPU, through `Buffer.dispatch` and `Buffer.combine`.

A case is one of two passes:

  forward   fresh routing, the forward pass of a layer and every decode step: `dispatch` of the
            activations with `topk_idx` and gate weights, then `combine` of the expert rows.
  replay    the same layer's backward pass: `dispatch` of the output gradients through the handle the
            forward left behind, then `combine` of the input gradients; the gate weights' values
            travel there and back as well.

The experts are the identity (the rows `dispatch` returned go straight into `combine`): what is measured is
the path of this framework, not a GEMM.  Every pass returns all it made: the received rows, weights and
ids, the handle's routing tensors where the pass is a fresh one, the combined rows and restored weights.
"""

from __future__ import annotations

import math

import torch

from nanoep_amd import Buffer, EPConfig

# Routing kinds, as in the repository's workloads and tests:
#   all       every token takes experts 0 .. K-1
#   uniform   K distinct experts, all equally likely
#   dropout   top-K of normal logits, a tenth of the choices masked (-1)
#   zipf      K distinct experts of popularity 1 / rank^1.2
#   biased    top-K of normal logits plus a per-expert bias of deviation 2
ROUTINGS = ("uniform", "dropout", "zipf", "biased")
MASKED_SHARE = 0.1

_DEFAULTS = {
    "mode": "forward",
    "routing": "dropout",
    "expand": True,
    "alignment": 1,
    "async_op": False,          # calls return an event that the caller's stream waits on
    "bias": False,              # combine adds a [T, H] bias (a shared expert's output)
    "restore_weights": False,   # combine is given the dispatched weights and returns them as [T, K]
    "multiple_reduction": False,
}


def _case(name, tokens, hidden, experts, topk, **options):
    return {"name": name, "tokens": tokens, "hidden": hidden, "experts": experts, "topk": topk, **_DEFAULTS, **options}


def listed():
    return [
        # the README's toy batch: the smallest call, all latency
        _case("toy-forward", 16, 256, 2, 2, routing="all"),
        # one decode step: 256 tokens in flight, the one shape the reference publishes latencies for
        _case("decode-forward", 256, 4096, 64, 8),
        # the forward-MoE example's batch: odd token count, compact layout, calls asynchronous, weights
        # restored at the source
        _case("example-compact-async", 129, 1024, 8, 3, expand=False, async_op=True, restore_weights=True),
        # a ragged prefill batch: odd sizes, K no power of two, row length no multiple of 1 KiB, padded
        # segments, a shared expert's output added by combine
        _case("ragged-forward", 1537, 2816, 60, 6, routing="biased", alignment=16, bias=True),
        # Mixtral's prefill batch: few experts, two rows a token
        _case("mixtral-forward", 4096, 4096, 8, 2, routing="uniform"),
        # DeepSeek-V3's prefill batch, forward
        _case("deepseek-v3-forward", 4096, 7168, 256, 8),
        # ... and its backward pass with segments padded for a grouped GEMM
        _case("deepseek-v3-a128-replay", 4096, 7168, 256, 8, mode="replay", alignment=128, restore_weights=True),
        # Qwen3-MoE's batch: padded segments, asynchronous calls with the caller on a stream of its own
        _case("qwen3-moe-async", 8192, 2048, 128, 8, routing="biased", alignment=128, async_op=True, restore_weights=True),
        # long batches of short rows, forward and backward: many tokens for the routing, one KiB a row
        _case("short-rows-forward", 32768, 512, 64, 8),
        _case("short-rows-replay", 32768, 1024, 64, 8, mode="replay"),
        # one rank's share of an EP=8 prefill, compact layout: the largest batch, forward and backward
        _case("ep8-share-forward", 32768, 7168, 32, 8, routing="zipf", expand=False),
        _case("ep8-share-replay", 32768, 7168, 32, 8, mode="replay", routing="zipf", expand=False, restore_weights=True),
    ]


def draw(rng):
    """A case from the ranges above: 1 to 32768 tokens, rows of 256 to 7168 elements, 2 to 256 experts,
    one to ten choices a token, and the options in about the shares they are used in."""
    most = max(_total_bytes(case) for case in listed())
    while True:
        tokens = int(round(math.exp(rng.uniform(0.0, math.log(32768)))))
        hidden = 256 * int(round(math.exp(rng.uniform(0.0, math.log(28)))))
        experts = int(round(math.exp(rng.uniform(math.log(2), math.log(256)))))
        topk = rng.choice([k for k in (1, 2, 3, 4, 6, 8, 8, 10) if k <= experts])
        expand = rng.random() < 0.75
        case = {
            "tokens": tokens, "hidden": hidden, "experts": experts, "topk": topk, **_DEFAULTS,
            "mode": rng.choice(("forward", "forward", "replay")),
            "routing": rng.choice(ROUTINGS),
            "expand": expand,
            "alignment": rng.choice((1, 1, 16, 128)) if expand else 1,
            "async_op": rng.random() < 0.25,
            "bias": rng.random() < 0.2,
            "restore_weights": rng.random() < 0.4,
            "multiple_reduction": rng.random() < 0.1,
        }
        if _total_bytes(case) <= most:
            return case


def _make_routing(case, generator):
    tokens, experts, topk = case["tokens"], case["experts"], case["topk"]
    if case["routing"] == "all":
        return (torch.arange(topk, device="cuda").repeat(tokens, 1).contiguous(),
                torch.full((tokens, topk), 1.0 / topk, device="cuda"))
    # The batch's load (how many choices each expert gets, how many are masked) belongs to the case, so
    # that the outputs have the case's shapes; the seed decides which token and which expert is which.
    load = torch.Generator(device="cuda").manual_seed(20)
    logits = torch.randn(tokens, experts, device="cuda", generator=load)
    if case["routing"] == "zipf":
        # adding Gumbel noise to the log popularity draws K experts without replacement
        rank = torch.arange(1, experts + 1, device="cuda", dtype=torch.float32)
        uniform = torch.rand(tokens, experts, device="cuda", generator=load).clamp_(1e-9, 1.0 - 1e-7)
        logits = -1.2 * rank.log() - torch.log(-torch.log(uniform))
    elif case["routing"] == "biased":
        logits = logits + 2.0 * torch.randn(experts, device="cuda", generator=load)
    token_of = torch.randperm(tokens, device="cuda", generator=generator)
    expert_of = torch.randperm(experts, device="cuda", generator=generator)
    chosen, idx = logits.topk(topk, dim=1)
    weights = torch.softmax(chosen, dim=1)[token_of]
    named = expert_of[idx][token_of]
    if case["routing"] == "dropout":
        masked = torch.rand(tokens, topk, device="cuda", generator=load) < MASKED_SHARE
        named = named.masked_fill(masked[token_of], -1)  # a masked choice keeps its weight
    return named.contiguous(), weights.contiguous()


def prepare(case, seed):
    generator = torch.Generator(device="cuda").manual_seed(seed)
    tokens, hidden = case["tokens"], case["hidden"]
    idx, weights = _make_routing(case, generator)

    def rows():
        return torch.randn(tokens, hidden, device="cuda", generator=generator, dtype=torch.float32).to(torch.bfloat16)

    config = EPConfig(num_experts=case["experts"], num_topk=case["topk"], hidden=hidden, num_max_tokens_per_rank=tokens)
    state = {
        "case": dict(case),
        "buffer": Buffer(None, config, allow_multiple_reduction=case["multiple_reduction"]),
        "x": rows(),
        "idx": idx,
        "weights": weights,
        "bias": rows() if case["bias"] else None,
        "handle": None,
    }
    if case["mode"] == "replay":
        # the forward pass that left the handle behind
        state["handle"] = _dispatch(state, async_op=False).handle
    return state


def _dispatch(state, async_op):
    case = state["case"]
    if state["handle"] is not None:
        return state["buffer"].dispatch(state["x"], handle=state["handle"], weights=state["weights"],
                                        zero_padding=case["expand"], async_op=async_op)
    return state["buffer"].dispatch(state["x"], topk_idx=state["idx"], weights=state["weights"], do_expand=case["expand"],
                                    alignment=case["alignment"], zero_padding=case["expand"], async_op=async_op)


def run(state):
    case = state["case"]
    received = _dispatch(state, case["async_op"])
    if received.event is not None:
        received.event.current_stream_wait()
    combined = state["buffer"].combine(received.x, received.handle, weights=received.topk_weights if case["restore_weights"] else None,
                                       bias=state["bias"], async_op=case["async_op"])
    if combined.event is not None:
        combined.event.current_stream_wait()
    outputs = {
        "received_x": received.x, "received_ids": received.topk_idx, "received_weights": received.topk_weights,
        "x": combined.x, "weights": combined.topk_weights,
    }
    if case["mode"] == "forward":
        handle = received.handle
        outputs.update(
            recv_metadata=handle.layout.recv_metadata, expert_counts=handle.layout.expert_counts,
            expert_offsets=handle.layout.expert_offsets, recv_rank_prefix=handle.layout.recv_rank_prefix,
            dst_slots=handle.dst_slots, send_counts=handle.send_counts, routing=handle.topk_idx,
        )
    return outputs


def _expected_rows(case):
    """Received rows N, valid choices A and padded capacity C, as expected values of the routing."""
    tokens, topk, experts = case["tokens"], case["topk"], case["experts"]
    keep = 1.0 - MASKED_SHARE if case["routing"] == "dropout" else 1.0
    received = tokens * (1.0 - (1.0 - keep) ** topk)
    assigned = tokens * topk * keep
    padding = min(experts, assigned) * (case["alignment"] - 1) / 2.0
    return received, assigned, assigned + padding


def _total_bytes(case):
    tokens, topk, row = case["tokens"], case["topk"], 2 * case["hidden"]
    received, assigned, capacity = _expected_rows(case)
    weight_rows = capacity if case["expand"] else received * topk
    # dispatch: source rows, ids and weights in; destination rows and weights out
    total = row * received + row * (capacity if case["expand"] else received) + 8 * tokens * topk + 4 * tokens * topk + 4 * weight_rows
    if not case["expand"]:
        total += 8 * received * topk  # local ids of the received rows
    if case["mode"] == "forward":
        # the handle: receive metadata, destination row of every token, the routing snapshot, counts and offsets
        total += 4 * received * (topk + 2) + 8 * tokens + 8 * tokens * topk + 16 * case["experts"]
    # combine: valid expert rows and the routing in, source rows out
    total += row * ((assigned if case["expand"] else received) + tokens) + 4 * received * (topk + 2)
    if case["bias"]:
        total += row * tokens
    if case["restore_weights"]:
        total += 4 * (assigned if case["expand"] else received * topk) + 4 * tokens * topk
    return total


def work(case):
    received, assigned, _ = _expected_rows(case)
    # one fp32 addition an element of every gathered row
    return {"bytes": _total_bytes(case), "flops": (assigned if case["expand"] else received) * case["hidden"]}


def tolerance(case):
    """Rows, ids and weights are moved, and a token's rows are summed in fp32 in ascending choice order and
    rounded once: the result is defined to the bit."""
    return "exact"
