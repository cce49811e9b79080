"""The work whose speed this framework answers for, as cases that can be timed one by one.

Four families, each through the public entry points:

  exchange     ElasticBuffer.dispatch (fresh: layout, host read-back of the row count, expand-permute) and combine of the
               experts' outputs; with "backward" also the training step's second half, a cached dispatch of the output
               gradient and a combine that carries the weight gradients on its return channel
  low_latency  the capacity layout that ElasticBuffer chooses for small batches of EP16-EP256 jobs, and its weighted combine
  mega         the W4A8 expert layer (fp8_fp4_mega_moe on the buffer's own inputs, mega_moe on BF16 rows)
  cast         the per-128 FP8 quantiser and dequantiser (per_token_cast_to_fp8, per_token_cast_back)

"world" / "rank": one rank's share of an expert-parallel job; "tokens" is then the number per source rank, and the call sees
the tokens of all of them, as the buffers expect.  Shapes are the ones of this repository's benchmark, protocol presets and
tests, and generic ones beside them.
"""

from __future__ import annotations

import math

import torch

import deepep_amd
from deepep_amd import megamoe, ops, utils

# Upper bounds of a drawn case, so that none costs more than the largest listed one.
_MOST_PAYLOAD_BYTES = 1 << 30     # rows * hidden * 2 of an exchange
_MOST_CAPACITY_BYTES = 1 << 30    # capacity rows * hidden * 2 of a low-latency call
_MOST_MEGA_FLOPS = 5.0e12
_MOST_WEIGHT_BYTES = 1 << 30


def listed():
    return [
        # The smallest call anybody makes: the smoke workload of the benchmark protocol. Launches and host time only.
        dict(name="decode 31x256", family="exchange", world=1, rank=0, tokens=31, hidden=256, topk=2, experts=8, dtype="bf16",
             weights=True, skew=0.0, masked=0.0, overlap=False, backward=False),
        # A decode step of a large MoE layer whose experts are all on this GPU.
        dict(name="decode 128x7168", family="exchange", world=1, rank=0, tokens=128, hidden=7168, topk=8, experts=256, dtype="bf16",
             weights=True, skew=0.0, masked=0.0, overlap=False, backward=False),
        # Ordinary chunked prefill with padding tokens in the batch (their routes are masked), sizes that are no powers of two.
        dict(name="chunk 1000x5120 masked", family="exchange", world=1, rank=0, tokens=1000, hidden=5120, topk=6, experts=160,
             dtype="bf16", weights=True, skew=0.0, masked=0.15, overlap=False, backward=False),
        # The headline prefill: BF16 tokens quantised inside the dispatch, skewed expert popularity.
        dict(name="prefill 4096x7168 fp8", family="exchange", world=1, rank=0, tokens=4096, hidden=7168, topk=8, experts=256,
             dtype="fp8_fused", weights=True, skew=1.2, masked=0.0, overlap=False, backward=False),
        # One EP8 rank's receive share of a prefill with pre-quantised tokens: most tokens own about one row here.
        dict(name="share ep8 8x2048 fp8", family="exchange", world=8, rank=3, tokens=2048, hidden=7168, topk=8, experts=256,
             dtype="fp8", weights=True, skew=0.0, masked=0.0, overlap=False, backward=False),
        # A training step's exchange, forward and backward, on the communication stream.
        dict(name="train 4096x4096 bf16", family="exchange", world=1, rank=0, tokens=4096, hidden=4096, topk=8, experts=128,
             dtype="bf16", weights=True, skew=0.6, masked=0.0, overlap=True, backward=True),
        # One EP64 rank's low-latency decode step, batch 96 per rank.
        dict(name="low latency ep64 96", family="low_latency", world=64, rank=5, tokens=96, hidden=7168, topk=6, experts=384,
             dtype="fp8", skew=0.0),
        # W4A8 layer in decode: few rows per expert, bound by streaming the weights.
        dict(name="mega decode 512", family="mega", world=8, rank=0, tokens=64, hidden=7168, inter=2048, topk=8, experts=256,
             shared=0, input="fp8"),
        # One EP64 rank's W4A8 share: about 340 rows for each of six experts, most of the output rows belong to nobody here.
        dict(name="mega share ep64", family="mega", world=64, rank=0, tokens=256, hidden=7168, inter=2048, topk=8, experts=384,
             shared=0, input="fp8"),
        # A smaller model from BF16 rows, with a shared expert and sizes that are no whole tiles.
        dict(name="mega 777x2880 shared", family="mega", world=1, rank=0, tokens=777, hidden=2880, inter=1408, topk=4, experts=32,
             shared=1, input="bf16"),
        # The largest: 8192 tokens, top-8 over 32 local experts.
        dict(name="mega prefill 8192", family="mega", world=1, rank=0, tokens=8192, hidden=7168, inter=2048, topk=8, experts=32,
             shared=0, input="fp8"),
        # Quantising and dequantising a batch outside the dispatch, a ragged token count.
        dict(name="cast 10007x5120", family="cast", tokens=10007, hidden=5120),
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _multiple(rng, step, low, high):
    return _log_int(rng, low // step, high // step) * step


def draw(rng):
    family = rng.choices(("exchange", "low_latency", "mega", "cast"), weights=(5, 1, 4, 1))[0]
    while True:
        if family == "exchange":
            dtype = rng.choice(("bf16", "fp8", "fp8_fused"))
            world = rng.choice((1, 1, 1, 2, 4, 8, 64))
            if world == 64:  # (small batches of such jobs take the low-latency path, except where the dispatch quantises)
                dtype = "fp8_fused"
            local = _log_int(rng, 2, 128) if world < 64 else rng.randint(1, 8)
            case = dict(family=family, world=world, rank=rng.randrange(world), tokens=_log_int(rng, 1, 8192),
                        hidden=_multiple(rng, 16 if dtype == "bf16" else 128, 256, 7168), topk=rng.randint(1, 10),
                        experts=world * local, dtype=dtype, weights=rng.random() < 0.7, skew=rng.choice((0.0, 0.6, 1.2)),
                        masked=rng.choice((0.0, 0.0, 0.15)), overlap=rng.random() < 0.3, backward=dtype == "bf16" and rng.random() < 0.4)
            rows = case["tokens"] * case["topk"]
            if case["topk"] <= case["experts"] <= 1024 and world * case["tokens"] <= 32768 and rows * case["hidden"] * 2 <= _MOST_PAYLOAD_BYTES:
                return case
        elif family == "low_latency":
            world = rng.choice((16, 32, 64, 128))
            dtype = rng.choice(("bf16", "fp16", "fp8"))
            case = dict(family=family, world=world, rank=rng.randrange(world), tokens=_log_int(rng, 1, 256),
                        hidden=_multiple(rng, 128, 1024, 7168), topk=rng.randint(2, 8), experts=world * rng.randint(1, 8),
                        dtype=dtype, skew=rng.choice((0.0, 0.6)))
            local = case["experts"] // world
            rows = world * case["tokens"] * min(case["topk"], local)
            if case["experts"] >= case["topk"] and rows * case["hidden"] * 2 <= _MOST_CAPACITY_BYTES:
                return case
        elif family == "mega":
            world = rng.choice((1, 1, 8, 64))
            local = _log_int(rng, 2, 64) if world < 64 else rng.randint(2, 8)
            case = dict(family=family, world=world, rank=rng.randrange(world), tokens=_log_int(rng, 1, 16384 // world),
                        hidden=_multiple(rng, 64, 1024, 8192), inter=_multiple(rng, 128, 256, 4096), topk=rng.randint(1, 8),
                        experts=world * local, shared=rng.choice((0, 0, 0, 1, 2)), input=rng.choice(("fp8", "bf16")))
            weight_bytes = (local + case["shared"]) * 3 * case["inter"] * case["hidden"] // 2
            if case["topk"] <= case["experts"] and work(case)["flops"] <= _MOST_MEGA_FLOPS and weight_bytes <= _MOST_WEIGHT_BYTES:
                return case
        else:
            case = dict(family=family, tokens=_log_int(rng, 1, 32768), hidden=_multiple(rng, 16, 128, 16384))
            if case["tokens"] * case["hidden"] <= 1 << 28:
                return case


class _State:
    """One call's inputs and the buffer they go through, released together."""

    def __init__(self, case, **fields):
        self.family = case["family"]
        self.buffer = None
        self.__dict__.update(fields)

    def __del__(self):
        if self.buffer is not None:
            self.buffer.destroy()


def _routes(gen, tokens, experts, topk, skew, masked=0.0):
    """Distinct top-k experts per token, expert e with popularity (e + 1)^-skew; masked: share of tokens that are padding."""
    padding = int(masked * tokens)
    popularity = -skew * torch.log(torch.arange(1, experts + 1, device="cuda", dtype=torch.float32))
    uniform = torch.rand((tokens, experts), generator=gen, device="cuda").clamp_(1e-20, 1.0 - 1e-7)
    idx = (popularity - torch.log(-torch.log(uniform))).topk(topk, dim=1).indices
    if padding:
        idx[torch.randperm(tokens, generator=gen, device="cuda")[:padding]] = -1
    return idx.contiguous()


def _share_routes(gen, case, masked=0.0):
    """Routes whose number of rows on this rank depends on the case alone (so do the shapes of what a call returns): with
    several ranks the seed decides which token goes where, not how many come here."""
    tokens = case["world"] * case["tokens"]
    if case["world"] == 1:
        return _routes(gen, tokens, case["experts"], case["topk"], case["skew"], masked)
    table = _routes(torch.Generator(device="cuda").manual_seed(0), tokens, case["experts"], case["topk"], case["skew"], masked)
    first, local = case["rank"] * case["experts"] // case["world"], case["experts"] // case["world"]
    if not bool(((table >= first) & (table < first + local)).any()):
        table[0, 0] = first
    return table[torch.randperm(tokens, generator=gen, device="cuda")].contiguous()


def _route_weights(gen, tokens, topk):
    return torch.softmax(torch.randn((tokens, topk), generator=gen, device="cuda"), dim=-1)


def _normal(gen, *shape, dtype=torch.bfloat16):
    return torch.randn(shape, generator=gen, device="cuda").to(dtype)


def _prepare_exchange(case, gen):
    world, rank, hidden, topk, experts = (case[k] for k in ("world", "rank", "hidden", "topk", "experts"))
    tokens, local = world * case["tokens"], experts // world
    idx = _share_routes(gen, case, case["masked"])
    rows = int(((idx >= rank * local) & (idx < (rank + 1) * local)).sum())
    x = _normal(gen, tokens, hidden)
    buffer = deepep_amd.ElasticBuffer(
        None, num_max_tokens_per_rank=case["tokens"], hidden=hidden, num_topk=topk, use_fp8_dispatch=case["dtype"] != "bf16",
        explicitly_destroy=True, rank=rank, world_size=world)
    return _State(
        case, buffer=buffer, x=utils.per_token_cast_to_fp8(x) if case["dtype"] == "fp8" else x, idx=idx, experts=experts,
        weights=_route_weights(gen, tokens, topk) if case["weights"] else None,
        expert_out=_normal(gen, rows, hidden),
        overlap=case["overlap"],
        grad_out=_normal(gen, tokens, hidden) if case["backward"] else None,
        grad_rows=_normal(gen, rows, hidden) if case["backward"] else None,
        grad_weights=_normal(gen, rows, dtype=torch.float32) if case["backward"] else None)


def _run_exchange(state):
    buffer, overlap = state.buffer, state.overlap
    received, _, received_weights, handle, event = buffer.dispatch(
        state.x, topk_idx=state.idx, topk_weights=state.weights, num_experts=state.experts, async_with_compute_stream=overlap)
    if overlap:
        event.current_stream_wait()
    combined, _, event = buffer.combine(state.expert_out, handle, async_with_compute_stream=overlap)
    if overlap:
        event.current_stream_wait()
    out = [received, received_weights, handle.expert_totals, handle.psum_num_recv_tokens_per_expert, handle.route_to_row,
           handle.weight_return_meta, handle.num_expanded_tokens, combined]
    if state.grad_out is not None:
        grad_expert_out, _, _, _, event = buffer.dispatch(state.grad_out, handle=handle, async_with_compute_stream=overlap)
        if overlap:
            event.current_stream_wait()
        grad_x, grad_topk_weights, event = buffer.combine(
            state.grad_rows, handle, topk_weights=state.grad_weights, async_with_compute_stream=overlap)
        if overlap:
            event.current_stream_wait()
        out += [grad_expert_out, grad_x, grad_topk_weights]
    return out


def _prepare_low_latency(case, gen):
    world, rank, hidden, topk, experts = (case[k] for k in ("world", "rank", "hidden", "topk", "experts"))
    tokens, local = world * case["tokens"], experts // world
    idx = _share_routes(gen, case)
    rows = int(((idx >= rank * local) & (idx < (rank + 1) * local)).sum())
    x = _normal(gen, tokens, hidden, dtype=torch.float16 if case["dtype"] == "fp16" else torch.bfloat16)
    buffer = deepep_amd.ElasticBuffer(
        None, num_bytes=8 << 30, num_max_tokens_per_rank=case["tokens"], hidden=hidden, num_topk=topk, explicitly_destroy=True,
        rank=rank, world_size=world)
    # the experts write the valid rows of the capacity layout; what lies behind them is never read
    expert_out = torch.zeros((world * case["tokens"] * min(topk, local), hidden), dtype=x.dtype, device="cuda")
    expert_out[:rows] = _normal(gen, rows, hidden, dtype=x.dtype)
    return _State(case, buffer=buffer, x=utils.per_token_cast_to_fp8(x) if case["dtype"] == "fp8" else x, idx=idx, experts=experts,
                  weights=_route_weights(gen, tokens, topk), expert_out=expert_out, rows=rows)


def _run_low_latency(state):
    received, _, _, handle, _ = state.buffer.dispatch(
        state.x, topk_idx=state.idx, topk_weights=state.weights, num_experts=state.experts)
    combined, _, _ = state.buffer.combine(state.expert_out, handle)
    rows = state.rows  # only the valid rows of the capacity layout are written
    received = tuple(t[:rows] for t in received) if isinstance(received, tuple) else received[:rows]
    return [received, handle.source_weights[:rows], handle.route_to_row, handle.send_counts, combined]


def _mxfp4(gen, experts, n, k):
    """Normal weights of scale 0.02 as packed e2m1 codes with a power-of-two scale per 32 of K (OCP MX)."""
    edges = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device="cuda")
    packed = torch.empty((experts, n, k // 2), dtype=torch.uint8, device="cuda")
    scales = torch.empty((experts, n, k // 64, 2), dtype=torch.uint8, device="cuda")
    for e in range(experts):
        w = torch.randn((n, k // 32, 32), generator=gen, device="cuda").mul_(0.02)
        exponent = torch.frexp(w.abs().amax(dim=-1, keepdim=True)).exponent - 3  # floor(log2(largest)) - 2
        w = torch.ldexp(w, -exponent)
        code = (torch.bucketize(w.abs(), edges, out_int32=True) + 8 * (w < 0)).to(torch.uint8).view(n, k)
        packed[e] = code[:, 0::2] | (code[:, 1::2] << 4)
        scales[e] = (exponent + 127).to(torch.uint8).view(n, k // 64, 2)
    return packed, scales


def _prepare_mega(case, gen):
    world, rank, hidden, inter, topk, experts = (case[k] for k in ("world", "rank", "hidden", "inter", "topk", "experts"))
    tokens, local = world * case["tokens"], experts // world
    buffer = megamoe.SymmBuffer(megamoe.LocalGroup(rank, world), experts, case["tokens"], topk, hidden, inter, case["shared"])
    l1, l2 = megamoe.transform_weights_for_mega_moe(_mxfp4(gen, local, 2 * inter, hidden), _mxfp4(gen, local, hidden, inter))
    shared = (None, None)
    if case["shared"]:
        shared = megamoe.transform_weights_for_mega_moe(
            _mxfp4(gen, case["shared"], 2 * inter, hidden), _mxfp4(gen, case["shared"], hidden, inter), shared=True)
    x = _normal(gen, tokens, hidden)
    idx = _routes(gen, tokens, experts, topk, 0.0).to(torch.int32)
    weights = _route_weights(gen, tokens, topk)
    y = torch.zeros((tokens, hidden), dtype=torch.bfloat16, device="cuda")
    buffer.prepare(tokens)
    if case["input"] == "fp8":
        codes, scales = ops.mx_quant(x)
        buffer.x.copy_(codes)
        buffer.x_sf.view(torch.uint8).copy_(scales)
        buffer.topk_idx.copy_(idx)
        buffer.topk_weights.copy_(weights)
        x = None
    return _State(case, buffer=buffer, x=x, idx=idx, weights=weights, l1=l1, l2=l2, shared_l1=shared[0], shared_l2=shared[1], y=y)


def _run_mega(state):
    if state.x is None:
        megamoe.fp8_fp4_mega_moe(state.y, state.l1, state.l2, state.buffer, state.shared_l1, state.shared_l2)
        return [state.y]
    y, counts = megamoe.mega_moe(state.x, state.idx, state.weights, state.l1, state.l2, state.buffer,
                                 shared_l1_weights=state.shared_l1, shared_l2_weights=state.shared_l2, out=state.y)
    return [y, counts]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    family = case["family"]
    if family == "exchange":
        return _prepare_exchange(case, gen)
    if family == "low_latency":
        return _prepare_low_latency(case, gen)
    if family == "mega":
        return _prepare_mega(case, gen)
    return _State(case, x=_normal(gen, case["tokens"], case["hidden"]))


def run(state):
    if state.family == "exchange":
        return _run_exchange(state)
    if state.family == "low_latency":
        return _run_low_latency(state)
    if state.family == "mega":
        return _run_mega(state)
    codes, scales = utils.per_token_cast_to_fp8(state.x)
    return [codes, scales, utils.per_token_cast_back(codes, scales)]


def _served(topk, share):
    """Expected share of tokens with at least one of their top-k routes here."""
    return 1.0 - (1.0 - share) ** topk


def work(case):
    """Bytes and operations of one pass: inputs read once, outputs written once (expected values of the routing)."""
    family, hidden = case["family"], case["hidden"]
    if family == "cast":
        values = case["tokens"] * hidden
        scales = case["tokens"] * -(-hidden // 128) * 4
        return {"bytes": values * (2 + 1) + scales + values * (1 + 2) + scales, "flops": 0}
    tokens, topk, share = case["world"] * case["tokens"], case["topk"], 1.0 / case["world"]
    routes = tokens * topk
    if family == "mega":
        touched = 1.0 - (1.0 - topk / case["experts"]) ** tokens  # share of the experts that any token goes to
        local = case["experts"] // case["world"] * touched + case["shared"]
        rows = routes * share + tokens * case["shared"]
        served = tokens if case["shared"] else tokens * _served(topk, share)
        weights = local * 3 * case["inter"] * hidden * (0.5 + 1.0 / 32)
        x_bytes = served * hidden * (33.0 / 32 if case["input"] == "fp8" else 2.0)
        return {"bytes": weights + x_bytes + routes * 8 + tokens * hidden * 2, "flops": rows * 6.0 * case["inter"] * hidden}
    kept = 1.0 - int(case.get("masked", 0.0) * tokens) / tokens
    rows, served = routes * share * kept, tokens * kept * _served(topk, share)
    scales = hidden // 128 * 4
    read = {"bf16": hidden * 2, "fp16": hidden * 2, "fp8_fused": hidden * 2, "fp8": hidden + scales}[case["dtype"]]
    written = hidden * 2 if case["dtype"] in ("bf16", "fp16") else hidden + scales
    weighted = 8 if case.get("weights", True) else 0
    dispatch = routes * 12 + served * read + rows * (written + 4 + weighted)
    combine = routes * 4 + rows * hidden * 2 + tokens * hidden * 2
    total, adds = dispatch + combine, rows * hidden
    if family == "low_latency":
        total, adds = total + rows * 4 + case["experts"] * 4, 2 * adds
    elif case["backward"]:
        total += served * read + rows * written + combine + rows * 4 + routes * 4
        adds *= 2
    return {"bytes": total, "flops": adds}


def tolerance(case):
    """Rows are moved, quantised and summed in a fixed order with single roundings: bit for bit.  The W4A8 layer sums
    products of 8- and 4-bit values in fp32 and rounds to BF16 and e4m3 in between."""
    return {"rel": 1e-2} if case["family"] == "mega" else "exact"
