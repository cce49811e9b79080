"""The native host path and the Python layer state the same rules twice (csrc/host.cpp returns None for a call that it does not
take, elastic.py then finds out why): seeded draws of calls, valid and faulty, made once through the native path and once with it
taken away, have to end alike: the same exception with the same text, or the same path, results and handle."""

import random

import pytest
import torch

pytestmark = pytest.mark.gpu


def _tensor_form(rng, t, others):
    """`t` in a form that a call may refuse."""
    form = rng.choice(["strided", "grad", "cpu", "short", "dtype"])
    if form == "strided":
        return torch.stack([t, t], dim=-1)[..., 0]
    if form == "grad":
        return t.clone().requires_grad_(True) if t.is_floating_point() and t.element_size() > 1 else t
    if form == "cpu":
        return t.cpu()
    if form == "short":
        return t[:-1].contiguous() if t.shape[0] > 1 else t[:, :-1].contiguous() if t.dim() == 2 else t
    return t.to(rng.choice(others))


# Argument: values, valid and faulty, that replace its default ("event": a recorded EventHandle).
OPTIONS = {
    "num_sms": (32, 64, 7, True, None), "num_qps": (2, 2, 1, False, "2"), "expert_alignment": (1, 1, True, 128), "do_cpu_sync": (True, True, False, 1),
    "do_expand": (True, True, False, 1), "do_handle_copy": (False, False, 1, None), "async_with_compute_stream": (True, True, True, 1, None),
    "allocate_on_comm_stream": (True, 0), "do_zero_padding": (True, 0), "use_tma_aligned_col_major_sf": (True, 0),
    "cumulative_local_expert_recv_stats": ("tensor",), "previous_event": ("event", "event", "event", 5),
}


def _draw_call(rng, gen):
    """(buffer options, positional payload, keyword arguments) of one dispatch: an ordinary call with at most two oddities."""
    odd = rng.sample(["x", "scales", "idx", "weights", "payload", "width", "topk", "experts", "capacity", "bound", "hidden", "num_topk", "combine_only",
                      "bytes", *OPTIONS, *OPTIONS], rng.choice((0, 0, 1, 1, 1, 2)))
    world = rng.choice((1, 1, 2, 4, 16, 16, 64))
    per_rank = rng.choice((1, 3, 17, 40, 256, 257) if world == 16 else (1, 3, 17, 40))
    tokens = max(world * per_rank - rng.choice((0, 0, 1)), 1)
    topk = rng.choice((1, 2, 6, 8, 16))
    if "topk" in odd:
        topk = 17 if per_rank <= 40 else 16
    experts = world * max(rng.choice((1, 2, 3, 8)), -(-topk // world))
    payload = rng.choice(("bf16", "bf16", "fp8"))
    if "payload" in odd:
        payload = rng.choice(("fp8_packed", "fp8_packed", "fp16", "fp16", "fp8_bare", "fp32"))
    width = rng.choice((128, 256, 384, 512))
    if "width" in odd:
        width = rng.choice((16, 48, 200, 8))
    x = torch.randn(tokens, width, generator=gen)
    blocks = -(-width // 128)
    if payload.startswith("fp8"):
        codes = x.cuda().to(torch.float8_e4m3fn)
        scales = torch.rand(tokens, blocks, generator=gen).cuda()
        if payload == "fp8_packed":
            scales = torch.randint(0, 1 << 30, (tokens, blocks), generator=gen, dtype=torch.int32).cuda()
        x = codes if payload == "fp8_bare" else (codes, _tensor_form(rng, scales, (torch.float64,)) if "scales" in odd else scales)
    else:
        x = x.to({"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}[payload]).cuda()
        if "x" in odd:
            x = _tensor_form(rng, x, (torch.float64,))
    idx = torch.stack([torch.randperm(experts, generator=gen)[:topk] for _ in range(tokens)]).cuda()
    idx[torch.rand(idx.shape, generator=gen).cuda() < 0.1] = -1
    weights = torch.rand(tokens, topk, generator=gen).cuda() if rng.random() < 0.7 else None
    if "idx" in odd:
        idx = _tensor_form(rng, idx, (torch.int32,))
    if "weights" in odd and weights is not None:
        weights = _tensor_form(rng, weights, (torch.float64, torch.bfloat16))
    kwargs = dict(topk_idx=idx, topk_weights=weights, num_experts=experts)
    if "experts" in odd:
        kwargs["num_experts"] = rng.choice((experts + 1, True, float(experts), world - 1, 1025 * world, None))
    bound = -(-tokens // world)
    if "capacity" in odd:
        kwargs["num_max_tokens_per_rank"] = rng.choice((bound, bound + 5, bound + 5, bound - 1, 0, True, float(bound), 256, 16384, 16385))
    for name, values in OPTIONS.items():
        if name in odd:
            kwargs[name] = rng.choice(values)
    options = dict(num_bytes=8 << 30 if world >= 16 and "bytes" not in odd else 4 << 20, rank=rng.randrange(world), world_size=world,
                   use_fp8_dispatch=rng.random() < 0.3 and width % 128 == 0, combine_only="combine_only" in odd)
    if "bound" in odd:
        options["num_max_tokens_per_rank"] = rng.choice((bound, bound + 7, max(bound - 1, 1)))
    if "hidden" in odd and width % 128 == 0:
        options["hidden"] = rng.choice((width, 1024))
    if "num_topk" in odd and topk <= 16:
        options["num_topk"] = rng.choice((topk, 3))
    return options, x, kwargs


def _draw_combine(rng):
    """How the combine behind a dispatch is called: applied to both sides' handles."""
    changes = {}
    if rng.random() < 0.3:
        changes["weights"] = rng.choice(("rows", "short", "float64", "cpu"))
    if rng.random() < 0.15:
        changes["rows"] = rng.choice(("short", "strided", "fp16", "fp32", "grad"))
    for name, values in (("num_sms", (64, 32, True)), ("num_qps", (2, 1, False)), ("bias", (0,)), ("async_with_compute_stream", (True, 1)),
                         ("allocate_on_comm_stream", (True, 0)), ("previous_event", ("event", 5))):
        if rng.random() < 0.1:
            changes[name] = rng.choice(values)
    return changes


def _outcome(function):
    try:
        return "done", function()
    except Exception as error:  # noqa: BLE001 - what is raised is what is compared
        return type(error).__name__, str(error)


def _bits(value, valid=None):
    if value is None or isinstance(value, (bool, int, str)):
        return value
    if isinstance(value, (tuple, list)):
        return [_bits(v, valid) for v in value]
    t = value.detach() if valid is None else value.detach()[:valid]
    return [str(value.dtype), list(value.shape), t.cpu().contiguous().view(torch.uint8).numpy().tobytes() if t.numel() else b""]


HANDLE = ("do_expand", "num_experts", "expert_alignment", "num_max_tokens_per_rank", "num_compute_units", "num_recv_tokens", "num_expanded_tokens",
          "num_recv_tokens_per_expert_list", "is_low_latency", "rank", "world_size", "num_tokens", "num_topk", "hidden", "metadata_only",
          "metadata_version", "psum_num_recv_tokens_per_scaleup_rank", "recv_src_metadata", "dst_buffer_slot_idx",
          "token_metadata_at_forward", "channel_linked_list", "expert_recv_counts")
TENSORS = ("topk_idx", "psum_num_recv_tokens_per_expert", "num_unaligned_recv_tokens_per_expert", "route_to_row", "weight_return_meta",
           "expert_totals", "expert_offsets", "send_counts")


def _side(native, options, x, kwargs, changes, gen_seed):
    """One draw through one of the two: what dispatch, a cached dispatch and combine did."""
    import deepep_amd
    from deepep_amd.event import EventHandle

    def event(given):
        return EventHandle() if given == "event" else torch.zeros(1) if given == "tensor" else given

    report = []
    made = _outcome(lambda: deepep_amd.ElasticBuffer(None, explicitly_destroy=True, **options))
    if made[0] != "done":
        return [made]
    buffer = made[1]
    try:
        if not native:
            buffer._exchange = None
        arguments = {k: event(v) if isinstance(v, str) else v for k, v in kwargs.items()}
        status, got = _outcome(lambda: buffer.dispatch(x, **arguments))
        if status != "done":
            return [(status, got, buffer._runtime.notify_failed)]
        received, nothing, received_weights, handle, overlap = got
        torch.cuda.synchronize()
        valid = int(handle.send_counts[-1]) if handle.is_low_latency else None
        report += [_bits(received, valid), nothing, _bits(received_weights, valid), overlap.event is None]
        report += [getattr(handle, name) for name in HANDLE]
        report += [_bits(getattr(handle, name)) for name in TENSORS]
        report.append(_bits(handle.source_weights, valid))
        rows, width = handle.num_expanded_tokens, handle.hidden
        y = torch.randn((rows, width), generator=torch.Generator().manual_seed(gen_seed)).bfloat16().cuda()
        if handle.is_low_latency:
            y[valid:] = 0
        y = {"short": lambda: y[: max(rows - 1, 0)], "strided": lambda: torch.stack([y, y], dim=-1)[..., 0], "fp16": y.half, "fp32": y.float,
             "grad": lambda: y.clone().requires_grad_(True)}.get(changes.get("rows"), lambda: y)()
        extra = {k: event(v) if isinstance(v, str) else v for k, v in changes.items() if k not in ("rows", "weights")}
        if "weights" in changes:
            w = torch.rand(rows, generator=torch.Generator().manual_seed(1)).cuda()
            extra["topk_weights"] = {"rows": w, "short": w[:-1], "float64": w.double(), "cpu": w.cpu()}[changes["weights"]]
        for call in (lambda: buffer.combine(y, handle, **extra)[:2], lambda: buffer.dispatch(x, handle=handle)[:3],
                     lambda: buffer.dispatch(x, handle=handle, topk_weights=kwargs["topk_weights"])[:3],
                     lambda: buffer.combine(y, handle)[:2]):
            status, got = _outcome(call)
            torch.cuda.synchronize()
            report.append((status, _bits(got) if status == "done" else got))
        report.append(buffer._runtime.notify_failed)
        return report
    finally:
        torch.cuda.synchronize()
        buffer.destroy()


@pytest.mark.parametrize("seed", range(40))
def test_native_path_and_python_layer_agree(seed):
    rng, gen = random.Random(seed), torch.Generator().manual_seed(seed)
    for draw in range(12):
        options, x, kwargs = _draw_call(rng, gen)
        changes = _draw_combine(rng)
        case = (seed, draw, options, {k: v for k, v in kwargs.items() if not isinstance(v, torch.Tensor)}, changes)
        print(case, flush=True)
        sides = [_side(native, options, x, kwargs, changes, seed) for native in (True, False)]
        assert len(sides[0]) == len(sides[1]), (case, sides)
        for at, (a, b) in enumerate(zip(*sides)):
            assert a == b, (case, at, str(a)[:300], str(b)[:300])


def test_bounds_of_the_native_path_are_the_python_layers():
    """Draws seldom touch them, so one by one: the largest value that is taken and the first that is not."""
    import deepep_amd

    for native in (True, False):
        buffer = deepep_amd.ElasticBuffer(None, num_bytes=4 << 20, explicitly_destroy=True)
        try:
            if not native:
                buffer._exchange = None
            for tokens, width, topk, experts, good in ((16384, 16, 1, 4, True), (16385, 16, 1, 4, False), (2, 7168, 1, 4, True), (2, 7184, 1, 4, False),
                                                       (2, 16, 16, 16, True), (2, 16, 17, 32, False), (2, 16, 1, 1024, True), (2, 16, 1, 1025, False)):
                x = torch.ones(tokens, width, dtype=torch.bfloat16, device="cuda")
                idx = torch.arange(topk, device="cuda").repeat(tokens, 1).contiguous()
                status, got = _outcome(lambda: buffer.dispatch(x, topk_idx=idx, num_experts=experts))
                assert (status == "done") == good and (good or status == "ValueError"), (native, tokens, width, topk, experts, got)
        finally:
            torch.cuda.synchronize()
            buffer.destroy()
