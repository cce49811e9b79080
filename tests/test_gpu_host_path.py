"""The native host path of ElasticBuffer (csrc/host.cpp) where it can go wrong: outputs allocated before the row count is known
and outgrown by it, row-major payloads that walk past their grid, the routing copy, ids per rank of the low-latency path,
handles that leave the native path, and memory that is handed out again behind asynchronous calls."""

import ctypes
import threading
import time

import numpy as np
import pytest
import torch

from oracle import combine as ocombine
from oracle import layout as olayout
from oracle import quant as oquant
from tests.gpu_util import bf16_bits, f32_bits, fp8_bits

pytestmark = pytest.mark.gpu


def _buffer(**options):
    import deepep_amd

    return deepep_amd.ElasticBuffer(None, explicitly_destroy=True, **options)


def _batch(tokens, hidden, topk, seed):
    gen = torch.Generator().manual_seed(seed)
    return torch.randn(tokens, hidden, generator=gen).bfloat16(), torch.rand(tokens, topk, generator=gen)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("world", [2, 4, 16])
def test_rows_of_a_share_far_from_the_expected_number(world, fp8):
    """One buffer, batches whose share of rows jumps: about the expected one, everything (outputs are outgrown, the payload is
    dispatched again), nothing, one row, everything again (sized by the batch before), and a batch of the one-launch size."""
    experts, topk, hidden = world * 4, 4, 256
    rank = world - 1
    local = range(rank * 4, rank * 4 + 4)
    rng = np.random.default_rng(world)
    buffer = _buffer(num_bytes=4 << 20, rank=rank, world_size=world, use_fp8_dispatch=fp8)
    try:
        for step, (tokens, kind) in enumerate([(1024, "usual"), (1024, "all"), (1024, "none"), (1024, "one"), (900, "all"), (1024, "usual"),
                                               (64, "all"), (64, "usual")]):
            ids = np.stack([rng.permutation(experts)[:topk] for _ in range(tokens)]).astype(np.int64)
            if kind == "all":
                ids = np.stack([rng.permutation(local)[:topk] for _ in range(tokens)]).astype(np.int64)
            elif kind != "usual":
                ids[np.isin(ids, local)] = -1
                if kind == "one":
                    ids[tokens - 1, topk - 1] = local[1]
            x, w = _batch(tokens, hidden, topk, step)
            idx = torch.from_numpy(ids).cuda()
            weights = w.cuda() if world < 16 or fp8 else None  # (with weights, EP16 and BF16 this would be a low-latency call)
            want = olayout.layout(ids, experts, rank * 4, 4)
            recv, _, recv_w, handle, _ = buffer.dispatch(x.cuda(), topk_idx=idx, topk_weights=weights, num_experts=experts)
            assert handle.num_expanded_tokens == want["num_rows"], (step, kind)
            assert handle.num_recv_tokens_per_expert_list == want["counts"].tolist()
            np.testing.assert_array_equal(handle.route_to_row.cpu().numpy(), want["route_to_row"])
            np.testing.assert_array_equal(handle.weight_return_meta.cpu().numpy(), want["row_to_route"])
            np.testing.assert_array_equal(handle.psum_num_recv_tokens_per_expert.cpu().numpy(), want["psum"])
            np.testing.assert_array_equal(handle.expert_offsets.cpu().numpy(), want["offsets"])
            assert torch.equal(handle.topk_idx, idx) and handle.topk_idx.data_ptr() != idx.data_ptr()
            if fp8:
                q, s = oquant.cast_to_fp8_torch(x)
                np.testing.assert_array_equal(fp8_bits(recv[0]), olayout.expand_rows(fp8_bits(q), want["row_to_route"], topk))
                np.testing.assert_array_equal(f32_bits(recv[1]), olayout.expand_rows(f32_bits(s), want["row_to_route"], topk))
            else:
                np.testing.assert_array_equal(bf16_bits(recv), olayout.expand_rows(bf16_bits(x), want["row_to_route"], topk))
            if weights is not None:
                np.testing.assert_array_equal(f32_bits(recv_w), olayout.expand_weights(w.numpy(), want["row_to_route"]).view(np.uint32))
            y = torch.randn(want["num_rows"], hidden).bfloat16()
            out, _, _ = buffer.combine(y.cuda(), handle)
            np.testing.assert_array_equal(bf16_bits(out), ocombine.combine(bf16_bits(y), want["route_to_row"]))
    finally:
        buffer.destroy()


@pytest.mark.parametrize("per_rank,skewed", [(3, False), (64, False), (64, True)])
def test_low_latency_ids_and_send_counts(per_rank, skewed):
    """Below and above the one-launch size, and with a share far above the expected one (row-major workgroups walk on)."""
    world, rank, experts, topk, hidden = 16, 9, 64, 8, 512
    rng = np.random.default_rng(per_rank)
    tokens = world * per_rank
    popularity = np.ones(experts)
    if skewed:
        popularity[rank * 4 : rank * 4 + 4] = 1000.0
    ids = np.stack([rng.choice(experts, topk, replace=False, p=popularity / popularity.sum()) for _ in range(tokens)]).astype(np.int64)
    x, w = _batch(tokens, hidden, topk, 5)
    want = olayout.layout(ids, experts, rank * 4, 4)
    buffer = _buffer(num_bytes=8 << 30, rank=rank, world_size=world)
    try:
        idx = torch.from_numpy(ids).cuda()
        recv, _, _, handle, _ = buffer.dispatch(x.cuda(), topk_idx=idx, topk_weights=w.cuda(), num_experts=experts)
        rows = want["num_rows"]
        np.testing.assert_array_equal(bf16_bits(recv[:rows]), olayout.expand_rows(bf16_bits(x), want["row_to_route"], topk))
        np.testing.assert_array_equal(f32_bits(handle.source_weights[:rows]), olayout.expand_weights(w.numpy(), want["row_to_route"]).view(np.uint32))
        sent = np.zeros(experts, np.int32)
        sent[rank * 4 : rank * 4 + 4] = want["psum"]
        sent[rank * 4 + 4 :] = rows
        np.testing.assert_array_equal(handle.send_counts.cpu().numpy(), sent)
        np.testing.assert_array_equal(handle.route_to_row.cpu().numpy(), want["route_to_row"])
        assert torch.equal(handle.topk_idx, idx)
        y = torch.zeros_like(recv)
        y[:rows] = recv[:rows]
        out, _, _ = buffer.combine(y, handle)
        np.testing.assert_array_equal(bf16_bits(out), ocombine.combine(bf16_bits(recv[:rows]), want["route_to_row"],
                                                                       olayout.expand_weights(w.numpy(), want["row_to_route"])))
    finally:
        buffer.destroy()


@pytest.mark.parametrize("world,tokens,experts,topk", [(1, 1, 1, 1), (1, 31, 8, 2), (1, 1000, 160, 6), (8, 2048, 256, 8), (16, 37, 496, 3),
                                                       (16, 256, 512, 5)])
def test_received_weights_and_maps_are_aligned_and_keep_little_else_alive(world, tokens, experts, topk):
    """Whatever they share an allocation with: addresses as a tensor of its own would have them, and no more than 64 KiB
    held through the weights beyond their own rows."""
    hidden, per_rank = 256, tokens if world < 16 else -(-tokens // world)
    x, w = _batch(per_rank * world if world >= 16 else tokens, hidden, topk, 8)
    idx = torch.stack([torch.randperm(experts)[:topk] for _ in range(x.shape[0])]).cuda()
    buffer = _buffer(num_bytes=8 << 30, rank=world - 1, world_size=world)
    try:
        recv, _, recv_w, handle, _ = buffer.dispatch(x.cuda(), topk_idx=idx, topk_weights=w.cuda(), num_experts=experts)
        assert handle.is_low_latency == (world == 16)
        weights = handle.source_weights if handle.is_low_latency else recv_w
        maps = [handle.topk_idx, handle.route_to_row] + ([] if handle.is_low_latency else [handle.weight_return_meta])
        for t in (weights, *maps):
            assert t.data_ptr() % 256 == 0
        held = weights.untyped_storage().nbytes()
        assert held <= 65536 or held <= 4 * recv.untyped_storage().nbytes() // (hidden * 2)
        if not handle.is_low_latency:
            want = olayout.layout(idx.cpu().numpy(), experts, (world - 1) * experts // world, experts // world)
            np.testing.assert_array_equal(f32_bits(weights), olayout.expand_weights(w.numpy(), want["row_to_route"]).view(np.uint32))
            np.testing.assert_array_equal(handle.weight_return_meta.cpu().numpy(), want["row_to_route"])
            np.testing.assert_array_equal(handle.expert_offsets.cpu().numpy(), want["offsets"])
    finally:
        buffer.destroy()


def test_changed_handles_and_unusual_tensors_take_the_slow_path():
    x, w = _batch(40, 256, 2, 1)
    idx = torch.stack([torch.randperm(8)[:2] for _ in range(40)]).cuda()
    buffer = _buffer(num_bytes=4 << 20)
    try:
        recv, _, _, handle, _ = buffer.dispatch(x.cuda(), topk_idx=idx, topk_weights=w.cuda(), num_experts=8)
        want, _, _ = buffer.combine(recv, handle)
        # inference mode: carried out step by step, the same results
        with torch.inference_mode():
            again, _, _, other, _ = buffer.dispatch(x.cuda(), topk_idx=idx, topk_weights=w.cuda(), num_experts=8)
            assert torch.equal(again, recv) and torch.equal(buffer.combine(again, handle)[0], want)
        assert torch.equal(buffer.combine(recv, other)[0], want)
        # a low-latency style handle: the saved weights multiply the rows
        handle.is_low_latency, handle.source_weights = True, torch.full((handle.num_expanded_tokens,), 2.0, device="cuda")
        assert torch.equal(buffer.combine(recv, handle)[0], (want.float() * 2).bfloat16())
        handle.is_low_latency = False
        with pytest.raises(ValueError, match="matching the handle"):
            buffer.combine(recv[:-1], handle)
        # an edit of the routing is found on the native path as well
        handle.expert_totals.add_(0)
        with pytest.raises(ValueError, match="Cached routing was modified: expert_totals"):
            buffer.combine(recv, handle)
        with pytest.raises(ValueError, match="Cached routing was modified"):
            buffer.dispatch(x.cuda(), handle=handle)
        other.route_to_row = other.route_to_row.clone()
        with pytest.raises(ValueError, match="Cached routing was modified: route_to_row"):
            buffer.combine(recv, other)
    finally:
        buffer.destroy()


@pytest.mark.parametrize("wait", ["caller", "other", "never"])
def test_memory_of_asynchronous_calls_is_not_handed_out_too_early(wait):
    """Everything an asynchronous call used is dropped right after it, behind a kernel that keeps the communication stream
    busy, and the allocator is asked for the same sizes at once: what the call wrote must still be right."""
    tokens, hidden, topk, experts = 512, 1024, 4, 16
    x, w = _batch(tokens, hidden, topk, 2)
    ids = torch.stack([torch.randperm(experts)[:topk] for _ in range(tokens)])
    want = olayout.layout(ids.numpy(), experts)
    rows = olayout.expand_rows(bf16_bits(x), want["row_to_route"], topk)
    buffer = _buffer(num_bytes=4 << 20)
    side = torch.cuda.Stream()
    try:
        idx, xd = ids.cuda(), x.cuda()
        _, _, _, handle, _ = buffer.dispatch(xd, topk_idx=idx, num_experts=experts)
        for _ in range(8):
            torch.cuda.synchronize()
            with torch.cuda.stream(buffer.get_comm_stream()):
                torch.cuda._sleep(2_000_000)
            payload = xd.clone()
            recv, _, _, _, event = buffer.dispatch(payload, handle=handle, async_with_compute_stream=True)
            if wait == "never":
                kept = recv  # waited for by hand below
            elif wait == "caller":
                event.current_stream_wait()
                kept = recv.clone()
                del recv
            else:
                with torch.cuda.stream(side):
                    event.current_stream_wait()
                    torch.cuda._sleep(1_000_000)
                    kept = recv.clone()
                del recv
            del payload, event
            noise = [torch.full((want["num_rows"], hidden), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(3)]
            noise += [torch.full((tokens, hidden), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(3)]
            buffer.get_comm_stream().synchronize()
            torch.cuda.synchronize()
            np.testing.assert_array_equal(bf16_bits(kept), rows)
            del noise, kept
            if wait == "never":
                del recv
    finally:
        torch.cuda.synchronize()
        buffer.destroy()


@pytest.mark.parametrize("wait", ["caller", "other", "never"])
def test_rows_of_an_outgrown_asynchronous_dispatch_outlive_their_tensor_while_they_are_read(wait):
    """The outputs made once the row count is known belong to the communication stream: dropped right behind their last use
    (queued, not run yet), their memory must not go to what that stream is given next."""
    world, experts, topk, tokens, hidden = 4, 16, 4, 4096, 1024
    x, _ = _batch(tokens, hidden, topk, 13)
    ids = np.stack([np.random.default_rng(13).permutation(4)[:topk] for _ in range(tokens)]).astype(np.int64)
    want = olayout.layout(ids, experts, 0, 4)
    xd, idx = x.cuda(), torch.from_numpy(ids).cuda()
    expected = xd[torch.from_numpy(want["row_to_route"]).cuda().long() // topk]
    side = torch.cuda.Stream()
    for _ in range(3):
        buffer = _buffer(num_bytes=4 << 20, rank=0, world_size=world)
        try:
            torch.cuda.synchronize()
            recv, _, _, _, event = buffer.dispatch(xd, topk_idx=idx, num_experts=experts, async_with_compute_stream=True)
            if wait == "never":
                kept = recv
            else:
                with torch.cuda.stream(side if wait == "other" else torch.cuda.current_stream()):
                    event.current_stream_wait()
                    torch.cuda._sleep(20_000_000)
                    kept = recv.clone()
            del recv, event
            with torch.cuda.stream(buffer.get_comm_stream()):
                noise = [torch.full((tokens * topk, hidden), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(3)]
            torch.cuda.synchronize()
            assert torch.equal(kept, expected)
            del noise, kept
        finally:
            torch.cuda.synchronize()
            buffer.destroy()


@pytest.mark.parametrize("fp8", [False, True])
def test_memory_of_an_outgrown_asynchronous_dispatch_is_not_handed_out_too_early(fp8):
    """A share several times the expected one, on the communication stream: the outputs it outgrew are let go inside the call,
    and the caller asks for memory of their size at once, on its own stream and without waiting for the event."""
    world, rank, experts, topk, tokens, hidden = 4, 1, 16, 4, 8192, 2048
    rng = np.random.default_rng(6)
    ids = np.stack([rank * 4 + rng.permutation(4)[:topk] for _ in range(tokens)]).astype(np.int64)
    x, w = _batch(tokens, hidden, topk, 6)
    want = olayout.layout(ids, experts, rank * 4, 4)
    rows = want["num_rows"]
    order = torch.from_numpy(want["row_to_route"]).cuda().long()
    xd, wd, idx = x.cuda(), w.cuda(), torch.from_numpy(ids).cuda()
    expected = (xd if not fp8 else oquant.cast_to_fp8_torch(x)[0].cuda().view(torch.uint8))[order // topk]
    for _ in range(4):
        # a new buffer each time: with the batch before as its guide the share would fit
        buffer = _buffer(num_bytes=4 << 20, rank=rank, world_size=world, use_fp8_dispatch=fp8)
        try:
            torch.cuda.synchronize()
            recv, _, recv_w, handle, event = buffer.dispatch(xd, topk_idx=idx, topk_weights=wd, num_experts=experts,
                                                             async_with_compute_stream=True)
            noise = [torch.full((n, hidden), 7.0, dtype=torch.bfloat16, device="cuda")
                     for n in (rows // 4, rows // 4 + rows // 16, rows // 3, rows // 8, rows // 8)]
            event.current_stream_wait()
            torch.cuda.synchronize()
            assert handle.num_expanded_tokens == rows == tokens * topk
            assert torch.equal(recv[0].view(torch.uint8) if fp8 else recv, expected)
            assert torch.equal(recv_w, wd.view(-1)[order])
            for block in noise:
                assert bool((block == 7.0).all())
            del recv, recv_w, handle, event, noise
        finally:
            torch.cuda.synchronize()
            buffer.destroy()


def test_outputs_made_after_the_wait_are_free_of_other_threads_work():
    """While an asynchronous dispatch waits for its row count, another thread uses the caller's stream: it fills memory of the size
    that the outputs turn out to need, late, and lets it go.  The outputs may well get that memory; the payload comes behind."""
    world, experts, topk, tokens, hidden = 4, 16, 4, 4096, 2048
    x, _ = _batch(tokens, hidden, topk, 10)
    ids = np.stack([np.random.default_rng(10).permutation(4)[:topk] for _ in range(tokens)]).astype(np.int64)
    want = olayout.layout(ids, experts, 0, 4)
    xd, idx = x.cuda(), torch.from_numpy(ids).cuda()
    expected = xd[torch.from_numpy(want["row_to_route"]).cuda().long() // topk]
    torch.empty((tokens * topk, hidden), dtype=torch.bfloat16, device="cuda")  # (so that the allocator has such a block)
    for _ in range(3):
        buffer = _buffer(num_bytes=4 << 20, rank=0, world_size=world)
        ready, queued = threading.Event(), []

        def other():
            ready.wait(30)
            time.sleep(0.005)
            block = torch.empty((tokens * topk, hidden), dtype=torch.bfloat16, device="cuda")
            torch.cuda._sleep(20_000_000)
            block.fill_(7.0)
            queued.append(time.perf_counter())

        thread = threading.Thread(target=other)
        try:
            torch.cuda.synchronize()
            thread.start()
            torch.cuda._sleep(200_000_000)  # about 90 ms: the layout, behind the caller's stream, waits for it
            ready.set()
            recv, _, _, handle, event = buffer.dispatch(xd, topk_idx=idx, num_experts=experts, async_with_compute_stream=True)
            returned = time.perf_counter()
            event.current_stream_wait()
            thread.join(timeout=60)
            torch.cuda.synchronize()
            assert handle.num_expanded_tokens == tokens * topk and queued and queued[0] < returned
            assert torch.equal(recv, expected)
            del recv, handle, event
        finally:
            thread.join(timeout=60)
            torch.cuda.synchronize()
            buffer.destroy()


def test_a_call_that_fails_behind_its_launch_leaves_its_buffer_closed():
    """The layout gives up waiting (forced by its own bound, every kernel ends normally): the asynchronous call raises with its
    payload queued on the communication stream, the caller's tensors go at once, and the buffer takes no further calls."""
    from deepep_amd import _lib

    tokens, hidden, topk, experts = 4096, 1024, 4, 16
    x, w = _batch(tokens, hidden, topk, 7)
    idx = torch.stack([torch.randperm(experts)[:topk] for _ in range(tokens)]).cuda()
    buffer = _buffer(num_bytes=4 << 20)
    try:
        workspace = buffer._runtime.workspace
        workspace.tune("layout_exchange_extra_rows", 1)
        workspace.tune("layout_exchange_ticks", 10_000)
        payload = x.cuda()
        with pytest.raises(_lib.NativeError, match="ran out of time"):
            buffer.dispatch(payload, topk_idx=idx, topk_weights=w.cuda(), num_experts=experts, async_with_compute_stream=True)
        del payload
        noise = [torch.full((tokens * topk, hidden), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
        buffer.get_comm_stream().synchronize()
        torch.cuda.synchronize()
        assert all(bool((block == 7.0).all()) for block in noise)
        with pytest.raises(RuntimeError, match="previous communication launch failed"):
            buffer.dispatch(x.cuda(), topk_idx=idx, num_experts=experts)
    finally:
        torch.cuda.synchronize()
        buffer.destroy()


def test_event_of_an_asynchronous_call_stands_in_for_torchs():
    x, _ = _batch(64, 256, 2, 3)
    idx = torch.stack([torch.randperm(8)[:2] for _ in range(64)]).cuda()
    buffer = _buffer(num_bytes=4 << 20)
    try:
        recv, _, _, handle, overlap = buffer.dispatch(x.cuda(), topk_idx=idx, num_experts=8, async_with_compute_stream=True)
        event = overlap.event.event
        torch.cuda.Stream().wait_event(event)
        event.wait()
        event.synchronize()
        assert event.query() and overlap.event._gpu_index == torch.cuda.current_device()
        assert overlap.event._marker.stream == buffer.get_comm_stream()
        out, _, second = buffer.combine(recv, handle, previous_event=overlap.event, async_with_compute_stream=True)
        with second(release_handle=True):
            pass
        assert second.event is None and second._lease is None
        assert torch.equal(out.float(), x.cuda().float() * 2)
    finally:
        buffer.destroy()


def test_event_of_an_asynchronous_call_is_torchs_own_and_marks_that_call_only():
    x, _ = _batch(64, 256, 2, 3)
    idx = torch.stack([torch.randperm(8)[:2] for _ in range(64)]).cuda()
    buffer = _buffer(num_bytes=4 << 20)
    try:
        comm = buffer.get_comm_stream()
        for sleep_first in (False, True):  # the value is still to come when the event is asked for, or is there already
            if sleep_first:
                with torch.cuda.stream(comm):
                    torch.cuda._sleep(2_000_000)
            recv, _, _, handle, overlap = buffer.dispatch(x.cuda(), topk_idx=idx, num_experts=8, async_with_compute_stream=True)
            event = overlap.event.event
            assert isinstance(event, torch.cuda.Event) and event is overlap.event.event and event.cuda_event != 0
            with torch.cuda.stream(comm):
                torch.cuda._sleep(200_000_000)  # about 0.1 s: what the stream is given later is not waited for
            event.synchronize()
            assert event.query() and not comm.query()
            torch.cuda.synchronize()
            # recorded again, it stands for what that stream has been given by then
            late = torch.zeros(4, device="cuda")
            torch.cuda.synchronize()
            with torch.cuda.stream(comm):
                torch.cuda._sleep(20_000_000)
                late.add_(1)
                event.record(comm)
            overlap.current_stream_wait()
            assert (late * 1).tolist() == [1.0] * 4
        with pytest.raises(Exception):
            event.elapsed_time(event)  # (made without timing, as before)
    finally:
        torch.cuda.synchronize()
        buffer.destroy()


@pytest.mark.parametrize("on_side_stream", [False, True])
def test_an_overlap_made_from_the_event_of_an_asynchronous_call_keeps_its_tensors(on_side_stream):
    """EventOverlap's public constructor with the event of a call: the given tensors are kept for the work and declared to
    whichever stream waits."""
    from deepep_amd.event import EventOverlap

    x, _ = _batch(64, 256, 2, 3)
    idx = torch.stack([torch.randperm(8)[:2] for _ in range(64)]).cuda()
    buffer = _buffer(num_bytes=4 << 20)
    try:
        xd = x.cuda()
        recv, _, _, handle, made = buffer.dispatch(xd, topk_idx=idx, num_experts=8, async_with_compute_stream=True)
        extra = torch.full((1 << 20,), 3.0, device="cuda")
        overlap = EventOverlap(made.event, extra_tensors=(extra,))
        calls = []
        overlap.register_hook_after_wait(lambda: calls.append(1) or "done")
        with torch.cuda.stream(torch.cuda.Stream() if on_side_stream else torch.cuda.current_stream()):
            assert overlap.current_stream_wait() == "done" and calls == [1]
            twice = recv.float() * 2
            total = extra.sum()
        del extra
        with overlap(release_handle=True):
            pass
        assert overlap.event is None and overlap._lease is None
        torch.cuda.synchronize()
        assert total.item() == 3.0 * (1 << 20)
        assert torch.equal(twice, xd.float()[handle.weight_return_meta.long() // 2] * 2)
    finally:
        torch.cuda.synchronize()
        buffer.destroy()


def test_asynchronous_calls_from_changing_streams_keep_their_order():
    """The caller's stream changes from call to call while the one before is still busy: every asynchronous call has to see
    its own caller's input, whichever stream raised the buffer's counter last."""
    tokens, hidden, topk, experts = 64, 256, 2, 8
    idx = torch.stack([torch.randperm(experts)[:topk] for _ in range(tokens)]).cuda()
    streams = [torch.cuda.Stream() for _ in range(3)]
    buffer = _buffer(num_bytes=4 << 20)
    try:
        _, _, _, handle, _ = buffer.dispatch(torch.zeros(tokens, hidden, dtype=torch.bfloat16, device="cuda"), topk_idx=idx, num_experts=experts)
        ones = torch.ones(tokens, hidden, dtype=torch.bfloat16, device="cuda")
        torch.cuda.synchronize()
        for order in ((0, 1, 2), (2, 1, 0), (0, 0, 1), (1, 2, 1)):
            results = []
            for at, which in enumerate(order):
                with torch.cuda.stream(streams[which]):
                    torch.cuda._sleep(3_000_000 if at == 0 else 1000)
                    x = ones * (at + 1 + which)
                    recv, _, _, _, event = buffer.dispatch(x, handle=handle, async_with_compute_stream=True)
                    out, _, done = buffer.combine(recv, handle, previous_event=event.event, async_with_compute_stream=True)
                    done.current_stream_wait()
                    results.append((out * 1, 2.0 * (at + 1 + which)))
            torch.cuda.synchronize()
            for out, want in results:
                assert torch.equal(out, torch.full_like(out, want)), order
    finally:
        torch.cuda.synchronize()
        buffer.destroy()


@pytest.mark.parametrize("first_in_the_graph", [False, True])
def test_asynchronous_cached_calls_in_a_hip_graph(first_in_the_graph):
    """Under capture streams are ordered by events: a cached dispatch and a combine on the communication stream, captured once
    and replayed on new payloads, with the program's own work between the replays.  With and without an asynchronous call of
    the buffer before the capture: counters are not taken under capture, where nothing may be allocated, but by the first call after."""
    tokens, hidden, topk, experts = 96, 512, 3, 8
    gen = torch.Generator().manual_seed(4)
    idx = torch.stack([torch.randperm(experts, generator=gen)[:topk] for _ in range(tokens)]).cuda()
    x = torch.zeros(tokens, hidden, dtype=torch.bfloat16, device="cuda")
    buffer = _buffer(num_bytes=4 << 20)
    try:
        _, _, _, handle, _ = buffer.dispatch(x, topk_idx=idx, num_experts=experts)
        if not first_in_the_graph:
            _, _, _, _, event = buffer.dispatch(x, handle=handle, async_with_compute_stream=True)
            event.current_stream_wait()
        torch.cuda.synchronize()
        side = torch.cuda.Stream()
        with torch.cuda.stream(side):
            buffer.combine(torch.zeros(handle.num_expanded_tokens, hidden, dtype=torch.bfloat16, device="cuda"), handle)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            recv, _, _, _, event = buffer.dispatch(x, handle=handle, async_with_compute_stream=True)
            event.current_stream_wait()
            out, _, event = buffer.combine(recv, handle, async_with_compute_stream=True)
            event.current_stream_wait()
        for _ in range(4):
            x.copy_(torch.randn(tokens, hidden, generator=gen).bfloat16())
            graph.replay()
            torch.cuda.synchronize()
            eager_rows, _, _, _, _ = buffer.dispatch(x, handle=handle)
            assert torch.equal(recv, eager_rows)
            assert torch.equal(out, buffer.combine(eager_rows, handle)[0])
            rows, _, _, _, event = buffer.dispatch(x, handle=handle, async_with_compute_stream=True)  # by the counters again
            event.current_stream_wait()
            assert torch.equal(rows, eager_rows)
    finally:
        torch.cuda.synchronize()
        buffer.destroy()


def test_stream_raise_stores_behind_earlier_work_and_refuses_bad_words():
    from deepep_amd import _lib

    lib = _lib.load()
    word = torch.zeros(2, dtype=torch.int64, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    word.fill_(3)
    assert lib.dpep_stream_raise(word.data_ptr(), 5_000_000_000, stream) == 0
    assert word.tolist() == [5_000_000_000, 3]
    for bad in (0, word.data_ptr() + 4):
        assert lib.dpep_stream_raise(bad, 1, stream) != 0


class _FreshDispatch(ctypes.Structure):
    _fields_ = [(name, ctypes.c_void_p) for name in (
        "topk_idx", "topk_idx_copy", "x", "scales", "topk_weights", "counts", "psum", "offsets", "route_to_row", "row_to_route", "num_rows",
        "send_counts", "out", "out_scales", "out_weights")] + [(name, ctypes.c_int32) for name in (
            "num_tokens", "num_topk", "num_experts", "expert_begin", "num_local", "row_bytes", "scale_cols", "quantize", "capacity_rows",
            "report_to_host")]


@pytest.mark.parametrize("report,short_by", [(2, 0), (2, 1), (2, 3000), (2, -2000), (2, "most unused"), (2, "just kept"), (1, 1), (1, 3000),
                                             (1, -5000)])
@pytest.mark.parametrize("quantize", [False, True])
@pytest.mark.parametrize("tokens,topk,experts,local", [(1000, 8, 32, 8), (4001, 1, 16, 4)])  # token-major and row-major payloads
def test_fresh_dispatch_into_outputs_that_are_too_small(tokens, topk, experts, local, quantize, report, short_by):
    """dpep_dispatch_fresh with capacities around the number of rows: all rows, the first ones, or (all or none: outputs too
    small or mostly unused) nothing."""
    from deepep_amd import _lib, ops

    hidden, begin = 256, local
    rng = np.random.default_rng(tokens)
    popularity = np.where((np.arange(experts) >= begin) & (np.arange(experts) < begin + local), 20.0, 1.0)
    ids = np.stack([rng.choice(experts, topk, replace=False, p=popularity / popularity.sum()) for _ in range(tokens)]).astype(np.int64)
    want = olayout.layout(ids, experts, begin, local)
    rows = want["num_rows"]
    if isinstance(short_by, str):
        short_by = -(rows // 2 + 1024 + (short_by == "most unused"))
    capacity = max(rows - short_by, 0)
    moved = min(capacity, rows) if report == 1 or capacity >= rows and capacity - rows <= rows // 2 + 1024 else 0
    x, w = _batch(tokens, hidden, topk, 9)
    device = dict(device="cuda")
    idx, xd, wd = torch.from_numpy(ids).cuda(), x.cuda(), w.cuda()
    meta = torch.zeros(3 * local + 2, dtype=torch.int32, **device)
    forward = torch.zeros(tokens * topk, dtype=torch.int32, **device)
    back = torch.zeros(tokens * topk, dtype=torch.int32, **device)
    size = max(rows, capacity)
    out = torch.full((size, hidden * (1 if quantize else 2)), 0x55, dtype=torch.uint8, **device)
    scales = torch.full((size, hidden // 128), 5.0, **device) if quantize else None
    weights = torch.full((size,), 5.0, **device)
    call = _FreshDispatch(
        idx.data_ptr(), None, xd.data_ptr(), None, wd.data_ptr(), meta.data_ptr(), meta[local:].data_ptr(), meta[2 * local :].data_ptr(),
        forward.data_ptr(), back.data_ptr(), meta[3 * local + 1 :].data_ptr(), None, out.data_ptr(),
        scales.data_ptr() if quantize else None, weights.data_ptr(), tokens, topk, experts, begin, local, hidden * 2, 0, int(quantize),
        capacity, report)
    workspace = ops.Workspace(1 << 20)
    try:
        stream = torch.cuda.current_stream().cuda_stream
        _lib.check(_lib.load().dpep_dispatch_fresh(workspace.handle, ctypes.byref(call), stream), "dispatch_fresh")
        assert ops.layout_wait(workspace) == (None, rows)
        torch.cuda.synchronize()
    finally:
        workspace.destroy()
    np.testing.assert_array_equal(forward.cpu().numpy().reshape(tokens, topk), want["route_to_row"])
    if quantize:
        codes, factors = oquant.cast_to_fp8_torch(x)
        np.testing.assert_array_equal(f32_bits(scales[:moved]), olayout.expand_rows(f32_bits(factors), want["row_to_route"], topk)[:moved])
        assert bool((scales[moved:] == 5.0).all())
        payload = fp8_bits(codes)
    else:
        payload = x.view(torch.uint8).numpy()
    np.testing.assert_array_equal(out[:moved].cpu().numpy(), olayout.expand_rows(payload, want["row_to_route"], topk)[:moved])
    np.testing.assert_array_equal(f32_bits(weights[:moved]), olayout.expand_weights(w.numpy(), want["row_to_route"]).view(np.uint32)[:moved])
    assert bool((out[moved:] == 0x55).all()) and bool((weights[moved:] == 5.0).all())


@pytest.mark.parametrize("world,tokens", [(8, 6000), (8, 240), (2, 3000)])
def test_storage_of_a_share_stays_close_to_its_rows(world, tokens):
    """Batches whose share jumps up and down: what a received tensor keeps alive follows its own number of rows."""
    experts, topk, hidden, local = world * 8, 4, 512, 8
    rng = np.random.default_rng(12)
    x, w = _batch(tokens, hidden, topk, 12)
    xd, wd = x.cuda(), w.cuda()
    buffer = _buffer(num_bytes=4 << 20, rank=0, world_size=world)
    try:
        for step, share in enumerate((1.0, 1.0, 0.02, 0.02, 10.0, 10.0, 0.0, 0.5, 1.0, 300.0, 300.0, 0.3)):
            popularity = np.where(np.arange(experts) < local, share + 1e-12, 1.0)
            ids = np.stack([rng.choice(experts, topk, replace=False, p=popularity / popularity.sum()) for _ in range(tokens)]).astype(np.int64)
            want = olayout.layout(ids, experts, 0, local)
            rows = want["num_rows"]
            recv, _, recv_w, handle, _ = buffer.dispatch(xd, topk_idx=torch.from_numpy(ids).cuda(), topk_weights=wd, num_experts=experts)
            kept = recv.untyped_storage().nbytes() / (hidden * 2)
            assert handle.num_expanded_tokens == rows == recv.shape[0] == recv_w.shape[0]
            assert kept <= (tokens * topk if world == 2 else rows * 1.5 + 1024 if tokens * topk > 2048 else 2048), (step, rows, kept)
            np.testing.assert_array_equal(bf16_bits(recv), olayout.expand_rows(bf16_bits(x), want["row_to_route"], topk))
            np.testing.assert_array_equal(f32_bits(recv_w), olayout.expand_weights(w.numpy(), want["row_to_route"]).view(np.uint32))
    finally:
        buffer.destroy()


def test_other_python_threads_run_while_a_dispatch_waits_for_its_row_count():
    """A wait as short as a busy stream's few ten microseconds is made without the GIL too."""
    x, _ = _batch(64, 256, 2, 3)
    idx = torch.stack([torch.randperm(8)[:2] for _ in range(64)]).cuda()
    xd = x.cuda()
    buffer = _buffer(num_bytes=4 << 20)
    turns, stop = [0], threading.Event()

    def other():
        while not stop.is_set():
            turns[0] += 1

    thread = threading.Thread(target=other)
    try:
        buffer.dispatch(xd, topk_idx=idx, num_experts=8)
        thread.start()
        let_in = 0
        for _ in range(20):
            torch.cuda.synchronize()
            torch.cuda._sleep(40_000)  # about 20 us
            before = turns[0]
            buffer.dispatch(xd, topk_idx=idx, num_experts=8)
            let_in += turns[0] > before
        assert let_in >= 15
    finally:
        stop.set()
        thread.join(timeout=60)
        buffer.destroy()


def test_outputs_that_a_share_outgrows_are_given_back_first():
    """A hot batch behind a cold one: the outputs made for the cold one's share are gone when those of the right size are made."""
    world, experts, topk, tokens, hidden = 4, 16, 4, 8192, 2048
    hot = torch.stack([torch.randperm(4)[:topk] for _ in range(tokens)]).cuda()
    x = torch.randn(tokens, hidden, device="cuda").bfloat16()
    buffer = _buffer(num_bytes=4 << 20, rank=0, world_size=world)
    try:
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        recv, _, _, handle, _ = buffer.dispatch(x, topk_idx=hot, num_experts=experts)
        peak = torch.cuda.max_memory_allocated() - before
        assert handle.num_expanded_tokens == tokens * topk
        payload = tokens * topk * hidden * 2
        assert payload <= recv.untyped_storage().nbytes() == payload and peak <= payload + (2 << 20)
    finally:
        buffer.destroy()
