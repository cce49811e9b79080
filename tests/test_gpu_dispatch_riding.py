"""A fresh dispatch whose payload rides in the layout's grid, at the sizes where that can go wrong (workgroups shared by one to four
rows' threads, rows wider and narrower than a workgroup, the longest chunks, top-k of a whole map, outputs that are too small), against the
two launches that any other store policy and a captured stream take: every output, bit for bit, and the rows against the oracle."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import layout as olayout
from tests.test_gpu_host_path import _FreshDispatch

pytestmark = pytest.mark.gpu


def _inputs(rng, tokens, topk, experts, row_bytes, scale_cols, quantize, masked):
    ids = np.argpartition(rng.random((tokens, experts)), topk - 1, axis=1)[:, :topk].astype(np.int64)
    ids[rng.random(ids.shape) < masked] = -1
    if quantize:  # (BF16 of moderate size)
        x = torch.from_numpy(rng.normal(size=(tokens, row_bytes // 2)).astype(np.float32)).bfloat16().cuda().view(torch.uint8)
    else:
        x = torch.from_numpy(rng.integers(0, 256, (tokens, row_bytes), dtype=np.uint8)).cuda()
    scales = torch.from_numpy(rng.random((tokens, scale_cols)).astype(np.float32)).cuda() if scale_cols else None
    return ids, x, scales, torch.from_numpy(rng.random((tokens, topk)).astype(np.float32)).cuda()


class _Call:
    """Outputs of their own and the call that fills them."""

    def __init__(self, idx, x, scales, weights, experts, begin, local, quantize, capacity, report):
        tokens, topk = idx.shape
        row_bytes, width = x.shape[1], x.shape[1] // 2
        scale_cols = width // 128 if quantize else 0 if scales is None else scales.shape[1]
        self.meta = torch.zeros(3 * local + 2, dtype=torch.int32, device="cuda")
        self.forward, self.back = (torch.full((tokens * topk,), -7, dtype=torch.int32, device="cuda") for _ in range(2))
        self.copy = torch.zeros_like(idx)
        self.out = torch.full((capacity, width if quantize else row_bytes), 0x55, dtype=torch.uint8, device="cuda")
        self.scales = torch.full((capacity, scale_cols), 5.0, device="cuda") if scale_cols else None
        self.weights = torch.full((capacity,), 5.0, device="cuda")
        self.keep = (idx, x, scales, weights)
        at = lambda tensor, by=0: None if tensor is None else tensor.data_ptr() + by
        self.call = _FreshDispatch(
            at(idx), at(self.copy), at(x), at(scales), at(weights), at(self.meta), at(self.meta, 4 * local), at(self.meta, 8 * local), at(self.forward),
            at(self.back), at(self.meta, 4 * (3 * local + 1)), None, at(self.out), at(self.scales), at(self.weights), tokens, topk, experts, begin,
            local, row_bytes, 0 if quantize or scales is None else scale_cols, int(quantize), capacity, report)

    def launch(self, workspace):
        from deepep_amd import _lib

        _lib.check(_lib.load().dpep_dispatch_fresh(workspace.handle, ctypes.byref(self.call), torch.cuda.current_stream().cuda_stream), "dispatch_fresh")

    def same_as(self, other, rows):
        for mine, theirs in ((self.meta, other.meta), (self.forward, other.forward), (self.back[:rows], other.back[:rows]), (self.copy, other.copy),
                             (self.out, other.out), (self.scales, other.scales), (self.weights, other.weights)):
            if mine is not None:
                assert torch.equal(mine, theirs)


# (report 1: the host is told and the first rows are kept; 2: all or none; 0: nobody is told)
@pytest.mark.parametrize("tokens,topk,experts,begin,local,row_bytes,scale_cols,quantize,report,spare", [
    (1100, 8, 32, 0, 32, 4096, 0, False, 1, 0),       # four column parts: four of them to a workgroup
    (4300, 2, 8, 0, 8, 4096, 3, False, 1, 0),         # two parts of 128 threads; scales
    (8200, 2, 16, 0, 16, 2560, 0, False, 1, 0),       # 160 vectors: 192 threads, one to a workgroup
    (700, 32, 64, 0, 64, 1536, 0, False, 1, 100),     # top-32, more room than rows
    (260, 16, 64, 0, 64, 9216, 0, False, 1, -300),    # the last rows have no room
    (420, 10, 40, 0, 40, 12128, 0, False, 1, 0),      # 758 vectors, not whole lines: parts that are not either
    (2100, 5, 24, 0, 24, 9232, 0, False, 1, 0),       # 577 in one part: two rounds from registers and one behind them
    (2100, 5, 24, 0, 24, 16368, 0, False, 1, 0),      # 1023: all that LDS is lent, and (the next) one more than that
    (2100, 5, 24, 0, 24, 16400, 0, False, 1, 0),
    (2040, 8, 256, 0, 256, 2176, 0, False, 1, 0),     # as many experts and routes per wave as ride
    (3900, 8, 256, 0, 256, 1088, 0, False, 1, 0),     # and more
    (1700, 12, 96, 48, 48, 4096, 5, False, 2, 0),     # half of the experts: all of the rows,
    (1700, 12, 96, 48, 48, 4096, 5, False, 2, -1),    # or none
    (10000, 3, 12, 0, 12, 2304, 0, True, 1, 0),       # quantised: 72 units, 128 threads
    (640, 8, 128, 0, 128, 14336, 0, True, 1, 0),      # 448 units in four parts
    (130, 32, 32, 0, 32, 40960, 0, True, 1, -64),     # 1280 units: parts of several rounds
    (3000, 20, 40, 0, 20, 2560, 0, True, 2, 0),
    (6000, 4, 256, 12, 4, 7168, 56, False, 0, 1000),  # row-major
    (6000, 4, 256, 12, 4, 7168, 0, False, 0, -100),
    (6000, 4, 256, 252, 4, 14336, 0, True, 0, 1000),
    (4000, 4, 1024, 800, 200, 464, 0, False, 0, 0),
    (32768, 2, 256, 0, 1, 256, 0, True, 0, 0),        # one expert
])
def test_riding_payload_equals_one_of_its_own_launch(tokens, topk, experts, begin, local, row_bytes, scale_cols, quantize, report, spare):
    from deepep_amd import _lib, ops

    rng = np.random.default_rng(tokens + topk)
    workspace = ops.Workspace(4 << 20)
    try:
        for turn in range(2):  # (the second finds the first one's words)
            ids, x, scales, weights = _inputs(rng, tokens, topk, experts, row_bytes, scale_cols, quantize, 0.1)
            want = olayout.layout(ids, experts, begin, local)
            # (the even share decides how the work is split, all or none: the capacity)
            capacity = want["num_rows"] + (want["num_rows"] // 8 + 256 if report == 2 and spare == 0 else spare)
            idx = torch.from_numpy(ids).cuda()
            args = (idx, x, scales, weights, experts, begin, local, quantize, capacity, report)
            riding, plain = _Call(*args), _Call(*args)
            riding.launch(workspace)
            if report:
                assert ops.layout_wait(workspace) == (None, want["num_rows"])
            before = ops.dispatch_store_policy("through")
            try:
                plain.launch(workspace)
                torch.cuda.synchronize()
            finally:
                ops.dispatch_store_policy(before)
            riding.same_as(plain, want["num_rows"])
            np.testing.assert_array_equal(riding.forward.cpu().numpy().reshape(tokens, topk), want["route_to_row"])
            if not quantize and report == 1 and spare >= 0:  # (a launch of its own by the default policy, into rows that begin 16 bytes behind a line)
                moved = torch.full((want["num_rows"] * row_bytes + 32,), 0x55, dtype=torch.uint8, device="cuda")
                _lib.check(_lib.load().dpep_dispatch_copy(
                    x.data_ptr(), None, None, riding.forward.data_ptr(), riding.back.data_ptr(), tokens, topk, want["num_rows"], row_bytes, 0,
                    moved.data_ptr() + 16, None, None, torch.cuda.current_stream().cuda_stream), "dispatch_copy")
                torch.cuda.synchronize()
                assert torch.equal(moved[16:-16].view(-1, row_bytes), riding.out[: want["num_rows"]])
                assert bool((moved[:16] == 0x55).all()) and bool((moved[-16:] == 0x55).all())
            if report == 2 and spare < 0:
                assert bool((riding.out == 0x55).all())
    finally:
        torch.cuda.synchronize()
        workspace.destroy()


# The payload may look for the layout's words `looks` times; with none it never sees one, as where the layout cannot start for whatever else
# runs, and everything that it moves follows from the ids alone.  (Ids drawn with repetition: a route's row counts the token's own earlier ones.)
@pytest.mark.parametrize("looks", [0, 1])
@pytest.mark.parametrize("tokens,topk,experts,begin,local,row_bytes,scale_cols,quantize,report,spare", [
    (1100, 8, 32, 0, 32, 4096, 0, False, 1, 0),       # four tokens' threads to a workgroup, the last workgroup not full
    (1101, 8, 32, 0, 32, 4096, 3, False, 1, -300),
    (420, 10, 40, 0, 40, 12128, 0, False, 1, 0),      # through LDS
    (2040, 8, 256, 0, 256, 2176, 0, False, 1, 0),     # as many experts as ride
    (700, 32, 64, 0, 64, 1536, 0, False, 1, 100),
    (1700, 12, 96, 48, 48, 4096, 5, False, 2, 0),     # all of the rows, or none
    (1700, 12, 96, 48, 48, 4096, 5, False, 2, -1),
    (640, 8, 128, 0, 128, 14336, 0, True, 1, 0),
    (3000, 20, 40, 0, 20, 2560, 0, True, 2, 0),
    (6000, 4, 256, 12, 4, 7168, 56, False, 0, 1000),  # row-major: fewer rows than the grid has
    (6000, 4, 256, 12, 4, 7168, 0, False, 0, -100),
    (6000, 4, 256, 252, 4, 14336, 0, True, 0, 1000),
    (1029, 4, 1024, 800, 200, 464, 0, False, 0, 0),   # a last step of 20 routes
    (32768, 2, 256, 0, 1, 256, 0, True, 0, 0),
])
def test_payload_that_gives_up_its_wait_works_its_rows_out(tokens, topk, experts, begin, local, row_bytes, scale_cols, quantize, report, spare, looks):
    from deepep_amd import ops

    rng = np.random.default_rng(tokens + topk + looks)
    workspace = ops.Workspace(4 << 20)
    try:
        workspace.tune("layout_payload_looks", looks)
        ids, x, scales, weights = _inputs(rng, tokens, topk, experts, row_bytes, scale_cols, quantize, 0.0)
        ids = np.where(rng.random(ids.shape) < 0.1, -1, rng.integers(0, experts, ids.shape))
        want = olayout.layout(ids, experts, begin, local)
        capacity = want["num_rows"] + (want["num_rows"] // 8 + 256 if report == 2 and spare == 0 else spare)
        idx = torch.from_numpy(ids).cuda()
        args = (idx, x, scales, weights, experts, begin, local, quantize, capacity, report)
        riding, plain = _Call(*args), _Call(*args)
        riding.launch(workspace)
        torch.cuda.synchronize()
        before = ops.dispatch_store_policy("through")
        try:
            plain.launch(workspace)
            torch.cuda.synchronize()
        finally:
            ops.dispatch_store_policy(before)
        riding.same_as(plain, want["num_rows"])
        np.testing.assert_array_equal(riding.forward.cpu().numpy().reshape(tokens, topk), want["route_to_row"])
    finally:
        torch.cuda.synchronize()
        workspace.destroy()


@pytest.mark.parametrize("looks", [64, 1])
def test_two_riding_grids_at_once(looks):
    """Two workspaces on two streams, each grid with several times the workgroups that the GPU holds, queued with nothing between them."""
    from deepep_amd import ops

    rng = np.random.default_rng(9)
    tokens, topk, experts = 4096, 8, 64
    workspaces = [ops.Workspace(4 << 20) for _ in range(2)]
    streams = [torch.cuda.Stream() for _ in range(2)]
    try:
        for workspace in workspaces:
            workspace.tune("layout_payload_looks", looks)
        batches = []
        for _ in range(2):
            ids, x, _, weights = _inputs(rng, tokens, topk, experts, 2048, 0, False, 0.1)
            want = olayout.layout(ids, experts, 0, experts)
            args = (torch.from_numpy(ids).cuda(), x, None, weights, experts, 0, experts, False, want["num_rows"], 0)
            batches.append((want["num_rows"], [_Call(*args) for _ in range(4)], _Call(*args)))
        torch.cuda.synchronize()
        for turn in range(4):
            for workspace, stream, (_, calls, _) in zip(workspaces, streams, batches):
                with torch.cuda.stream(stream):
                    calls[turn].launch(workspace)
        torch.cuda.synchronize()
        before = ops.dispatch_store_policy("through")
        try:
            for workspace, (_, _, plain) in zip(workspaces, batches):
                plain.launch(workspace)
            torch.cuda.synchronize()
        finally:
            ops.dispatch_store_policy(before)
        for rows, calls, plain in batches:
            for call in calls:
                call.same_as(plain, rows)
    finally:
        torch.cuda.synchronize()
        for workspace in workspaces:
            workspace.destroy()


def test_captured_dispatch_takes_two_launches():
    """Replays with new ids, ordinary calls between them: a payload that waited for words would find those of the replay before."""
    from deepep_amd import ops

    rng = np.random.default_rng(4)
    tokens, topk, experts, local = 6000, 4, 256, 4
    workspace = ops.Workspace(4 << 20)
    try:
        ids, x, _, weights = _inputs(rng, tokens, topk, experts, 2048, 0, False, 0.0)
        idx = torch.from_numpy(ids).cuda()
        args = (idx, x, None, weights, experts, 0, local, False, 2000, 0)
        captured, eager = _Call(*args), _Call(*args)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            captured.launch(workspace)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            captured.launch(workspace)
        for turn in range(4):
            fresh = _inputs(rng, tokens, topk, experts, 2048, 0, False, 0.05 * turn)[0]
            idx.copy_(torch.from_numpy(fresh))
            want = olayout.layout(fresh, experts, 0, local)
            captured.out.fill_(0x55), captured.weights.fill_(5.0), eager.out.fill_(0x55), eager.weights.fill_(5.0)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            eager.launch(workspace)
            torch.cuda.synchronize()
            captured.same_as(eager, want["num_rows"])
            np.testing.assert_array_equal(captured.forward.cpu().numpy().reshape(tokens, topk), want["route_to_row"])
    finally:
        torch.cuda.synchronize()
        workspace.destroy()
