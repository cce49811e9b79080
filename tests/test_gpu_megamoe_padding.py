"""The grouped GEMMs that leave out padding.  The 128-row one with two workgroups to a CU, at the sizes where it can go wrong: row counts on both sides of its 32-row
tiles, k that ends inside a span of four k tiles, inside a k tile and behind one MFMA step, column tiles and waves of nothing but
padding, more tiles than workgroups.  A k sum is taken in the same order as in the few-rows kernel, so the two give the same bits; both
against the fp32 oracle within the path's 2e-2."""

import numpy as np
import pytest
import torch

from oracle import megamoe as mm

pytestmark = pytest.mark.gpu

EDGES = (1, 31, 32, 33, 0, 64, 65, 96, 97, 127, 128, 129, 160, 256, 257)


def _forward(ops, x, l1, l2, shared, idx, weights, hidden, inter, local, tile_rows, few_rows_waves=4, experts=None, fill=0, paired=0, kernels=None):
    dev = "cuda"
    num_shared = 0 if shared is None else shared[0][0].shape[0]

    def prepared(l, n, gate_up):
        return ops.megamoe_prepare_weights(torch.from_numpy(l[0]).to(dev), torch.from_numpy(l[1]).reshape(l[0].shape[0], n, -1).to(dev), gate_up)

    w1, s1 = prepared(l1, 2 * inter, True)
    w2, s2 = prepared(l2, hidden, False)
    shared_weights = (*prepared(shared[0], 2 * inter, True), *prepared(shared[1], hidden, False)) if num_shared else None
    ws = ops.Workspace(ops.megamoe_workspace_bytes(len(idx), idx.shape[1], hidden, inter, local, num_shared))
    ws.tune("gemm_tile_rows", tile_rows)
    ws.tune("gemm_few_rows_waves", few_rows_waves)
    ws.tune("gemm_paired", paired)
    ws.tune("gemm_zero_fill", fill)
    if paired:
        kernels = (("paired", "paired_streamed")[paired - 1],) * 2
    if kernels:
        assert ops.megamoe_gemm_kernels(len(idx), hidden, inter, idx.shape[1], experts or local, local, num_shared, ws=ws) == kernels
    y = torch.full((len(idx), hidden), float("nan"), dtype=torch.bfloat16, device=dev)
    counts = torch.empty((local,), dtype=torch.int32, device=dev)
    ops.megamoe_forward(ws, torch.from_numpy(x[0]).to(dev).view(torch.float8_e4m3fn), torch.from_numpy(x[1]).to(dev), torch.from_numpy(idx).to(dev),
                        torch.from_numpy(weights).to(dev), w1, s1, w2, s2, experts or local, 0, local, y, counts, shared=shared_weights, intermediate=inter)
    torch.cuda.synchronize()
    ws.destroy()
    return y, counts.cpu().numpy()


@pytest.mark.parametrize("hidden,inter,rows,num_shared", [
    (64, 128, EDGES, 0),                # the smallest sizes: one k step in the first GEMM, one k tile in the second
    (576, 384, EDGES, 0),               # k ends behind one step of a k tile; the first GEMM's fourth column tile is all padding
    (1152, 1152, EDGES, 1),             # nine k tiles of ten: the last span holds one, its scale bytes sit two words up; a shared expert
    (320, 640, EDGES[:8], 0),           # ten k tiles of 64 in the first GEMM, a last column tile with one live wave in the second
    (2624, 1280, (40,) * 70, 0),        # 700 and 770 tiles for 512 workgroups
    (512, 512, (2, 0, 700, 5), 2),      # experts of many and of few row tiles, every tile of exactly four items
])
def test_paired_kernel_at_its_edges(hidden, inter, rows, num_shared):
    from deepep_amd import ops

    rng = np.random.default_rng(hidden * 7 + inter)
    local = len(rows)
    idx = rng.permutation(np.repeat(np.arange(local, dtype=np.int32), rows))[:, None].copy()
    x = mm.mx_quantize(rng.normal(size=(len(idx), hidden)).astype(np.float32))
    weights = rng.random((len(idx), 1)).astype(np.float32)

    def quantised(experts, n, k):  # (a few distinct matrices: quantising one takes the oracle a while)
        few = mm.quantize_weight_mxfp4((rng.normal(size=(min(experts, 4), n, k)) * 0.02).astype(np.float32))
        return tuple(np.ascontiguousarray(part[np.arange(experts) % len(part)]) for part in few)

    l1, l2 = quantised(local, 2 * inter, hidden), quantised(local, hidden, inter)
    shared = (quantised(num_shared, 2 * inter, hidden), quantised(num_shared, hidden, inter)) if num_shared else None
    want, _ = _forward(ops, x, l1, l2, shared, idx, weights, hidden, inter, local, 32)
    for paired in (1, 2):  # weights cached, and past the caches
        got, counts = _forward(ops, x, l1, l2, shared, idx, weights, hidden, inter, local, 128, paired=paired)
        np.testing.assert_array_equal(counts, np.bincount(idx.ravel(), minlength=local))
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), paired
    if len(idx) * hidden * inter < 2e9 and not num_shared:
        oracle = mm.round_bf16(mm.local_reference(mm.mx_dequantize(*x), idx, weights, mm.unpack_weight(*l1), mm.unpack_weight(*l2), 0))
        assert mm.relative_frobenius(got.float().cpu().numpy(), oracle) <= 2e-2


@pytest.mark.parametrize("hidden,inter,rows,one_wave", [  # one_wave: the kernels that one-wave workgroups run
    (64, 128, (3, 1), ("few_rows", "few_rows")),           # one k tile in both GEMMs
    (960, 640, (5, 0, 2), ("one_wave", "one_wave")),       # eight k tiles, the last half padding; five
    (1664, 1152, (33, 1, 32), ("one_wave", "one_wave")),   # 13 and nine: four and three spans of four
    (2368, 3200, (5, 0, 33), ("few_rows", "one_wave")),    # 19 and 25: five and seven spans
    (2624, 2176, (1,) * 66, ("few_rows", "few_rows")),     # more experts than a wave has lanes
])
def test_few_rows_kernels_at_their_edges(hidden, inter, rows, one_wave):
    """k tiles of every number behind the last whole span, and a span loop of none, one and several rounds: one-wave workgroups (without
    LDS where the launch is small) and four-wave ones against the 64-row kernel, bit for bit."""
    from deepep_amd import ops

    rng = np.random.default_rng(hidden)
    local = len(rows)
    idx = rng.permutation(np.repeat(np.arange(local, dtype=np.int32), rows))[:, None].copy()
    x = mm.mx_quantize(rng.normal(size=(len(idx), hidden)).astype(np.float32))
    weights = rng.random((len(idx), 1)).astype(np.float32)

    def random_weights(n, k):  # (codes and scale bytes of any matrix will do: the kernels are held against each other)
        return rng.integers(0, 256, (local, n, k // 2), dtype=np.uint8), rng.integers(118, 122, (local, n, k // 32), dtype=np.uint8)

    l1, l2 = random_weights(2 * inter, hidden), random_weights(hidden, inter)
    want, _ = _forward(ops, x, l1, l2, None, idx, weights, hidden, inter, local, 64)
    for waves in (1, 4):
        got, counts = _forward(ops, x, l1, l2, None, idx, weights, hidden, inter, local, 32, waves,
                               kernels=one_wave if waves == 1 else ("few_rows",) * 2)
        np.testing.assert_array_equal(counts, rows)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), waves


@pytest.mark.parametrize("tokens,hidden,topk,experts", [
    (70, 64, 4, 4),       # hardly more tokens than fillers; rows of 8 chunks, less than a lane each
    (1000, 576, 2, 16),   # 72 chunks: a lane has one or two
    (330, 1664, 4, 16),   # several tiles to a workgroup's XCD
])
def test_one_wave_launches_fill(tokens, hidden, topk, experts):
    """Two of the experts are here, with more than 64 rows each: the launch has fillers, and the rows of the other tokens are zero whoever wrote them."""
    from deepep_amd import ops

    rng = np.random.default_rng(tokens)
    inter, local = 256, 2
    idx = np.argsort(rng.random((tokens, experts)), axis=1)[:, :topk].astype(np.int32)
    if topk == experts:
        idx[::3] = np.where(idx[::3] < local, -1, idx[::3])
    x = mm.mx_quantize(rng.normal(size=(tokens, hidden)).astype(np.float32))
    weights = rng.random((tokens, topk)).astype(np.float32)

    def random_weights(n, k):
        return rng.integers(0, 256, (local, n, k // 2), dtype=np.uint8), rng.integers(118, 122, (local, n, k // 32), dtype=np.uint8)

    l1, l2 = random_weights(2 * inter, hidden), random_weights(hidden, inter)
    want, _ = _forward(ops, x, l1, l2, None, idx, weights, hidden, inter, local, 32, 1, experts)
    got, _ = _forward(ops, x, l1, l2, None, idx, weights, hidden, inter, local, 32, 1, experts, fill=1)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    unserved = ~((idx >= 0) & (idx < local)).any(1)
    assert unserved.any() and not got.cpu()[torch.from_numpy(unserved)].any()


@pytest.mark.parametrize("tokens,hidden,topk,experts,local", [
    (1, 64, 1, 8, 1),         # one row of sixteen pieces
    (37, 192, 16, 64, 1),     # four rows to a wave: as many ids as it has lanes
    (38, 192, 17, 64, 1),     # and more, which are not looked at
    (333, 1088, 3, 16, 2),    # 80 pieces a row: waves with one row and with two; the last workgroup is not full
    (1500, 576, 4, 64, 8),    # 48 pieces; a layout of several workgroups
    (2500, 320, 4, 64, 3),    # two waves with the same rows; layout and preparation are neighbours in one grid
])
def test_rows_of_other_ranks_are_not_prepared(tokens, hidden, topk, experts, local):
    """Padded rows, most tokens without a local expert: served rows against the oracle, the others zero."""
    from deepep_amd import ops

    rng = np.random.default_rng(tokens)
    inter = 128
    idx = np.argsort(rng.random((tokens, experts)), axis=1)[:, :topk].astype(np.int32)
    idx[-1] = np.arange(topk)  # the last row is served
    x = mm.mx_quantize(rng.normal(size=(tokens, hidden)).astype(np.float32))
    weights = rng.random((tokens, topk)).astype(np.float32)
    l1, l2 = (mm.quantize_weight_mxfp4((rng.normal(size=(local, n, k)) * 0.02).astype(np.float32)) for n, k in ((2 * inter, hidden), (hidden, inter)))
    got, _ = _forward(ops, x, l1, l2, None, idx, weights, hidden, inter, local, 0, experts=experts)
    oracle = mm.round_bf16(mm.local_reference(mm.mx_dequantize(*x), idx, weights, mm.unpack_weight(*l1), mm.unpack_weight(*l2), 0))
    got, served = got.float().cpu().numpy(), (idx < local).any(1)
    assert not got[~served].any()
    for row in np.flatnonzero(served):
        assert mm.relative_frobenius(got[row], oracle[row]) <= 2e-2, row
