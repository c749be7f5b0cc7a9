"""The mid-size fp8 expert kernels (tiles of up to 64 rows, three workgroups per CU): the same
bits as the kernels they stand in for, which other tests hold to the oracle."""
import dataclasses

import numpy as np
import pytest
import torch

from _util import say
from vllm_neuron_amd import ops, synthetic
from vllm_neuron_amd.config import MoEConfig

pytestmark = pytest.mark.gpu


def _experts(tpid, b2e, B, T, K, E, S, mt, xq, xs, w):
    tiles, num, mx = ops.build_tiles(tpid, b2e, B, T, K, E, S, mt)
    NB = tpid.numel()
    hq, hs = ops.expert_gate_up(xq, xs, w, tpid, NB, tiles, num, mx, mt)
    return hq, hs, ops.expert_down(hq, hs, w, T, NB, tiles, num, mx, mt)


# Expert counts that give every tile height around a 16-row fragment and a 64-row tile; mt 128
# runs the ring kernel. H and I: one group of four K blocks, several, and odd numbers of them.
# 64-row tiles always take these kernels, 32-row tiles from 512 items of a product (mid32: bit 0
# gate_up, bit 1 down).
@pytest.mark.parametrize("H,I,S,chan,mid32", [(512, 512, 0, False, 0), (1024, 1536, 1, False, 1),
                                              (1536, 512, 2, True, 0), (512, 8192, 1, False, 1),
                                              (4096, 512, 1, False, 2), (4096, 1536, 1, True, 3)])
@pytest.mark.parametrize("mt", [32, 64])
def test_row_tiles_equal_ring_kernel(cuda, mt, H, I, S, chan, mid32):
    counts = [1, 15, 16, 17, 0, 31, 32, 33, 48, 49, 63, 64, 65, 130]
    E, T = len(counts), sum(counts)
    say("mid row tiles", mt, H, I, S, chan, T)
    w = synthetic.make_weights(MoEConfig(H, I, E, 1, n_shared=S), 3, device=cuda)
    if chan:
        g = torch.Generator(device=cuda).manual_seed(9)
        c = lambda *s: torch.rand(*s, device=cuda, generator=g) + 0.5
        w = dataclasses.replace(w, w13_chan=c(E, 2 * I), w2_chan=c(E, H), shared_w13_chan=c(S, 2 * I),
                                shared_w2_chan=c(S, H))
    ids = torch.from_numpy(np.random.default_rng(1).permutation(np.repeat(np.arange(E), counts))
                           .astype(np.int32).reshape(T, 1)).to(cuda)
    m = ops.blockwise_mapping(ids=ids, n_experts=E, block_size=256)
    tpid, b2e = m["token_position_to_id"].clone(), m["block_to_expert"]
    tpid[(tpid >= 0).nonzero()[5]] = -1  # a hole inside a tile: its h row is not written
    tiles = ops.build_tiles(tpid, b2e, 256, T, 1, E, S, 32)[2]
    assert (tiles * (I // 128) >= 512) + 2 * (tiles * (H // 256) >= 512) == mid32
    xq, xs = ops.act_quant(synthetic.hidden_states(T, H, 3).to(cuda))
    got = _experts(tpid, b2e, 256, T, 1, E, S, mt, xq, xs, w)
    ref = _experts(tpid, b2e, 256, T, 1, E, S, 128, xq, xs, w)
    live = torch.cat([tpid >= 0, torch.ones(S * T, dtype=torch.bool, device=cuda)])
    for a, b in zip(got, ref):
        as_int = torch.int16 if a.dtype == torch.bfloat16 else torch.uint8
        assert torch.equal(a.view(as_int)[live], b.view(as_int)[live])
    assert float(got[2][live].float().abs().max()) > 0


# 16-row tiles of enough experts (items >= 1024): the mid-size kernels.
def test_sixteen_row_tiles_equal_ring_kernel(cuda):
    E, K, H, I, T = 128, 4, 2048, 1024, 96
    say("mid 16-row tiles")
    w = synthetic.make_weights(MoEConfig(H, I, E, K), 4, device=cuda)
    rng = np.random.default_rng(2)
    ids = torch.from_numpy(np.stack([rng.choice(E, K, replace=False) for _ in range(T)]).astype(np.int32)).to(cuda)
    m = ops.blockwise_mapping(ids=ids, n_experts=E, block_size=16)
    tpid, b2e = m["token_position_to_id"], m["block_to_expert"]
    xq, xs = ops.act_quant(synthetic.hidden_states(T, H, 4).to(cuda))
    assert ops.build_tiles(tpid, b2e, 16, T, K, E, 0, 16)[2] * min(I // 128, H // 256) >= 1024
    got = _experts(tpid, b2e, 16, T, K, E, 0, 16, xq, xs, w)
    ref = _experts(tpid, b2e, 16, T, K, E, 0, 128, xq, xs, w)
    live = tpid >= 0
    for a, b in zip(got, ref):
        as_int = torch.int16 if a.dtype == torch.bfloat16 else torch.uint8
        assert torch.equal(a.view(as_int)[live], b.view(as_int)[live])


# 33 to 76 rows per expert: the layer against the op-by-op path's block kernels. A zero weight
# scale repeats the previous block's ratio in both. Above 40 rows a router bias spreads the
# experts over every count of 16-row fragments and several tiles.
@pytest.mark.parametrize("T,S,zero", [(513, 1, False), (577, 0, True), (640, 1, True), (641, 1, False),
                                      (1000, 0, True), (1216, 2, False)])
def test_layer_block_tiles_equal_block_kernels(cuda, T, S, zero):
    E, K, H, I = 128, 8, 1024, 512
    cfg = MoEConfig(H, I, E, K, n_shared=S, scoring="sigmoid", grouped=True, renorm=True)
    say("mid block tiles", T, S, zero)
    w = synthetic.make_weights(cfg, 5, device=cuda)
    if zero:
        w.w13_scale[:, :, 0] = 0
        w.w13_scale[3, :, 2] = 0
        w.w2_scale[:, 1, 3] = 0
    x = synthetic.hidden_states(T, H, 5).to(cuda)
    tall = T * K > 40 * E
    if tall:
        g = torch.Generator(device=cuda).manual_seed(6)
        bias = torch.randn(E, device=cuda, generator=g) * (x.float() @ w.router_w.float().t()).std()
        w = dataclasses.replace(w, router_bias=bias)
    out, ids, wts, _ = ops.layer_forward(x, w, cfg, return_routing=True)
    if tall:
        c = torch.bincount(ids.flatten(), minlength=E).tolist()
        assert set(range(1, 9)) <= {-(-n // 16) for n in c} and max(c) > 128
    m = ops.blockwise_mapping(ids=ids, n_experts=E, block_size=256)
    tpid, b2e = m["token_position_to_id"], m["block_to_expert"]
    NB = tpid.numel()
    xq, xs = ops.act_quant(x)
    assert ops.use_block_kernels(T, K, E) and T * K <= 76 * E
    tiles, num, mx = ops.build_block_tiles(tpid, b2e, 256, T, K, E, S)
    hq, hs = ops.expert_gate_up_block(xq, xs, w, tpid, NB, tiles, num, mx)
    y = ops.expert_down_block(hq, hs, w, T, NB, tiles, num, mx)
    ref = ops.combine(y, m["inv_pos"], wts, T, H, NB, S)
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))


# The operators' block tile lists of up to 128 rows against those of up to 256 on the block
# kernels, whose rows' results do not depend on the tile. The last two cases (H not a multiple of 512,
# channel scales) run the block kernels on both.
@pytest.mark.parametrize("H,I,S,chan", [(512, 512, 0, False), (1024, 1536, 1, False), (2560, 512, 2, False),
                                        (768, 512, 0, False), (512, 512, 1, True)])
def test_tall_tile_lists_equal_block_lists(cuda, H, I, S, chan):
    counts = [1, 16, 17, 0, 33, 64, 65, 81, 97, 112, 113, 127, 128, 129, 256, 257, 300]
    E, T = len(counts), sum(counts)
    say("tall tile lists", H, I, S, chan, T)
    w = synthetic.make_weights(MoEConfig(H, I, E, 1, n_shared=S), 7, device=cuda)
    if chan:
        g = torch.Generator(device=cuda).manual_seed(9)
        c = lambda *s: torch.rand(*s, device=cuda, generator=g) + 0.5
        w = dataclasses.replace(w, w13_chan=c(E, 2 * I), w2_chan=c(E, H), shared_w13_chan=c(S, 2 * I),
                                shared_w2_chan=c(S, H))
    ids = torch.from_numpy(np.random.default_rng(1).permutation(np.repeat(np.arange(E), counts))
                           .astype(np.int32).reshape(T, 1)).to(cuda)
    m = ops.blockwise_mapping(ids=ids, n_experts=E, block_size=64)
    tpid, b2e = m["token_position_to_id"].clone(), m["block_to_expert"]
    tpid[(tpid >= 0).nonzero()[5]] = -1  # a hole inside a tile: its h row is not written
    xq, xs = ops.act_quant(synthetic.hidden_states(T, H, 7).to(cuda))
    live = torch.cat([tpid >= 0, torch.ones(S * T, dtype=torch.bool, device=cuda)])
    got = []
    for rows in (128, 256):
        tiles, num, mx = ops.build_block_tiles(tpid, b2e, 64, T, 1, E, S, rows)
        hq, hs = ops.expert_gate_up_block(xq, xs, w, tpid, tpid.numel(), tiles, num, mx, rows)
        y = ops.expert_down_block(hq, hs, w, T, tpid.numel(), tiles, num, mx, rows)
        n = int(num[0])
        got.append((hq[live].view(torch.uint8), hs[live], y[live].view(torch.int16)))
        assert n <= mx and int(tiles[: 4 * n].view(n, 4)[:, 2].max()) <= rows
    for a, b in zip(*got):
        assert torch.equal(a, b)
    assert float(y[live].float().abs().max()) > 0
