"""The MXFP4 block kernels: of the layer's block tiles (above 32 routed rows per expert, enough
items), and of 32- and 64-row tiles of at least 512 work items.

Same scaled MFMAs in the same K order and the same epilogue arithmetic as the ring kernels,
so results are held bit for bit to those on 16-row tiles, which always run them (and which
test_gpu_mx.py checks against the oracle)."""
import dataclasses

import pytest
import torch

from _util import say
from test_gpu_mx import make_mx_weights
from vllm_neuron_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _skew(w, counts_bias):
    return dataclasses.replace(w, router_bias=torch.tensor(counts_bias, device=w.w13.device))


def _ring_experts(x, ids, wts, w, act, gl, ul, B=256):
    """ops.mx_experts on 16-row tiles."""
    T, K = ids.shape
    E, H = w.n_experts, w.hidden
    m = ops.blockwise_mapping(ids=ids.contiguous(), n_experts=E, top_k=K, block_size=B)
    tpid, b2e = m["token_position_to_id"], m["block_to_expert"]
    NB = tpid.numel()
    xq, xs = ops.act_quant_mx(x)
    tiles, num, mx = ops.build_tiles(tpid, b2e, B, T, K, E, 0, 16)
    hq, hs = ops.expert_gate_up_mx(xq, xs, w, tpid, NB, tiles, num, mx, 16, NB, act, gl, ul)
    y = ops.expert_down_mx(hq, hs, w, T, NB, tiles, num, mx, 16)
    return ops.combine(y, m["inv_pos"], wts.contiguous(), T, H, NB, 0)


# T * K / E > 32 in all of them. H = I = 512: one scale group, two steps; 1536 x 1024: odd
# numbers of groups; 768: not a multiple of 512, which stays on the row-tile kernels. 1025
# tokens run block tiles, the others have too few items for them.
@pytest.mark.parametrize("T,E,K,H,I,act,bias,skew", [
    (67, 2, 1, 512, 512, "swish", True, [0.0, -60.0]),         # one expert holds all 67 rows, one none
    (129, 4, 2, 512, 512, "silu", False, [30.0, 0.0, 0.0, -30.0]),  # a 129-row expert: two 65-row tiles
    (128, 3, 1, 1536, 1024, "swish", True, [0.0, 0.0, 0.0]),
    (97, 1, 1, 1024, 512, "swish", True, [0.0]),               # a 97-row tile (four 32-row groups)
    (257, 8, 2, 512, 1536, "swish", True, [3.0, 2.0, 1.0, 0.0, 0.0, -1.0, -2.0, -40.0]),
    (1025, 16, 4, 1024, 1024, "swish", True, [0.0] * 16),
    (300, 8, 2, 768, 512, "swish", True, [0.0] * 8),
])
def test_layer_equals_ring_kernels(cuda, T, E, K, H, I, act, bias, skew):
    say("mx block layer", T, E, K, H, I, act)
    w = _skew(make_mx_weights(E, H, I, 11, cuda, bias=bias), skew)
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(cuda)
    gl, ul = ((None, 7.0), (-6.0, 8.0)) if act == "swish" else ((None, None), (None, None))
    assert T * K > 32 * E
    out, ids, wts, _ = ops.layer_forward_mx(x, w, K, act, gl, ul, return_routing=True)
    ref = _ring_experts(x, ids, wts, w, act, gl, ul)
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))
    assert bool(torch.isfinite(out.float()).all()) and float(out.float().abs().max()) > 0


# Enough items for block tiles: experts of every count of 16-row fragments, of two and three tiles,
# and of none (each token names its expert in the first E columns).
@pytest.mark.parametrize("H,I,act,bias", [(512, 1536, "swish", True), (1024, 1024, "silu", False),
                                          (1536, 2048, "swish", True)])
def test_layer_block_tiles_of_every_height(cuda, H, I, act, bias):
    counts = [1, 15, 16, 17, 32, 33, 48, 49, 64, 65, 80, 81, 96, 97, 112, 113, 127, 128, 0, 129, 256, 257]
    E, T = len(counts), sum(counts)
    say("mx block tiles", H, I, act, T)
    assert _lib.load().moe_layer_mx_tile_rows(T, H, I, E, 1, 256) == 128
    w = make_mx_weights(E, H, I, 19, cuda, bias=bias)
    w = dataclasses.replace(w, router_w=torch.eye(E, H, dtype=torch.bfloat16, device=cuda), router_bias=None)
    g = torch.Generator().manual_seed(T)
    e = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=g)]
    x = torch.randn(T, H, generator=g)
    x[:, :E] = 8.0 * torch.nn.functional.one_hot(e, E)
    x = x.to(torch.bfloat16).to(cuda)
    gl, ul = ((None, 7.0), (-6.0, 8.0)) if act == "swish" else ((None, None), (None, None))
    out, ids, wts, _ = ops.layer_forward_mx(x, w, 1, act, gl, ul, return_routing=True)
    assert torch.equal(ids.flatten().cpu().long(), e)
    ref = _ring_experts(x, ids, wts, w, act, gl, ul)
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))
    assert bool(torch.isfinite(out.float()).all()) and float(out.float().abs().max()) > 0


# 5 to 32 rows per expert: row tiles (the layer's, and the operator path's at 32 or 64 rows).
# on_block: the products on the block kernels, bit 0 gate_up, bit 1 down (the same for both lists).
@pytest.mark.parametrize("T,E,K,H,I,act,B,rows,on_block", [
    (160, 128, 4, 512, 512, "swish", 256, 32, 1),
    (700, 160, 4, 512, 1024, "silu", 256, 32, 3),
    (700, 136, 4, 1024, 1024, "silu", 256, 64, 3),   # 20 rows per expert; the operator path: 32 rows
    (1200, 160, 4, 1024, 512, "swish", 256, 64, 3),  # 30 rows per expert: 64 rows in both
    (250, 64, 4, 2560, 1536, "swish", 256, 32, 2),
    (900, 128, 4, 1024, 512, "swish", 16, 64, 3),   # 16-slot blocks: every tile at most 16 rows
    (200, 40, 4, 512, 512, "swish", 256, 32, 0),    # too few items: the ring kernels
])
def test_row_tiles_equal_ring_kernels(cuda, T, E, K, H, I, act, B, rows, on_block):
    say("mx block row tiles", T, E, K, H, I, act, B)
    lib = _lib.load()
    assert lib.moe_layer_mx_tile_rows(T, H, I, E, K, B) == rows
    for mt in (rows, ops.choose_mt(T, K, E)):
        tiles = lib.moe_max_tiles(T, K, E, lib.moe_num_blocks(T, K, E, B), B, 0, mt)
        assert lib.moe_mx_row_tile_kernels(H, I, E, tiles, mt) == on_block
    w = make_mx_weights(E, H, I, 13, cuda)
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(cuda)
    gl, ul = ((None, 7.0), (-6.0, 8.0)) if act == "swish" else ((None, None), (None, None))
    assert 4 * E < T * K <= 32 * E
    out, ids, wts, _ = ops.layer_forward_mx(x, w, K, act, gl, ul, return_routing=True, block_size=B)
    heights = torch.bincount(ids.flatten(), minlength=E).clamp(max=rows)
    assert B < 64 or int(heights.max()) > 16
    ref = _ring_experts(x, ids, wts, w, act, gl, ul, B)
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))
    got = ops.mx_experts(x, ids, wts, w, act, gl, ul, block_size=B)
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))


# Above four tokens the norm's own pass writes the MXFP8 codes: the same bits as the layer
# without its norm on the normalized rows.
@pytest.mark.parametrize("T,residual,actual", [(5, False, 480), (77, True, 512), (600, True, 500)])
def test_norm_pass_quantizes(cuda, T, residual, actual):
    say("mx norm pass", T, residual, actual)
    w = make_mx_weights(16, 512, 512, 17, cuda)
    g = torch.Generator().manual_seed(T)
    rnd = lambda *s: torch.randn(*s, generator=g)
    x, res = (rnd(T, 512).to(torch.bfloat16).to(cuda) for _ in range(2))
    gamma = (1 + 0.1 * rnd(512)).to(cuda)
    res = res if residual else None
    got = ops.layer_forward_mx(x, w, 4, gamma=gamma, eps=1e-5, hidden_actual=actual, residual=res)
    out, rsum = got if residual else (got, None)
    xn, _, _, v = ops.rms_norm_quant(x, gamma, 1e-5, actual, res)
    ref = ops.layer_forward_mx(xn, w, 4)
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))
    assert rsum is None or torch.equal(rsum.view(torch.int16), v.view(torch.int16))
