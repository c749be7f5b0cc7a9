"""The prefill-sized MXFP4 expert GEMMs of the layer (above 32 routed rows per expert).

Same scaled MFMAs in the same K order and the same epilogue arithmetic as the row-tile
kernels, so the layer's output is held bit for bit to the op-by-op path, which runs the
row-tile kernels (those are checked against the oracle in test_gpu_mx.py)."""
import dataclasses

import pytest
import torch

from _util import say
from test_gpu_mx import make_mx_weights
from vllm_neuron_amd import ops

pytestmark = pytest.mark.gpu


def _skew(w, counts_bias):
    return dataclasses.replace(w, router_bias=torch.tensor(counts_bias, device=w.w13.device))


# T * K / E > 32 in all of them. H = I = 512: one scale group, two steps; 1536 x 1024: odd
# numbers of groups; 768: not a multiple of 512, which stays on the row-tile kernels.
@pytest.mark.parametrize("T,E,K,H,I,act,bias,skew", [
    (67, 2, 1, 512, 512, "swish", True, [0.0, -60.0]),         # one expert holds all 67 rows, one none
    (129, 4, 2, 512, 512, "silu", False, [30.0, 0.0, 0.0, -30.0]),  # a 129-row expert: two 65-row tiles
    (128, 3, 1, 1536, 1024, "swish", True, [0.0, 0.0, 0.0]),
    (97, 1, 1, 1024, 512, "swish", True, [0.0]),               # a 97-row tile (four 32-row groups)
    (257, 8, 2, 512, 1536, "swish", True, [3.0, 2.0, 1.0, 0.0, 0.0, -1.0, -2.0, -40.0]),
    (1025, 16, 4, 1024, 1024, "swish", True, [0.0] * 16),
    (300, 8, 2, 768, 512, "swish", True, [0.0] * 8),
])
def test_layer_equals_row_tile_path(cuda, T, E, K, H, I, act, bias, skew):
    say("mx block layer", T, E, K, H, I, act)
    w = _skew(make_mx_weights(E, H, I, 11, cuda, bias=bias), skew)
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(cuda)
    gl, ul = ((None, 7.0), (-6.0, 8.0)) if act == "swish" else ((None, None), (None, None))
    assert T * K > 32 * E
    out, ids, wts, _ = ops.layer_forward_mx(x, w, K, act, gl, ul, return_routing=True)
    ref = ops.mx_experts(x, ids, wts, w, act, gl, ul)
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))
    assert bool(torch.isfinite(out.float()).all()) and float(out.float().abs().max()) > 0
