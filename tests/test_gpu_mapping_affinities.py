"""The blockwise mapping from dense affinities and the block-tile list of a mapping, at the
edges of their chunked passes: token counts around a 256-token chunk, expert counts whose
rows are not whole 16-byte pieces, block counts around the tile builder's LDS capacity."""
import numpy as np
import pytest
import torch

import test_gpu_kernels
from _util import say
from oracle import blockwise as BW
from vllm_neuron_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,E,B,mask", [
    (1, 1, 1, 4, False), (255, 3, 7, 16, True), (256, 8, 160, 256, False), (257, 2, 5, 64, True),
    (1500, 8, 160, 256, False), (777, 8, 257, 32, True), (300, 4, 1024, 16, False)])
def test_mapping_from_affinities_bit_exact(cuda, T, K, E, B, mask):
    say("mapping from affinities", T, K, E, B, mask)
    rng = np.random.default_rng(T + E)
    aff = np.zeros((T, E), np.float32)
    for t in range(T):
        aff[t, rng.choice(E, K, replace=False)] = rng.uniform(-1.0, 1.0, K).astype(np.float32)
    pm = (rng.uniform(size=T) < 0.8) if mask else None
    # one row in, so that rows start at any 4-byte offset of a 16-byte piece when E % 4 != 0
    store = torch.zeros(T + 1, E, device=cuda)
    store[1:] = torch.from_numpy(aff)
    got = ops.blockwise_mapping(affinities=store[1:], top_k=K, block_size=B,
                                padding_mask=None if pm is None else torch.from_numpy(pm).to(cuda))
    am, tpid, b2e, cond = BW.build_blockwise_mapping(aff, E, K, B, padding_mask=pm)
    for name, ref in (("affinities_masked", am), ("token_position_to_id", tpid),
                      ("block_to_expert", b2e), ("conditions", cond)):
        assert np.array_equal(got[name].cpu().numpy().reshape(-1), np.asarray(ref).reshape(-1)), name


# 1553 blocks (B = 6: no 16-byte pieces), 2048 and 2115 blocks: at and past the capacity
@pytest.mark.parametrize("T,K,E,B,S", [(2300, 4, 24, 6, 1), (4066, 8, 16, 16, 1), (4200, 8, 16, 16, 2),
                                       (40, 1, 2, 8, 0)])
def test_block_tiles_of_many_blocks(cuda, T, K, E, B, S):
    test_gpu_kernels.test_block_tiles_cover_every_slot_once(cuda, T, K, E, B, S)
