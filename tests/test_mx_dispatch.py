"""Which kernels the MXFP4 experts run, by sizes: host rules, no GPU needed. The results of both
kernels are the same bits (test_gpu_mx_block.py); these are the sizes where one of them was
measured slower."""
import pytest

from vllm_neuron_amd import _lib

RING, GATE_UP, DOWN, BOTH = 0, 1, 2, 3


def _plan(T, H, I, E, K, B=256):
    """(rows per tile, products on the block kernels) of the layer on row tiles."""
    lib = _lib.load()
    mt = lib.moe_layer_mx_tile_rows(T, H, I, E, K, B)
    tiles = lib.moe_max_tiles(T, K, E, lib.moe_num_blocks(T, K, E, B), B, 0, mt)
    return mt, lib.moe_mx_row_tile_kernels(H, I, E, tiles, mt)


# GPT-OSS-20B (32 experts, top-4, 2880 padded to 3072): one tile per expert is 768 gate_up and 384
# down items. Three whole rounds of the ring kernels' 256 workgroups, and 64-row tiles whose down
# would stay on the ring.
@pytest.mark.parametrize("T,rows,on_block", [
    (32, 16, RING), (33, 32, RING), (64, 32, RING), (80, 32, DOWN), (135, 32, DOWN), (160, 64, BOTH),
    (256, 64, BOTH)])
def test_gpt_oss_20b_row_tiles(T, rows, on_block):
    assert _plan(T, 3072, 3072, 32, 4) == (rows, on_block)


@pytest.mark.parametrize("T,H,I,E,rows,on_block", [
    (48, 4096, 4096, 24, 32, RING),        # 768 gate_up items of K = 4096
    (108, 1024, 1024, 96, 32, GATE_UP),    # of K = 1024: the block kernel even at 768; down on the ring
    (144, 1024, 512, 128, 32, BOTH),       # 584 and 584 items: below 1024 of 64-row tiles, up to 16 rows
    (96, 2048, 1024, 64, 32, BOTH), (256, 2048, 1024, 64, 32, BOTH), (272, 2048, 1024, 64, 64, BOTH),
    (256, 2048, 1024, 128, 64, BOTH),      # 8 rows, 1152 and 1152 items of 64-row tiles
    (320, 1024, 2048, 64, 64, GATE_UP),    # 20 rows per expert: 64-row tiles, down on the ring
    (160, 3072, 3072, 128, 64, BOTH)])     # GPT-OSS-120B
def test_row_tiles(T, H, I, E, rows, on_block):
    assert _plan(T, H, I, E, 4) == (rows, on_block)


# Above 32 rows per expert: block tiles of up to 128 rows, but 64-row tiles on the ring kernels
# where one round of those holds both products (tall tiles are then longer chains of the same work).
@pytest.mark.parametrize("T,H,I,E,K,rows", [
    (66, 512, 512, 4, 2, 64), (260, 512, 512, 16, 2, 64), (160, 1024, 1024, 8, 2, 64),  # 33 to 40 rows
    (512, 512, 512, 4, 2, 64), (600, 1024, 1024, 8, 2, 64),
    (256, 3072, 3072, 4, 2, 64), (300, 3072, 3072, 4, 2, 128),  # 288 and 336 gate_up items
    (1024, 1536, 512, 16, 2, 64), (1200, 1536, 512, 16, 2, 128),  # 288 and 324 down items
    (257, 3072, 3072, 32, 4, 128), (2048, 3072, 3072, 128, 4, 128)])
def test_block_tiles(T, H, I, E, K, rows):
    lib = _lib.load()
    assert lib.moe_layer_mx_tile_rows(T, H, I, E, K, 256) == rows
    if rows == 64:
        assert _plan(T, H, I, E, K) == (64, RING)
