"""Rows per tile of the fp8 layer, by sizes: host rules, no GPU needed. The results of all tile
heights are the same bits (test_gpu_mid_tiles.py); these are the sizes where one of them was
measured slower."""
from types import SimpleNamespace

import pytest
import torch

from vllm_neuron_amd import _lib, ops


def _rows(T, H, I, E, K, S=0, B=256):
    return _lib.load().moe_layer_tile_rows(T, H, I, E, K, S, B)


RING, GATE_UP, DOWN, BOTH = 0, 1, 2, 3


# 16-row tiles: the mid-size kernels from 1024 items, 2048 where K is above 5120.
@pytest.mark.parametrize("T,H,I,E,on_mid", [
    (2, 7168, 2048, 384, RING), (4, 7168, 2048, 384, RING),      # 35 tiles: 560 gate_up and 980 down items
    (8, 7168, 2048, 384, DOWN), (8, 7168, 2048, 256, DOWN), (14, 7168, 2048, 384, DOWN),  # 1104 to 1920 gate_up
    (15, 7168, 2048, 384, BOTH), (64, 7168, 2048, 256, BOTH),
    (9, 5120, 1536, 160, DOWN), (10, 5120, 1536, 160, BOTH)])    # 936 and 1044 gate_up items of K = 5120
def test_sixteen_row_kernels(T, H, I, E, on_mid):
    lib = _lib.load()
    assert _rows(T, H, I, E, 8, 1) == 16
    tiles = lib.moe_max_tiles(T, 8, E, lib.moe_num_blocks(T, 8, E, 256), 256, 1, 16)
    assert lib.moe_row_tile_kernels(H, I, tiles, 16) == on_mid


# 5 to 24 rows per expert: 64-row tiles only where both products have 512 items of them.
@pytest.mark.parametrize("T,H,I,E,K,S,rows", [
    (16, 4096, 14336, 8, 2, 0, 16), (24, 4096, 14336, 8, 2, 0, 32),  # 1008 gate_up, 144 down items
    (96, 4096, 14336, 8, 2, 0, 32), (112, 4096, 14336, 8, 2, 0, 64),
    (96, 7168, 2048, 32, 8, 1, 64),   # 47 tiles: 752 and 1316
    (257, 7168, 2048, 256, 8, 1, 64), (200, 5120, 1536, 160, 8, 1, 64),
    (20, 1024, 512, 8, 2, 0, 32), (100, 1024, 512, 8, 2, 0, 64),  # the small layer
    (200, 2048, 768, 128, 8, 0, 32)])  # I not a multiple of 512
def test_row_tiles(T, H, I, E, K, S, rows):
    assert _rows(T, H, I, E, K, S) == rows


# Above 32: 128-row block tiles up to 76 rows per expert, where their gate_up items fill the chip twice.
@pytest.mark.parametrize("T,H,I,E,K,S,rows", [
    (1537, 7168, 2048, 384, 8, 1, 128), (1901, 7168, 2048, 384, 8, 1, 128), (3648, 7168, 2048, 384, 8, 1, 128),
    (3649, 7168, 2048, 384, 8, 1, 256), (641, 5120, 1536, 160, 8, 1, 128), (8192, 7168, 2048, 256, 8, 1, 256),
    (136, 7168, 2048, 32, 8, 1, 128),                                   # 41 x 16 items
    (160, 1024, 512, 8, 2, 0, 256), (520, 2048, 768, 128, 8, 0, 256)])  # 10 x 4; I not a multiple of 512
def test_block_tiles(T, H, I, E, K, S, rows):
    assert _rows(T, H, I, E, K, S) == rows


# The operators' block tile lists are as tall as the layer's; channel scales keep 256 rows.
@pytest.mark.parametrize("T,H,I,E,K,S,rows", [
    (1500, 5120, 1536, 160, 8, 0, 128), (250, 5120, 1536, 40, 8, 1, 128),  # 57 tiles, 684 items
    (560, 2048, 1024, 48, 6, 2, 128), (400, 2048, 768, 48, 6, 2, 256), (1700, 5120, 1536, 160, 8, 0, 256)])
def test_operators_take_the_layers_block_tiles(T, H, I, E, K, S, rows):
    w = SimpleNamespace(hidden=H, w13=torch.empty(E, 2 * I, 0), n_shared=S, has_channel_scales=False)
    assert ops.use_block_kernels(T, K, E)
    assert ops.block_tile_rows(T, K, E, w) == rows == _rows(T, H, I, E, K, S)
    w.has_channel_scales = True
    assert ops.block_tile_rows(T, K, E, w) == 256
