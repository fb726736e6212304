"""The 64- and 128-slot INT4 prefill tiles (int4_tile_kernel) against the
oracle: shapes from one k-tile up (128 columns), every group size, with and
without zero points, ragged tiles, skewed experts of many tiles. Bars: the
layer's (tests/helpers.py)."""
import numpy as np
import pytest

from helpers import awq_layer
from test_gpu_layer import check_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seq,hidden,inter,group,n_experts,top_k,n_shared", [
    (256, 1280, 896, 32, 64, 6, 2), (283, 1280, 896, 128, 64, 6, 2), (257, 1280, 896, 64, 64, 6, 0),
    (597, 1280, 896, 32, 64, 6, 1), (598, 1280, 896, 32, 64, 6, 1),   # the rule's edge (56 rows per expert)
    (256, 128, 128, 32, 40, 6, 1), (300, 256, 128, 64, 64, 4, 1),      # 64 slots, 1 .. 2 k-tiles of 128
    (300, 128, 256, 128, 5, 1, 1), (1000, 384, 128, 32, 6, 3, 2), (700, 640, 384, 64, 8, 2, 1),  # 128 slots
])
def test_int4_tiles(dev, seq, hidden, inter, group, n_experts, top_k, n_shared):
    from uocr_hip import synth
    L = synth.random_layer(seed=seq + hidden, hidden=hidden, inter=inter, n_experts=n_experts, top_k=top_k,
                           n_shared=n_shared, group=group)
    x = synth.bf16_normal(np.random.default_rng(seq), (seq, hidden), 1.0)
    check_parity(L, x, dev, sample=16, label=f"int4 tile H={hidden} I={inter} g={group}")


@pytest.mark.parametrize("seq,group,n_experts,top_k", [(256, 32, 40, 6), (300, 64, 48, 6), (270, 128, 32, 6), (600, 32, 4, 2)])
def test_int4_tiles_zero_points(dev, seq, group, n_experts, top_k):
    from uocr_hip import synth
    # (the last: 300 rows per expert at a shape of the 128-slot tiles)
    hidden, inter = (1280, 896) if n_experts > 4 else (384, 256)
    L = awq_layer(seed=group, group=group, n_experts=n_experts, top_k=top_k, n_shared=1, hidden=hidden, inter=inter)
    x = synth.bf16_normal(np.random.default_rng(seq), (seq, hidden), 1.0)
    check_parity(L, x, dev, sample=16, label=f"int4 tile zeros g={group}")


@pytest.mark.parametrize("seq,hidden,inter,n_experts,top_k", [
    (400, 1280, 896, 64, 6), (300, 256, 256, 64, 6), (1024, 640, 256, 64, 6),
])
def test_int4_tiles_skewed(dev, seq, hidden, inter, n_experts, top_k):
    """Popular experts own several tiles, others none: the live tiles are a small
    part of the list's capacity."""
    from uocr_hip import synth
    L = synth.random_layer(seed=seq, hidden=hidden, inter=inter, n_experts=n_experts, top_k=top_k, n_shared=1, group=32,
                           router_bias=synth.zipf_bias(n_experts) * 4)
    x = synth.bf16_normal(np.random.default_rng(seq), (seq, hidden), 1.0)
    x[:, 0] = 1.0
    check_parity(L, x, dev, sample=16, label=f"int4 tile skew H={hidden} I={inter}")
