"""The prefill-sized tiles of the unquantised matrices (dense_tile_kernel)
against the oracle: the batch sizes where its tiles change, ragged last tiles,
and layer shapes outside the decoder's. Bars: the layer's (tests/helpers.py)."""
import numpy as np
import pytest

from test_gpu_layer import check_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seq,hidden,inter,n_shared", [
    (65, 1280, 128, 2), (128, 256, 896, 2), (129, 1280, 128, 14), (1023, 128, 128, 1), (1024, 384, 128, 3),
    (1025, 384, 128, 3), (1300, 1280, 128, 1), (3300, 1280, 128, 1),
    (96, 1280, 128, 2), (97, 1280, 128, 2), (97, 640, 896, 2),  # the smallest batch on 64-slot tiles
])
def test_shared_mlp_tiles(dev, seq, hidden, inter, n_shared):
    from uocr_hip import synth
    L = synth.random_layer(seed=seq, hidden=hidden, inter=inter, n_experts=8, top_k=2, n_shared=n_shared, group=32)
    synth.with_bf16_shared(L, seed=seq + 1)
    x = synth.bf16_normal(np.random.default_rng(seq), (seq, hidden), 1.0)
    check_parity(L, x, dev, sample=24, label=f"shared H={hidden} I={inter} S={n_shared}")


@pytest.mark.parametrize("seq,hidden,inter", [(256, 384, 128), (400, 128, 384), (700, 640, 256), (1111, 1280, 896)])
def test_routed_expert_tiles(dev, seq, hidden, inter):
    """128-slot tiles (more than 56 rows per expert)."""
    from uocr_hip import synth
    L = synth.random_layer_bf16(seed=seq, hidden=hidden, inter=inter, n_experts=6, top_k=3, n_shared=1)
    x = synth.bf16_normal(np.random.default_rng(seq), (seq, hidden), 1.0)
    check_parity(L, x, dev, sample=24, label=f"routed H={hidden} I={inter}")


@pytest.mark.parametrize("seq,hidden,inter,n_experts,top_k,zipf", [
    (256, 1280, 896, 64, 6, False), (283, 1280, 896, 64, 6, False),  # the decoder's shapes, 128 columns per workgroup
    (597, 1280, 896, 64, 6, False), (598, 1280, 896, 64, 6, False),  # the rule's edge (56 rows per expert)
    (300, 1280, 896, 64, 6, True),                                   # experts of several 64-slot tiles, and of none
    (300, 128, 128, 64, 2, False), (257, 384, 128, 40, 6, True),     # down with 64 columns per workgroup
])
def test_routed_expert_tiles_of_64_slots(dev, seq, hidden, inter, n_experts, top_k, zipf):
    from uocr_hip import synth
    L = synth.random_layer_bf16(seed=seq, hidden=hidden, inter=inter, n_experts=n_experts, top_k=top_k, n_shared=1,
                                router_bias=synth.zipf_bias(n_experts) if zipf else None)
    x = synth.bf16_normal(np.random.default_rng(seq), (seq, hidden), 1.0)
    if zipf:
        x[:, 0] = 1.0
    check_parity(L, x, dev, sample=24, label=f"routed64 H={hidden} E={n_experts} zipf={zipf}")
