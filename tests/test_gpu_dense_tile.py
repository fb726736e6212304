"""The prefill-sized tiles of the unquantised matrices (dense_tile_kernel)
against the oracle: the batch sizes where its tiles change, ragged last tiles,
and layer shapes outside the large-tile kernel's (routed experts through its
128-slot tiles). Bars: the layer's (tests/helpers.py)."""
import numpy as np
import pytest

from test_gpu_layer import check_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seq,hidden,inter,n_shared", [
    (65, 1280, 128, 2), (128, 256, 896, 2), (129, 1280, 128, 14), (1023, 128, 128, 1), (1024, 384, 128, 3),
    (1025, 384, 128, 3), (1300, 1280, 128, 1), (3300, 1280, 128, 1),
])
def test_shared_mlp_tiles(dev, seq, hidden, inter, n_shared):
    from uocr_hip import synth
    L = synth.random_layer(seed=seq, hidden=hidden, inter=inter, n_experts=8, top_k=2, n_shared=n_shared, group=32)
    synth.with_bf16_shared(L, seed=seq + 1)
    x = synth.bf16_normal(np.random.default_rng(seq), (seq, hidden), 1.0)
    check_parity(L, x, dev, sample=24, label=f"shared H={hidden} I={inter} S={n_shared}")


@pytest.mark.parametrize("seq,hidden,inter", [(256, 384, 128), (400, 128, 384), (700, 640, 256), (1111, 1280, 896)])
def test_routed_expert_tiles(dev, seq, hidden, inter):
    from uocr_hip import synth
    L = synth.random_layer_bf16(seed=seq, hidden=hidden, inter=inter, n_experts=6, top_k=3, n_shared=1)
    x = synth.bf16_normal(np.random.default_rng(seq), (seq, hidden), 1.0)
    check_parity(L, x, dev, sample=24, label=f"routed H={hidden} I={inter}")
