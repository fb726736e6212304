"""The MFMA router (bf16 router matrix, more than 64 tokens or unquantised
experts): routing ids and weights bit-exact with the CPU oracle at the edges of
its 16-token tiles, 16-expert waves and hidden sizes, with every input form."""
import numpy as np
import pytest

from test_gpu_layer import run_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seq,hidden,n_experts,top_k,rms,dtype", [
    (65, 1280, 64, 6, False, "bf16"),
    (80, 1280, 64, 6, False, "f32"),
    (257, 1280, 64, 8, True, "f32"),
    (255, 1280, 17, 4, True, "f32"),
    (300, 1280, 5, 1, False, "bf16"),
    (271, 128, 64, 6, False, "f32"),
    (272, 128, 64, 6, True, "f32"),
    (273, 1792, 48, 6, True, "f32"),
    (256, 1792, 64, 6, False, "bf16"),
    (289, 896, 16, 2, True, "f32"),
])
def test_mfma_router_bit_exact(dev, seq, hidden, n_experts, top_k, rms, dtype):
    import oracle as O
    from uocr_hip import MoELayerInt4, synth

    print(f"[router] seq={seq} H={hidden} E={n_experts} K={top_k} rms={rms} {dtype}", flush=True)
    L = synth.random_layer(seed=seq + hidden, hidden=hidden, inter=128, n_experts=n_experts, top_k=top_k,
                           n_shared=1, group=32, rms=rms)
    rng = np.random.default_rng(seq)
    x = synth.bf16_normal(rng, (seq, hidden), 1.0)
    if dtype == "f32":  # values scaled by 2^-3 .. 2^2, zeros, one tiny row
        x = rng.standard_normal((seq, hidden), dtype=np.float32)
        x *= np.exp2(rng.integers(-3, 3, size=x.shape)).astype(np.float32)
        x[0, ::3] = 0.0
        x[1] *= np.float32(2.0 ** -30)
    layer = MoELayerInt4(L)
    ids, w, out = run_layer(layer, x, dtype, dev)
    assert layer.status() == 0
    ids_o, w_o, _ = O.moe_layer(L, x, sel=np.arange(1, dtype=np.int32))
    assert np.array_equal(ids, ids_o), np.argwhere(ids != ids_o)[:5]
    assert np.array_equal(w.view(np.uint32), w_o.view(np.uint32))
    assert np.isfinite(out).all()
    layer.close()
