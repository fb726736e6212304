"""The calls that a user of uocr_hip makes, at the sizes they are made with.

Five families, each through a public entry point:

* ``moe``          MoELayer.forward on INT4 routed experts: the decoder's MoE
                   block, from one decoding request to a 4096-token prefill.
* ``moe_bf16``     the same on the default (unquantised bf16) expert format.
* ``rswa_decode``  batched R-SWA decode attention over the requests' caches.
* ``rswa_prefill`` ragged prefill: the cache write, then causal attention.
* ``ops``          the MoE block through the operator mirrors, call by call.

Shapes are the decoder's (hidden 1280, 64 experts of width 896, top-6, shared
MLP of width 1792, 10 heads of 128) as synth.py and bench.py hold them.
"""
import math
import types

import numpy as np
import torch

import sys
import os

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "unlimited-ocr.cpp_amd"))

from uocr_hip import MoELayer, _lib, ops  # noqa: E402

H, I, E, K, S = 1280, 896, 64, 6, 2
SI = S * I
EPS = 1e-6
ZIPF = [1.5 * -1.1 * math.log(e + 1) for e in range(E)]


def listed():
    def moe(name, seq, **kw):
        c = dict(name=name, kind="moe", seq=seq, group=32, zeros=False, shared="int4", rms=False, x="bf16",
                 router="bf16", zipf=False)
        c.update(kw)
        return c

    return [
        # one request generating: the smallest call, latency counts
        moe("decode_1", 1),
        # a batch of 16 requests generating (bench.py's headline)
        moe("decode_16", 16),
        # 64 requests in the engine's own layer form: f32 hidden states, fused
        # RMSNorm and residual, shared MLP as the checkpoint holds it
        moe("decode_64_engine", 64, rms=True, x="f32", shared="bf16"),
        # a large decode batch, or a short prompt, on AWQ experts (zero points,
        # group 128, the f32 router that the fold leaves)
        moe("decode_150_awq", 150, group=128, zeros=True, rms=True, x="f32", router="f32"),
        # one page's prompt: the 273 visual tokens and a few words
        moe("prefill_283_engine", 283, rms=True, x="f32", shared="bf16"),
        # ragged prefill of several pages or prompts
        moe("prefill_1024", 1024),
        # the largest prefill, with popular experts (Zipf)
        moe("prefill_4096_zipf", 4096, zipf=True),
        # the default expert format, decoding and in prefill
        dict(name="bf16_decode_16", kind="moe_bf16", seq=16),
        dict(name="bf16_prefill_1111", kind="moe_bf16", seq=1111),
        # attention of 16 generating requests with full and part-full caches
        dict(name="rswa_decode_16", kind="rswa_decode", batch=16, most=1128, heads=10, kv_heads=10, head_dim=128),
        # attention of four prompts' prefill
        dict(name="rswa_prefill_4", kind="rswa_prefill", batch=4, most=1000, heads=10, kv_heads=10, head_dim=128),
        # a program written against the operators: 16 prompts of 64 tokens
        dict(name="ops_1024", kind="ops", seq=1024, group=128, zeros=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["moe"] * 5 + ["moe_bf16", "rswa_decode", "rswa_prefill", "ops"])
    if kind == "moe":
        seq = _log(rng, 1, 4096)
        awq = rng.random() < 0.3
        rms = rng.random() < 0.5
        return dict(kind=kind, seq=seq, group=rng.choice([32, 64, 128]), zeros=awq,
                    shared=rng.choice(["int4", "bf16"]), rms=rms, x="f32" if rms else rng.choice(["bf16", "f32"]),
                    router="f32" if awq and rng.random() < 0.7 else "bf16", zipf=seq >= 512 and rng.random() < 0.5)
    if kind == "moe_bf16":
        return dict(kind=kind, seq=_log(rng, 1, 2048))
    if kind == "ops":
        return dict(kind=kind, seq=_log(rng, 1, 1024), group=rng.choice([32, 64, 128]), zeros=rng.random() < 0.5)
    heads, kv_heads, head_dim = rng.choice([(10, 10, 128), (10, 10, 128), (8, 2, 64)])
    if kind == "rswa_decode":
        return dict(kind=kind, batch=_log(rng, 1, 32), most=rng.randint(150, 1300), heads=heads, kv_heads=kv_heads,
                    head_dim=head_dim)
    return dict(kind=kind, batch=rng.randint(1, 4), most=rng.randint(60, 1000), heads=heads, kv_heads=kv_heads,
                head_dim=head_dim)


# ---- inputs -----------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * std


def _bf16(t):
    return t.to(torch.bfloat16)


def _bits(t):
    """bf16 tensor -> host array of its bits."""
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def _int4(g, n, rows, cols, group, zeros):
    """n reference-layout INT4 matrices: nibbles uniform, scales |N(0, 0.003)|."""
    ng = cols // group
    q = torch.randint(0, 256, (n, rows, cols // 2), generator=g, device="cuda", dtype=torch.uint8)
    s = _bf16(_randn(g, n, rows, ng, std=0.003).abs()).float()
    if zeros:
        z = torch.randint(5, 11, (n, rows, ng), generator=g, device="cuda").float()
    else:
        z = torch.full((n, rows, ng), 8.0, device="cuda")
    return q, s, z


def _weights(case, g):
    """Device tensors of one layer's weights (the sources of both the layer and the exact result)."""
    w = types.SimpleNamespace()
    router = _randn(g, E, H, std=0.02)
    if case.get("zipf"):
        router[:, 0] = torch.tensor(ZIPF, device="cuda")
    w.router = _bf16(router)
    w.router_f32 = None
    if case.get("router") == "f32":  # the fold's per-column scale
        w.router_f32 = w.router.float() * (0.5 + 1.5 * torch.rand(H, generator=g, device="cuda"))
    if case["kind"] == "moe_bf16":
        w.gate, w.up = (_bf16(_randn(g, E, I, H, std=0.02)) for _ in range(2))
        w.down = _bf16(_randn(g, E, H, I, std=0.02))
    else:
        w.gate, w.up = (_int4(g, E, I, H, case["group"], case["zeros"]) for _ in range(2))
        w.down = _int4(g, E, H, I, case["group"], case["zeros"])
    if case.get("shared") == "int4":
        w.sgate, w.sup = (_int4(g, 1, SI, H, case["group"], case["zeros"]) for _ in range(2))
        w.sdown = _int4(g, 1, H, SI, case["group"], case["zeros"])
    else:
        w.sgate, w.sup = (_bf16(_randn(g, SI, H, std=0.02)) for _ in range(2))
        w.sdown = _bf16(_randn(g, H, SI, std=0.02))
    w.rms = 0.5 + 1.5 * torch.rand(H, generator=g, device="cuda") if case.get("rms") else None
    return w


def _input(case, g):
    x = _randn(g, case["seq"], H)
    if case["kind"] == "ops":
        return x
    if case.get("zipf"):
        x[:, 0] = 1.0
    x = _bf16(x)
    return x.float() if case.get("x") == "f32" else x


def _host_int4(t, group):
    q, s, z = (a.cpu().numpy() for a in t)
    return [types.SimpleNamespace(packed=q[i], scales=s[i], zeros=z[i], rows=q.shape[1], cols=2 * q.shape[2],
                                  group=group) for i in range(q.shape[0])]


def _host_bf16(t):
    b = _bits(t)
    return [types.SimpleNamespace(data=m) for m in (b if b.ndim == 3 else b[None])]


def _layer(case, w):
    L = types.SimpleNamespace(hidden=H, inter=I, n_experts=E, top_k=K, n_shared=S, group=case.get("group", 32),
                              norm_topk_prob=0, routed_scaling_factor=1.0, scoring_sigmoid=0,
                              router_bf16=_bits(w.router), rms_eps=EPS,
                              router_f32=None if w.router_f32 is None else w.router_f32.cpu().numpy(),
                              rms_weight=None if w.rms is None else w.rms.cpu().numpy())
    if case["kind"] == "moe_bf16":
        L.gate_w, L.up_w, L.down_w = _host_bf16(w.gate), _host_bf16(w.up), _host_bf16(w.down)
    else:
        L.gate, L.up, L.down = (_host_int4(t, case["group"]) for t in (w.gate, w.up, w.down))
    if case.get("shared") == "int4":
        L.shared_gate, L.shared_up, L.shared_down = (_host_int4(t, case["group"])[0]
                                                     for t in (w.sgate, w.sup, w.sdown))
    else:
        L.shared_gate_w, L.shared_up_w, L.shared_down_w = (_host_bf16(t)[0] for t in (w.sgate, w.sup, w.sdown))
    return MoELayer(L)


def _lens(case):
    """Rows of each request: the longest, and others between a quarter of it and all."""
    most = case["most"]
    return [max(1, int(most * (1.0 - 0.75 * (j * 0.6180339887 % 1.0)))) for j in range(case["batch"])]


def _table(t):
    """The engine's device table of INT4 matrices (ops.RefInt4Table's fields)."""
    q, s, z = t
    n, rows, half = q.shape
    r = object.__new__(ops.RefInt4Table)
    r.rows, r.cols, r.ng = rows, 2 * half, s.shape[2]
    r.group = r.cols // r.ng
    r.packed, r.scales, r.zeros = q, s, z
    r.pstride, r.sstride = rows * half, rows * r.ng
    return r


def prepare(case, seed):
    g = _gen(seed)
    st = types.SimpleNamespace(case=case)
    if case["kind"] in ("moe", "moe_bf16"):
        w = _weights(case, g)
        n = case["seq"]
        st.x = _input(case, g)
        st.layer = _layer(case, w)
        st.ws = st.layer.alloc_workspace(n)
        st.out = torch.empty(n, H, device="cuda")
        st.ids = torch.empty(n, K, dtype=torch.int32, device="cuda")
        st.weights = torch.empty(n, K, device="cuda")
    elif case["kind"] == "ops":
        w = _weights(case, g)
        n = case["seq"]
        st.x = _input(case, g)
        st.router, st.sgate, st.sup, st.sdown = (t.view(torch.int16) for t in (w.router, w.sgate, w.sup, w.sdown))
        st.gate, st.up, st.down = _table(w.gate), _table(w.up), _table(w.down)
        f = lambda *s: torch.empty(*s, device="cuda")  # noqa: E731
        i = lambda *s: torch.empty(*s, dtype=torch.int32, device="cuda")  # noqa: E731
        st.logits, st.ids, st.weights = f(n, E), i(n, K), f(n, K)
        st.tok, st.tok_w, st.count, st.act = i(E, n), f(E, n), i(E), f(E, n, I)
        st.g, st.u, st.h, st.y, st.out = f(n, SI), f(n, SI), f(n, SI), f(n, H), f(n, H)
    else:
        b, cap, st_ = case["batch"], case["most"], case["kv_heads"] * case["head_dim"]
        n = _lens(case)
        st.lens = torch.tensor(n, dtype=torch.int32, device="cuda")
        if case["kind"] == "rswa_decode":
            st.k, st.v = _randn(g, b, cap, st_), _randn(g, b, cap, st_)
            st.slots = torch.arange(b, dtype=torch.int32, device="cuda")
            st.q = _randn(g, b, case["heads"] * case["head_dim"])
        else:
            total = sum(n)
            st.k, st.v = torch.zeros(b, cap, st_, device="cuda"), torch.zeros(b, cap, st_, device="cuda")
            st.k_new, st.v_new = _randn(g, total, st_), _randn(g, total, st_)
            st.q = _randn(g, total, case["heads"] * case["head_dim"])
            st.slots = torch.cat([torch.full((m,), j, dtype=torch.int32) for j, m in enumerate(n)]).cuda()
            st.pos = torch.cat([torch.arange(m, dtype=torch.int32) for m in n]).cuda()
        st.out = torch.empty_like(st.q)
    return st


# ---- one pass ---------------------------------------------------------------

def run(st):
    case = st.case
    if case["kind"] in ("moe", "moe_bf16"):
        st.layer.forward(st.x, st.out, st.ws, st.ids, st.weights)
        return {"out": st.out, "ids": st.ids, "weights": st.weights}
    if case["kind"] == "ops":
        n = case["seq"]
        ops.matmul_t_bf16(st.x, st.router, st.logits)
        ops.moe_router_topk(st.logits, K, 0, 1.0, 0, st.ids, st.weights, st.tok, st.tok_w, st.count, n)
        st.out.zero_()
        ops.moe_grouped_gate_up_int4(st.x, st.gate, st.up, st.tok, st.count, n, st.act)
        ops.moe_grouped_down_int4(st.act, st.down, st.tok, st.tok_w, st.count, n, st.out)
        ops.matmul_t_bf16(st.x, st.sgate, st.g)
        ops.matmul_t_bf16(st.x, st.sup, st.u)
        ops.silu_mul(st.g, st.u, st.h)
        ops.matmul_t_bf16(st.h, st.sdown, st.y)
        ops.add_scaled(st.out, st.y, 1.0)
        return {"out": st.out, "ids": st.ids, "weights": st.weights}
    lib = _lib.load()
    stream = torch.cuda.current_stream().cuda_stream
    b, cap = case["batch"], case["most"]
    kv, hd = case["kv_heads"], case["head_dim"]
    if case["kind"] == "rswa_decode":
        _lib.check(lib.uocr_hip_rswa_attention_batch(
            st.q.data_ptr(), st.k.data_ptr(), st.v.data_ptr(), st.lens.data_ptr(), st.slots.data_ptr(), b, cap,
            case["heads"], kv, hd, st.out.data_ptr(), stream))
        return {"out": st.out}
    n = st.q.shape[0]
    _lib.check(lib.uocr_hip_rswa_write_prefill_ragged(
        st.k_new.data_ptr(), st.v_new.data_ptr(), st.k.data_ptr(), st.v.data_ptr(), st.slots.data_ptr(),
        st.pos.data_ptr(), n, cap, kv, hd, stream))
    _lib.check(lib.uocr_hip_rswa_attention_ragged(
        st.q.data_ptr(), st.k.data_ptr(), st.v.data_ptr(), st.slots.data_ptr(), st.pos.data_ptr(), n, cap,
        case["heads"], kv, hd, st.out.data_ptr(), stream))
    return {"out": st.out, "k": st.k, "v": st.v}


# ---- what a pass cannot do without ------------------------------------------

def work(case):
    if case["kind"] in ("moe", "moe_bf16", "ops"):
        n = case["seq"]
        touched = E * (1.0 - (1.0 - K / E) ** n)
        per = 3 * H * I
        if case["kind"] == "moe_bf16":
            weights = (touched + S) * per * 2
        else:
            int4 = per * (0.5 + (4 if case["zeros"] else 2) / case["group"])
            weights = touched * int4 + S * (int4 if case.get("shared") == "int4" else per * 2)
        rows = n * H * ((2 if case.get("x", "bf16") == "bf16" and case["kind"] != "ops" else 4) + 4)
        router = E * H * (4 if case.get("router") == "f32" else 2)
        return {"bytes": weights + rows + router, "flops": n * (2.0 * per * (K + S) + 2.0 * E * H)}
    hd, heads, kv = case["head_dim"], case["heads"], case["kv_heads"]
    b, lens = case["batch"], _lens(case)
    rows = sum(lens)
    if case["kind"] == "rswa_decode":
        return {"bytes": 4.0 * (rows * 2 * kv * hd + 2 * b * heads * hd), "flops": 4.0 * hd * heads * rows}
    pairs = sum(n * (n + 1) // 2 for n in lens)
    return {"bytes": 4.0 * rows * (2 * heads * hd + 4 * kv * hd), "flops": 4.0 * hd * heads * pairs}


def tolerance(case):
    # about four times the error against exact(): attention 1.8e-7 (32-bit
    # sums, and the hardware's exp2); the operators 8.4e-4 (f16 operands
    # rounded once more per call); with the residual in the sum 1.5e-4; the
    # MoE block alone 2.9e-4 (f16 activations)
    if case["kind"].startswith("rswa"):
        return {"rel": 2e-6, "max": 2e-5}
    if case["kind"] == "ops":
        return {"rel": 3.4e-3, "max": 3.4e-2}
    if case.get("rms"):
        return {"rel": 6e-4, "max": 6e-3}
    return {"rel": 1.2e-3, "max": 1.2e-2}


# ---- the same in 64 bits ----------------------------------------------------

def _deq(t, i):
    q, s, z = (a[i] for a in t)
    v = torch.stack([q & 15, q >> 4], dim=-1).flatten(1).double()
    n = v.shape[1] // s.shape[1]
    return (v - z.double().repeat_interleave(n, 1)) * s.double().repeat_interleave(n, 1)


def _mlp(x, gate, up, down):
    g = x @ gate.T.contiguous()
    return (g * torch.sigmoid(g) * (x @ up.T.contiguous())) @ down.T.contiguous()


def exact(case, seed):
    g = _gen(seed)
    if case["kind"] in ("moe", "moe_bf16", "ops"):
        w = _weights(case, g)
        x0 = _input(case, g).double()
        x = x0
        if w.rms is not None:
            x = x0 / torch.sqrt((x0 * x0).mean(1, keepdim=True) + EPS) * w.rms.double()
        router = (w.router if w.router_f32 is None else w.router_f32).double()
        p = torch.softmax(x @ router.T.contiguous(), 1)
        weights, ids = torch.topk(p, K, dim=1)
        mat = (lambda t, e: t[e].double()) if case["kind"] == "moe_bf16" else _deq
        out = torch.zeros_like(x)
        for e in range(E):
            tok, j = torch.nonzero(ids == e, as_tuple=True)
            if len(tok):
                y = _mlp(x[tok], mat(w.gate, e), mat(w.up, e), mat(w.down, e))
                out[tok] += weights[tok, j][:, None] * y
        if case.get("shared") == "int4":
            out += _mlp(x, _deq(w.sgate, 0), _deq(w.sup, 0), _deq(w.sdown, 0))
        else:
            out += _mlp(x, w.sgate.double(), w.sup.double(), w.sdown.double())
        if w.rms is not None:
            out += x0
        return {"out": out, "ids": ids.int(), "weights": weights}
    st = prepare(case, seed)
    b, cap, hd, kv, heads = case["batch"], case["most"], case["head_dim"], case["kv_heads"], case["heads"]
    rep = heads // kv
    out = torch.empty(st.q.shape, dtype=torch.float64, device="cuda")
    k, v = st.k.clone(), st.v.clone()
    at = 0
    for j, n in enumerate(st.lens.tolist()):
        if case["kind"] == "rswa_prefill":
            k[j, :n], v[j, :n] = st.k_new[at:at + n], st.v_new[at:at + n]
            rows = slice(at, at + n)
        else:
            rows = slice(j, j + 1)
        at += n
        q = st.q[rows].double().view(-1, heads, hd)
        for h in range(heads):
            kh = k[j, :n].view(n, kv, hd)[:, h // rep].double()
            vh = v[j, :n].view(n, kv, hd)[:, h // rep].double().contiguous()
            s = q[:, h].contiguous() @ kh.T.contiguous() / math.sqrt(hd)
            if case["kind"] == "rswa_prefill":
                s = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), -math.inf)
            out[rows, h * hd:(h + 1) * hd] = torch.softmax(s, 1) @ vh
    if case["kind"] == "rswa_decode":
        return {"out": out}
    return {"out": out, "k": None, "v": None}  # the caches hold copies
