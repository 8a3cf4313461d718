"""The work a program has this backend do, as cases that can be timed and checked.

The sizes are gpt-oss's own (2880-wide stream, 64 query and 8 key/value heads of 64, 32 or
128 MXFP4 experts of which 4 run per token) at the contexts and prompt lengths of the
benchmark configurations and the tests.  Ten of the twelve listed cases are single layers
or blocks through the C ABI or its Python wrapper, on weights and workspaces that a program
keeps; two are whole calls of the model that return logits.

Layer weights are uploaded from GGUF bytes made from the seed, with scales that give rows
of about the magnitude of a trained model's (the projections' outputs are of order one).
exact() evaluates the same bytes in 64 bits in plain torch.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tt-lab_amd"))
import ttlab_amd  # noqa: E402

N = 2880                      # residual stream, expert hidden
HEADS, KV_HEADS, HEAD = 64, 8, 64
QKV_ROWS, Q_WIDTH = 5120, 4096
WINDOW = 128                  # sliding window of the even layers
USED = 4                      # experts per token
VOCAB = 201088
EPS = 1e-5
EMIN, EMAX = 116, 121         # E8M0 of the layers' weights: rms about 0.02


def listed():
    return [
        # One token, one expert matrix at a time: the stacked gate|up matvec of decode, over
        # 16 resident matrices in rotation so that the weights come from memory as they do
        # while a token passes through the layers.
        {"name": "matvec_5760", "kind": "matvec", "rows": 5760, "matrices": 16, "bias": True},
        # One token through the MoE layers of the 20b shape (norm, router, top-4, experts,
        # combine): the largest part of a decode step.
        {"name": "moe_decode_20b", "kind": "moe_decode", "experts": 32, "layers": 6},
        # One token's attention in every layer (sliding and full in turn) at context 2048,
        # the context of the decode benchmark.
        {"name": "attn_decode_2048", "kind": "attn_decode", "position": 2047, "layers": 24},
        # The Q/K/V projection of one 512-token prompt pass.
        {"name": "qkv_prompt_512", "kind": "projection", "rows": QKV_ROWS, "cols": N, "tokens": 512,
         "residual": False},
        # The output projection with its residual add for a short prompt (a Harmony
        # template with a one-line question).
        {"name": "output_prompt_77", "kind": "projection", "rows": N, "cols": Q_WIDTH, "tokens": 77,
         "residual": True},
        # Attention of the last 512-token pass of a 2048-token prompt, one sliding and one
        # full layer.
        {"name": "attn_prompt_2048", "kind": "attn_prompt", "first": 1536, "tokens": 512, "layers": 2},
        # The MoE layer (router and experts) of one 512-token prompt pass, 20b shape.
        {"name": "moe_prompt_512", "kind": "moe_prompt", "experts": 32, "tokens": 512},
        # The same for a short prompt at the 120b shape: about one token per expert that is
        # hit, so the weights are read for few tokens.
        {"name": "moe_prompt_40_120b", "kind": "moe_prompt", "experts": 128, "tokens": 40},
        # Batched experts with the routing given (balanced), bf16 activations: the prefill
        # benchmark configuration.
        {"name": "experts_bf16_512", "kind": "experts", "experts": 32, "tokens": 512, "dtype": "bf16",
         "balanced": True},
        # The same on the opt-in scaled path (MXFP8 activations).
        {"name": "experts_mxfp8_512", "kind": "experts", "experts": 32, "tokens": 512, "dtype": "bf16_mxfp8",
         "balanced": True},
        # One decode step of the whole 20b model at context 2048, token in, logits out.
        {"name": "forward_20b", "kind": "forward", "layers": 24, "position": 2047},
        # A 2048-token prompt through the whole 20b model, tokens in, last logits out.
        {"name": "prompt_20b", "kind": "prompt", "layers": 24, "tokens": 2048},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    kind = rng.choice(["matvec", "moe_decode", "attn_decode", "projection", "projection", "attn_prompt", "moe_prompt",
                       "moe_prompt", "experts", "experts", "forward", "prompt"])
    if kind == "matvec":
        return {"kind": kind, "rows": 16 * _log(rng, 1, 360), "matrices": rng.randint(1, 16),
                "bias": rng.random() < 0.5}
    if kind == "moe_decode":
        return {"kind": kind, "experts": rng.choice([32, 128]), "layers": rng.randint(1, 4)}
    if kind == "attn_decode":
        return {"kind": kind, "position": _log(rng, 1, 4096) - 1, "layers": 2 * rng.randint(1, 12)}
    if kind == "projection":
        rows, cols = rng.choice([(QKV_ROWS, N), (N, Q_WIDTH)])
        return {"kind": kind, "rows": rows, "cols": cols, "tokens": _log(rng, 1, 512), "residual": cols == Q_WIDTH}
    if kind == "attn_prompt":
        return {"kind": kind, "first": rng.choice([0, rng.randint(1, 1536)]), "tokens": _log(rng, 1, 512), "layers": 2}
    if kind == "moe_prompt":
        return {"kind": kind, "experts": rng.choice([32, 32, 128]), "tokens": _log(rng, 1, 512)}
    if kind == "experts":
        return {"kind": kind, "experts": 32, "tokens": _log(rng, 1, 512),
                "dtype": rng.choice(["bf16", "bf16_mxfp8", "f32", "f32_mxfp8"]), "balanced": False}
    if kind == "forward":
        return {"kind": kind, "layers": 2 * rng.randint(1, 12), "position": _log(rng, 1, 4096) - 1}
    return {"kind": kind, "layers": 2 * rng.randint(1, 6), "tokens": _log(rng, 2, 2048)}


# ---- inputs from a seed ----------------------------------------------------------------


class _Rng:
    """Values of one seed on the GPU, in a fixed order."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed) * 1000003 + 17)

    def normal(self, *shape, sigma=1.0, mean=0.0):
        return torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32) * sigma + mean

    def ints(self, lo, hi, *shape, dtype=torch.int32):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=dtype)

    def mxfp4(self, experts, rows):
        """GGUF MXFP4 blocks: an E8M0 byte, then 16 bytes of E2M1 codes."""
        b = self.ints(0, 256, experts, rows, N // 32, 17, dtype=torch.uint8)
        b[..., 0] = self.ints(EMIN, EMAX + 1, experts, rows, N // 32, dtype=torch.uint8)
        return b

    def q8(self, rows, cols):
        """GGUF Q8_0 blocks: an fp16 scale, then 32 int8; rms about 0.02."""
        b = self.ints(0, 256, rows, cols // 32, 34, dtype=torch.uint8)
        d = (self.normal(rows, cols // 32, sigma=0.1, mean=1.0).abs() * 2.7e-4).to(torch.float16)
        b[..., :2] = d.view(torch.uint8).view(rows, cols // 32, 2)
        return b


def _moe_tensors(r, experts):
    return {
        "router": r.normal(experts, N, sigma=0.02), "router_b": r.normal(experts, sigma=0.1),
        "gate": r.mxfp4(experts, N), "up": r.mxfp4(experts, N), "down": r.mxfp4(experts, N),
        "gate_b": r.normal(experts, N, sigma=0.1), "up_b": r.normal(experts, N, sigma=0.1),
        "down_b": r.normal(experts, N, sigma=0.1), "norm": r.normal(N, sigma=0.05, mean=1.0),
    }


def _routing(r, case):
    n, experts = case["tokens"], case["experts"]
    if case["balanced"]:
        # every expert equally often, each token's experts distinct
        base = torch.randperm(n, generator=r.g, device="cuda") % experts
        idx = (base[:, None] + (experts // USED) * torch.arange(USED, device="cuda")[None, :]) % experts
    else:
        idx = r.normal(n, experts).argsort(dim=1)[:, :USED]
    return idx.to(torch.int32).contiguous(), torch.softmax(r.normal(n, USED), 1).contiguous()


def _inputs(case, seed):
    """The case's inputs as torch tensors on the GPU (weights as GGUF bytes)."""
    r, k = _Rng(seed), case["kind"]
    if k == "matvec":
        return {"w": r.mxfp4(case["matrices"], case["rows"]),
                "b": r.normal(case["matrices"], case["rows"], sigma=0.1) if case["bias"] else None, "x": r.normal(N)}
    if k == "moe_decode":
        return {"layers": [_moe_tensors(r, case["experts"]) for _ in range(case["layers"])],
                "x": r.normal(case["layers"], N, sigma=2.0)}
    if k == "attn_decode":
        # a cache with room past the position, as a program allocates it
        cap = (case["position"] + 1 + 64 + 63) // 64 * 64
        return {"capacity": cap, "q": r.normal(case["layers"], HEADS, HEAD),
                "k": r.normal(case["layers"], cap, KV_HEADS, HEAD), "v": r.normal(case["layers"], cap, KV_HEADS, HEAD),
                "sinks": r.normal(case["layers"], HEADS)}
    if k == "projection":
        return {"w": r.q8(case["rows"], case["cols"]), "b": r.normal(case["rows"], sigma=0.1),
                "x": r.normal(case["tokens"], case["cols"]),
                "res": r.normal(case["tokens"], case["rows"]) if case["residual"] else None}
    if k == "attn_prompt":
        cap = case["first"] + case["tokens"]
        return {"capacity": cap, "q": r.normal(case["layers"], case["tokens"], HEADS, HEAD),
                "k": r.normal(case["layers"], cap, KV_HEADS, HEAD), "v": r.normal(case["layers"], cap, KV_HEADS, HEAD),
                "sinks": r.normal(case["layers"], HEADS)}
    if k == "moe_prompt":
        return {"layer": _moe_tensors(r, case["experts"]), "x": r.normal(case["tokens"], N)}
    assert k == "experts"
    t = _moe_tensors(r, case["experts"])
    x = r.normal(case["tokens"], N)
    idx, w = _routing(r, case)
    return {"layer": t, "x": x.to(torch.bfloat16) if case["dtype"].startswith("bf16") else x, "idx": idx, "wts": w}


# ---- what a program holds, and one pass ---------------------------------------------------


class _Ptr:
    """A torch tensor as the wrapper's buffer arguments see one."""

    def __init__(self, t):
        self.t = t
        self.ptr = t.data_ptr()
        self.nbytes = t.numel() * t.element_size()

    @property
    def p(self):
        return C.c_void_p(self.ptr)


_DEV = []


def _device():
    if not _DEV:
        _DEV.append(ttlab_amd.Device(0))
    return _DEV[0]


def _check(rc):
    if rc != 0:
        raise ttlab_amd.TtlError(ttlab_amd.load_library().ttl_last_error().decode())


def _mxfp4(dev, t):
    h = C.c_void_p()
    _check(dev.lib.ttl_mxfp4_upload_dev(dev.ctx, t.data_ptr(), t.shape[1], N, t.shape[0], C.byref(h)))
    return ttlab_amd.Mxfp4(dev, h.value)


class _State:
    """The case's handles and buffers; device handles are given back with the state."""

    def __init__(self):
        self.handles, self.model = [], None

    def __del__(self):
        for h in self.handles:
            h.free()
        if self.model is not None:
            self.model.close()


def _layer(dev, st, t, norm):
    desc = ttlab_amd.MoeLayerDesc()
    desc.hidden = desc.expert_hidden = N
    desc.experts, desc.used = t["gate"].shape[0], USED
    for name in ("gate", "up", "down"):
        h = _mxfp4(dev, t.pop(name))
        st.handles.append(h)
        setattr(desc, name, h.handle)
    desc.router_weight, desc.router_bias = t["router"].data_ptr(), t["router_b"].data_ptr()
    desc.gate_bias, desc.up_bias, desc.down_bias = (t[n].data_ptr() for n in ("gate_b", "up_b", "down_b"))
    if norm:
        desc.input_norm, desc.input_norm_epsilon = t["norm"].data_ptr(), EPS
    st.handles[-1].keep = t  # the f32 tensors live as long as the layer
    return desc


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, device="cuda", dtype=dtype)


def prepare(case, seed):
    st, k = _State(), case["kind"]
    st.case = case
    if k in ("forward", "prompt"):
        # the model with the generator's weights for this seed
        tokens = case["position"] + 1 if k == "forward" else case["tokens"]
        st.model = ttlab_amd.Model(layers=case["layers"], experts=32, vocab=VOCAB, capacity=(tokens + 64 + 63) // 64 * 64,
                                   seed=0x77000003 + int(seed))
        rng = np.random.RandomState(int(seed) % (1 << 32))
        if k == "forward":
            if case["position"]:
                st.model.fill_kv_synthetic(case["position"], 0x78000300 + int(seed))
            st.token = int(rng.randint(VOCAB))
        else:
            st.tokens = rng.randint(0, VOCAB, case["tokens"]).astype(np.int32)
        return st
    dev = st.dev = _device()
    t = _inputs(case, seed)
    torch.cuda.synchronize()  # the library works on a stream of its own
    if k == "matvec":
        st.w = _mxfp4(dev, t.pop("w"))
        st.handles.append(st.w)
        st.out = _empty(case["matrices"], case["rows"])
        st.bias = None if t["b"] is None else _Ptr(t["b"])
        st.x, st.y = _Ptr(t["x"]), [_Ptr(row) for row in st.out]
    elif k == "moe_decode":
        st.layers = [_layer(dev, st, lt, True) for lt in t.pop("layers")]
        n = len(st.layers)
        st.out = [_empty(n, N), _empty(n, USED, dtype=torch.int32), _empty(n, USED)]
        st.args = [tuple(_Ptr(b[i]) for b in [t["x"]] + st.out) for i in range(n)]
    elif k == "attn_decode":
        st.out = _empty(case["layers"], HEADS, HEAD)
        st.position = _Ptr(torch.tensor([case["position"]], dtype=torch.int32, device="cuda"))
        st.ws = _Ptr(_empty(max(1, dev.lib.ttl_attention_workspace_bytes(t["capacity"]) // 4)))
        st.args = [tuple(_Ptr(b[i]) for b in (t["q"], t["k"], t["v"], t["sinks"], st.out))
                   for i in range(case["layers"])]
    elif k == "projection":
        h = C.c_void_p()
        _check(dev.lib.ttl_q8_upload_dev(dev.ctx, t["w"].data_ptr(), case["rows"], case["cols"], None, C.byref(h)))
        dev.sync()
        st.w = ttlab_amd.Q8(dev, h.value, case["rows"], case["cols"])
        st.handles.append(st.w)
        del t["w"]
        st.ws = _empty(dev.lib.ttl_matmul_q8_0_workspace_bytes(case["tokens"], case["cols"]), dtype=torch.uint8)
        st.out = _empty(case["tokens"], case["rows"])
    elif k == "attn_prompt":
        st.out = _empty(case["layers"], case["tokens"], HEADS, HEAD)
        st.args = [tuple(_Ptr(b[i]) for b in (t["q"], t["k"], t["v"], t["sinks"])) + (_Ptr(st.out[i]),)
                   for i in range(case["layers"])]
    elif k == "moe_prompt":
        st.layer = _layer(dev, st, t.pop("layer"), False)
        st.ws = _empty(dev.lib.ttl_moe_prefill_batch_workspace_bytes(case["tokens"], case["experts"], USED),
                       dtype=torch.uint8)
        st.out = [_empty(case["tokens"], N), _empty(case["tokens"], USED, dtype=torch.int32),
                  _empty(case["tokens"], USED)]
    else:
        st.layer = _layer(dev, st, t.pop("layer"), False)
        st.dtype = {"f32": ttlab_amd.TTL_DTYPE_F32, "bf16": ttlab_amd.TTL_DTYPE_BF16,
                    "f32_mxfp8": ttlab_amd.TTL_DTYPE_F32_AS_MXFP8,
                    "bf16_mxfp8": ttlab_amd.TTL_DTYPE_BF16_AS_MXFP8}[case["dtype"]]
        st.ws = _Ptr(_empty(dev.moe_prefill_workspace_bytes(case["tokens"], case["experts"], USED, st.dtype),
                            dtype=torch.uint8))
        st.out = _empty(case["tokens"], N)
        st.x, st.idx, st.wts, st.y = _Ptr(t["x"]), _Ptr(t["idx"]), _Ptr(t["wts"]), _Ptr(st.out)
    st.t = t
    torch.cuda.synchronize()
    return st


def run(st):
    case, k = st.case, st.case["kind"]
    if k == "forward":
        return st.model.forward(st.token, case["position"])
    if k == "prompt":
        return st.model.prefill(st.tokens)
    dev, lib = st.dev, st.dev.lib
    if k == "matvec":
        for e in range(case["matrices"]):
            dev.matvec_mxfp4(st.w, st.bias, st.x, st.y[e], e)
    elif k == "moe_decode":
        for desc, (x, out, idx, wts) in zip(st.layers, st.args):
            dev.moe_decode(desc, x, out, idx, wts)
    elif k == "attn_decode":
        for i, (q, kc, vc, sinks, out) in enumerate(st.args):
            dev.attention_decode(q, kc, vc, sinks, st.position, st.t["capacity"], i, st.ws, out)
    elif k == "projection":
        t = st.t
        _check(lib.ttl_matmul_q8_0(dev.ctx, st.w.handle, t["b"].data_ptr(), t["x"].data_ptr(), case["tokens"],
                                   t["res"].data_ptr() if case["residual"] else None, st.out.data_ptr(),
                                   st.ws.data_ptr(), st.ws.numel()))
    elif k == "attn_prompt":
        for i, (q, kc, vc, sinks, out) in enumerate(st.args):
            dev.attention_prefill(q, kc, vc, sinks, case["first"], case["tokens"], st.t["capacity"], i, out)
    elif k == "moe_prompt":
        _check(lib.ttl_moe_prefill(dev.ctx, C.byref(st.layer), st.t["x"].data_ptr(), case["tokens"],
                                   st.out[0].data_ptr(), st.out[1].data_ptr(), st.out[2].data_ptr(), st.ws.data_ptr(),
                                   st.ws.numel()))
    else:
        dev.moe_prefill_experts(st.layer, st.x, st.dtype, case["tokens"], st.idx, st.wts, st.y, st.ws)
    return st.out


# ---- the least a pass needs ------------------------------------------------------------------

MX_ROW, Q8_ROW = N // 32 * 17, N // 32 * 34   # bytes of one 2880-wide MXFP4 / Q8_0 row


def _span(position, layer):
    return min(position + 1, WINDOW) if layer % 2 == 0 else position + 1


def _moe_work(n, experts, router=True):
    """(bytes, flops) of n tokens through one MoE layer; the experts that n tokens hit in
    expectation under even routing (all of them for a balanced batch)."""
    hit = experts * (1.0 - (1.0 - USED / experts) ** n)
    b = hit * (3 * N * MX_ROW + 3 * N * 4) + n * N * 8
    f = n * USED * 3 * 2.0 * N * N
    if router:
        b += experts * (N + 1) * 4
        f += n * 2.0 * experts * N
    return b, f


def _attn_work(first, n, layer):
    spans = sum(_span(first + i, layer) for i in range(n))
    lo = first + 1 - _span(first, layer)
    return (first + n - lo) * KV_HEADS * HEAD * 8 + n * HEADS * HEAD * 8, spans * HEADS * HEAD * 4.0


def work(case):
    k = case["kind"]
    if k == "matvec":
        m, r = case["matrices"], case["rows"]
        return {"bytes": m * r * (MX_ROW + 4 + (4 if case["bias"] else 0)) + N * 4, "flops": 2.0 * m * r * N}
    if k == "moe_decode":
        b, f = _moe_work(1, case["experts"])
        return {"bytes": case["layers"] * (b + N * 4), "flops": case["layers"] * f}
    if k == "attn_decode":
        w = [_attn_work(case["position"], 1, i) for i in range(case["layers"])]
        return {"bytes": sum(b for b, _ in w), "flops": sum(f for _, f in w)}
    if k == "projection":
        n, r, c = case["tokens"], case["rows"], case["cols"]
        return {"bytes": r * c // 32 * 34 + 4 * r + 4 * n * (c + r * (2 if case["residual"] else 1)),
                "flops": 2.0 * n * r * c}
    if k == "attn_prompt":
        w = [_attn_work(case["first"], case["tokens"], i) for i in range(case["layers"])]
        return {"bytes": sum(b for b, _ in w), "flops": sum(f for _, f in w)}
    if k == "moe_prompt":
        b, f = _moe_work(case["tokens"], case["experts"])
        return {"bytes": b, "flops": f}
    if k == "experts":
        b, f = _moe_work(case["tokens"], case["experts"], router=False)
        return {"bytes": b, "flops": f}
    n = 1 if k == "forward" else case["tokens"]
    first = case["position"] if k == "forward" else 0
    proj = QKV_ROWS * Q8_ROW + N * (Q_WIDTH // 32 * 34) + 4 * (QKV_ROWS + N)
    b, f = VOCAB * N * 2 + VOCAB * 4 + n * Q8_ROW, 2.0 * VOCAB * N
    for i in range(case["layers"]):
        mb, mf = _moe_work(n, 32)
        ab, af = _attn_work(first, n, i)
        # keys and values are read where the pass did not make them itself, and written
        b += mb - n * N * 8 + proj + first * KV_HEADS * HEAD * 8 * (1 if i % 2 else 0) + n * KV_HEADS * HEAD * 8
        f += mf + af + n * 2.0 * (QKV_ROWS * N + N * Q_WIDTH)
    return {"bytes": b, "flops": f}


def tolerance(case):
    # relative 2-norm between two correct 32-bit computations with their sums in another
    # order: about four times what a pass differs from exact() by, never below 2e-6
    k = case["kind"]
    if k in ("matvec", "projection", "attn_decode", "attn_prompt"):
        return {"rel": 3e-6, "max": 1e-4}
    if k in ("moe_decode", "moe_prompt"):
        # the routing's indices are whole numbers and exact
        return {"rel": 5e-6, "max": 2e-4}
    if k == "experts":
        if case["dtype"].endswith("mxfp8"):
            # the hidden is rounded to 3 fraction bits: a value whose sum lies at a
            # rounding boundary moves by a whole step
            return {"rel": 1e-2, "max": 0.2}
        return {"rel": 5e-6, "max": 2e-4}
    # whole models: a change in the last bits travels through every later layer and now and
    # then swaps two experts whose router logits nearly tie.  The prefill and the decode
    # steps over the same tokens, two correct orders of the same sums, gave logits 2e-4 to
    # 2.3e-3 apart (64 to 700 tokens).
    return {"rel": 9e-3, "max": 5e-2}


# ---- 64-bit values ------------------------------------------------------------------------------

_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _dq_mxfp4(blocks):
    """GGUF MXFP4 rows [rows][90][17] in 64 bits [rows][2880]: code byte j holds elements j
    (low nibble) and j + 16."""
    table = torch.tensor(_E2M1 + tuple(-v for v in _E2M1), dtype=torch.float64, device=blocks.device)
    scale = torch.exp2(blocks[..., 0].double() - 127.0)
    codes = blocks[..., 1:].long()
    v = torch.cat([table[codes & 15], table[codes >> 4]], dim=-1)
    return (v * scale[..., None]).reshape(blocks.shape[0], -1)


def _dq_q8(blocks):
    d = blocks[..., :2].contiguous().view(torch.float16).double()
    return (blocks[..., 2:].contiguous().view(torch.int8).double() * d).reshape(blocks.shape[0], -1)


def _swiglu(gate, up):
    x, y = torch.clamp(gate, max=7.0), torch.clamp(up, -7.0, 7.0)
    return x / (1.0 + torch.exp(-1.702 * x)) * (y + 1.0)


def _mxfp8(x):
    """Rows of 2880 as E4M3 times a power of two per 32 values (the smallest at which the
    block's largest magnitude is at most 448), nearest even, in 64 bits."""
    b = x.reshape(x.shape[0], -1, 32)
    m = b.abs().amax(-1, keepdim=True)
    f, e = torch.frexp(m)  # m = f 2^e with f in [0.5, 1): the exponent is e - 1
    ex = torch.where(m > 0, e - 9 + (f > 0.875).to(e.dtype), torch.zeros_like(e)).clamp(min=-127)
    s = torch.ldexp(b, -ex)
    _, es = torch.frexp(s)
    step = torch.exp2(torch.clamp(es - 1, min=-6).double() - 3.0)
    return torch.ldexp(torch.round(s / step) * step, ex).reshape(x.shape)


def _experts64(t, x, idx, wts, quant=None):
    """Expert order, as the batch sums them."""
    out = torch.zeros(x.shape[0], N, dtype=torch.float64, device="cuda")
    xq = quant(x) if quant else x
    for e in range(t["gate"].shape[0]):
        tok, rank = (idx == e).nonzero(as_tuple=True)
        if tok.numel() == 0:
            continue
        xe = xq[tok]
        g = xe @ _dq_mxfp4(t["gate"][e]).T.contiguous() + t["gate_b"][e].double()
        u = xe @ _dq_mxfp4(t["up"][e]).T.contiguous() + t["up_b"][e].double()
        h = _swiglu(g, u)
        if quant:
            h = quant(h)
        d = h @ _dq_mxfp4(t["down"][e]).T.contiguous() + t["down_b"][e].double()
        out.index_add_(0, tok, d * wts[tok, rank].double()[:, None])
    return out


def _route64(t, x):
    top, idx = (x @ t["router"].double().T.contiguous() + t["router_b"].double()).topk(USED, dim=1)
    return idx, torch.softmax(top, 1)


def _attn64(q, kc, vc, sinks, first, layer):
    """q [n][64][64] at positions first ..; softmax with the head's sink in the denominator."""
    n = q.shape[0]
    kd, vd = kc[:first + n].double(), vc[:first + n].double()
    pos = torch.arange(first + n, device="cuda")[None, :]
    at = first + torch.arange(n, device="cuda")[:, None]
    mask = (pos > at) | ((pos <= at - WINDOW) if layer % 2 == 0 else torch.zeros_like(pos > at))
    out = torch.empty(n, HEADS, HEAD, dtype=torch.float64, device="cuda")
    for h in range(HEADS):
        g = h // (HEADS // KV_HEADS)
        s = (q[:, h].double() @ kd[:, g].T.contiguous()) / 8.0
        s = torch.cat([s.masked_fill(mask, -math.inf), sinks[h].double().expand(n, 1)], 1)
        out[:, h] = torch.softmax(s, 1)[:, :-1] @ vd[:, g].contiguous()
    return out


def exact(case, seed):
    k = case["kind"]
    if k in ("forward", "prompt"):
        # the weights are the framework's own generator's, and 24 layers of them in 64 bits
        # take longer than a check should
        return None
    t = _inputs(case, seed)
    if k == "matvec":
        x = t["x"].double()
        y = torch.stack([_dq_mxfp4(w) @ x for w in t["w"]])
        return y if t["b"] is None else y + t["b"].double()
    if k == "moe_decode":
        outs, wts = [], []
        for i, lt in enumerate(t["layers"]):
            x = t["x"][i:i + 1].double()
            x = x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * lt["norm"].double()
            idx, w = _route64(lt, x)
            outs.append(_experts64(lt, x, idx, w))
            wts.append(w)
        return [torch.cat(outs), None, torch.cat(wts)]
    if k == "attn_decode":
        return torch.cat([_attn64(t["q"][i:i + 1], t["k"][i], t["v"][i], t["sinks"][i], case["position"], i)
                          for i in range(case["layers"])])
    if k == "projection":
        y = t["x"].double() @ _dq_q8(t["w"]).T.contiguous() + t["b"].double()
        return y if t["res"] is None else y + t["res"].double()
    if k == "attn_prompt":
        return torch.stack([_attn64(t["q"][i], t["k"][i], t["v"][i], t["sinks"][i], case["first"], i)
                            for i in range(case["layers"])])
    x = t["x"].double()
    if k == "moe_prompt":
        idx, w = _route64(t["layer"], x)
        return [_experts64(t["layer"], x, idx, w), None, w]
    return _experts64(t["layer"], x, t["idx"], t["wts"], _mxfp8 if case["dtype"].endswith("mxfp8") else None)
