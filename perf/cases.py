"""The work that a user of this framework has it do, as cases that can be timed and compared.

Every case goes through the session layer of the C ABI (``include/mnb_hip.h``), the way the ONNX
Runtime plugin runs a node: constants uploaded (and laid out) once, activations and results in
device memory, calls ordered on the session's stream and returning once enqueued.

Kinds
  norm     the two RMSNorms of a decoder layer (SkipSimplifiedLayerNormalization with the residual
           sum, SimplifiedLayerNormalization without)
  linear   MatMulNBits nodes: 4- or 8-bit weights, blocks of 16 to 128, with or without zero
           points, fp16 or fp32 activations, accuracy_level 0 or 4 (int8 activations)
  qmoe     one fused mixture-of-experts block: routing, int4 experts with SwiGLU, combine
  gqa      one attention node: rotary embedding, append to the KV cache, causal attention

Sizes: the Phi-3.5-mini layer, the gpt-oss expert block, the accuracy_level 4 node and the head
layouts of this repository's benchmark and tests, and generic ones around them.
"""

import ctypes
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "onnxruntime-ep-vulkan_amd"))
import mnb  # noqa: E402

# (K, N) of the Phi-3.5-mini decoder layer's nodes: qkv, o, gate_up, down
LAYER = "3072x9216,3072x3072,3072x16384,8192x3072"


def _linear(name, m, nodes, layers=1, bits=4, block=32, zp=True, dtype="f16", level=0):
    case = {"kind": "linear", "m": m, "nodes": nodes, "layers": layers, "bits": bits,
            "block": block, "zp": zp, "dtype": dtype, "level": level}
    return dict(case, name=name) if name else case


def _norm(name, rows, hidden, dtype="f16"):
    case = {"kind": "norm", "rows": rows, "hidden": hidden, "dtype": dtype}
    return dict(case, name=name) if name else case


def _qmoe(name, tokens, hidden, inter, experts, k, block=32, fusion=1):
    case = {"kind": "qmoe", "tokens": tokens, "hidden": hidden, "inter": inter,
            "experts": experts, "k": k, "block": block, "fusion": fusion}
    return dict(case, name=name) if name else case


def _gqa(name, batch, seq, past, arena, nq, nkv, d):
    """``arena``: extent of a KV buffer updated in place; 0: a new present of past + seq."""
    case = {"kind": "gqa", "batch": batch, "seq": seq, "past": past, "arena": arena, "nq": nq,
            "nkv": nkv, "d": d}
    return dict(case, name=name) if name else case


def listed():
    return [
        # the smallest calls of a token: one row through the two norms of a layer
        _norm("norm_token", 1, 3072),
        # one token of one sequence: four layers' linears, weights streamed once
        _linear("linear_token", 1, LAYER, layers=4),
        # a few sequences decoded together
        _linear("linear_batch", 8, LAYER, layers=4),
        # a larger decode batch, or a draft of several tokens for several sequences
        _linear("linear_batch_large", 48, LAYER, layers=4),
        # the whole prompt of a request through one layer
        _linear("linear_prompt", 2048, LAYER),
        # a short prompt of odd length on a model quantised to 8 bits without zero points
        _linear("linear_prompt_8bit", 333, "2880x2880,2880x5760", bits=8, block=64, zp=False),
        # int8 activations (accuracy_level 4): a decode batch on one node with 128-blocks
        _linear("int8_batch", 16, "8192x3072", layers=4, block=128, level=4),
        # int8 activations: a prompt
        _linear("int8_prompt", 512, "3072x8192", level=4),
        # mixture of experts: a decode batch, nearly every expert routed to
        _qmoe("experts_batch", 64, 2880, 2880, 32, 4),
        # mixture of experts: a prompt
        _qmoe("experts_prompt", 1024, 2880, 2880, 32, 4),
        # attention of a decode batch over long, ragged caches updated in place
        _gqa("attention_token", 8, 1, 3500, 4096, 32, 8, 128),
        # attention of a prompt without a past
        _gqa("attention_prompt", 1, 2048, 0, 0, 32, 32, 96),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["norm", "linear", "linear", "linear8", "linear32", "int8", "qmoe", "gqa",
                       "gqa"])
    if kind == "norm":
        dtype = rng.choice(["f16", "f16", "f32"])
        hidden = 8 * rng.randint(64, 1024 if dtype == "f16" else 512)
        return _norm(None, _log(rng, 1, 4096), hidden, dtype)
    if kind in ("linear", "int8", "linear32", "linear8"):
        block = rng.choice([32, 32, 64, 128] + ([16] if kind == "linear8" else []))
        k = 256 * rng.randint(4, 32) if rng.random() < 0.7 else max(64, block) * rng.randint(5, 36)
        if kind == "linear" and block == 32 and rng.random() < 0.2:
            k += 32                                      # a last group of one block
        n = 128 * rng.randint(4, 64) if rng.random() < 0.6 else rng.randint(300, 6000)
        m = _log(rng, 1, 256 if kind == "linear32" else 2048)
        return _linear(None, m, "%dx%d" % (k, n), layers=2 if m <= 16 else 1,
                       bits=8 if kind == "linear8" else 4, block=block, zp=rng.random() < 0.6,
                       dtype="f32" if kind == "linear32" else "f16",
                       level=4 if kind == "int8" else 0)
    if kind == "qmoe":
        experts, k = rng.choice([(32, 4), (8, 2), (16, 2), (64, 6)])
        block = rng.choice([32, 32, 64])
        return _qmoe(None, _log(rng, 1, 1024), 64 * rng.randint(12, 45), 64 * rng.randint(8, 45),
                     experts, k, block, rng.choice([1, 1, 2]))
    nq, nkv, d = rng.choice([(32, 8, 128), (32, 32, 96), (8, 2, 64), (16, 16, 128), (64, 8, 64)])
    if rng.random() < 0.5:                               # decode, or a few drafted tokens
        batch = _log(rng, 1, 16)
        past = _log(rng, 64, 4000)
        seq = rng.choice([1, 1, 1, 2, 4])
        arena = past + seq + rng.randint(0, 512)
    else:                                                # a prompt, or a chunk of one
        batch, seq = rng.choice([1, 1, 2]), _log(rng, 16, 1500)
        past = rng.choice([0, 0, _log(rng, 32, 1024)])
        arena = past + seq + rng.randint(0, 300) if rng.random() < 0.5 else 0
    return _gqa(None, batch, seq, past, arena, nq, nkv, d)


# ---- the session and the handles a program keeps --------------------------------------------

_kept = {}


def _session():
    """The process's one session: device-only calls return once enqueued on its stream."""
    if "s" not in _kept:
        s = ctypes.c_void_p()
        mnb.check(mnb.load().mnb_session_create(0, ctypes.byref(s)))
        mnb.check(mnb.load().mnb_session_set_async(s, 1))
        _kept["s"] = s
    return _kept["s"]


class _Handle:
    """A weights handle, released with its owner."""

    def __init__(self, release):
        self.h, self._release = ctypes.c_void_p(), release

    def __del__(self):
        if self.h:
            self._release(self.h)


def _up(t):
    """(pointer, bytes) of a tensor's host copy, with the tensor that keeps it alive."""
    t = t.cpu().contiguous()
    return t, ctypes.c_void_p(t.data_ptr()), t.numel() * t.element_size()


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _dt(case):
    return torch.float32 if case.get("dtype") == "f32" else torch.float16


def _nodes(case):
    return [tuple(int(v) for v in n.split("x")) for n in case["nodes"].split(",")]


def _quantised(gen, n, k, bits, block, zp, dtype, experts=None):
    """Codes, scales and zero points as a quantiser leaves roughly normal weights: codes gathered
    about the zero point, scales within a factor of three of one another."""
    lead = (n,) if experts is None else (experts, n)
    mid, top = 1 << (bits - 1), (1 << bits) - 1
    spread = (mid - 1) / 3.0
    codes = torch.randn(*lead, k // block, block, device="cuda", generator=gen).mul_(spread)
    codes = codes.add_(mid).round_().clamp_(0, top).to(torch.uint8)
    if bits == 4:
        codes = codes[..., 0::2] | (codes[..., 1::2] << 4)
    scales = torch.rand(*lead, k // block, device="cuda", generator=gen)
    scales = ((0.5 + scales) * (1.2 / (spread * math.sqrt(k)))).to(dtype)
    zeros = None
    if zp:
        z = torch.randint(mid - 1, mid + 2, (n, k // block), device="cuda", generator=gen)
        z = z.to(torch.uint8)
        if bits == 4:
            if z.shape[1] % 2:
                z = torch.cat([z, torch.zeros(n, 1, dtype=torch.uint8, device="cuda")], 1)
            z = z[:, 0::2] | (z[:, 1::2] << 4)
        zeros = z.contiguous()
    return codes.contiguous(), scales, zeros


def _linear_data(case, seed):
    gen, dtype, out = _gen(seed), _dt(case), []
    for _ in range(case["layers"]):
        for k, n in _nodes(case):
            w = _quantised(gen, n, k, case["bits"], case["block"], case["zp"], dtype)
            a = torch.randn(case["m"], k, device="cuda", generator=gen).to(dtype)
            out.append((k, n, w, a))
    return out


def _norm_data(case, seed):
    gen, dtype = _gen(seed), _dt(case)
    r, h = case["rows"], case["hidden"]

    def rnd(*shape):
        return torch.randn(*shape, device="cuda", generator=gen)

    return {"x": rnd(r, h).to(dtype), "skip": (2.0 * rnd(r, h)).to(dtype),
            "g1": (1.0 + 0.2 * rnd(h)).to(dtype), "g2": (1.0 + 0.2 * rnd(h)).to(dtype)}


def _qmoe_data(case, seed):
    gen = _gen(seed)
    h, i, e, block = case["hidden"], case["inter"], case["experts"], case["block"]
    w1, s1, _ = _quantised(gen, 2 * i, h, 4, block, False, torch.float16, e)
    w2, s2, _ = _quantised(gen, h, i, 4, block, False, torch.float16, e)
    b1 = (0.1 * torch.randn(e, 2 * i, device="cuda", generator=gen)).to(torch.float16)
    b2 = (0.1 * torch.randn(e, h, device="cuda", generator=gen)).to(torch.float16)
    x = torch.randn(case["tokens"], h, device="cuda", generator=gen).to(torch.float16)
    logits = torch.randn(case["tokens"], e, device="cuda", generator=gen).to(torch.float16)
    return {"w1": w1, "s1": s1, "b1": b1, "w2": w2, "s2": s2, "b2": b2, "x": x, "logits": logits}


def _gqa_data(case, seed):
    gen = _gen(seed)
    b, s, nq, nkv, d = case["batch"], case["seq"], case["nq"], case["nkv"], case["d"]
    qkv = torch.randn(b, s, (nq + 2 * nkv) * d, device="cuda", generator=gen).to(torch.float16)
    extent = case["arena"] or case["past"]
    pk = torch.randn(b, nkv, extent, d, device="cuda", generator=gen).to(torch.float16)
    pv = torch.randn(b, nkv, extent, d, device="cuda", generator=gen).to(torch.float16)
    # ragged: the first sequence has the whole past, the others between a quarter and all of it
    past = torch.rand(b, device="cuda", generator=gen).mul_(0.75).add_(0.25).mul_(case["past"])
    past = past.long()
    past[0] = case["past"]
    if not case["arena"]:
        past[:] = case["past"]
    pos = torch.arange(case["past"] + s, device="cuda", dtype=torch.float64)
    inv = 10000.0 ** (-torch.arange(0, d, 2, device="cuda", dtype=torch.float64) / d)
    angle = pos[:, None] * inv[None]
    return {"qkv": qkv, "pk": pk, "pv": pv, "past": past, "seqlens": (past + s - 1).int(),
            "cos": angle.cos().half(), "sin": angle.sin().half()}


# ---- prepare and run ------------------------------------------------------------------------

def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def _prepare_linear(case, seed):
    lib, s, calls, outs = mnb.load(), _session(), [], []
    for k, n, (b, sc, z), a in _linear_data(case, seed):
        p = mnb.problem(0, n, k, case["bits"], case["block"], case["zp"],
                        mnb.DTYPE_F32 if case["dtype"] == "f32" else mnb.DTYPE_F16, case["level"])
        w = _Handle(lib.mnb_weights_release)
        (hb, pb, nb), (hs, ps, ns) = _up(b), _up(sc)
        hz, pz, nz = _up(z) if z is not None else (None, None, 0)
        mnb.check(lib.mnb_weights_upload(s, ctypes.byref(p), pb, nb, ps, ns, pz, nz,
                                         ctypes.byref(w.h)))
        rc = lib.mnb_weights_prepack(w.h, None)          # as the plugin does at Compile
        if rc != mnb.MNB_ERR_UNSUPPORTED:
            mnb.check(rc)
        y = torch.empty(case["m"], n, dtype=a.dtype, device="cuda")
        calls.append((w, a, y, ctypes.c_void_p(a.data_ptr()), ctypes.c_void_p(y.data_ptr())))
        outs.append(y)
    return {"kind": "linear", "m": case["m"], "calls": calls, "outs": outs}


def _run_linear(state):
    run_device, s, m = mnb.load().mnb_session_run_device, _session(), state["m"]
    for w, _, _, pa, py in state["calls"]:
        mnb.check(run_device(s, w.h, m, pa, py))
    return state["outs"]


def _prepare_norm(case, seed):
    lib, s, d = mnb.load(), _session(), _norm_data(case, seed)
    st = {"kind": "norm", "rows": case["rows"], "d": d}
    for name, gamma, skip in (("w1", "g1", 1), ("w2", "g2", 0)):
        p = mnb.RmsNormProblem(0, case["hidden"], 1e-5, skip, 0, skip,
                               mnb.DTYPE_F32 if case["dtype"] == "f32" else mnb.DTYPE_F16)
        w = _Handle(lib.mnb_rmsnorm_weights_release)
        hg, pg, ng = _up(d[gamma])
        mnb.check(lib.mnb_rmsnorm_weights_upload(s, ctypes.byref(p), pg, ng, None, 0,
                                                 ctypes.byref(w.h)))
        st[name] = w
    st["y1"], st["sum"], st["y2"] = (torch.empty_like(d["x"]) for _ in range(3))
    st["p"] = [ctypes.c_void_p(t.data_ptr())
               for t in (d["x"], d["skip"], st["y1"], st["sum"], st["y2"])]
    return st


def _run_norm(state):
    f, s, r = mnb.load().mnb_session_run_rmsnorm, _session(), state["rows"]
    x, skip, y1, total, y2 = state["p"]
    mnb.check(f(s, state["w1"].h, r, x, 1, skip, 1, y1, 1, total, 1))
    mnb.check(f(s, state["w2"].h, r, total, 1, None, 0, y2, 1, None, 0))
    return [state["y1"], state["sum"], state["y2"]]


def _prepare_qmoe(case, seed):
    lib, s, d = mnb.load(), _session(), _qmoe_data(case, seed)
    p = mnb.qmoe_problem(0, case["hidden"], case["inter"], case["experts"], case["k"],
                         case["block"], case["fusion"])
    w = _Handle(lib.mnb_qmoe_weights_release)
    host = [_up(d[n]) for n in ("w1", "s1", "b1", "w2", "s2", "b2")]
    args = [v for _, ptr, size in host for v in (ptr, size)]
    mnb.check(lib.mnb_qmoe_weights_upload(s, ctypes.byref(p), 0, *args, ctypes.byref(w.h)))
    mnb.check(lib.mnb_qmoe_weights_prepack(w.h, None))   # as the plugin does at Compile
    y = torch.empty_like(d["x"])
    return {"kind": "qmoe", "tokens": case["tokens"], "w": w, "x": d["x"], "logits": d["logits"],
            "y": y, "p": [ctypes.c_void_p(t.data_ptr()) for t in (d["x"], d["logits"], y)]}


def _run_qmoe(state):
    x, logits, y = state["p"]
    mnb.check(mnb.load().mnb_session_run_qmoe(_session(), state["w"].h, state["tokens"], x, 1,
                                              logits, 1, y, 1))
    return state["y"]


def _prepare_gqa(case, seed):
    lib, s, d = mnb.load(), _session(), _gqa_data(case, seed)
    b, sq, nq, nkv, hd = case["batch"], case["seq"], case["nq"], case["nkv"], case["d"]
    extent = case["arena"] or case["past"]
    present = case["arena"] or case["past"] + sq
    shape = mnb.gqa_problem(b, sq, extent, present, int(d["cos"].shape[0]), nq, nkv, hd, hd)
    c = _Handle(lib.mnb_gqa_caches_release)
    (hc, pc, nc), (hs, ps, ns) = _up(d["cos"]), _up(d["sin"])
    mnb.check(lib.mnb_gqa_caches_upload(s, ctypes.byref(shape), pc, nc, ps, ns, ctypes.byref(c.h)))
    out = torch.empty(b, sq, nq * hd, dtype=torch.float16, device="cuda")
    if case["arena"]:
        rk, rv = d["pk"], d["pv"]
    else:
        rk = torch.empty(b, nkv, present, hd, dtype=torch.float16, device="cuda")
        rv = torch.empty_like(rk)
    p = [ctypes.c_void_p(t.data_ptr() or None)
         for t in (d["qkv"], d["pk"], d["pv"], d["seqlens"], out, rk, rv)]
    return {"kind": "gqa", "c": c, "shape": shape, "d": d, "outs": [out, rk, rv], "p": p}


_GQA_DEVICE = (mnb.GQA_ON_DEVICE_QKV | mnb.GQA_ON_DEVICE_PAST | mnb.GQA_ON_DEVICE_SEQLENS
               | mnb.GQA_ON_DEVICE_OUT | mnb.GQA_ON_DEVICE_PRESENT)


def _run_gqa(state):
    qkv, pk, pv, sl, out, rk, rv = state["p"]
    mnb.check(mnb.load().mnb_session_run_gqa(
        _session(), state["c"].h, ctypes.byref(state["shape"]), qkv, pk, pv, sl, None, None, out,
        rk, rv, _GQA_DEVICE))
    return state["outs"]


_RUN = {"linear": _run_linear, "norm": _run_norm, "qmoe": _run_qmoe, "gqa": _run_gqa}


def run(state):
    return _RUN[state["kind"]](state)


# ---- what a pass cannot do without, and what it should return -------------------------------

def _gqa_pasts(case):
    """Mean past length: the first sequence's is whole, the others' 0.625 of it on average."""
    if not case["arena"]:
        return float(case["past"])
    return case["past"] * (1.0 + 0.625 * (case["batch"] - 1)) / case["batch"]


def work(case):
    size = 4 if case.get("dtype") == "f32" else 2
    if case["kind"] == "norm":
        rows, h = case["rows"], case["hidden"]
        return {"bytes": size * (5 * rows * h + 2 * h), "flops": 8.0 * rows * h}
    if case["kind"] == "linear":
        total = flops = 0
        for k, n in _nodes(case):
            blocks = k // case["block"]
            total += n * k * case["bits"] // 8 + size * n * blocks + size * case["m"] * (k + n)
            if case["zp"]:
                total += n * ((blocks * case["bits"] + 7) // 8)
            flops += 2 * case["m"] * n * k
        return {"bytes": total * case["layers"], "flops": flops * case["layers"]}
    if case["kind"] == "qmoe":
        t, h, i, e = case["tokens"], case["hidden"], case["inter"], case["experts"]
        hit = e * (1.0 - (1.0 - case["k"] / e) ** t)     # experts that some token is routed to
        expert = 3 * h * i // 2 + 2 * 3 * h * i // case["block"] + 2 * (2 * i + h)
        return {"bytes": hit * expert + 2 * t * (2 * h + e), "flops": 6.0 * t * case["k"] * h * i}
    b, s, nq, nkv, d = case["batch"], case["seq"], case["nq"], case["nkv"], case["d"]
    past = _gqa_pasts(case)
    moved = b * s * (2 * nq + 2 * nkv) * d + 2 * b * nkv * d * (past + s)
    if not case["arena"]:
        moved += 2 * b * nkv * d * past                  # the past, copied into the new present
    return {"bytes": 2 * moved, "flops": 4.0 * b * nq * d * s * (past + (s + 1) / 2)}


def tolerance(case):
    # fp16 results: two sums that differ in their last bits round to neighbouring fp16 values now
    # and then (2^-10 of the value at most); a result's own rounding is 2^-11, 2e-4 in 2-norm.
    if case["kind"] == "qmoe":
        # three fp16 roundings in series (h, the activation, the expert outputs)
        return {"rel": 2e-3, "max": 1e-2}
    if case.get("dtype") == "f32":
        return {"rel": 1e-5, "max": 1e-4}
    if case["kind"] == "gqa":
        return {"rel": 1e-3, "max": 5e-3}
    return {"rel": 8e-4, "max": 4e-3}


def _unpack(codes, bits):
    if bits == 4:
        codes = torch.stack([codes & 15, codes >> 4], -1).flatten(-2)
    return codes


def _dequantised(w, k, bits, block, experts=False):
    codes, scales, zeros = w
    q = _unpack(codes, bits).double()                    # [.., n, blocks, block]
    if zeros is None:
        q -= 1 << (bits - 1)
    else:
        z = _unpack(zeros.unsqueeze(-1), bits).flatten(1)[:, :k // block]
        q -= z.double().unsqueeze(-1)
    return q.mul_(scales.double().unsqueeze(-1)).flatten(-2)


def exact(case, seed):
    return globals()["_exact_" + case["kind"]](case, seed)


def _exact_linear(case, seed):
    out = []
    for k, n, w, a in _linear_data(case, seed):
        x = a.double()
        if case["level"] == 4:
            # the level's definition: int8 codes of each (row, block), rounded half to even in fp32
            g = a.float().reshape(case["m"], k // case["block"], case["block"])
            top = g.abs().amax(-1, keepdim=True)
            code = (g * (127.0 / top)).round().clamp(-127, 127)
            code = torch.where(top > 0, code, torch.zeros_like(code))
            x = (code.double() * (top / 127.0).double()).reshape(case["m"], k)
        out.append(x @ _dequantised(w, k, case["bits"], case["block"]).t())
    return out


def _rms(x, gamma):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5) * gamma.double()


def _exact_norm(case, seed):
    d = _norm_data(case, seed)
    total = d["x"].double() + d["skip"].double()
    stored = total.to(_dt(case)).double()                # the second norm reads the stored sum
    return [_rms(total, d["g1"]), total, _rms(stored, d["g2"])]


def _exact_qmoe(case, seed):
    d, k, inter = _qmoe_data(case, seed), case["k"], case["inter"]
    prob = d["logits"].double().softmax(-1)
    weight, expert = prob.sort(dim=-1, descending=True, stable=True)
    weight, expert = weight[:, :k], expert[:, :k]
    weight = weight / weight.sum(-1, keepdim=True)
    x = d["x"].double()
    y = torch.zeros_like(x)
    for e in range(case["experts"]):
        row, slot = (expert == e).nonzero(as_tuple=True)
        if not row.numel():
            continue
        w1 = _dequantised((d["w1"][e], d["s1"][e], None), case["hidden"], 4, case["block"])
        w2 = _dequantised((d["w2"][e], d["s2"][e], None), inter, 4, case["block"])
        h = x[row] @ w1.t() + d["b1"][e].double()
        gate, lin = (h[:, 0::2], h[:, 1::2]) if case["fusion"] == 1 else (h[:, :inter], h[:, inter:])
        gate, lin = gate.clamp(max=7.0), lin.clamp(-7.0, 7.0)
        alpha = 1.7020000219345093                       # 1.702 as the fp32 attribute holds it
        act = gate * torch.sigmoid(alpha * gate) * (lin + 1.0)
        y.index_add_(0, row, weight[row, slot].unsqueeze(1) * (act @ w2.t() + d["b2"][e].double()))
    return y


def _exact_gqa(case, seed):
    d = _gqa_data(case, seed)
    b, s, nq, nkv, hd = case["batch"], case["seq"], case["nq"], case["nkv"], case["d"]
    present = case["arena"] or case["past"] + s
    qkv = d["qkv"].double().reshape(b, s, nq + 2 * nkv, hd)
    rk = torch.zeros(b, nkv, present, hd, dtype=torch.float64, device="cuda")
    rv = torch.zeros_like(rk)
    rk[:, :, :d["pk"].shape[2]], rv[:, :, :d["pv"].shape[2]] = d["pk"].double(), d["pv"].double()
    out = torch.empty(b, s, nq * hd, dtype=torch.float64, device="cuda")
    half = hd // 2
    for i in range(b):
        p = int(d["past"][i])
        c, sn = d["cos"][p:p + s].double().unsqueeze(1), d["sin"][p:p + s].double().unsqueeze(1)

        def turn(x):
            lo, hi = x[..., :half], x[..., half:]
            return torch.cat([lo * c - hi * sn, hi * c + lo * sn], -1)

        q = turn(qkv[i, :, :nq])
        rk[i, :, p:p + s] = turn(qkv[i, :, nq:nq + nkv]).transpose(0, 1)
        rv[i, :, p:p + s] = qkv[i, :, nq + nkv:].transpose(0, 1)
        seen = torch.arange(p + s, device="cuda")[None] <= p + torch.arange(s, device="cuda")[:, None]
        # the new keys enter the scores as they are stored
        keys, values = rk[i, :, :p + s].half().double(), rv[i, :, :p + s]
        for g in range(nkv):
            rows = slice(g * (nq // nkv), (g + 1) * (nq // nkv))
            score = q[:, rows].transpose(0, 1) @ keys[g].t() * hd ** -0.5
            score.masked_fill_(~seen, -math.inf)
            att = score.softmax(-1) @ values[g]
            out[i].reshape(s, nq, hd)[:, rows] = att.transpose(0, 1)
    return [out, rk, rv]
