"""Performance cases of the W4A16 group-128 path: what a program that uses it has it do.

Two kinds of use are covered.  Most cases are single blocks through the launcher API (qe_amd.launch_*): the MLP and
the attention layer of a prefill chunk, decode attention with its O projection, one decode projection, the LM head
with sampling.  Two are whole calls of the engine: prefill of a prompt, and a short generation.

Every case is a dict of plain values; "kind" says which path it takes:

  mlp        rows of a prefill chunk: RMSNorm, gate/up + SwiGLU, down + residual, over `layers` layers
             path "tiled" / "packed": W4A16 on the tiled copy or the .qwenbin layout, "w4a8": Q8_1 activations
  attention  rows of a prefill chunk at position `base`: RMSNorm, QKV, bias + RoPE + KV append, causal attention,
             O + residual
  decode_attention  one token at position `pos`: split flash decode over the KV cache, O + residual
             path "fused": partials, then combine inside the O projection; "plain": the separate launches
  gemv       one decode projection, fp16 activation
  head       final RMSNorm, LM head and greedy sampling of one token
  prefill    Engine.prefill of a prompt
  generate   Engine.prefill of a short prompt, then Engine.decode

Sizes are those of Qwen2.5-1.5B (hidden 1536, intermediate 8960, 12 query and 2 key/value heads of 128, vocabulary
151936), the model the engine's default configuration describes; drawn cases also take other widths the launchers
accept.
"""
from __future__ import annotations

import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "qwen-engine_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import qe_amd  # noqa: E402

H, I, V, NQ, NKV, HD = 1536, 8960, 151936, 12, 2, 128
THETA = 1000000.0
EPS = 1e-6
DEV = "cuda"


def listed():
    return [
        # one decode projection called on its own: the smallest call of the API, where launching it counts
        {"name": "gemv_gate", "kind": "gemv", "n": I, "k": H, "residual": False},
        # the last step of every generated token: the largest matrix of the model, read once
        {"name": "lm_head", "kind": "head", "vocab": V, "hidden": H},
        # a token generated deep in a long conversation: reading the KV cache dominates the layer's attention
        {"name": "decode_attn_16k", "kind": "decode_attention", "nq": NQ, "nkv": NKV, "pos": 16000, "max_seq": 32768,
         "path": "fused"},
        # a prompt of a few words: weights are read for a handful of rows
        {"name": "mlp_9", "kind": "mlp", "m": 9, "hidden": H, "inter": I, "layers": 4, "path": "packed"},
        # the prompt length of the decode benchmark
        {"name": "mlp_128", "kind": "mlp", "m": 128, "hidden": H, "inter": I, "layers": 2, "path": "tiled"},
        # a page of text, not a round number of rows
        {"name": "mlp_1000", "kind": "mlp", "m": 1000, "hidden": H, "inter": I, "layers": 1, "path": "tiled"},
        # a long document in one chunk (prefill_chunk is the caller's choice)
        {"name": "mlp_4096", "kind": "mlp", "m": 4096, "hidden": H, "inter": I, "layers": 1, "path": "tiled"},
        # the int8 prefill path on a medium prompt
        {"name": "mlp_w4a8_300", "kind": "mlp", "m": 300, "hidden": H, "inter": I, "layers": 1, "path": "w4a8"},
        # the attention layer of a medium prompt, weights as the file has them
        {"name": "attn_509", "kind": "attention", "m": 509, "base": 0, "max_seq": 4096, "nq": NQ, "nkv": NKV,
         "path": "packed"},
        # one chunk late in a long prompt: the whole cache is visible to every row
        {"name": "attn_1024_at_15k", "kind": "attention", "m": 1024, "base": 15000, "max_seq": 32768, "nq": NQ,
         "nkv": NKV, "path": "tiled"},
        # time to first token of a long prompt through the engine, in the default chunks
        {"name": "prefill_3000", "kind": "prefill", "prompt": 3000, "max_seq": 4096},
        # a short answer through the engine, the benchmark's prompt length
        {"name": "generate_128_48", "kind": "generate", "prompt": 128, "steps": 48, "max_seq": 4096},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "head", "decode_attention", "mlp", "mlp", "mlp", "attention", "attention", "prefill",
                       "generate"])
    if kind == "gemv":
        return {"kind": kind, "n": _log_int(rng, 256, 17920), "k": 128 * rng.randint(4, 72),
                "residual": rng.random() < 0.5}
    if kind == "head":
        return {"kind": kind, "vocab": _log_int(rng, 32000, V), "hidden": rng.choice([1024, 1280, H, 2048])}
    if kind == "decode_attention":
        nq, nkv = rng.choice([(NQ, NKV), (NQ, NKV), (16, 4), (8, 8)])
        return {"kind": kind, "nq": nq, "nkv": nkv, "pos": _log_int(rng, 500, 32000), "max_seq": 32768,
                "path": rng.choice(["fused", "plain"])}
    if kind == "mlp":
        path = rng.choice(["tiled", "tiled", "packed", "w4a8"])
        unit = 256 if path == "tiled" else 128
        m = _log_int(rng, 2, 4096 if path != "w4a8" else 1500)
        hidden, inter = (H, I) if rng.random() < 0.35 else (unit * rng.randint(1024 // unit, 2048 // unit),
                                                          unit * rng.randint(2048 // unit, I // unit))
        return {"kind": kind, "m": m, "hidden": hidden, "inter": inter,
                "layers": rng.choice([3, 5]) if m < 100 else 1, "path": path}
    if kind == "attention":
        nq, nkv = rng.choice([(NQ, NKV), (NQ, NKV), (16, 4), (8, 8)])
        m = _log_int(rng, 8, 2048)
        base = rng.choice([0, 0, _log_int(rng, 100, 15000)])
        while m * (base + m // 2) > 1024 * 15512:
            base //= 2
        return {"kind": kind, "m": m, "base": base, "max_seq": 32768, "nq": nq, "nkv": nkv,
                "path": rng.choice(["tiled", "packed"])}
    if kind == "prefill":
        return {"kind": kind, "prompt": _log_int(rng, 5, 3000), "max_seq": 4096}
    return {"kind": kind, "prompt": _log_int(rng, 5, 1000), "steps": rng.randint(8, 32), "max_seq": 4096}


# ---- inputs ------------------------------------------------------------------------------------------------------
class _Rand:
    def __init__(self, seed):
        self.gen = torch.Generator(device=DEV)
        self.gen.manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0):
        return (torch.randn(shape, device=DEV, generator=self.gen) * std + mean).half()

    def w4(self, n, k):
        """Packed weights and group scales that keep the variance of their input."""
        qw = torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k // 8), dtype=torch.int32, device=DEV, generator=self.gen)
        sc = (torch.randn((n, k // 128), device=DEV, generator=self.gen).abs() / math.sqrt(21.5 * k)).half()
        return qw, sc


def _mlp_inputs(c, seed):
    r = _Rand(seed)
    x = r.normal(c["m"], c["hidden"])
    layers = [{"gamma": r.normal(c["hidden"], std=0.1, mean=1.0), "gate_up": r.w4(2 * c["inter"], c["hidden"]),
               "down": r.w4(c["hidden"], c["inter"])} for _ in range(c["layers"])]
    return x, layers


def _attention_inputs(c, seed):
    r = _Rand(seed)
    hid, qd, kvd = c["nq"] * HD, c["nq"] * HD, c["nkv"] * HD
    return {"x": r.normal(c["m"], hid), "gamma": r.normal(hid, std=0.1, mean=1.0), "q": r.w4(qd, hid),
            "k": r.w4(kvd, hid), "v": r.w4(kvd, hid), "o": r.w4(hid, qd), "q_bias": r.normal(qd, std=0.1),
            "k_bias": r.normal(kvd, std=0.1), "v_bias": r.normal(kvd, std=0.1),
            "kc": r.normal(c["nkv"], c["max_seq"], HD), "vc": r.normal(c["nkv"], c["max_seq"], HD)}


def _decode_attention_inputs(c, seed):
    r = _Rand(seed)
    qd = c["nq"] * HD
    return {"q": r.normal(qd, std=1.5), "kc": r.normal(c["nkv"], c["max_seq"], HD),
            "vc": r.normal(c["nkv"], c["max_seq"], HD), "o": r.w4(qd, qd), "res": r.normal(qd)}


def _gemv_inputs(c, seed):
    r = _Rand(seed)
    return {"x": r.normal(c["k"]), "w": r.w4(c["n"], c["k"]), "res": r.normal(c["n"]) if c["residual"] else None}


def _head_inputs(c, seed):
    r = _Rand(seed)
    return {"x": r.normal(c["hidden"], std=3.0), "gamma": r.normal(c["hidden"], std=0.1, mean=1.0),
            "w": r.w4(c["vocab"], c["hidden"])}


def _control(pos):
    """Device control block (256 bytes): token_id, seq_pos, temperature 0, rng_seed."""
    ctl = torch.zeros(64, dtype=torch.int32, device=DEV)
    ctl[1] = pos
    return ctl


def _empty(*shape, dtype=torch.float16):
    return torch.empty(shape, dtype=dtype, device=DEV)


# ---- what a program keeps, and one pass --------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case, "stream": torch.cuda.current_stream().cuda_stream}
    if kind in ("prefill", "generate"):
        cfg = qe_amd.default_config()
        cfg.max_seq_len = case["max_seq"]
        st["engine"] = qe_amd.Engine(cfg, seed=seed)
        g = torch.Generator()
        g.manual_seed(seed)
        st["tokens"] = torch.randint(0, cfg.vocab_size, (case["prompt"],), generator=g).tolist()
        return st
    if kind in ("mlp", "attention"):
        qe_amd.gemm_reserve_workspace(st["stream"])  # the stream's split-K workspace, once per program
    if kind == "mlp":
        m, hid, inter = case["m"], case["hidden"], case["inter"]
        st["x"], layers = _mlp_inputs(case, seed)
        if case["path"] == "tiled":
            for L in layers:
                L["gate_up"] = qe_amd.w4_tiled(*L["gate_up"], 2 * inter, hid, stream=st["stream"])
                L["down"] = qe_amd.w4_tiled(*L["down"], hid, inter, stream=st["stream"])
        st.update(layers=layers, norm=_empty(m, hid), mlp=_empty(m, inter),
                  h=[_empty(m, hid) for _ in range(case["layers"])])
        if case["path"] == "w4a8":
            st["q8"] = [(_empty(m, k, dtype=torch.int8), _empty(m, k // 128, dtype=torch.float32),
                         _empty(m, k // 8, dtype=torch.int32)) for k in (hid, inter)]
        return st
    if kind == "attention":
        m, qd, kvd = case["m"], case["nq"] * HD, case["nkv"] * HD
        st.update(_attention_inputs(case, seed))
        if case["path"] == "tiled":
            for w, n in (("q", qd), ("k", kvd), ("v", kvd), ("o", qd)):
                st[w] = qe_amd.w4_tiled(*st[w], n, qd, stream=st["stream"])
        st.update(ctl=_control(case["base"]), norm=_empty(m, qd), dq=_empty(m, qd), dk=_empty(m, kvd),
                  dv=_empty(m, kvd), attn=_empty(m, qd), y=_empty(m, qd))
        st["view"] = qe_amd.make_qkv_view(*st["q"], st["dq"], *st["k"], st["dk"], *st["v"], st["dv"])
        return st
    if kind == "decode_attention":
        qd = case["nq"] * HD
        st.update(_decode_attention_inputs(case, seed))
        st.update(ctl=_control(case["pos"]), part_o=_empty(case["nq"] * 16 * HD, dtype=torch.float32),
                  part_lse=_empty(case["nq"] * 32, dtype=torch.float32), attn=_empty(qd), y=_empty(qd),
                  q8=_empty(qd, dtype=torch.int8), q8s=_empty(qd // 128, dtype=torch.float32),
                  q8sum=_empty(qd // 8, dtype=torch.int32))
        return st
    if kind == "gemv":
        st.update(_gemv_inputs(case, seed))
        st["y"] = _empty(case["n"])
        return st
    if kind == "head":
        st.update(_head_inputs(case, seed))
        parts = qe_amd.LM_HEAD_SAMPLE_PARTS
        st.update(ctl=_control(5), logits=_empty(case["vocab"]), val=_empty(parts, dtype=torch.float32),
                  idx=_empty(parts, dtype=torch.int32))
        return st
    raise ValueError(kind)


def run(st):
    c, s = st["case"], st["stream"]
    kind = c["kind"]
    if kind == "mlp":
        return _run_mlp(st, c, s)
    if kind == "attention":
        return _run_attention(st, c, s)
    if kind == "decode_attention":
        return _run_decode_attention(st, c, s)
    if kind == "gemv":
        qe_amd.launch_gemv_w4a16(st["w"][0], st["w"][1], st["x"], st["res"], st["y"], c["n"], c["k"], stream=s)
        return st["y"]
    if kind == "head":
        qe_amd.launch_rmsnorm_gemv_lm_head_sample_w4a16(st["x"], st["gamma"], None, st["w"][0], st["w"][1],
                                                        st["logits"], st["val"], st["idx"], st["ctl"], None,
                                                        vocab_size=c["vocab"], hidden_size=c["hidden"], stream=s)
        return {"logits": st["logits"], "token": st["ctl"][:1]}
    e = st["engine"]
    e.prefill(st["tokens"])
    if kind == "generate":
        e.decode(c["steps"])
    return {"logits": e.logits(), "hidden": e.hidden_row0()}


def _run_mlp(st, c, s):
    m, hid, inter = c["m"], c["hidden"], c["inter"]
    x, norm, mlp = st["x"], st["norm"], st["mlp"]
    for L, h in zip(st["layers"], st["h"]):
        qe_amd.launch_rmsnorm_fp16(x, L["gamma"], norm, m, stream=s, hidden_size=hid)
        if c["path"] == "tiled":
            qe_amd.launch_gemm_prefill_dual_gate_up_swiglu_w4a16_tiled(*L["gate_up"], norm, mlp, m, stream=s,
                                                                       hidden_size=hid, intermediate_size=inter)
            qe_amd.launch_gemm_prefill_w4a16_tiled(*L["down"], mlp, x, h, m, hid, inter, stream=s)
        elif c["path"] == "packed":
            qe_amd.launch_gemm_prefill_dual_gate_up_swiglu_w4a16(*L["gate_up"], norm, mlp, m, stream=s,
                                                                 hidden_size=hid, intermediate_size=inter)
            qe_amd.launch_gemm_prefill_w4a16(*L["down"], mlp, x, h, m, hid, inter, stream=s)
        else:
            qh, qi = st["q8"]
            qe_amd.launch_quantize_fp16_to_q8_1(norm, *qh, m * hid, stream=s)
            qe_amd.launch_gemm_prefill_dual_gate_up_swiglu_w4a8(*L["gate_up"], *qh, mlp, m, stream=s,
                                                                hidden_size=hid, intermediate_size=inter)
            qe_amd.launch_quantize_fp16_to_q8_1(mlp, *qi, m * inter, stream=s)
            qe_amd.launch_gemm_prefill_w4a8(*L["down"], *qi, x, h, m, hid, inter, stream=s)
        x = h
    return {"mlp": mlp, "y": x}


def _run_attention(st, c, s):
    m, nq, nkv, qd = c["m"], c["nq"], c["nkv"], c["nq"] * HD
    qe_amd.launch_rmsnorm_fp16(st["x"], st["gamma"], st["norm"], m, stream=s, hidden_size=qd)
    qkv = qe_amd.launch_gemm_prefill_qkv_w4a16_tiled if c["path"] == "tiled" else qe_amd.launch_gemm_prefill_qkv_w4a16
    qkv(st["view"], st["norm"], m, stream=s, in_features=qd, num_q_heads=nq, num_kv_heads=nkv, head_dim=HD)
    qe_amd.launch_qkv_bias_rope_kv_append(st["dq"], st["dk"], st["dv"], st["q_bias"], st["k_bias"], st["v_bias"],
                                          st["kc"], st["vc"], st["ctl"], m, stream=s, num_q_heads=nq,
                                          num_kv_heads=nkv, head_dim=HD, max_seq_len=c["max_seq"], rotary_dim=HD,
                                          rope_theta=THETA)
    qe_amd.launch_attention_gqa_prefill(st["dq"], st["kc"], st["vc"], st["attn"], st["ctl"], m, stream=s,
                                        num_q_heads=nq, num_kv_heads=nkv, head_dim=HD, max_seq_len=c["max_seq"],
                                        hidden_size=qd)
    o = qe_amd.launch_gemm_prefill_w4a16_tiled if c["path"] == "tiled" else qe_amd.launch_gemm_prefill_w4a16
    o(*st["o"], st["attn"], st["x"], st["y"], m, qd, qd, stream=s)
    new = slice(c["base"], c["base"] + m)
    return {"attn": st["attn"], "y": st["y"], "k": st["kc"][:, new], "v": st["vc"][:, new]}


def _run_decode_attention(st, c, s):
    nq, nkv, qd = c["nq"], c["nkv"], c["nq"] * HD
    if c["path"] == "fused":
        qe_amd.launch_attention_gqa_flash_decode_partials(st["q"], st["kc"], st["vc"], st["part_o"], st["part_lse"],
                                                          st["ctl"], stream=s, num_q_heads=nq, num_kv_heads=nkv,
                                                          head_dim=HD, max_seq_len=c["max_seq"])
        qe_amd.launch_attention_combine_gemv_o_w4a8(st["part_o"], st["part_lse"], st["o"][0], st["o"][1], st["res"],
                                                    st["y"], attn_out=st["attn"], d_control=st["ctl"],
                                                    out_features=qd, num_q_heads=nq, head_dim=HD,
                                                    max_seq_len=c["max_seq"], stream=s)
    else:
        qe_amd.launch_attention_gqa_flash_decode(st["q"], st["kc"], st["vc"], st["part_o"], st["part_lse"],
                                                 st["attn"], st["ctl"], stream=s, num_q_heads=nq, num_kv_heads=nkv,
                                                 head_dim=HD, max_seq_len=c["max_seq"], out_q8=st["q8"],
                                                 out_scale=st["q8s"], out_sum8=st["q8sum"])
        qe_amd.launch_gemv_w4a8(st["o"][0], st["o"][1], st["q8"], st["q8s"], st["q8sum"], st["res"], st["y"], qd, qd,
                                stream=s)
    return {"attn": st["attn"], "y": st["y"]}


# ---- what a pass cannot do without -------------------------------------------------------------------------------
def _w_bytes(n, k):
    return n * k // 2 + n * (k // 128) * 2


def work(case):
    c, kind = case, case["kind"]
    if kind == "mlp":
        m, hid, inter, n = c["m"], c["hidden"], c["inter"], c["layers"]
        return {"bytes": n * (_w_bytes(2 * inter, hid) + _w_bytes(hid, inter) + 4 * m * hid + 2 * m * inter),
                "flops": n * 2.0 * m * 3 * hid * inter}
    if kind == "attention":
        m, qd, kvd, end = c["m"], c["nq"] * HD, c["nkv"] * HD, c["base"] + c["m"]
        visible = m * c["base"] + m * (m + 1) / 2
        return {"bytes": 2 * _w_bytes(qd, qd) + 2 * _w_bytes(kvd, qd) + 6 * m * qd + 4 * end * kvd + 4 * m * kvd,
                "flops": 2.0 * m * qd * (2 * qd + 2 * kvd) + 4.0 * visible * qd}
    if kind == "decode_attention":
        qd, kvd, n = c["nq"] * HD, c["nkv"] * HD, c["pos"] + 1
        return {"bytes": 4 * n * kvd + _w_bytes(qd, qd) + 8 * qd, "flops": 4.0 * n * qd + 2.0 * qd * qd}
    if kind == "gemv":
        return {"bytes": _w_bytes(c["n"], c["k"]) + 2 * c["k"] + (4 if c["residual"] else 2) * c["n"],
                "flops": 2.0 * c["n"] * c["k"]}
    if kind == "head":
        return {"bytes": _w_bytes(c["vocab"], c["hidden"]) + 4 * c["hidden"] + 2 * c["vocab"],
                "flops": 2.0 * c["vocab"] * c["hidden"]}
    # engine: 28 layers, tied LM head; the prompt's rows, then one pass over all weights a generated token
    p, layers, kvd = c["prompt"], 28, NKV * HD
    layer_w = 2 * _w_bytes(H, H) + 2 * _w_bytes(kvd, H) + _w_bytes(2 * I, H) + _w_bytes(H, I)
    layer_mac = H * (2 * H + 2 * kvd) + 3 * H * I
    head = _w_bytes(V, H)
    kv_row = 4 * kvd
    nbytes = layers * (layer_w + p * kv_row) + head
    flops = 2.0 * p * layers * layer_mac + layers * 2.0 * p * (p + 1) * H + 2.0 * V * H
    if kind == "generate":
        n = c["steps"]
        nbytes += n * (layers * layer_w + head) + layers * kv_row * (n * p + n * (n + 1) // 2)
        flops += n * 2.0 * (layers * layer_mac + V * H) + layers * 4.0 * H * (n * p + n * (n + 1) / 2)
    return {"bytes": float(nbytes), "flops": flops}


def tolerance(case):
    """About four times the error against 64 bits (blocks) or the difference another GEMM tiling makes (engine)."""
    kind = case["kind"]
    if kind == "mlp":  # layers feed each other; w4a8: a changed rounding moves an int8 activation by a whole step
        n = case["layers"] - 1
        if case["path"] == "w4a8":
            return {"rel": 1e-2 + 3e-3 * n, "max": 0.2}
        return {"rel": 3e-3 + 1e-3 * n, "max": 0.1}
    if kind == "attention":
        return {"rel": 4e-3, "max": 0.05}
    if kind == "decode_attention":
        return {"rel": 2e-3, "max": 0.02}
    if kind == "gemv":
        return {"rel": 1e-3, "max": 0.02}
    if kind == "head":
        return {"rel": 5e-3, "max": 0.05}
    return {"rel": 2e-3, "max": 0.02}


# ---- the same in 64 bits -----------------------------------------------------------------------------------------
def _dequant(qw, sc, row0=0, rows=None):
    """(q - 8) * scale of packed weights, float64 [rows][K]; nibble j of a word holds element (0, 2, 4, 6, 1, 3, 5,
    7)[j] of its 8 (element order q0 q4 q1 q5 q2 q6 q3 q7 from the low nibble up)."""
    qw = qw[row0:] if rows is None else qw[row0:row0 + rows]
    sc = sc[row0:] if rows is None else sc[row0:row0 + rows]
    shifts = torch.tensor([0, 8, 16, 24, 4, 12, 20, 28], device=qw.device, dtype=torch.int32)
    q = (qw.unsqueeze(-1) >> shifts) & 15
    q = q.reshape(qw.shape[0], -1).double() - 8.0
    return (q.reshape(qw.shape[0], -1, 128) * sc.double().unsqueeze(-1)).reshape(qw.shape[0], -1)


def _matmul_w4(x, w):
    """x [M, K] float64 times the transposed weights, a block of rows at a time."""
    qw, sc = w
    return torch.cat([x @ _dequant(qw, sc, r, 4096).T for r in range(0, qw.shape[0], 4096)], dim=1)


def _q8(x):
    """Q8_1 round trip of rows: 128-groups, scale max|x|/127, half away from zero."""
    g = x.reshape(x.shape[0], -1, 128)
    d = (g.abs().amax(dim=-1, keepdim=True) / 127.0).clamp_min(1e-8)
    y = g / d
    return (torch.sign(y) * torch.floor(y.abs() + 0.5) * d).reshape(x.shape)


def _rms(x, gamma):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + EPS) * gamma.double()


def _rope(x, pos):
    """NeoX rotation of [M, heads, 128] at positions pos [M]."""
    i = torch.arange(HD // 2, device=x.device, dtype=torch.float64)
    ang = pos.double()[:, None] * (THETA ** (-2.0 * i / HD))[None, :]
    cs, sn = ang.cos()[:, None, :], ang.sin()[:, None, :]
    a, b = x[..., :HD // 2], x[..., HD // 2:]
    return torch.cat([a * cs - b * sn, a * sn + b * cs], dim=-1)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "mlp":
        x, layers = _mlp_inputs(c, seed)
        x = x.double()
        act = _q8 if c["path"] == "w4a8" else (lambda t: t)
        for L in layers:
            norm = _rms(x, L["gamma"])
            if c["path"] == "w4a8":
                norm = norm.half().double()  # the quantizer's input is the rounded norm
            gu = _matmul_w4(act(norm), L["gate_up"])
            g, u = gu[:, 0::2], gu[:, 1::2]
            mlp = g * torch.sigmoid(g) * u
            if c["path"] == "w4a8":
                mlp = mlp.half().double()
            x = _matmul_w4(act(mlp), L["down"]) + x
        return {"mlp": mlp, "y": x}
    if kind == "attention":
        t = _attention_inputs(c, seed)
        m, nq, nkv, base = c["m"], c["nq"], c["nkv"], c["base"]
        x = t["x"].double()
        norm = _rms(x, t["gamma"])
        pos = torch.arange(base, base + m, device=x.device)
        q = _rope((_matmul_w4(norm, t["q"]) + t["q_bias"].double()).reshape(m, nq, HD), pos)
        k = _rope((_matmul_w4(norm, t["k"]) + t["k_bias"].double()).reshape(m, nkv, HD), pos).transpose(0, 1)
        v = (_matmul_w4(norm, t["v"]) + t["v_bias"].double()).reshape(m, nkv, HD).transpose(0, 1)
        kc = torch.cat([t["kc"][:, :base].double(), k], dim=1)
        vc = torch.cat([t["vc"][:, :base].double(), v], dim=1)
        attn = torch.empty(m, nq, HD, dtype=torch.float64, device=x.device)
        key = torch.arange(base + m, device=x.device)
        for h in range(nq):
            g = h // (nq // nkv)
            for r in range(0, m, 512):
                s = (q[r:r + 512, h] @ kc[g].T) / math.sqrt(HD)
                s = s.masked_fill(key[None, :] > pos[r:r + 512, None], -math.inf)
                attn[r:r + 512, h] = torch.softmax(s, dim=-1) @ vc[g]
        attn = attn.reshape(m, nq * HD)
        return {"attn": attn, "y": _matmul_w4(attn, t["o"]) + x, "k": k, "v": v}
    if kind == "decode_attention":
        t = _decode_attention_inputs(c, seed)
        nq, nkv, n = c["nq"], c["nkv"], c["pos"] + 1
        q = t["q"].double().reshape(nkv, nq // nkv, HD)
        kc, vc = t["kc"][:, :n].double(), t["vc"][:, :n].double()
        p = torch.softmax(q @ kc.transpose(1, 2) / math.sqrt(HD), dim=-1)
        attn = (p @ vc).reshape(1, nq * HD)
        y = _matmul_w4(_q8(attn), t["o"]) + t["res"].double()
        return {"attn": attn.reshape(-1), "y": y.reshape(-1)}
    if kind == "gemv":
        t = _gemv_inputs(c, seed)
        y = _matmul_w4(_q8(t["x"].double().reshape(1, -1)), t["w"]).reshape(-1)
        return y if t["res"] is None else y + t["res"].double()
    if kind == "head":
        t = _head_inputs(c, seed)
        norm = _rms(t["x"].double().reshape(1, -1), t["gamma"]).half().double()
        return {"logits": _matmul_w4(_q8(norm), t["w"]).reshape(-1), "token": None}
    return None  # the engine makes its own weights
