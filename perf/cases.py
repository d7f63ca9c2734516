"""The work that a program built on this framework has it do, as a list of cases to time.

Every case goes through a public entry point: spock_amd.ops, the C ABI of include/spock_hip.h (through
spock_amd._lib, as a C program would call it), or spock_amd.model.Session.  Shapes are the framework's own: 16 DeltaNet
heads of 128, hidden 1024, MLP 3584, 8 query and 2 KV heads of 256, vocabulary 248320.

`run` leaves its input tensors alone, except where the entry point updates state in place (decode steps, conv
history, KV rows).  `exact` restates the mathematics in torch float64.
"""
from __future__ import annotations

import ctypes as C
import math
import tempfile

import numpy as np
import torch

from spock_amd import _lib, model, ops

HEADS, DIM, HIDDEN, INTER, CONV = 16, 128, 1024, 3584, 6144
VAL = HEADS * DIM
Q_HEADS, KV_HEADS, HEAD_DIM, ROT = 8, 2, 256, 64
EPS = 1e-6
LAYERS = 18  # rows of the (A_log, dt_bias) table
# the layer-input and MLP projections of one decode token, as (rows, columns)
CHAIN = "6144x1024,2048x1024,3584x1024,3584x1024;1024x2048,1024x3584"


def listed():
    return [
        # a short prompt of one layer in the reference's own float32 interface: latency of two launches
        {"name": "chunk_f32_104", "kind": "chunk", "dtype": "f32", "lens": "104", "init": False, "l2": False},
        # one ordinary prompt that continues a sequence: 128 state columns times a chain of 32 chunks
        {"name": "chunk_f16_2048", "kind": "chunk", "dtype": "f16", "lens": "2048", "init": True, "l2": False},
        # a server's packed batch of prompts, ragged lengths: the largest chunk-rule call
        {"name": "chunk_f16_pack8", "kind": "chunk", "dtype": "f16", "lens": "2504,3608,3930,7547,1061,7884,4357,3987",
         "init": False, "l2": False},
        # one decode step of a serving batch: 64 sequences' states read and written once
        {"name": "dn_step_b64", "kind": "dn_step", "batch": 64},
        # one token through a DeltaNet layer at batch 1: four dependent launches
        {"name": "dn_layer_decode", "kind": "dn_layer"},
        # one token through an attention layer at batch 1, with an ordinary context
        {"name": "attn_layer_decode_1500", "kind": "attn_layer", "pos": 1500},
        # the decode projections of one layer, in two dependent calls
        {"name": "gemv_chain", "kind": "gemv", "shapes": CHAIN},
        # the tied lm_head over the whole vocabulary with the greedy token
        {"name": "lm_head_248320", "kind": "lm_head", "vocab": 248320},
        # a 512-token prompt through a DeltaNet mixer on the matrix cores
        {"name": "dn_prompt_512", "kind": "dn_prompt", "tokens": 512},
        # a longer prompt through an MLP on the matrix cores
        {"name": "mlp_prompt_2000", "kind": "mlp_prompt", "tokens": 2000},
        # a prompt through an attention mixer
        {"name": "attn_prompt_1000", "kind": "attn_prompt", "tokens": 1000, "pos0": 0},
        # a whole call: a session's default prefill of a 512-token prompt, then greedy tokens (four layers of the model)
        {"name": "session_512_32", "kind": "session", "tokens": 512, "new": 32, "matrix": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["chunk", "chunk", "chunk", "dn_step", "attn_layer", "gemv", "lm_head", "dn_prompt", "mlp_prompt",
                       "attn_prompt", "session"])
    if kind == "chunk":
        f32 = rng.random() < 0.25
        lens = [_log_int(rng, 16, 8000)]
        for _ in range(rng.choice([0, 0, 1, 3, 7, 11])):
            lens.append(_log_int(rng, 16, 4000))
        while sum(lens) > (8000 if f32 else 32000):
            lens.pop()
        return {"kind": kind, "dtype": "f32" if f32 else "f16", "lens": ",".join(map(str, lens)),
                "init": rng.random() < 0.5, "l2": rng.random() < 0.4}
    if kind == "dn_step":
        return {"kind": kind, "batch": _log_int(rng, 1, 200)}
    if kind == "attn_layer":
        return {"kind": kind, "pos": _log_int(rng, 1, 4000)}
    if kind == "gemv":
        stage = lambda n, k: ",".join("%dx%d" % (_log_int(rng, 16, 7000), k) for _ in range(n))  # noqa: E731
        return {"kind": kind, "shapes": ";".join(stage(rng.randint(1, 4), 64 * rng.randint(8, 56)) for _ in range(2))}
    if kind == "lm_head":
        return {"kind": kind, "vocab": _log_int(rng, 4000, 248000)}
    if kind == "attn_prompt":
        return {"kind": kind, "tokens": _log_int(rng, 16, 2000), "pos0": rng.choice([0, 0, _log_int(rng, 1, 1000)])}
    if kind == "session":
        matrix = rng.random() < 0.5
        return {"kind": kind, "tokens": _log_int(rng, 16, 500), "new": 0 if matrix else rng.randint(1, 32), "matrix": matrix}
    return {"kind": kind, "tokens": _log_int(rng, 16, 4000)}


# ---- inputs -------------------------------------------------------------------------------------------------


class _Rand:
    """Normal values on the GPU from one seed, one stream of draws."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def f32(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device="cuda") * std

    def f16(self, *shape, std=1.0):
        return self.f32(*shape, std=std).half()

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, generator=self.g, device="cuda") * (hi - lo) + lo


def _empty(*shape, dtype=torch.float16):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def _lens(case):
    return [int(x) for x in case["lens"].split(",")]


def _chunk_inputs(case, seed):
    """q, k (unit rows, or raw where the call normalises them), v ~ N(0, 1), log-decays and write strengths as a
    trained layer has them: -softplus(N(0, 1)) and sigmoid(N(0, 1))."""
    r, n, lens = _Rand(seed), sum(_lens(case)), _lens(case)
    q, k, v = (r.f32(HEADS, n, DIM) for _ in range(3))
    if not case["l2"]:
        q, k = (x / torch.sqrt((x * x).sum(-1, keepdim=True) + EPS) for x in (q, k))
    if case["dtype"] == "f16":
        q, k, v = q.half(), k.half(), v.half()
    g = -torch.nn.functional.softplus(r.f32(HEADS, n))
    beta = torch.sigmoid(r.f32(HEADS, n))
    init = r.f32(len(lens), HEADS, DIM, DIM, std=0.1) if case["init"] else None
    return q.contiguous(), k.contiguous(), v.contiguous(), g, beta, init


def _dn_weights(r):
    return {"a_log": r.uniform(LAYERS, HEADS, lo=-1.0, hi=1.0), "dt": r.f16(LAYERS, HEADS, std=0.1).float(),
            "conv_w": r.f16(CONV, 4, std=0.3), "nw": r.uniform(DIM, lo=0.5, hi=1.5)}


def _alb(w):
    return torch.stack([w["a_log"], w["dt"]], dim=-1).contiguous()


def _step_inputs(batch, seed):
    r = _Rand(seed)
    d = _dn_weights(r)
    d.update(qkv=r.f16(batch, CONV), state=r.f32(batch, HEADS, DIM, DIM, std=0.1), conv=r.f16(batch, CONV, 4),
             a=r.f16(batch, HEADS), b=r.f16(batch, HEADS), z=r.f16(batch, VAL))
    return d


def _mats(r, *shapes):
    return [r.f16(n, k, std=0.02) for n, k in shapes]


def _layer_inputs(seed):
    """A DeltaNet layer's weights with the state of a sequence under way."""
    r = _Rand(seed)
    d = _dn_weights(r)
    d["Win"] = _mats(r, (CONV, HIDDEN), (VAL, HIDDEN), (HEADS, HIDDEN), (HEADS, HIDDEN))
    d["Wout"], = _mats(r, (HIDDEN, VAL))
    d.update(_mlp_weights(r))
    d.update(h=r.f16(1, HIDDEN), norm=r.f16(HIDDEN, std=0.1), state=r.f32(1, HEADS, DIM, DIM, std=0.1),
             conv=r.f16(1, CONV, 4))
    return d


def _mlp_weights(r):
    gate, up, down = _mats(r, (INTER, HIDDEN), (INTER, HIDDEN), (HIDDEN, INTER))
    return {"gate": gate, "up": up, "down": down, "post": r.f16(HIDDEN, std=0.1)}


def _rope(max_seq):
    ang = torch.arange(max_seq, dtype=torch.float64)[:, None] * (1e7 ** (-torch.arange(32, dtype=torch.float64) / 32))[None]
    return torch.stack([torch.cos(ang), torch.sin(ang)], dim=-1).reshape(max_seq, ROT).float().cuda()


def _attn_inputs(seed, tokens, pos0, max_seq, mlp):
    r = _Rand(seed)
    d = {"Win": _mats(r, (2 * Q_HEADS * HEAD_DIM, HIDDEN), (KV_HEADS * HEAD_DIM, HIDDEN), (KV_HEADS * HEAD_DIM, HIDDEN))}
    d["Wout"], = _mats(r, (HIDDEN, Q_HEADS * HEAD_DIM))
    d.update(h=r.f16(tokens, HIDDEN), norm=r.f16(HIDDEN, std=0.1), qn=r.f16(HEAD_DIM, std=0.1), kn=r.f16(HEAD_DIM, std=0.1),
             rope=_rope(max_seq), kv=torch.zeros(max_seq, 1024, dtype=torch.float16, device="cuda"))
    d["kv"][:pos0] = r.f16(pos0, 1024)
    if mlp:
        d.update(_mlp_weights(r))
    return d


def _stages(case):
    return [[tuple(map(int, s.split("x"))) for s in st.split(",")] for st in case["shapes"].split(";")]


# ---- argument structs of the C ABI ----------------------------------------------------------------------------


def _p(t):
    return None if t is None else t.data_ptr()


def _gemv_in(kind, x, x2=None):
    a = _lib.SpkGemvInput()
    a.kind, a.in_dim, a.x, a.x2 = kind, x.shape[-1], _p(x), _p(x2)
    return a


def _gemv_out(*items):
    arr = (_lib.SpkGemvOutput * len(items))()
    for o, (W, y, res, up) in zip(arr, items):
        o.W, o.y, o.residual, o.out_dim, o.W_up = _p(W), _p(y), _p(res), W.shape[0], _p(up)
    return arr


def _step_args(d, qkv, z, a, b, layer):
    s = _lib.SpkDecodeArgs()
    s.batch, s.num_heads, s.layer_idx = qkv.shape[0], HEADS, layer
    s.qkv, s.qkv_stride, s.conv_state, s.conv_state_stride = _p(qkv), CONV, _p(d["conv"]), CONV * 4
    s.conv_weight, s.a, s.b, s.ab_stride, s.a_log_bias = _p(d["conv_w"]), _p(a), _p(b), HEADS, _p(d["alb"])
    s.state, s.state_stride, s.z, s.z_stride, s.norm_weight = _p(d["state"]), HEADS * DIM * DIM, _p(z), VAL, _p(d["nw"])
    return s


def _attn_args(d, qg, k, v, out, max_seq, positions, tokens):
    d["attn_ws"] = torch.zeros(_lib.lib().spk_attention_workspace_size(positions, tokens), dtype=torch.uint8, device="cuda")
    a = _lib.SpkAttnArgs()
    a.qg, a.k, a.v, a.q_norm_w, a.k_norm_w, a.rope = _p(qg), _p(k), _p(v), _p(d["qn"]), _p(d["kn"]), _p(d["rope"])
    a.kv_cache, a.max_seq, a.out = _p(d["kv"]), max_seq, _p(out)
    a.workspace, a.workspace_bytes = _p(d["attn_ws"]), d["attn_ws"].numel()
    return a


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _ok(rc, what):
    _lib.check(rc, what)


def _mlp_decode(d):
    d["m"], d["y"] = _empty(1, INTER), _empty(1, HIDDEN)
    return [("gate_up", _gemv_in(_lib.SPK_GEMV_IN_RMSNORM, d["h2"], d["post"]), _gemv_out((d["gate"], d["m"], None, d["up"]))),
            ("down", _gemv_in(_lib.SPK_GEMV_IN_PLAIN, d["m"]), _gemv_out((d["down"], d["y"], d["h2"], None)))]


# ---- prepare --------------------------------------------------------------------------------------------------


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def _prepare_chunk(case, seed):
    q, k, v, g, beta, init = _chunk_inputs(case, seed)
    lens, n = _lens(case), q.shape[1]
    s = dict(q=q, k=k, v=v, g=g, beta=beta, init=init, l2=case["l2"], cu=None, cu_dev=None)
    if len(lens) > 1:
        s["cu"] = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        s["cu_dev"] = torch.from_numpy(s["cu"]).cuda()
    s["core"] = _empty(HEADS, n, DIM, dtype=torch.float32)
    s["state"] = _empty(len(lens), HEADS, DIM, DIM, dtype=torch.float32)
    s["ws"] = _empty(ops.chunk_workspace_bytes(HEADS, n, len(lens)), dtype=torch.uint8)
    s["kind"] = "chunk"
    return s


def _prepare_dn_step(case, seed):
    d = _step_inputs(case["batch"], seed)
    d["alb"], d["kind"] = _alb(d), "dn_step"
    return d


def _prepare_dn_layer(case, seed):
    d = _layer_inputs(seed)
    d["alb"], d["kind"] = _alb(d), "dn_layer"
    d["qkv"], d["z"], d["a"], d["b"], d["h2"] = (_empty(1, n) for n in (CONV, VAL, HEADS, HEADS, HIDDEN))
    d["arrive"] = torch.zeros(1024, dtype=torch.int32, device="cuda")
    d["inproj"] = (_gemv_in(_lib.SPK_GEMV_IN_RMSNORM, d["h"], d["norm"]),
                   _gemv_out(*((W, y, None, None) for W, y in zip(d["Win"], (d["qkv"], d["z"], d["a"], d["b"])))),
                   _step_args(d, d["qkv"], d["z"], d["a"], d["b"], 3))
    d["gemvs"] = [("out_proj", _gemv_in(_lib.SPK_GEMV_IN_PLAIN, d["qkv"][:, 2 * VAL:]),
                   _gemv_out((d["Wout"], d["h2"], d["h"], None)))] + _mlp_decode(d)
    return d


def _prepare_attn_layer(case, seed):
    pos, max_seq = case["pos"], 4096
    d = _attn_inputs(seed, 1, pos, max_seq, True)
    d["kind"] = "attn_layer"
    d["qg"], d["k"], d["v"], d["out"], d["h2"] = (_empty(1, n) for n in (4096, 512, 512, 2048, HIDDEN))
    d["pos"] = torch.tensor([pos], dtype=torch.int32, device="cuda")
    a = _attn_args(d, d["qg"], d["k"], d["v"], d["out"], max_seq, max_seq, 1)
    a.pos_dev = _p(d["pos"])
    d["inproj"] = (_gemv_in(_lib.SPK_GEMV_IN_RMSNORM, d["h"], d["norm"]),
                   _gemv_out(*((W, y, None, None) for W, y in zip(d["Win"], (d["qg"], d["k"], d["v"])))), a,
                   _gemv_out((d["Wout"], d["h2"], d["h"], None)))
    d["gemvs"] = _mlp_decode(d)
    return d


def _prepare_gemv(case, seed):
    r, stages = _Rand(seed), []
    for st in _stages(case):
        xs = {k: r.f16(k) for k in {k for _, k in st}}
        items = [(W, xs[W.shape[1]], _empty(W.shape[0])) for W in _mats(r, *st)]
        stages.append(items)
    return {"kind": "gemv", "stages": stages}


def _prepare_lm_head(case, seed):
    r = _Rand(seed)
    W, = _mats(r, (case["vocab"], HIDDEN))
    return {"kind": "lm_head", "W": W, "x": r.f16(HIDDEN), "logits": _empty(case["vocab"]),
            "token": _empty(1, dtype=torch.int32),
            "ws": _empty(ops.lm_head_workspace_bytes(case["vocab"]), dtype=torch.uint8)}


def _prepare_dn_prompt(case, seed):
    d, n = _layer_inputs(seed), case["tokens"]
    d["alb"], d["kind"], d["h"] = _alb(d), "dn_prompt", _Rand(seed + (1 << 40)).f16(n, HIDDEN)
    d["xn"], d["qkv"], d["z"], d["a"], d["b"] = (_empty(n, c) for c in (HIDDEN, CONV, VAL, HEADS, HEADS))
    d["q"], d["k"], d["v"] = (_empty(HEADS, n, DIM) for _ in range(3))
    d["g"], d["beta"] = (_empty(HEADS, n, dtype=torch.float32) for _ in range(2))
    d["core"], d["out_state"] = _empty(HEADS, n, DIM, dtype=torch.float32), _empty(1, HEADS, DIM, DIM, dtype=torch.float32)
    d["ws"] = _empty(ops.chunk_workspace_bytes(HEADS, n), dtype=torch.uint8)
    d["gated"], d["y"] = _empty(n, VAL), _empty(n, HIDDEN)
    return d


def _prepare_mlp_prompt(case, seed):
    r, n = _Rand(seed), case["tokens"]
    d = _mlp_weights(r)
    d.update(kind="mlp_prompt", h=r.f16(n, HIDDEN), xn=_empty(n, HIDDEN), ga=_empty(n, INTER), ua=_empty(n, INTER),
             y=_empty(n, HIDDEN))
    return d


def _prepare_attn_prompt(case, seed):
    n, pos0 = case["tokens"], case["pos0"]
    max_seq = pos0 + n
    d = _attn_inputs(seed, n, pos0, max_seq, False)
    d["kind"], d["pos0"] = "attn_prompt", pos0
    d["xn"], d["qg"], d["k"], d["v"], d["out"], d["y"] = (_empty(n, c) for c in (HIDDEN, 4096, 512, 512, 2048, HIDDEN))
    d["attn"] = _attn_args(d, d["qg"], d["k"], d["v"], d["out"], max_seq, max_seq, n)
    return d


def _prepare_session(case, seed):
    with tempfile.TemporaryDirectory() as tmp:
        model.write_synthetic_artifact(tmp, layers=4, vocab=32768, seed=seed % 1000003)
        s = model.Session(tmp, max_seq=1024, matrix_prefill=case["matrix"])
    prompt = np.random.default_rng(seed).integers(0, s.vocab, case["tokens"]).astype(np.int32)
    return {"kind": "session", "session": s, "prompt": prompt, "new": case["new"]}


_PREPARE = {"chunk": _prepare_chunk, "dn_step": _prepare_dn_step, "dn_layer": _prepare_dn_layer,
            "attn_layer": _prepare_attn_layer, "gemv": _prepare_gemv, "lm_head": _prepare_lm_head,
            "dn_prompt": _prepare_dn_prompt, "mlp_prompt": _prepare_mlp_prompt, "attn_prompt": _prepare_attn_prompt,
            "session": _prepare_session}


# ---- run ------------------------------------------------------------------------------------------------------


def run(s):
    return _RUN[s["kind"]](s)


def _run_chunk(s):
    core, state = ops.chunk_prefill(s["q"], s["k"], s["v"], s["g"], s["beta"], initial_state=s["init"], cu_seqlens=s["cu"],
                                    use_qk_l2norm=s["l2"], out_core=s["core"], out_state=s["state"], workspace=s["ws"],
                                    cu_seqlens_dev=s["cu_dev"])
    return {"core": core, "state": state}


def _run_dn_step(d):
    ops.decode_step(d["qkv"], d["state"], d["conv"], d["conv_w"], d["a"], d["b"], d["alb"], d["z"], d["nw"], layer_idx=3)
    return {"qkv": d["qkv"], "state": d["state"], "conv": d["conv"]}


def _run_gemvs(gemvs, st):
    for what, gi, go in gemvs:
        _ok(_lib.lib().spk_gemv_fused(C.byref(gi), go, 1, st), what)


def _run_dn_layer(d):
    st, (gi, go, step) = _stream(), d["inproj"]
    _ok(_lib.lib().spk_deltanet_inproj_step(C.byref(gi), go, C.byref(step), _p(d["arrive"]), st), "inproj step")
    _run_gemvs(d["gemvs"], st)
    return {n: d[n] for n in ("qkv", "state", "conv", "h2", "m", "y")}


def _run_attn_layer(d):
    st, (gi, go, a, oo) = _stream(), d["inproj"]
    _ok(_lib.lib().spk_attention_inproj(C.byref(gi), go, C.byref(a), st), "attention inproj")
    _ok(_lib.lib().spk_attention_decode_oproj(C.byref(a), oo, st), "attention decode")
    _run_gemvs(d["gemvs"], st)
    return {n: d[n] for n in ("out", "kv", "h2", "m", "y")}


def _run_gemv(s):
    for items in s["stages"]:
        ops.matvec_f16_batched(items)
    return [y for items in s["stages"] for _, _, y in items]


def _run_lm_head(s):
    token = ops.lm_head_argmax(s["W"], s["x"], logits=s["logits"], out=s["token"], workspace=s["ws"])
    return {"token": token, "logits": s["logits"]}


def _gemm(x, W, y, st, residual=None):
    n, k = x.shape
    _ok(_lib.lib().spk_gemm_f16(_p(x), k, _p(W), k, _p(y), W.shape[0], _p(residual), n, W.shape[0], k, st), "gemm")


def _rmsnorm(x, w, y, st):
    _ok(_lib.lib().spk_rmsnorm_f16(_p(x), _p(w), _p(y), x.shape[0], HIDDEN, st), "rmsnorm")


def _run_dn_prompt(d):
    L, st, n = _lib.lib(), _stream(), d["h"].shape[0]
    _rmsnorm(d["h"], d["norm"], d["xn"], st)
    for W, y in zip(d["Win"], (d["qkv"], d["z"], d["a"], d["b"])):
        _gemm(d["xn"], W, y, st)
    _ok(L.spk_deltanet_prefill_conv(_p(d["qkv"]), CONV, _p(d["conv"]), _p(d["conv_w"]), n, _p(d["q"]), _p(d["k"]), _p(d["v"]),
                                    st), "conv")
    _ok(L.spk_deltanet_prefill_gbeta(_p(d["a"]), _p(d["b"]), HEADS, _p(d["alb"]), 3, n, _p(d["g"]), _p(d["beta"]), st), "g/beta")
    ops.chunk_prefill(d["q"], d["k"], d["v"], d["g"], d["beta"], initial_state=d["state"], out_core=d["core"],
                      out_state=d["out_state"], workspace=d["ws"])
    _ok(L.spk_deltanet_norm_gate(_p(d["core"]), n, _p(d["z"]), VAL, _p(d["nw"]), 0.0, n, _p(d["gated"]), VAL, st), "norm gate")
    _gemm(d["gated"], d["Wout"], d["y"], st, residual=d["h"])
    return {n: d[n] for n in ("y", "gated", "out_state", "conv")}


def _run_mlp_prompt(d):
    st = _stream()
    _rmsnorm(d["h"], d["post"], d["xn"], st)
    _gemm(d["xn"], d["gate"], d["ga"], st)
    _gemm(d["xn"], d["up"], d["ua"], st)
    _ok(_lib.lib().spk_silu_gate_f16(_p(d["ga"]), _p(d["ua"]), _p(d["ga"]), d["ga"].numel(), st), "silu gate")
    _gemm(d["ga"], d["down"], d["y"], st, residual=d["h"])
    return {"m": d["ga"], "y": d["y"]}


def _run_attn_prompt(d):
    st = _stream()
    _rmsnorm(d["h"], d["norm"], d["xn"], st)
    for W, y in zip(d["Win"], (d["qg"], d["k"], d["v"])):
        _gemm(d["xn"], W, y, st)
    _ok(_lib.lib().spk_attention_prefill(C.byref(d["attn"]), d["pos0"], d["h"].shape[0], st), "attention prefill")
    _gemm(d["out"], d["Wout"], d["y"], st, residual=d["h"])
    return {"out": d["out"], "kv": d["kv"], "y": d["y"]}


def _run_session(s):
    m = s["session"]
    m.reset()
    tokens = [m.prefill(s["prompt"])]
    if s["new"]:
        tokens += m.decode(s["new"]).tolist()
    logits, hidden = m.last_output()
    return {"tokens": np.asarray(tokens, dtype=np.int64), "logits": logits.view(np.float16), "hidden": hidden.view(np.float16)}


_RUN = {"chunk": _run_chunk, "dn_step": _run_dn_step, "dn_layer": _run_dn_layer, "attn_layer": _run_attn_layer,
        "gemv": _run_gemv, "lm_head": _run_lm_head, "dn_prompt": _run_dn_prompt, "mlp_prompt": _run_mlp_prompt,
        "attn_prompt": _run_attn_prompt, "session": _run_session}


# ---- work -----------------------------------------------------------------------------------------------------


def work(case):
    """One pass: inputs and weights read once, outputs written once; activations between a block's own calls are not
    counted.  The chunk rule counts the recurrence's three products per token and head (K S, the update, Q S)."""
    kind = case["kind"]
    state, mlp = HEADS * DIM * DIM * 4, 3 * HIDDEN * INTER
    if kind == "chunk":
        n, s, e = sum(_lens(case)), len(_lens(case)), 4 if case["dtype"] == "f32" else 2
        return {"bytes": HEADS * n * (3 * DIM * e + 8 + DIM * 4) + state * s * (2 if case["init"] else 1),
                "flops": HEADS * n * 6 * DIM * DIM}
    if kind == "dn_step":
        b = case["batch"]
        return {"bytes": b * (2 * state + CONV * (2 + 2 + 8 + 8) + VAL * 2 + HEADS * 4), "flops": b * HEADS * 6 * DIM * DIM}
    dn_w, attn_w = HIDDEN * (CONV + 2 * VAL + 2 * HEADS), HIDDEN * (4096 + 1024 + 2048)
    if kind == "dn_layer":
        w = dn_w + mlp
        return {"bytes": 2 * w + 2 * state + CONV * 24, "flops": 2 * w + HEADS * 6 * DIM * DIM}
    if kind == "attn_layer":
        w, p = attn_w + mlp, case["pos"] + 1
        return {"bytes": 2 * w + p * 2048, "flops": 2 * w + p * Q_HEADS * HEAD_DIM * 4}
    if kind == "gemv":
        w = sum(n * k for st in _stages(case) for n, k in st)
        return {"bytes": 2 * w, "flops": 2 * w}
    if kind == "lm_head":
        w = case["vocab"] * HIDDEN
        return {"bytes": 2 * w + 2 * case["vocab"], "flops": 2 * w}
    n = case["tokens"]
    if kind == "dn_prompt":
        return {"bytes": 2 * dn_w + 4 * n * HIDDEN + 2 * state, "flops": 2 * n * dn_w + n * HEADS * 6 * DIM * DIM}
    if kind == "mlp_prompt":
        return {"bytes": 2 * mlp + 4 * n * HIDDEN, "flops": 2 * n * mlp}
    if kind == "attn_prompt":
        pairs = n * case["pos0"] + n * (n + 1) // 2
        return {"bytes": 2 * attn_w + 4 * n * HIDDEN + (case["pos0"] + 2 * n) * 2048,
                "flops": 2 * n * attn_w + pairs * Q_HEADS * HEAD_DIM * 4}
    w = 3 * (dn_w + mlp) + attn_w + mlp  # three DeltaNet layers and one of attention
    head = 32768 * HIDDEN
    return {"bytes": 2 * (w + head) * (1 + case["new"]) + 6 * state * case["new"],
            "flops": 2 * w * (n + case["new"]) + 2 * head * (1 + case["new"])}


# ---- tolerance and the 64-bit answers ---------------------------------------------------------------------------


def tolerance(case):
    kind = case["kind"]
    if kind == "chunk":  # 32-bit sums over 64 tokens and 128 dims, carried through a chain of chunks
        return {"rel": 4e-6, "max": 2e-4}
    if kind in ("dn_prompt", "mlp_prompt", "attn_prompt"):  # 16-bit activations between 32-bit accumulations
        return {"rel": 2e-3, "max": 5e-2}
    if kind == "session" and case["matrix"]:  # the same through four layers; a token may fall in a tie
        return {"rel": 1e-2, "max": 0.2, "differ": 0.01}
    # the entry points of the decode path, and the session's default mode, promise the bits of a stated order of sums
    return "exact"


def exact(case, seed):
    f = _EXACT.get(case["kind"])
    return None if f is None else f(case, seed)


def _d(t):
    return t.double()


def _silu(x):
    return x * torch.sigmoid(x)


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _recur(q, k, v, g, beta, S):
    """The gated delta rule token by token: q, k, v [B][n][128], g, beta [B][n], S [B][128][128]; q is scaled here."""
    out, q, decay = torch.empty_like(v), q / math.sqrt(DIM), torch.exp(g)
    for t in range(q.shape[1]):
        S = S * decay[:, t, None, None]
        delta = (v[:, t] - (S * k[:, t, :, None]).sum(1)) * beta[:, t, None]
        S = S + k[:, t, :, None] * delta[:, None, :]
        out[:, t] = (S * q[:, t, :, None]).sum(1)
    return out, S


def _exact_chunk(case, seed):
    q, k, v, g, beta, init = _chunk_inputs(case, seed)
    q, k, v, g, beta = map(_d, (q, k, v, g, beta))
    if case["l2"]:
        q, k = (x / torch.sqrt((x * x).sum(-1, keepdim=True) + EPS) for x in (q, k))
    lens = _lens(case)
    top, at = max(lens), np.concatenate([[0], np.cumsum(lens)]).tolist()
    pad = lambda x: torch.cat([torch.nn.functional.pad(x[:, a:a + n], (0, 0) * (x.dim() - 2) + (0, top - n))  # noqa: E731
                               for a, n in zip(at, lens)])
    S = _d(init).reshape(-1, DIM, DIM) if init is not None else q.new_zeros(len(lens) * HEADS, DIM, DIM)
    # padding tokens have g = beta = k = 0: they leave the state alone
    out, S = _recur(pad(q), pad(k), pad(v), pad(g), pad(beta), S)
    core = torch.cat([out[HEADS * i:HEADS * (i + 1), :n] for i, n in enumerate(lens)], dim=1)
    return {"core": core, "state": S.reshape(len(lens), HEADS, DIM, DIM)}


def _gbeta(d, a, b, layer):
    g = -torch.exp(_d(d["a_log"][layer])) * torch.nn.functional.softplus(a + _d(d["dt"][layer]))
    return g, torch.sigmoid(b)


def _conv_qkv(d, x, hist):
    """Causal conv of 4 taps, SiLU and the unit rows of q and k: x [B][n][6144], hist [B][6144][4]."""
    w = torch.cat([hist[:, :, 1:].transpose(1, 2), x], dim=1)
    n = x.shape[1]
    y = _silu(sum(w[:, i:i + n] * _d(d["conv_w"])[:, i] for i in range(4)))
    q, k, v = (t.reshape(x.shape[0], n, HEADS, DIM) for t in y.split(VAL, dim=-1))
    q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + EPS) for t in (q, k))
    # the 4 newest raw inputs stay as the next call's history
    return q, k, v, torch.cat([hist.transpose(1, 2), x], dim=1)[:, -4:].transpose(1, 2)


def _mixer(d, qkv, z, a, b, state, hist, layer=3):
    """DeltaNet mixer over n tokens of each sequence: gated output [B][n][2048], state, history, and q, k."""
    q, k, v, hist = _conv_qkv(d, qkv, hist)
    g, beta = _gbeta(d, a, b, layer)
    flat = lambda t: t.transpose(1, 2).reshape(-1, t.shape[1], *t.shape[3:])  # noqa: E731
    out, S = _recur(flat(q), flat(k), flat(v), flat(g), flat(beta), state.reshape(-1, DIM, DIM))
    B, n = qkv.shape[:2]
    out = _rms(out.reshape(B, HEADS, n, DIM).transpose(1, 2), _d(d["nw"])).reshape(B, n, VAL) * _silu(z)
    return out, S.reshape(state.shape), hist, q.reshape(B, n, VAL), k.reshape(B, n, VAL)


def _exact_dn_step(case, seed):
    d = _step_inputs(case["batch"], seed)
    one = lambda t: _d(t)[:, None]  # noqa: E731
    out, S, hist, q, k = _mixer(d, one(d["qkv"]), one(d["z"]), one(d["a"]), one(d["b"]), _d(d["state"]), _d(d["conv"]))
    return {"qkv": torch.cat([q, k, out], dim=-1)[:, 0], "state": S, "conv": hist}


def _mlp(d, h):
    xn = _rms(h, 1 + _d(d["post"]))
    m = _silu(xn @ _d(d["gate"]).T) * (xn @ _d(d["up"]).T)
    return m, h + m @ _d(d["down"]).T


def _exact_dn_layer(case, seed):
    d = _layer_inputs(seed)
    h = _d(d["h"])
    xn = _rms(h, 1 + _d(d["norm"]))
    ins = [(xn @ _d(W).T)[None] for W in d["Win"]]
    out, S, hist, q, k = _mixer(d, *ins, _d(d["state"]), _d(d["conv"]))
    h2 = h + out[0] @ _d(d["Wout"]).T
    m, y = _mlp(d, h2)
    return {"qkv": torch.cat([q, k, out], dim=-1)[0], "state": S, "conv": hist, "h2": h2, "m": m, "y": y}


def _attend(d, h, pos0):
    """Attention mixer of the rows of h at positions pos0..: gated output [n][2048] and the KV rows."""
    n = h.shape[0]
    xn = _rms(h, 1 + _d(d["norm"]))
    qg, k, v = (xn @ _d(W).T for W in d["Win"])
    qg = qg.reshape(n, Q_HEADS, 2, HEAD_DIM)
    q, k = _rms(qg[:, :, 0], 1 + _d(d["qn"])), _rms(k.reshape(n, KV_HEADS, HEAD_DIM), 1 + _d(d["kn"]))
    cs = _d(d["rope"])[pos0:pos0 + n].reshape(n, 1, ROT // 2, 2)

    def turn(x):
        a, b, c, s = x[..., :32], x[..., 32:64], cs[..., 0], cs[..., 1]
        return torch.cat([a * c - b * s, b * c + a * s, x[..., 64:]], dim=-1)

    q, k = turn(q), turn(k)
    kv = _d(d["kv"])
    kv[pos0:pos0 + n] = torch.cat([k.reshape(n, 512), v], dim=-1)
    out = torch.empty(n, Q_HEADS, HEAD_DIM, dtype=torch.float64, device=h.device)
    future = torch.arange(pos0 + n, device=h.device)[None] > torch.arange(pos0, pos0 + n, device=h.device)[:, None]
    for i in range(Q_HEADS):
        j = (i // (Q_HEADS // KV_HEADS)) * HEAD_DIM
        sc = (q[:, i] @ kv[:pos0 + n, j:j + HEAD_DIM].T / math.sqrt(HEAD_DIM)).masked_fill(future, -math.inf)
        out[:, i] = torch.softmax(sc, dim=-1) @ kv[:pos0 + n, 512 + j:512 + j + HEAD_DIM]
    return (out * torch.sigmoid(qg[:, :, 1])).reshape(n, -1), kv


def _exact_attn_layer(case, seed):
    d = _attn_inputs(seed, 1, case["pos"], 4096, True)
    out, kv = _attend(d, _d(d["h"]), case["pos"])
    h2 = _d(d["h"]) + out @ _d(d["Wout"]).T
    m, y = _mlp(d, h2)
    return {"out": out, "kv": kv, "h2": h2, "m": m, "y": y}


def _exact_gemv(case, seed):
    return [_d(W) @ _d(x) for items in _prepare_gemv(case, seed)["stages"] for W, x, _ in items]


def _exact_lm_head(case, seed):
    r = _Rand(seed)
    W, = _mats(r, (case["vocab"], HIDDEN))
    x = _d(r.f16(HIDDEN))
    return {"token": None, "logits": torch.cat([_d(w) @ x for w in W.split(32768)])}


def _exact_dn_prompt(case, seed):
    d = _layer_inputs(seed)
    h = _d(_Rand(seed + (1 << 40)).f16(case["tokens"], HIDDEN))
    xn = _rms(h, 1 + _d(d["norm"]))
    out, S, hist, _, _ = _mixer(d, *((xn @ _d(W).T)[None] for W in d["Win"]), _d(d["state"]), _d(d["conv"]))
    return {"y": h + out[0] @ _d(d["Wout"]).T, "gated": out[0], "out_state": S, "conv": hist}


def _exact_mlp_prompt(case, seed):
    r = _Rand(seed)
    d = _mlp_weights(r)
    m, y = _mlp(d, _d(r.f16(case["tokens"], HIDDEN)))
    return {"m": m, "y": y}


def _exact_attn_prompt(case, seed):
    d = _attn_inputs(seed, case["tokens"], case["pos0"], case["pos0"] + case["tokens"], False)
    out, kv = _attend(d, _d(d["h"]), case["pos0"])
    return {"out": out, "kv": kv, "y": _d(d["h"]) + out @ _d(d["Wout"]).T}


# no 64-bit answer for a session: its logits follow the greedy tokens that 16-bit ties decide
_EXACT = {"chunk": _exact_chunk, "dn_step": _exact_dn_step, "dn_layer": _exact_dn_layer, "attn_layer": _exact_attn_layer,
          "gemv": _exact_gemv, "lm_head": _exact_lm_head, "dn_prompt": _exact_dn_prompt, "mlp_prompt": _exact_mlp_prompt,
          "attn_prompt": _exact_attn_prompt}
