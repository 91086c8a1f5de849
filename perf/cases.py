"""What this library is measured on: the calls a streaming speech-to-text
program makes, through the library's Python binding, over the sizes it makes
them at.

Kinds of case (the "kind" of a case dict):

  decode   single-query attention of a token over the decoder's K/V ring with
           the token's row appended: one layer as the decoder's own loop calls
           it ("layer"), or every layer and stream in one call ("step")
  prefill  causal attention of a prompt's tokens over one layer of the ring,
           their rows appended
  window   sliding-window attention of an encoder chunk's frames over one
           layer of the encoder ring, their rows appended
  ffn      a layer's MLP on quantized weights: norm, SwiGLU, down projection
           and residual, for one token or for several rows
  token    one decoder token: embedding, all layers, logits, argmax
  prompt   the decoder's prefill of a prompt: all layers, the last row's logits
  encoder  a chunk of audio: conv stem, all encoder layers into the output
           ring, and the adapter over the groups of frames it completes

Weights are valid blocks of the formats a model file holds ("q4km": Q4_K with
Q6_K where such files have it; "q8_0": every matrix Q8_0), with random codes,
zero mean and the spread of a trained layer.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "voxtral.cpp_amd"))
import vkv  # noqa: E402

# decoder and encoder shapes of bench.py and the tests
LAYERS, CAP, KVH, HD, QH = 26, 8192, 8, 128, 32
KV_DIM, Q_DIM, DIM, HIDDEN, VOCAB = KVH * HD, QH * HD, 3072, 9216, 131072
E_LAYERS, E_CAP, E_HEADS, E_HD, E_WIN = 32, vkv.ENC_KV_CAP, 32, 64, vkv.ENC_WINDOW
E_KV, E_DIM, E_HIDDEN, N_MEL, DOWN, RING = E_HEADS * E_HD, 1280, 5120, 128, 4, 256
EPS, THETA = 1e-5, 1e6

KV_TYPE = {"f32": vkv.F32, "f16": vkv.F16, "q8_0": vkv.Q8_0}
KV_BYTES = {"f32": 4.0, "f16": 2.0, "q8_0": 34 / 32}
Q4, Q6, Q8 = vkv.Q4_K, vkv.Q6_K, vkv.Q8_0
DEC_MATS = {"q": (Q4, Q_DIM, DIM), "k": (Q4, KV_DIM, DIM), "v": (Q6, KV_DIM, DIM),
            "o": (Q4, DIM, Q_DIM), "w1": (Q4, HIDDEN, DIM), "w3": (Q4, HIDDEN, DIM),
            "w2": (Q6, DIM, HIDDEN)}
ENC_MATS = {"q": (Q4, E_KV, E_DIM), "k": (Q4, E_KV, E_DIM), "v": (Q6, E_KV, E_DIM),
            "o": (Q4, E_DIM, E_KV), "w1": (Q4, E_HIDDEN, E_DIM), "w3": (Q4, E_HIDDEN, E_DIM),
            "w2": (Q6, E_DIM, E_HIDDEN)}


def listed():
    return [
        # one layer of a token early in a session: the smallest call there is
        dict(name="layer_f16_1025", kind="decode", call="layer", kv="f16", streams=1, layers=1,
             fill=1024),
        # a long session: the ring is full and each token evicts the oldest
        dict(name="step_f16_full", kind="decode", call="step", kv="f16", streams=1, layers=LAYERS,
             fill=12345),
        # a server with eight streams over q8_0 rings, all wrapped: the most bytes
        dict(name="step_q8_0_8_streams", kind="decode", call="step", kv="q8_0", streams=8,
             layers=LAYERS, fill=9000),
        # a layer's attention for a prompt on the q8_0 ring such a server keeps
        dict(name="prefill_q8_0_199", kind="prefill", kv="q8_0", n=199, pos0=38),
        # a layer's attention for a steady chunk over the default f32 encoder ring
        dict(name="window_f32_16", kind="window", kv="f32", frames=16, q_start=3008),
        # the MLP of one token
        dict(name="ffn_token_q4km", kind="ffn", weights="q4km", side="decoder", rows=1),
        # the MLP of an encoder's last, ragged run, on a Q8_0 file
        dict(name="ffn_encoder_q8_0_61", kind="ffn", weights="q8_0", side="encoder", rows=61),
        # one 80 ms step of live audio
        dict(name="encoder_live_4", kind="encoder", weights="q4km", kv="f32", frames=4, q_start=1296),
        # the start-up block, and each block of a recording that is there whole
        dict(name="encoder_block_128", kind="encoder", weights="q4km", kv="f32", frames=128,
             q_start=1280),
        # one token of a long session
        dict(name="token_q4km_full", kind="token", weights="q4km", fill=12345),
        # the prompt every session starts with
        dict(name="prompt_38", kind="prompt", weights="q4km", kv="f16", n=38, pos0=0),
        # a session taken up again with the text that it had
        dict(name="prompt_503", kind="prompt", weights="q4km", kv="f16", n=503, pos0=0),
    ]


def _log(rng, lo, hi):
    """a size from lo to hi, spread over its logarithm"""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "window", "ffn", "ffn", "token", "prompt",
                       "encoder", "encoder"])
    weights = rng.choice(["q4km", "q4km", "q8_0"])
    if kind == "decode":
        fill = _log(rng, 1, 3 * CAP)
        if rng.random() < 0.5:
            return dict(kind=kind, call="layer", kv=rng.choice(["f16", "f32", "q8_0"]), streams=1,
                        layers=1, fill=fill)
        kv = rng.choice(["f16", "q8_0"])
        return dict(kind=kind, call="step", kv=kv, streams=_log(rng, 1, 8 if kv == "q8_0" else 4),
                    layers=LAYERS, fill=fill)
    if kind == "prefill":
        return dict(kind=kind, kv=rng.choice(["f16", "f32", "q8_0"]), n=_log(rng, 2, 503),
                    pos0=rng.choice([0, 0, 38, 541]))
    if kind == "window":
        return dict(kind=kind, kv=rng.choice(["f16", "f32"]), frames=_log(rng, 1, 128),
                    q_start=_log(rng, 1, 6000) - 1)
    if kind == "ffn":
        return dict(kind=kind, weights=weights, side=rng.choice(["decoder", "encoder"]),
                    rows=_log(rng, 1, 503))
    if kind == "token":
        return dict(kind=kind, weights=weights, fill=_log(rng, 38, 3 * CAP))
    if kind == "prompt":
        return dict(kind=kind, weights=weights, kv="f16",
                    n=_log(rng, 2, 503 if weights == "q4km" else 251), pos0=0)
    return dict(kind=kind, weights=weights, kv=rng.choice(["f16", "f32"]),
                frames=rng.choice([4, 4, 8, 16, 32, _log(rng, 1, 128)]),
                q_start=4 * (_log(rng, 1, 1500) - 1))


# ---- inputs --------------------------------------------------------------
def _gen(seed, *parts):
    g = torch.Generator(device="cuda")
    h = seed & 0xffffffff
    for p in parts:
        h = (h * 1000003 + 17 * int(p) + 12345) & 0x7fffffffffff
    g.manual_seed(h)
    return g


def _blocks(dtype, rows, n_in, g, gain=0.7):
    """random blocks of a [rows][n_in] matrix: zero mean, std about gain / sqrt(n_in)"""
    std = gain / math.sqrt(n_in)
    if dtype == Q8:
        nb = rows * (n_in // 32)
        w = torch.randint(-127, 128, (nb, 34), dtype=torch.int8, device="cuda",
                          generator=g).view(torch.uint8)
        d = torch.empty(nb, device="cuda").uniform_(0.6, 1.4, generator=g) * (std / 73)
        w[:, 0:2] = d.half().view(torch.uint8).view(nb, 2)
        return w.view(-1)
    nb = rows * (n_in // 256)
    w = torch.randint(0, 256, (nb, vkv.KQ_BLOCK_BYTES[dtype]), dtype=torch.uint8, device="cuda",
                      generator=g)
    d = torch.empty(nb, device="cuda").uniform_(0.6, 1.4, generator=g)
    if dtype == Q4:
        d = (d * (std / 200)).half()
        w[:, 0:2] = d.view(torch.uint8).view(nb, 2)
        w[:, 2:4] = (d.float() * 7.5).half().view(torch.uint8).view(nb, 2)
        sc = torch.randint(20, 64, (nb, 8), dtype=torch.uint8, device="cuda", generator=g)
        # scale and min of a sub-block alike: the codes' mean (7.5) maps to zero
        lo, hi = sc[:, :4], sc[:, 4:]
        w[:, 4:8] = lo | ((hi >> 4) << 6)
        w[:, 8:12] = lo | ((hi >> 4) << 6)
        w[:, 12:16] = (hi & 15) | ((hi & 15) << 4)
        return w.view(-1)
    sc = torch.randint(20, 128, (nb, 16), dtype=torch.int8, device="cuda", generator=g)
    sign = torch.randint(0, 2, (nb, 16), dtype=torch.int8, device="cuda", generator=g) * 2 - 1
    w[:, 192:208] = (sc * sign).view(torch.uint8)
    w[:, 208:210] = (d * (std / 1450)).half().view(torch.uint8).view(nb, 2)
    return w.view(-1)


def _type(weights, dtype):
    return Q8 if weights == "q8_0" else dtype


def _mats(table, weights, g, names=None):
    # the projections back into the residual stream are a fifth of the others,
    # so that a deep stack adds up to what one layer's input is
    return {k: _blocks(_type(weights, dt), r, n, g, 0.15 if k in ("o", "w2") else 0.7)
            for k, (dt, r, n) in table.items() if names is None or k in names}


def _norm(n, g):
    return torch.empty(n, device="cuda").uniform_(0.5, 1.5, generator=g)


def _al(t):
    return (t.data_ptr() + 255) & ~255


def _ws(n_bytes):
    return torch.empty(n_bytes + 512, dtype=torch.uint8, device="cuda")


def _rows(seed, which, stream, layer, n, width):
    return torch.randn(n, width, device="cuda", generator=_gen(seed, 7, which, stream, layer))


def _stream():
    return torch.cuda.current_stream().cuda_stream


class _Mem:
    """device memory of `owner` as a tensor's base: the tensor and its views
    keep this object, and so the owner, alive"""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (int(ptr), False), "shape": tuple(shape),
                                         "typestr": typestr, "strides": None, "version": 3}


def _views(cache, kv):
    """the cache's K and V storage as tensors [stream][layer][slot][row]"""
    lay = cache.layout
    w = {"f32": cache.kv_dim, "f16": cache.kv_dim, "q8_0": cache.row_bytes}[kv]
    ts = {"f32": "<f4", "f16": "<f2", "q8_0": "|u1"}[kv]
    shape = (cache.n_streams, cache.n_layers, cache.capacity, w)
    return [torch.as_tensor(_Mem(cache, p, shape, ts), device="cuda") for p in (lay.k_base, lay.v_base)]


def _fill_cache(cache, seed, first, last):
    """rows of positions [first, last) in every stream and layer"""
    n, cap, width = last - first, cache.capacity, cache.kv_dim
    if n <= 0:
        return
    segs = [(a, b - a) for a, b in _slots(first, n, cap)]
    for s in range(cache.n_streams):
        for l in range(cache.n_layers):
            k, v = (_rows(seed, i, s, l, n, width) for i in (0, 1))
            cache.append(s, l, 1, segs, k.data_ptr(), v.data_ptr(), hip_stream=_stream())
    torch.cuda.synchronize()   # the source rows are freed on return


def _ring(cap, used, pos):
    r = vkv.new_ring(cap)
    r.used, r.next_absolute_position, r.oldest_absolute_position = used, pos, pos - used
    return r


def _ring_copy(r):
    c = vkv.Ring()
    ctypes.pointer(c)[0] = r
    return c


def _fill(case):
    """positions a decoder ring holds, and the next one (streams differ a little)"""
    return [(min(CAP, case["fill"] + 37 * s), case["fill"] + 37 * s)
            for s in range(case.get("streams", 1))]


# ---- decode / prefill / window -------------------------------------------
def _prepare_decode(case, seed):
    ns, nl = case["streams"], case["layers"]
    st = dict(case=case)
    c = st["cache"] = vkv.Cache(n_streams=ns, n_layers=nl, capacity=CAP, n_kv_heads=KVH, head_dim=HD,
                                n_q_heads=QH, dtype=KV_TYPE[case["kv"]])
    for s, (used, pos) in enumerate(_fill(case)):
        segs = [(a, b - a) for a, b in _slots(pos - used, used, CAP)]
        for l in range(nl):
            k, v = (_rows(seed, i, s, l, used, KV_DIM) for i in (0, 1))
            c.append(s, l, 1, segs, k.data_ptr(), v.data_ptr(), hip_stream=_stream())
    torch.cuda.synchronize()
    st["q"], st["k"], st["v"] = _decode_inputs(case, seed)
    st["out"] = torch.empty(ns, nl, Q_DIM, device="cuda")
    st["rings"] = [_ring(CAP, u, p) for u, p in _fill(case)]
    st["pos"] = [p for _, p in _fill(case)]
    kv = _views(c, case["kv"])
    st["rows"] = [t[s, :, p % CAP] for t in kv for s, p in enumerate(st["pos"])]
    return st


def _decode_inputs(case, seed):
    g = _gen(seed, 1)
    return [torch.randn(case["streams"], case["layers"], w, device="cuda", generator=g)
            for w in (Q_DIM, KV_DIM, KV_DIM)]


def _run_decode(st):
    case, c = st["case"], st["cache"]
    a = (st["q"].data_ptr(), st["k"].data_ptr(), st["v"].data_ptr(), st["out"].data_ptr())
    scale = HD ** -0.5
    if case["call"] == "layer":
        ring = _ring_copy(st["rings"][0])
        plan = vkv.decoder_plan(ring, st["pos"][0], 1)
        c.decoder_layer_step(0, plan, st["pos"][0], 0, 1, *a, scale, rope_theta=THETA,
                             hip_stream=_stream())
        vkv.decoder_commit(ring, plan)
    else:
        rings = (vkv.Ring * len(st["rings"]))(*st["rings"])
        c.decoder_step_rope(0, rings, st["pos"], 0, case["layers"], *a, scale, THETA,
                            hip_stream=_stream())
    return dict(out=st["out"], rows=st["rows"])


def _prepare_prefill(case, seed):
    st = dict(case=case)
    c = st["cache"] = vkv.Cache(n_streams=1, n_layers=1, capacity=CAP, n_kv_heads=KVH, head_dim=HD,
                                n_q_heads=QH, dtype=KV_TYPE[case["kv"]])
    n, pos0 = case["n"], case["pos0"]
    _fill_cache(c, seed, 0, pos0)
    st["q"], st["k"], st["v"] = _prefill_inputs(n, Q_DIM, KV_DIM, seed)
    st["out"] = torch.empty(n, Q_DIM, device="cuda")
    st["ring"] = _ring(CAP, pos0, pos0)
    st["rows"] = [t[0, 0, pos0:pos0 + n] for t in _views(c, case["kv"])]
    return st


def _prefill_inputs(n, qw, kw, seed):
    g = _gen(seed, 2)
    return [torch.randn(n, w, device="cuda", generator=g) for w in (qw, kw, kw)]


def _run_prefill(st):
    st["cache"].decoder_prefill(0, _ring_copy(st["ring"]), 0, 1, st["case"]["n"], st["q"].data_ptr(),
                                st["k"].data_ptr(), st["v"].data_ptr(), st["out"].data_ptr(),
                                HD ** -0.5, hip_stream=_stream())
    return dict(out=st["out"], rows=st["rows"])


def _slots(first, n, cap):
    """ring slots of n rows from row `first`, as at most two ranges"""
    s, head = first % cap, min(n, cap - first % cap)
    return ([(s, s + head)] if n > 0 else []) + ([(0, n - head)] if n > head else [])


def _prepare_window(case, seed):
    st = dict(case=case)
    c = st["cache"] = vkv.Cache(n_streams=1, n_layers=1, capacity=E_CAP, n_kv_heads=E_HEADS,
                                head_dim=E_HD, n_q_heads=E_HEADS, dtype=KV_TYPE[case["kv"]])
    n, q0 = case["frames"], case["q_start"]
    _fill_cache(c, seed, max(0, q0 - E_WIN), q0)
    st["q"], st["k"], st["v"] = _prefill_inputs(n, E_KV, E_KV, seed)
    st["out"] = torch.empty(n, E_KV, device="cuda")
    st["rows"] = [t[0, 0, a:b] for t in _views(c, case["kv"]) for a, b in _slots(q0, n, E_CAP)]
    return st


def _run_window(st):
    case = st["case"]
    plan = vkv.enc_plan(case["q_start"], case["frames"], E_CAP, E_WIN)
    st["cache"].enc_step(0, plan, E_WIN, 0, 1, st["q"].data_ptr(), st["k"].data_ptr(),
                         st["v"].data_ptr(), st["out"].data_ptr(), E_HD ** -0.5,
                         hip_stream=_stream())
    return dict(out=st["out"], rows=st["rows"])


# ---- the MLP block --------------------------------------------------------
def _ffn_shape(case):
    dec = case["side"] == "decoder"
    return (DEC_MATS if dec else ENC_MATS), (DIM if dec else E_DIM), (HIDDEN if dec else E_HIDDEN)


def _ffn_inputs(case, seed):
    mats, dim, _ = _ffn_shape(case)
    g = _gen(seed, 3)
    st = _mats(mats, case["weights"], g, ("w1", "w2", "w3"))
    st["norm"] = _norm(dim, g)
    st["x"] = torch.randn(case["rows"], dim, device="cuda", generator=g)
    # the decoder's ada scale, the encoder's norm and output biases
    st["extra"] = torch.empty(2, dim, device="cuda").uniform_(-0.3, 0.3, generator=g)
    return st


def _prepare_ffn(case, seed):
    _, dim, hidden = _ffn_shape(case)
    st = dict(_ffn_inputs(case, seed), case=case)
    st["h"] = torch.empty(case["rows"], hidden, device="cuda")
    st["y"] = torch.empty(case["rows"], dim, device="cuda")
    st["wb"] = max(vkv.matmul_workspace(case["rows"], dim), vkv.matmul_workspace(case["rows"], hidden))
    st["ws"] = _ws(st["wb"])
    return st


def _run_ffn(st):
    case = st["case"]
    mats, dim, hidden = _ffn_shape(case)
    dt = {k: _type(case["weights"], mats[k][0]) for k in mats}
    x, h, y, norm = (st[k].data_ptr() for k in ("x", "h", "y", "norm"))
    e0, e1 = st["extra"][0].data_ptr(), st["extra"][1].data_ptr()
    dec = case["side"] == "decoder"
    up = [(st["w1"].data_ptr(), dt["w1"], hidden, h), (st["w3"].data_ptr(), dt["w3"], hidden, None)]
    sp = _stream()
    if case["rows"] == 1 and dec:
        vkv.matvec(x, dim, up, norm_w_ptr=norm, ada_ptr=e0, eps=EPS, epilogue=vkv.MV_SWIGLU,
                   hip_stream=sp)
        vkv.matvec(h, hidden, [(st["w2"].data_ptr(), dt["w2"], dim, y, x)], hip_stream=sp)
    else:
        ws, wb = _al(st["ws"]), st["wb"]
        vkv.matmul(x, case["rows"], dim, up, ws, wb, norm_w_ptr=norm, norm_b_ptr=None if dec else e0,
                   ada_ptr=e0 if dec else None, eps=EPS, epilogue=vkv.MV_SWIGLU, hip_stream=sp)
        vkv.matmul(h, case["rows"], hidden,
                   [(st["w2"].data_ptr(), dt["w2"], dim, y, x, None if dec else e1)], ws, wb,
                   hip_stream=sp)
    return dict(h=st["h"], y=st["y"])


# ---- the decoder ----------------------------------------------------------
def _dec_weights(case, seed):
    """per layer: matrices, norms and ada scale; the embedding table (tied to
    the logits) and the final norm"""
    g = _gen(seed, 4)
    ls = []
    for _ in range(LAYERS):
        m = _mats(DEC_MATS, case["weights"], g)
        m["n1"], m["n2"] = _norm(DIM, g), _norm(DIM, g)
        m["ada"] = torch.empty(DIM, device="cuda").uniform_(-0.3, 0.3, generator=g)
        ls.append(m)
    return ls, _blocks(_type(case["weights"], Q6), VOCAB, DIM, g), _norm(DIM, g)


def _dec_model(case, ls, table, out_norm):
    arr = (vkv.DecLayer * LAYERS)()
    dt = {k: _type(case["weights"], DEC_MATS[k][0]) for k in DEC_MATS}
    for l, m in enumerate(ls):
        p = {k: t.data_ptr() for k, t in m.items()}
        arr[l] = vkv.DecLayer(p["n1"], p["q"], p["k"], p["v"], p["o"], dt["q"], dt["k"], dt["v"],
                              dt["o"], p["n2"], p["ada"], p["w1"], p["w2"], p["w3"], dt["w1"],
                              dt["w2"], dt["w3"])
    tt = _type(case["weights"], Q6)
    return vkv.DecModel(LAYERS, DIM, HIDDEN, QH, KVH, HD, VOCAB, EPS, THETA, table.data_ptr(), tt,
                        out_norm.data_ptr(), table.data_ptr(), tt,
                        ctypes.cast(arr, ctypes.POINTER(vkv.DecLayer))), arr


def _dec_inputs(case, seed):
    g = _gen(seed, 5)
    n = case.get("n", 1)
    ids = torch.randint(0, VOCAB, (n,), device="cuda", generator=g)
    return [int(i) for i in ids.tolist()], torch.randn(RING, DIM, device="cuda", generator=g)


def _prepare_dec(case, seed):
    st = dict(case=case)
    st["w"] = _dec_weights(case, seed)
    st["model"], st["arr"] = _dec_model(case, *st["w"])
    kv = case.get("kv", "f16")
    c = st["cache"] = vkv.Cache(n_streams=1, n_layers=LAYERS, capacity=CAP, n_kv_heads=KVH,
                                head_dim=HD, n_q_heads=QH, dtype=KV_TYPE[kv])
    pos = case["fill"] if case["kind"] == "token" else case["pos0"]
    used = min(CAP, pos)
    _fill_cache(c, seed, pos - used, pos)
    st["ring"], st["pos"] = _ring(CAP, used, pos), pos
    st["ids"], st["audio"] = _dec_inputs(case, seed)
    st["aring"] = vkv.RowRing(st["audio"].data_ptr(), RING, DIM)
    st["logits"] = torch.empty(VOCAB, device="cuda")
    st["tok"] = torch.empty(1, dtype=torch.int32, device="cuda")
    n = len(st["ids"])
    st["wb"] = (vkv.decoder_token_workspace(st["model"]) if case["kind"] == "token"
                else vkv.decoder_prompt_workspace(st["model"], n))
    st["ws"] = _ws(st["wb"])
    # the workspace's first rows hold the residual stream after the call
    off = _al(st["ws"]) - st["ws"].data_ptr()
    st["x"] = st["ws"][off:off + 4 * n * DIM].view(torch.float32).view(n, DIM)
    s = pos % CAP
    st["rows"] = [t[0, :, s:s + n] for t in _views(c, kv)]
    return st


def _run_dec(st):
    ring = _ring_copy(st["ring"])
    if st["case"]["kind"] == "token":
        vkv.decoder_token(st["cache"], 0, ring, st["model"], st["ids"][0],
                          st["audio"].data_ptr() + 4 * DIM * (st["pos"] % RING),
                          st["logits"].data_ptr(), st["tok"].data_ptr(), _al(st["ws"]), st["wb"],
                          hip_stream=_stream())
    else:
        vkv.decoder_prompt(st["cache"], 0, ring, st["model"], st["ids"], st["aring"],
                           st["logits"].data_ptr(), st["tok"].data_ptr(), _al(st["ws"]), st["wb"],
                           hip_stream=_stream())
    return dict(logits=st["logits"], x=st["x"], rows=st["rows"])


# ---- the encoder ----------------------------------------------------------
def _enc_weights(case, seed):
    g = _gen(seed, 6)

    def vec(n, s=0.1):
        return torch.randn(n, device="cuda", generator=g) * s

    ls = []
    for _ in range(E_LAYERS):
        m = _mats(ENC_MATS, case["weights"], g)
        m["n1"], m["n2"] = _norm(E_DIM, g), _norm(E_DIM, g)
        m["n1b"], m["n2b"], m["ob"], m["w2b"] = (vec(E_DIM) for _ in range(4))
        m["qb"], m["vb"] = vec(E_KV), vec(E_KV)
        ls.append(m)
    top = dict(norm=_norm(E_DIM, g), norm_b=vec(E_DIM), b0=vec(E_DIM), b1=vec(E_DIM))
    top["c0"] = (torch.randn(E_DIM, N_MEL, 3, device="cuda", generator=g) * 0.05).half()
    top["c1"] = (torch.randn(E_DIM, E_DIM, 3, device="cuda", generator=g) * 0.02).half()
    top["a0"] = _blocks(_type(case["weights"], Q4), DIM, E_DIM * DOWN, g)
    top["a2"] = _blocks(_type(case["weights"], Q4), DIM, DIM, g)
    return ls, top


def _groups(case):
    """the adapter groups that the chunk completes"""
    g0, g1 = case["q_start"] // DOWN, (case["q_start"] + case["frames"]) // DOWN
    return g0, g1 - g0


def _enc_inputs(case, seed):
    plan = vkv.enc_plan(case["q_start"], case["frames"], E_CAP, E_WIN)
    g = _gen(seed, 8)
    return plan, torch.randn(N_MEL, plan.conv_mel_end - plan.conv_mel_start, device="cuda", generator=g)


def _prepare_enc(case, seed):
    st = dict(case=case)
    ls, top = st["w"] = _enc_weights(case, seed)
    dt = {k: _type(case["weights"], ENC_MATS[k][0]) for k in ENC_MATS}
    arr = st["arr"] = (vkv.EncLayer * E_LAYERS)()
    for l, m in enumerate(ls):
        p = {k: t.data_ptr() for k, t in m.items()}
        arr[l] = vkv.EncLayer(p["n1"], p["n1b"], p["q"], p["k"], p["v"], p["o"], dt["q"], dt["k"],
                              dt["v"], dt["o"], p["qb"], p["vb"], p["ob"], p["n2"], p["n2b"], p["w1"],
                              p["w2"], p["w3"], dt["w1"], dt["w2"], dt["w3"], p["w2b"])
    st["model"] = vkv.EncModel(E_LAYERS, E_DIM, E_HIDDEN, E_HEADS, E_HD, EPS, THETA,
                               top["norm"].data_ptr(), top["norm_b"].data_ptr(),
                               ctypes.cast(arr, ctypes.POINTER(vkv.EncLayer)))
    n, q0 = case["frames"], case["q_start"]
    c = st["cache"] = vkv.Cache(n_streams=1, n_layers=E_LAYERS, capacity=E_CAP, n_kv_heads=E_HEADS,
                                head_dim=E_HD, n_q_heads=E_HEADS, dtype=KV_TYPE[case["kv"]])
    _fill_cache(c, seed, max(0, q0 - E_WIN), q0)
    st["plan"], st["mel"] = _enc_inputs(case, seed)
    st["x"] = torch.empty(n, E_DIM, device="cuda")
    st["enc"] = torch.zeros(RING, E_DIM, device="cuda")
    st["emb"] = torch.zeros(RING, DIM, device="cuda")
    st["enc_r"] = vkv.RowRing(st["enc"].data_ptr(), RING, E_DIM)
    st["emb_r"] = vkv.RowRing(st["emb"].data_ptr(), RING, DIM)
    st["enc_rows"] = [st["enc"][a:b] for a, b in _slots(q0, n, RING)]
    st["emb_rows"] = [st["emb"][a:b] for a, b in _slots(*_groups(case), RING)]
    at = _type(case["weights"], Q4)
    st["ad"] = vkv.Adapter(top["a0"].data_ptr(), top["a2"].data_ptr(), at, at, E_DIM, DIM, DOWN)
    conv_len = st["mel"].shape[1]
    st["cb"] = vkv.enc_conv_stem_workspace(conv_len, N_MEL, E_DIM, n)
    st["eb"] = vkv.encoder_chunk_workspace(st["model"], n)
    st["ab"] = vkv.adapter_workspace(st["ad"], max(1, _groups(case)[1]))
    st["cw"], st["ew"], st["aw"] = _ws(st["cb"]), _ws(st["eb"]), _ws(st["ab"])
    return st


def _run_enc(st):
    case, plan, sp = st["case"], st["plan"], _stream()
    top = st["w"][1]
    vkv.enc_conv_stem(st["mel"].data_ptr(), N_MEL, plan, top["c0"].data_ptr(), top["b0"].data_ptr(),
                      top["c1"].data_ptr(), top["b1"].data_ptr(), E_DIM, st["x"].data_ptr(),
                      _al(st["cw"]), st["cb"], hip_stream=sp)
    vkv.encoder_chunk_ring(st["cache"], 0, plan, E_WIN, st["model"], st["x"].data_ptr(), st["enc_r"],
                           _al(st["ew"]), st["eb"], hip_stream=sp)
    g0, n = _groups(case)
    if n > 0:
        vkv.adapter_commit(st["ad"], st["enc_r"], st["emb_r"], g0, n, _al(st["aw"]), st["ab"],
                           hip_stream=sp)
    return dict(x=st["x"], enc=st["enc_rows"], emb=st["emb_rows"])


_PREPARE = dict(decode=_prepare_decode, prefill=_prepare_prefill, window=_prepare_window,
                ffn=_prepare_ffn, token=_prepare_dec, prompt=_prepare_dec, encoder=_prepare_enc)
_RUN = dict(decode=_run_decode, prefill=_run_prefill, window=_run_window, ffn=_run_ffn,
            token=_run_dec, prompt=_run_dec, encoder=_run_enc)


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["case"]["kind"]](state)


# ---- the work a pass cannot do without -----------------------------------
def _mat_bytes(table, weights, names=None):
    return sum(r * n // 256 * vkv.KQ_BLOCK_BYTES[_type(weights, dt)]
               for k, (dt, r, n) in table.items() if names is None or k in names)


def _mat_params(table, names=None):
    return sum(r * n for k, (_, r, n) in table.items() if names is None or k in names)


def _pairs(n, keys, window=0):
    """(query, key) pairs of n causal queries, the last one over `keys` keys"""
    per = [keys - (n - 1 - i) for i in range(n)]
    return sum(min(p, window) if window else p for p in per)


def work(case):
    kind = case["kind"]
    if kind == "decode":
        b = f = 0
        for used, _ in _fill(case):
            keys = min(CAP, used + 1)
            b += case["layers"] * (2 * keys * KV_DIM * KV_BYTES[case["kv"]]
                                   + 2 * KV_DIM * (4 + KV_BYTES[case["kv"]]) + 8 * Q_DIM)
            f += case["layers"] * 4 * keys * Q_DIM
        return dict(bytes=b, flops=f)
    if kind == "prefill":
        n, keys = case["n"], case["n"] + case["pos0"]
        return dict(bytes=2 * keys * KV_DIM * KV_BYTES[case["kv"]] + 8 * n * KV_DIM + 8 * n * Q_DIM,
                    flops=4 * _pairs(n, keys) * Q_DIM)
    if kind == "window":
        n, keys = case["frames"], min(case["q_start"], E_WIN - 1) + case["frames"]
        return dict(bytes=2 * keys * E_KV * KV_BYTES[case["kv"]] + 8 * n * E_KV + 8 * n * E_KV,
                    flops=4 * _pairs(n, keys, E_WIN) * E_KV)
    if kind == "ffn":
        mats, dim, _ = _ffn_shape(case)
        names = ("w1", "w2", "w3")
        return dict(bytes=_mat_bytes(mats, case["weights"], names) + 8 * case["rows"] * dim,
                    flops=2 * case["rows"] * _mat_params(mats, names))
    if kind in ("token", "prompt"):
        n = case.get("n", 1)
        keys = min(CAP, case["fill"] + 1) if kind == "token" else case["pos0"] + n
        head = VOCAB * DIM // 256 * vkv.KQ_BLOCK_BYTES[_type(case["weights"], Q6)]
        kvb = KV_BYTES[case.get("kv", "f16")]
        return dict(bytes=LAYERS * (_mat_bytes(DEC_MATS, case["weights"]) + 2 * keys * KV_DIM * kvb)
                    + head + 4 * n * DIM + 4 * VOCAB,
                    flops=2 * n * LAYERS * _mat_params(DEC_MATS) + 2 * VOCAB * DIM
                    + 4 * LAYERS * _pairs(n, keys) * Q_DIM)
    n, q0 = case["frames"], case["q_start"]
    keys = min(q0, E_WIN - 1) + n
    conv = 3 * E_DIM * (N_MEL + E_DIM)
    at = vkv.KQ_BLOCK_BYTES[_type(case["weights"], Q4)] / 256
    ad = DIM * (E_DIM * DOWN + DIM)
    g = max(0, _groups(case)[1])
    return dict(bytes=E_LAYERS * (_mat_bytes(ENC_MATS, case["weights"])
                                  + 2 * keys * E_KV * KV_BYTES[case["kv"]])
                + 2 * conv + (at * ad if g else 0) + 4 * n * (2 * N_MEL + E_DIM) + 4 * g * DIM,
                flops=E_LAYERS * (2 * n * _mat_params(ENC_MATS) + 4 * _pairs(n, keys, E_WIN) * E_KV)
                + 2 * n * 3 * E_DIM * (2 * N_MEL + E_DIM) + 2 * g * ad)


def tolerance(case):
    """About four times the largest difference measured between a path, the same
    path on the library's alternative kernels (other chunks, other sums) and
    64 bits, over these cases and draws."""
    kind, kv = case["kind"], case.get("kv")
    if kind in ("token", "prompt", "encoder"):
        # every product rounds its input to 8 bits: where one sum is rounded
        # otherwise, codes flip in all layers that follow (0.4 to 1.8 % measured)
        return dict(rel=0.03, max=0.3)
    if kind == "ffn":
        # one flipped code of the second product's input: 7e-5, 4e-3
        return dict(rel=3e-4, max=2e-2)
    if kv == "f16":
        # f16 queries and softmax weights: 3e-4, 1.5e-3; a rotated key's rows
        # may round to the next f16
        return dict(rel=1.2e-3, max=6e-3)
    if kv == "q8_0" and kind == "decode":
        # an 8-bit query, f16 weights in some kernels: 2e-4, 5e-3; codes of a
        # rotated key's row on a tie: 4e-5 of them
        return dict(rel=8e-4, max=2e-2, differ=2e-4)
    # 32 bits throughout: 7e-7, 5e-6
    return dict(rel=3e-6, max=2e-5)


# ---- 64 bits --------------------------------------------------------------
def _deq(dtype, blocks, rows, n_in):
    """the values of a [rows][n_in] matrix's blocks, in 64 bits"""
    f16 = lambda t: t.contiguous().view(torch.float16).double()  # noqa: E731
    if dtype == Q8:
        w = blocks.view(-1, 34)
        return (f16(w[:, 0:2]) * w[:, 2:].contiguous().view(torch.int8).double()).view(rows, n_in)
    w = blocks.view(-1, vkv.KQ_BLOCK_BYTES[dtype])
    nb = w.shape[0]
    if dtype == Q4:
        d, dmin = f16(w[:, 0:2]), f16(w[:, 2:4])
        s0, s1, s2 = w[:, 4:8], w[:, 8:12], w[:, 12:16]
        sc = torch.cat([s0 & 63, (s2 & 15) | ((s0 >> 6) << 4)], 1).double()
        mn = torch.cat([s1 & 63, (s2 >> 4) | ((s1 >> 6) << 4)], 1).double()
        qs = w[:, 16:].reshape(nb, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(nb, 8, 32).double()
        return (q * (d * sc)[:, :, None] - (dmin * mn)[:, :, None]).view(rows, n_in)
    ql = w[:, :128].reshape(nb, 2, 1, 2, 32)
    nib = torch.cat([ql & 15, ql >> 4], 2).view(nb, 2, 4, 32)
    qh = w[:, 128:192].reshape(nb, 2, 1, 32)
    top = torch.cat([(qh >> (2 * g)) & 3 for g in range(4)], 2)
    q = (nib | (top << 4)).double() - 32
    sc = w[:, 192:208].contiguous().view(torch.int8).double().view(nb, 2, 4, 2, 1)
    return (q.view(nb, 2, 4, 2, 16) * sc * f16(w[:, 208:210])[:, :, None, None, None]).view(rows, n_in)


def _image(h, q80):
    """the 8-bit image of a product's input rows that the weight formats
    define, as values: Q8_K for the k-quants, q8_0 for Q8_0"""
    n = h.shape[-1]
    b = h.float().view(-1, 32 if q80 else 256)
    amax, at = b.abs().max(1, keepdim=True)
    if q80:
        d = (amax / 127).half().double()
        q = torch.round(b * torch.where(amax > 0, 127 / amax, torch.zeros_like(amax))).double()
    else:
        iscale = -127 / b.gather(1, at)
        q = torch.where(amax > 0, torch.clamp(torch.round(iscale * b), max=127), 0 * b).double()
        d = torch.where(amax > 0, 1 / iscale, 0 * amax).double()
    return (q * d).view(-1, n)


def _mul(x, blocks, spec, weights):
    dt = _type(weights, spec[0])
    return _image(x, dt == Q8) @ _deq(dt, blocks, spec[1], spec[2]).T


def _rms(x, w, b=None, ada=None):
    h = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()
    if b is not None:
        h = h + b.double()
    return h if ada is None else h + h * ada.double()


def _silu(x):
    return x / (1 + torch.exp(-x))


def _gelu(x):
    return 0.5 * x * (1 + torch.erf(x * 0.5 ** 0.5))


def _rope64(x, pos, hd):
    """RoPE of rows [n][heads * hd] at pos [n], the angle by the f32 running product"""
    ts = torch.tensor(np.float32(THETA) ** np.float32(-2.0 / hd), device="cuda")
    t, a = pos.float(), []
    for _ in range(hd // 2):
        a.append(t)
        t = t * ts
    a = torch.stack(a, 1).double()[:, None]
    y = x.view(x.shape[0], -1, hd // 2, 2)
    c, s = a.cos(), a.sin()
    return torch.stack([y[..., 0] * c - y[..., 1] * s, y[..., 0] * s + y[..., 1] * c], -1).view(x.shape)


def _q8_rows(x):
    """q8_0 cache rows of x [n][w]: (bytes [n][w / 32 * 34], values)"""
    b = x.float().view(x.shape[0], -1, 32)
    amax = b.abs().amax(2, keepdim=True)
    d = amax / 127
    idd = torch.where(d > 0, 1 / d, torch.zeros_like(d))
    y = b * idd
    q = torch.sign(y) * torch.floor(y.abs() + 0.5)
    dh = d.half()
    by = torch.cat([dh.view(torch.uint8), q.to(torch.int8).view(torch.uint8)], 2)
    return by.view(x.shape[0], -1), (q.double() * dh.double()).view(x.shape)


def _stored(x, kv):
    """rows as the cache holds them: (the output's form, values in 64 bits)"""
    if kv == "q8_0":
        return _q8_rows(x)
    y = x.half() if kv == "f16" else x.float()
    return y, y.double()


def _attn64(q, k, v, qpos, kpos, heads, kvh, window=0):
    n, m, hd = q.shape[0], k.shape[0], q.shape[1] // heads
    ok = kpos[None] <= qpos[:, None]
    if window:
        ok &= kpos[None] > qpos[:, None] - window
    out = []
    qh, kh, vh = q.view(n, heads, hd), k.view(m, kvh, hd), v.view(m, kvh, hd)
    for h in range(heads):
        s = qh[:, h] @ kh[:, h * kvh // heads].T * hd ** -0.5
        out.append(torch.softmax(s.masked_fill(~ok, -math.inf), 1) @ vh[:, h * kvh // heads])
    return torch.stack(out, 1).view(n, -1)


def _arange(a, b):
    return torch.arange(a, b, device="cuda")


def _exact_decode(case, seed):
    q, k, v = _decode_inputs(case, seed)
    kv, out, rows = case["kv"], [], [[], []]
    for s, (used, pos) in enumerate(_fill(case)):
        at = torch.tensor([pos], device="cuda")
        for l in range(case["layers"]):
            qr, kr = (_rope64(t[s, l][None].double(), at, HD) for t in (q, k))
            if kv == "q8_0":   # such a ring's query is quantized as its rows are
                qr = _q8_rows(qr)[1]
            keep = min(used, CAP - 1)
            old = [_stored(_rows(seed, i, s, l, used, KV_DIM), kv)[1][used - keep:] for i in (0, 1)]
            new = [_stored(t, kv) for t in (kr, v[s, l][None])]
            out.append(_attn64(qr, *(torch.cat([o, n[1]]) for o, n in zip(old, new)), at,
                               _arange(pos - keep, pos + 1), QH, KVH))
            for i in (0, 1):
                rows[i].append(new[i][0][0])
    shape = (case["streams"], case["layers"], -1)
    rows = [torch.stack(r).view(shape) for r in rows]
    return dict(out=torch.stack(out).view(*shape[:2], Q_DIM), rows=[r[s] for r in rows for s in range(shape[0])])


def _exact_prefill(case, seed):
    q, k, v = _prefill_inputs(case["n"], Q_DIM, KV_DIM, seed)
    n, p, kv = case["n"], case["pos0"], case["kv"]
    new = [_stored(t, kv) for t in (k, v)]
    old = [_stored(_rows(seed, i, 0, 0, p, KV_DIM), kv)[1] for i in (0, 1)]
    out = _attn64(q.double(), *(torch.cat([o, t[1]]) for o, t in zip(old, new)), _arange(p, p + n),
                  _arange(0, p + n), QH, KVH)
    return dict(out=out, rows=[t[0] for t in new])


def _cut(rows, first, cap):
    """rows in the pieces that _slots makes of them"""
    return list(rows.split([b - a for a, b in _slots(first, rows.shape[0], cap)]))


def _exact_window(case, seed):
    n, q0, kv = case["frames"], case["q_start"], case["kv"]
    q, k, v = _prefill_inputs(n, E_KV, E_KV, seed)
    p = min(q0, E_WIN)
    new = [_stored(t, kv) for t in (k, v)]
    old = [_stored(_rows(seed, i, 0, 0, p, E_KV), kv)[1] for i in (0, 1)]
    out = _attn64(q.double(), *(torch.cat([o, t[1]]) for o, t in zip(old, new)), _arange(q0, q0 + n),
                  _arange(q0 - p, q0 + n), E_HEADS, E_HEADS, E_WIN)
    return dict(out=out, rows=[r for t in new for r in _cut(t[0], q0, E_CAP)])


def _exact_ffn(case, seed):
    mats, _, _ = _ffn_shape(case)
    i, wt, dec = _ffn_inputs(case, seed), case["weights"], case["side"] == "decoder"
    x, e = i["x"].double(), i["extra"]
    h = _rms(x, i["norm"], None if dec else e[0], e[0] if dec else None)
    h = _silu(_mul(h, i["w1"], mats["w1"], wt)) * _mul(h, i["w3"], mats["w3"], wt)
    y = x + _mul(h, i["w2"], mats["w2"], wt) + (0 if dec else e[1].double())
    return dict(h=h, y=y)


def _exact_dec(case, seed):
    ls, table, out_norm = _dec_weights(case, seed)
    ids, audio = _dec_inputs(case, seed)
    wt, kv, n = case["weights"], case.get("kv", "f16"), len(ids)
    pos = case["fill"] if case["kind"] == "token" else case["pos0"]
    used = min(CAP, pos)
    at = _arange(pos, pos + n)
    tt = _type(wt, Q6)
    rb = DIM // 256 * vkv.KQ_BLOCK_BYTES[tt]
    x = _deq(tt, table.view(VOCAB, rb)[torch.tensor(ids, device="cuda")], n, DIM) + audio[at % RING].double()
    rows = [[], []]
    for l, m in enumerate(ls):
        h = _rms(x, m["n1"])
        q, k, v = (_mul(h, m[i], DEC_MATS[i], wt) for i in "qkv")
        q, k = _rope64(q, at, HD), _rope64(k, at, HD)
        keep = min(used, CAP - n)
        new = [_stored(t, kv) for t in (k, v)]
        old = [_stored(_rows(seed, i, 0, l, used, KV_DIM), kv)[1][used - keep:] for i in (0, 1)]
        a = _attn64(q, *(torch.cat([o, t[1]]) for o, t in zip(old, new)), at,
                    _arange(pos - keep, pos + n), QH, KVH)
        x = x + _mul(a, m["o"], DEC_MATS["o"], wt)
        h = _rms(x, m["n2"], ada=m["ada"])
        h = _silu(_mul(h, m["w1"], DEC_MATS["w1"], wt)) * _mul(h, m["w3"], DEC_MATS["w3"], wt)
        x = x + _mul(h, m["w2"], DEC_MATS["w2"], wt)
        for i in (0, 1):
            rows[i].append(new[i][0])
    h = _image(_rms(x[-1:], out_norm), tt == Q8)
    step = VOCAB // 8
    logits = torch.cat([(h @ _deq(tt, table.view(VOCAB, rb)[i:i + step].reshape(-1), step, DIM).T)[0]
                        for i in range(0, VOCAB, step)])
    return dict(logits=logits, x=x, rows=[torch.stack(r) for r in rows])


def _exact_enc(case, seed):
    ls, top = _enc_weights(case, seed)
    plan, mel = _enc_inputs(case, seed)
    wt, kv, n, q0 = case["weights"], case["kv"], case["frames"], case["q_start"]
    conv = torch.nn.functional.conv1d
    pad = torch.nn.functional.pad
    y = _gelu(conv(pad(mel.half().double()[None], (2, 0)), top["c0"].double(), top["b0"].double()))
    # a window of odd length is padded on the right to complete its last frame
    y = conv(pad(y.half().double(), (1, y.shape[2] % 2)), top["c1"].double(), top["b1"].double(), stride=2)
    s = plan.conv_slice_start
    x = _gelu(y)[0].T[s:s + n].contiguous()
    p = min(q0, E_WIN)
    at = _arange(q0, q0 + n)
    for l, m in enumerate(ls):
        h = _rms(x, m["n1"], m["n1b"])
        q, k, v = (_mul(h, m[i], ENC_MATS[i], wt) for i in "qkv")
        q, k, v = _rope64(q + m["qb"].double(), at, E_HD), _rope64(k, at, E_HD), v + m["vb"].double()
        old = [_stored(_rows(seed, i, 0, l, p, E_KV), kv)[1] for i in (0, 1)]
        a = _attn64(q, *(torch.cat([o, _stored(t, kv)[1]]) for o, t in zip(old, (k, v))), at,
                    _arange(q0 - p, q0 + n), E_HEADS, E_HEADS, E_WIN)
        x = x + _mul(a, m["o"], ENC_MATS["o"], wt) + m["ob"].double()
        h = _rms(x, m["n2"], m["n2b"])
        h = _silu(_mul(h, m["w1"], ENC_MATS["w1"], wt)) * _mul(h, m["w3"], ENC_MATS["w3"], wt)
        x = x + _mul(h, m["w2"], ENC_MATS["w2"], wt) + m["w2b"].double()
    enc = _rms(x, top["norm"], top["norm_b"])
    g0, g = _groups(case)
    emb = []
    if g > 0:
        h = _gelu(_mul(enc[:g * DOWN].reshape(g, -1), top["a0"], (Q4, DIM, E_DIM * DOWN), wt))
        emb = _cut(_mul(h, top["a2"], (Q4, DIM, DIM), wt), g0, RING)
    return dict(x=x, enc=_cut(enc, q0, RING), emb=emb)


_EXACT = dict(decode=_exact_decode, prefill=_exact_prefill, window=_exact_window, ffn=_exact_ffn,
              token=_exact_dec, prompt=_exact_dec, encoder=_exact_enc)


def exact(case, seed):
    with torch.no_grad():
        return _EXACT[case["kind"]](case, seed)
