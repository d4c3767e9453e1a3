"""What a user of this framework has it do, as measurable cases.

Each case is one pass through public entry points (the C ABI bound by
taraference_amd.capi, or DecodeModel):

  gemv     tf_quantize_q8 + tf_gemv_q4k_q8: the smallest call, one projection
           of one token;
  ffn      the decode MLP block of several layers (norm + Q8, gate/up + SiLU,
           Q8, down into the residual), each layer with its own weights, as
           a decode step walks them;
  head     the decode head: RMSNorm + Q8 + Q6_K lm_head + argmax;
  flash    one token's attention over a long f16 K/V cache, with the Q8 of
           its output for the wo projection;
  gemm     one prompt projection on raw GGUF weights (Q4_K or Q6_K);
  attn     causal prompt attention over the cache, fresh or continued;
  prefill  a prompt through a whole model (DecodeModel.prefill);
  decode   teacher-forced decode steps of a whole model after a prompt
           (DecodeModel.generate, graph replay): a Qwen2.5-3B-width Q4_K_M
           model on the persistent step, and the Qwen2.5-0.5B layout, whose
           896-wide matrices are Q5_0 / Q8_0.

Widths are those of the Qwen2.5 0.5B, 3B and 7B shapes (taraference_amd.synth);
whole models keep the real widths and vocabulary and a few layers.
"""
import math

import numpy as np
import torch

from taraference_amd import capi
from taraference_amd.model import DecodeModel

Q4K, Q6K, Q5_0, Q8_0 = 12, 14, 6, 8
BLOCK = {Q4K: 144, Q6K: 210, Q5_0: 22, Q8_0: 34}   # bytes of a block
WIDTH = {Q4K: 256, Q6K: 256, Q5_0: 32, Q8_0: 32}   # its values

EMBD = {"0.5b": 896, "3b": 2048, "7b": 3584}
FF = {"0.5b": 4864, "3b": 11008, "7b": 18944}
HEADS = {"0.5b": (14, 2, 64), "3b": (16, 2, 128), "7b": (28, 4, 128)}
VOCAB = {"0.5b": 151936, "3b": 151936, "7b": 152064}
EPS, THETA = 1e-6, 1e6


def listed():
    return [
        # one projection of one token at the smallest model's width: launch latency
        {"name": "gemv_q4k_896", "kind": "gemv", "k": 896, "n": 4864},
        # the MLP of three consecutive 3B layers in a decode step (down alternates Q4_K / Q6_K)
        {"name": "ffn_decode_3b", "kind": "ffn", "e": 2048, "f": 11008, "layers": 3},
        # the 3B lm_head with its argmax, the largest single matrix of a token
        {"name": "head_3b", "kind": "head", "k": 2048, "n": 151936},
        # one token of a 7B model at a full 32K context
        {"name": "flash_7b_32k", "kind": "flash", "size": "7b", "ctx": 32768},
        # gate or up of a 512-token prompt
        {"name": "gemm_q4k_512", "kind": "gemm", "type": Q4K, "k": 2048, "n": 11008, "t": 512},
        # a short question to a 7B model: few tokens, weights dominate
        {"name": "gemm_q4k_37", "kind": "gemm", "type": Q4K, "k": 3584, "n": 3584, "t": 37},
        # ffn_down of a prompt whose length is no multiple of anything
        {"name": "gemm_q6k_300", "kind": "gemm", "type": Q6K, "k": 11008, "n": 2048, "t": 300},
        # a fresh 512-token prompt
        {"name": "attn_3b_512", "kind": "attn", "size": "3b", "pos": 0, "t": 512},
        # a prompt chunk deep in a long document
        {"name": "attn_7b_8k", "kind": "attn", "size": "7b", "pos": 8000, "t": 256},
        # a prompt through two 3B layers and the head: time to first token
        {"name": "prefill_3b", "kind": "prefill", "size": "3b", "layers": 2, "pos": 0, "t": 700},
        # sixteen decode steps after a 500-token prompt
        {"name": "decode_3b", "kind": "decode", "size": "3b", "layers": 2, "ctx": 500, "t": 16},
        # the same of the 896-wide layout
        {"name": "decode_05b", "kind": "decode", "size": "0.5b", "layers": 6, "ctx": 120, "t": 16},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "ffn", "head", "flash", "gemm", "gemm", "gemm", "attn", "attn",
                       "prefill", "prefill", "decode", "decode"])
    if kind == "gemv":
        return {"kind": kind, "k": 32 * _log(rng, 8, 344), "n": _log(rng, 64, 11008)}
    if kind == "ffn":
        e, f = 256 * rng.randint(1, 14), 256 * _log(rng, 4, 43)
        return {"kind": kind, "e": e, "f": f, "layers": rng.randint(1, 3)}
    if kind == "head":
        return {"kind": kind, "k": 256 * rng.randint(2, 8), "n": _log(rng, 1000, 151936)}
    if kind == "flash":
        return {"kind": kind, "size": rng.choice(["0.5b", "3b", "7b"]),
                "ctx": _log(rng, 100, 32768)}
    if kind == "gemm":
        ty = rng.choice([Q4K, Q6K])
        k = 256 * _log(rng, 1, 43)
        t = _log(rng, 1, 512)
        n = _log(rng, 77, max(78, min(11008, 2048 * 11008 // k)))
        return {"kind": kind, "type": ty, "k": k, "n": n, "t": t}
    if kind == "attn":
        size = rng.choice(["0.5b", "3b", "7b", "7b"])
        if size == "0.5b":
            return {"kind": kind, "size": size, "pos": rng.randint(0, 600),
                    "t": _log(rng, 5, 400)}
        return {"kind": kind, "size": size, "pos": rng.choice([0, _log(rng, 10, 8000)]),
                "t": _log(rng, 5, 256)}
    if kind == "prefill":
        return {"kind": kind, "size": "3b", "layers": rng.randint(1, 2),
                "pos": rng.choice([0, rng.randint(1, 300)]), "t": _log(rng, 10, 700)}
    size = rng.choice(["0.5b", "3b"])
    return {"kind": kind, "size": size, "layers": rng.randint(1, 6 if size == "0.5b" else 2),
            "ctx": _log(rng, 20, 120 if size == "0.5b" else 500), "t": rng.randint(2, 16)}


# ------------------------------------------------------------------ inputs

def _gen(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * (seed % 2000003) + 17 * len(case["kind"]))
    return g


def _uni(g, n, lo, hi):
    return (torch.rand(n, generator=g, device="cuda") * (hi - lo) + lo).half()


def _ints(g, lo, hi, shape):
    return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.int32)


def _bytes(h):
    return h.contiguous().view(torch.uint8).reshape(h.numel(), 2)


def _matrix(g, ty, k, n):
    """n columns of k weights of spread about 0.02 (mean about 0), as GGUF
    stores them: uint8 [n, column bytes]."""
    nb = -(-k // WIDTH[ty])
    m = n * nb
    b = torch.randint(0, 256, (m, BLOCK[ty]), generator=g, device="cuda", dtype=torch.uint8)
    if ty == Q4K:
        # w = d sc q - dmin mn with dmin mn about d sc 7.5: 6-bit scales over their range
        d = _uni(g, m, 6e-5, 2e-4)
        sc = _ints(g, 0, 64, (m, 8))
        mn = (sc * 15 + 8) // 16
        b[:, 0:2] = _bytes(d)
        b[:, 2:4] = _bytes((d.float() * 8).half())
        b[:, 4:8] = ((sc[:, :4]) | ((sc[:, 4:] >> 4) << 6)).to(torch.uint8)
        b[:, 8:12] = ((mn[:, :4]) | ((mn[:, 4:] >> 4) << 6)).to(torch.uint8)
        b[:, 12:16] = ((sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)).to(torch.uint8)
    elif ty == Q6K:
        b[:, 208:210] = _bytes(_uni(g, m, 8e-6, 2.4e-5))  # int8 scales over their whole range
    elif ty == Q5_0:
        b[:, 0:2] = _bytes(_uni(g, m, 1e-3, 4e-3))
    else:
        b[:, 0:2] = _bytes(_uni(g, m, 1e-4, 5e-4))
    return b.reshape(n, nb * BLOCK[ty])


def _act(g, t, k):
    """t rows of k activations, some channels several times larger."""
    ch = torch.exp(0.5 * torch.randn(k, generator=g, device="cuda"))
    return (torch.randn((t, k), generator=g, device="cuda") * ch).contiguous()


def _norm(g, k):
    return 1 + 0.1 * torch.randn(k, generator=g, device="cuda")


def _compact(w, k):
    n, nb = w.shape[0], k // 256
    c = torch.empty(n * nb * 212, dtype=torch.uint8, device="cuda")
    capi.call("tf_q6k_compact_repack", w.data_ptr(), c.data_ptr(), k, n, w.shape[1],
              capi.stream_ptr())
    return c


def _cache(g, seq, width):
    return torch.randn((seq, width), generator=g, device="cuda").half()


def _empty(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device="cuda")


def _ffn_inputs(case, g):
    e, f = case["e"], case["f"]
    layers = []
    for i in range(case["layers"]):
        ty = Q6K if i % 2 else Q4K
        layers.append({"norm": _norm(g, e), "gate": _matrix(g, Q4K, e, f),
                       "up": _matrix(g, Q4K, e, f), "ty": ty, "down": _matrix(g, ty, f, e)})
    return layers, _act(g, 1, e)[0].contiguous()


def _model_inputs(case, g):
    size = case["size"]
    e, f, (h, kv, hd) = EMBD[size], FF[size], HEADS[size]
    small = size == "0.5b"
    wt, vt = (Q5_0, Q8_0) if small else (Q4K, Q6K)
    layers = []
    for i in range(case["layers"]):
        dt = Q6K if i % 2 else Q4K
        shapes = {"wq": (wt, e, h * hd), "wk": (wt, e, kv * hd), "wv": (vt, e, kv * hd),
                  "wo": (wt, h * hd, e), "gate": (wt, e, f), "up": (wt, e, f),
                  "down": (dt, f, e)}
        L = {n: (_matrix(g, *s), s) for n, s in shapes.items()}
        L["attn_norm"], L["ffn_norm"] = _norm(g, e), _norm(g, e)
        for n, w in (("bq", h * hd), ("bk", kv * hd), ("bv", kv * hd)):
            L[n] = 0.02 * torch.randn(w, generator=g, device="cuda")
        layers.append(L)
    et = Q8_0 if small else Q6K
    emb = (_matrix(g, et, e, VOCAB[size]), (et, e, VOCAB[size]))
    n_tok = case["t"] + (case["ctx"] if case["kind"] == "decode" else case["pos"])
    tokens = torch.randint(0, VOCAB[size], (n_tok,), generator=g, device="cuda").tolist()
    return layers, emb, _norm(g, e), tokens


class _DeviceView:
    """A device buffer of a model; a tensor made of it keeps the model."""

    def __init__(self, owner, ptr, shape, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": kind,
                                         "version": 2, "strides": None}


def _view(owner, ptr, shape, kind):
    return torch.as_tensor(_DeviceView(owner, ptr, shape, kind), device="cuda")


def prepare(case, seed):
    g = _gen(case, seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "gemv":
        k, n = case["k"], case["n"]
        s.update(w=_matrix(g, Q4K, k, n), x=_act(g, 1, k), bias=0.02 * torch.randn(
            n, generator=g, device="cuda"), xq=_empty(k, dtype=torch.int8), xd=_empty(k // 32),
            out=_empty(n))
    elif kind == "ffn":
        layers, x = _ffn_inputs(case, g)
        e, f = case["e"], case["f"]
        for L in layers:
            L["cb"] = L["down"].shape[1]
            if L["ty"] == Q6K:
                L["down"], L["cb"] = _compact(L["down"], f), f // 256 * 212
        # norm_quant takes 128-value multiples up to 8192
        s.update(layers=layers, x0=x, x=_empty(e), xb=_empty(e), q=_empty(max(e, f),
                 dtype=torch.int8), d=_empty(max(e, f) // 32), h=[_empty(f) for _ in layers])
    elif kind == "head":
        k, n = case["k"], case["n"]
        s.update(w=_compact(_matrix(g, Q6K, k, n), k), x=_act(g, 1, k), norm=_norm(g, k),
                 out=_empty(n), key=torch.zeros(1024, dtype=torch.int64, device="cuda"),
                 tok=_empty(1, dtype=torch.int32))
    elif kind == "flash":
        h, kv, hd = HEADS[case["size"]]
        ns = capi.load().tf_flash_decode_n_split(kv, case["ctx"])
        s.update(q=_act(g, 1, h * hd), k=_cache(g, case["ctx"], kv * hd),
                 v=_cache(g, case["ctx"], kv * hd), part=_empty(h * ns * (2 + hd)), ns=ns,
                 out=_empty(h * hd), q8=_empty(h * hd, dtype=torch.int8), d8=_empty(h * hd // 32))
    elif kind == "gemm":
        s.update(w=_matrix(g, case["type"], case["k"], case["n"]),
                 x=_act(g, case["t"], case["k"]), out=_empty(case["t"], case["n"]))
    elif kind == "attn":
        h, kv, hd = HEADS[case["size"]]
        L = case["pos"] + case["t"]
        s.update(q=_act(g, case["t"], h * hd), k=_cache(g, L, kv * hd), v=_cache(g, L, kv * hd),
                 out=_empty(case["t"], h * hd))
    else:
        layers, emb, norm, tokens = _model_inputs(case, g)
        size = case["size"]
        h, kv, hd = HEADS[size]

        def host(wm):
            w, (ty, _, _) = wm
            return w.cpu().numpy(), int(w.shape[1]), ty

        def rows(L):
            return {n: host(v) if isinstance(v, tuple) else v.cpu().numpy()
                    for n, v in L.items()}

        cfg = dict(n_layer=len(layers), n_embd=EMBD[size], n_ff=FF[size], n_head=h, n_kv=kv,
                   head_dim=hd, n_vocab=VOCAB[size], rope_theta=THETA, rms_eps=EPS,
                   max_seq=len(tokens) + 8)
        m = DecodeModel(cfg, (rows(L) for L in layers), host(emb),
                        output_norm=norm.cpu().numpy())
        done = len(tokens) - case["t"]  # what the program has run before: the prompt so far
        if done:
            if size == "0.5b":
                m.generate(tokens[:done], 1)
            else:
                m.prefill(tokens[:done])
        lib, shape = m.lib, (len(tokens), kv * hd)
        s.update(m=m, tokens=tokens[done:], pos=done,
                 logits=_view(m, lib.tf_model_logits(m.h), (VOCAB[size],), "<f4"),
                 k=[_view(m, lib.tf_model_k_cache(m.h, i), shape, "<f2")
                    for i in range(len(layers))],
                 v=[_view(m, lib.tf_model_v_cache(m.h, i), shape, "<f2")
                    for i in range(len(layers))])
    torch.cuda.synchronize()
    return s


# ------------------------------------------------------------------ the pass

def run(s):
    c = s["case"]
    kind = c["kind"]
    st = capi.stream_ptr()
    call = capi.call
    P = capi.ptr
    if kind == "gemv":
        k, n = c["k"], c["n"]
        call("tf_quantize_q8", P(s["x"]), P(s["xq"]), P(s["xd"]), k, st)
        call("tf_gemv_q4k_q8", P(s["w"]), P(s["xq"]), P(s["xd"]), P(s["out"]), k, n,
             s["w"].shape[1], 1, P(s["bias"]), 0, None, st)
        return s["out"]
    if kind == "ffn":
        e, f, x, xb, q, d = c["e"], c["f"], s["x"], s["xb"], s["q"], s["d"]
        x.copy_(s["x0"])
        for L, h in zip(s["layers"], s["h"]):
            call("tf_norm_quant", P(x), P(L["norm"]), EPS, P(xb), P(q), P(d), e, st)
            call("tf_gemv_q4k_ffn", P(L["gate"]), P(L["up"]), P(q), P(d), P(h), e, f,
                 e // 256 * 144, st)
            call("tf_quantize_q8", P(h), P(q), P(d), f, st)
            call("tf_gemv_q4k_q8" if L["ty"] == Q4K else "tf_gemv_q6k_down_splitk", P(L["down"]),
                 P(q), P(d), P(x), f, e, L["cb"], 0, None, 2, None, st)
        return {"x": x, "h": s["h"]}
    if kind == "head":
        k, n = c["k"], c["n"]
        call("tf_gemv_q6k_head_argmax", P(s["w"]), P(s["x"]), P(s["norm"]), EPS, P(s["out"]), k, n,
             k // 256 * 212, P(s["key"]), st)
        call("tf_argmax_key_finalize", P(s["key"]), P(s["tok"]), st)
        return {"logits": s["out"], "token": s["tok"]}
    if kind == "flash":
        h, kv, hd = HEADS[c["size"]]
        call("tf_flash_decode", P(s["q"]), P(s["k"]), P(s["v"]), P(s["part"]), None, P(s["out"]),
             P(s["q8"]), P(s["d8"]), h, kv, hd, c["ctx"] - 1, None, s["ns"], hd ** -0.5, st)
        return {"out": s["out"], "q8": s["q8"], "d8": s["d8"]}
    if kind == "gemm":
        call("tf_gemm_q4k_f32" if c["type"] == Q4K else "tf_gemm_q6k_f32", P(s["w"]), P(s["x"]),
             P(s["out"]), c["k"], c["n"], s["w"].shape[1], c["t"], st)
        return s["out"]
    if kind == "attn":
        h, kv, hd = HEADS[c["size"]]
        call("tf_attn_prefill", P(s["q"]), P(s["k"]), P(s["v"]), P(s["out"]), h, kv, hd, c["pos"],
             c["t"], hd ** -0.5, st)
        return s["out"]
    if kind == "prefill":
        s["m"].prefill(s["tokens"], s["pos"])
    else:
        s["m"].generate(s["tokens"], 1, pos0=s["pos"])
    return {"logits": s["logits"], "k": [t[s["pos"]:] for t in s["k"]],
            "v": [t[s["pos"]:] for t in s["v"]]}


# ------------------------------------------------------------------ its cost

def _mat_bytes(ty, k, n):
    return n * (k // WIDTH[ty]) * BLOCK[ty]


def _model_cost(case):
    """(bytes of the layers' weights, of the head, parameters of a layer)."""
    size = case["size"]
    e, f, (h, kv, hd) = EMBD[size], FF[size], HEADS[size]
    small = size == "0.5b"
    wt, vt = (Q5_0, Q8_0) if small else (Q4K, Q6K)
    w = 0
    for i in range(case["layers"]):
        w += _mat_bytes(wt, e, h * hd + kv * hd + 2 * f) + _mat_bytes(vt, e, kv * hd)
        w += _mat_bytes(wt, h * hd, e) + _mat_bytes(Q6K if i % 2 else Q4K, f, e)
    return (w, _mat_bytes(Q8_0 if small else Q6K, e, VOCAB[size]),
            e * (2 * h * hd + 2 * kv * hd + 3 * f))


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        k, n = case["k"], case["n"]
        return {"bytes": _mat_bytes(Q4K, k, n) + 4 * k + 8 * n, "flops": 2 * k * n}
    if kind == "ffn":
        e, f = case["e"], case["f"]
        b = sum(2 * _mat_bytes(Q4K, e, f) + _mat_bytes(Q6K if i % 2 else Q4K, f, e) + 4 * e
                for i in range(case["layers"]))
        return {"bytes": b + 8 * e + 4 * f, "flops": 6 * e * f * case["layers"]}
    if kind == "head":
        k, n = case["k"], case["n"]
        return {"bytes": _mat_bytes(Q6K, k, n) + 8 * k + 4 * n, "flops": 2 * k * n}
    if kind == "flash":
        h, kv, hd = HEADS[case["size"]]
        L = case["ctx"]
        return {"bytes": 4 * L * kv * hd + 9 * h * hd, "flops": 4 * L * h * hd}
    if kind == "gemm":
        k, n, t = case["k"], case["n"], case["t"]
        return {"bytes": _mat_bytes(case["type"], k, n) + 4 * t * (k + n), "flops": 2 * k * n * t}
    if kind == "attn":
        h, kv, hd = HEADS[case["size"]]
        p, t = case["pos"], case["t"]
        return {"bytes": 4 * (p + t) * kv * hd + 8 * t * h * hd,
                "flops": 4 * h * hd * (t * p + t * (t + 1) // 2)}
    w, head, par = _model_cost(case)
    size = case["size"]
    e, (h, kv, hd) = EMBD[size], HEADS[size]
    n, t = case["layers"], case["t"]
    p = case["pos"] if kind == "prefill" else case["ctx"]
    pairs = t * p + t * (t + 1) // 2
    flops = n * (2 * par * t + 4 * h * hd * pairs)
    if kind == "prefill":
        return {"bytes": w + head + n * 4 * kv * hd * (p + t) + 4 * VOCAB[size],
                "flops": flops + 2 * e * VOCAB[size]}
    return {"bytes": t * (w + head) + n * 4 * kv * hd * pairs + 4 * t * VOCAB[size],
            "flops": flops + 2 * t * e * VOCAB[size]}


def tolerance(case):
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        return {"rel": 1e-5}          # sums of 32 bits
    if kind == "ffn":
        # a value at the edge of two Q8 steps may round either way; each such
        # value moves the outputs by about 1e-3, and the layers after it by more
        return {"rel": 1.5e-2, "max": 1e-1}
    if kind == "head":
        return {"rel": 2e-3}          # one such value of the normalized row
    if kind == "flash":
        return {"rel": 1e-5, "differ": 5e-3}
    if kind == "attn":
        return {"rel": 1e-5}
    if kind == "prefill":
        return {"rel": 6e-3, "max": 5e-2}  # the head's Q8, and f16 K/V rows
    # Q8 at four places of every layer: two of the runtime's decode paths, which
    # add in another order, are 1.3e-2 apart after three layers
    return {"rel": 2.5e-2, "max": 2.5e-1}


# ------------------------------------------------------------------ in 64 bits

def _f16(b):
    return b.contiguous().view(torch.float16)[..., 0].double()


def _weights(w, ty, k):
    """float64 [n, k] of a matrix (a last partial super-block is not read)."""
    n, nb = w.shape[0], k // WIDTH[ty]
    b = w[:, : nb * BLOCK[ty]].reshape(n * nb, BLOCK[ty])
    if ty == Q4K:
        s = b[:, 4:16].int()
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = b[:, 16:].reshape(-1, 4, 32)
        q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        v = (_f16(b[:, 0:2])[:, None] * sc)[..., None] * q
        v -= (_f16(b[:, 2:4])[:, None] * mn)[..., None]
    elif ty == Q6K:
        ql, qh = b[:, :128].int().reshape(-1, 2, 64), b[:, 128:192].int().reshape(-1, 2, 32)
        lo, hi = ql[:, :, :32], ql[:, :, 32:]
        q = torch.stack([lo & 15 | (qh & 3) << 4, hi & 15 | (qh >> 2 & 3) << 4,
                         lo >> 4 | (qh >> 4 & 3) << 4, hi >> 4 | (qh >> 6 & 3) << 4], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        v = (_f16(b[:, 208:210])[:, None] * sc)[..., None] * (q.reshape(-1, 16, 16).double() - 32)
    elif ty == Q5_0:
        qh = b[:, 2:6].contiguous().view(torch.int32).long()
        bit = (qh >> torch.arange(32, device=b.device)) & 1
        nib = torch.cat([b[:, 6:] & 15, b[:, 6:] >> 4], 1).long()
        v = _f16(b[:, 0:2])[:, None] * (nib + 16 * bit - 16).double()
    else:
        v = _f16(b[:, 0:2])[:, None] * b[:, 2:].contiguous().view(torch.int8).double()
    return v.reshape(n, nb * WIDTH[ty])


def _q8(x):
    """Rows of x as the Q8 activation holds them: 32-value groups, 8 bits."""
    v = x.reshape(-1, 32)
    d = v.abs().amax(1, keepdim=True) / 127
    return torch.where(d > 0, torch.round(v / d.clamp_min(1e-300)) * d, 0 * v).reshape(x.shape)


def _q8_parts(x):
    v = x.reshape(-1, 32)
    d = v.abs().amax(1, keepdim=True) / 127
    return torch.round(v / d.clamp_min(1e-300)).reshape(-1).to(torch.int8), d[:, 0]


def _mul(x, wm):
    """x W for rows x, with W (bytes, (type, k, n))."""
    w, (ty, k, n) = wm
    out = []
    for i in range(0, n, 16384):  # columns at a time: the vocabulary in 64 bits is large
        W = _weights(w[i:i + 16384], ty, k)
        out.append(x[:, : W.shape[1]] @ W.T)
    return torch.cat(out, 1)


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _silu(x):
    return x / (1 + torch.exp(-x))


def _softmax_attn(q, k, v, pos, h, kv, hd):
    """Causal attention of rows q at positions pos.. over k, v [L, kv hd]."""
    t, L = q.shape[0], k.shape[0]
    out = torch.empty(t, h * hd, dtype=torch.float64, device=q.device)
    see = torch.arange(L, device=q.device)[None] <= pos + torch.arange(t, device=q.device)[:, None]
    for i in range(h):
        j = i // (h // kv)
        a = (q[:, i * hd:(i + 1) * hd] @ k[:, j * hd:(j + 1) * hd].T.contiguous()) / math.sqrt(hd)
        a = torch.softmax(a.masked_fill(~see, -math.inf), 1)
        out[:, i * hd:(i + 1) * hd] = a @ v[:, j * hd:(j + 1) * hd]
    return out


def _rope(x, n, hd):
    t = x.shape[0]
    half = hd // 2
    f = THETA ** (-2.0 * torch.arange(half, device=x.device, dtype=torch.float64) / hd)
    a = torch.arange(t, device=x.device, dtype=torch.float64)[:, None] * f
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    x = x.reshape(t, n, hd)
    x0, x1 = x[..., :half], x[..., half:]
    return torch.cat([x0 * c - x1 * s, x0 * s + x1 * c], -1).reshape(t, n * hd)


def _model64(case, seed):
    layers, emb, norm, tokens = _model_inputs(case, _gen(case, seed))
    size = case["size"]
    h, kv, hd = HEADS[size]
    first = len(tokens) - case["t"]
    quant = torch.zeros(len(tokens), 1, dtype=torch.bool, device="cuda")
    if case["kind"] == "decode":  # the decode steps quantize their activations
        quant[0 if size == "0.5b" else first:] = True

    def mul(x, wm):
        # Q5_0 matrices and a Q6_K v take the activation in 32 bits
        ty = wm[1][0]
        if ty == Q8_0 or (ty != Q5_0 and wm is not vmat):
            x = torch.where(quant, _q8(x), x)
        return _mul(x, wm)

    w, (ty, k, _) = emb
    x = _weights(w[torch.tensor(tokens, device="cuda")], ty, k)
    ks, vs = [], []
    for L in layers:
        vmat = L["wv"]
        a = _rms(x, L["attn_norm"])
        q = _rope(mul(a, L["wq"]) + L["bq"].double(), h, hd)
        k_ = _rope(mul(a, L["wk"]) + L["bk"].double(), kv, hd)
        v_ = mul(a, vmat) + L["bv"].double()
        ks.append(k_[first:])
        vs.append(v_[first:])
        o = _softmax_attn(q, k_.half().double(), v_.half().double(), 0, h, kv, hd)
        x = x + mul(o, L["wo"])
        a = _rms(x, L["ffn_norm"])
        x = x + mul(_silu(mul(a, L["gate"])) * mul(a, L["up"]), L["down"])
    # Past the first Q8 of an activation there is no one value in 64 bits: a value
    # at the edge of two steps rounds either way, which moves all that follows by
    # 1e-3.  In a prompt that is the head's input, in a decode step the input of
    # every layer but the first's q, k and v.
    if case["kind"] == "decode":
        ks[1:], vs[1:] = [None] * (len(ks) - 1), [None] * (len(vs) - 1)
    return {"logits": None, "k": ks, "v": vs}


def exact(case, seed):
    kind = case["kind"]
    g = _gen(case, seed)
    if kind == "gemv":
        w, x = _matrix(g, Q4K, case["k"], case["n"]), _act(g, 1, case["k"])
        bias = 0.02 * torch.randn(case["n"], generator=g, device="cuda")
        return _mul(_q8(x.double()), (w, (Q4K, case["k"], case["n"])))[0] + bias.double()
    if kind == "ffn":
        # the first layer's h: past it a value at the edge of two Q8 steps rounds
        # either way, which moves all that follows by 1e-3
        layers, x = _ffn_inputs(case, g)
        e, f, L = case["e"], case["f"], layers[0]
        a = _q8(_rms(x.double()[None], L["norm"]))
        h = _silu(_mul(a, (L["gate"], (Q4K, e, f)))) * _mul(a, (L["up"], (Q4K, e, f)))
        return {"x": None, "h": [h[0]] + [None] * (len(layers) - 1)}
    if kind == "head":
        w = _matrix(g, Q6K, case["k"], case["n"])
        x = _act(g, 1, case["k"])
        lg = _mul(_q8(_rms(x.double(), _norm(g, case["k"]))), (w, (Q6K, case["k"], case["n"])))[0]
        return {"logits": lg, "token": None}
    if kind == "flash":
        h, kv, hd = HEADS[case["size"]]
        q = _act(g, 1, h * hd)
        k, v = _cache(g, case["ctx"], kv * hd), _cache(g, case["ctx"], kv * hd)
        o = _softmax_attn(q.double(), k.double(), v.double(), case["ctx"] - 1, h, kv, hd)[0]
        return {"out": o, "q8": None, "d8": _q8_parts(o)[1]}
    if kind == "gemm":
        k, n = case["k"], case["n"]
        w = _matrix(g, case["type"], k, n)
        return _mul(_act(g, case["t"], k).double(), (w, (case["type"], k, n)))
    if kind == "attn":
        h, kv, hd = HEADS[case["size"]]
        L = case["pos"] + case["t"]
        q = _act(g, case["t"], h * hd)
        k, v = _cache(g, L, kv * hd), _cache(g, L, kv * hd)
        return _softmax_attn(q.double(), k.double(), v.double(), case["pos"], h, kv, hd)
    return _model64(case, seed)
