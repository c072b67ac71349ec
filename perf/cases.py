"""Performance cases: the work that a user of this engine has it do, through
its public entry points (the C ABI of include/draco_hip.h and the drivers of
dracohip over it).

A case is a dict of plain values.  `prepare` makes what a serving program
holds before the call (weights resident on the device, the session's state,
the inputs), `run` makes one call as such a program does, `exact` is the same
result in 64-bit arithmetic by plain torch / numpy.

Weights are random GGUF blocks: every quant and scale byte uniform, the block
scale set so that the weights have mean about 0 and standard deviation about
`std` (0.02 unless a matrix says otherwise), with 25% spread from block to
block.  Activations and states are normal, as behind an RMSNorm.
"""
import ctypes as ct
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dracomancer-llmengine_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from dracohip import driver as _driver  # noqa: E402
from dracohip import lib as _lib  # noqa: E402
from dracohip import models as _models  # noqa: E402
from dracohip import qwen35 as _qwen  # noqa: E402

Q8_0, Q5_K, Q6_K, Q4_K, F32 = 0, 3, 4, 5, 9
CODE = {"q8_0": Q8_0, "q5_k": Q5_K, "q6_k": Q6_K, "q4_k": Q4_K}
BLOCK = {Q8_0: (32, 34), Q5_K: (256, 176), Q6_K: (256, 210), Q4_K: (256, 144)}  # values, bytes
GEMM_ENTRY = {"q8_0": "m5_gemm_q80", "q5_k": "m5_gemm_q5k", "q6_k": "m5_gemm_q6k", "q4_k": "m5_gemm_q4k"}

# The shapes of the repository's own configurations: the dense ones by their
# layer shape and formats, with the depth and vocabulary that a case names.
DENSE = {
    "smollm2-360m": dict(base=_models.SMOL360M, codes=_models.SMOL360M.codes),
    "llama-3.2-1b": dict(base=_models.LLAMA1B, codes=_models.LLAMA1B.codes),
    # the Q5_K_M mix of the repository's small test model at the 1B layer shape
    "llama-3.2-1b-q5": dict(base=_models.LLAMA1B, codes=dict(_models.TINY_Q5.codes, emb=Q5_K, out=Q5_K)),
}
MOE = _models.QWEN3_MOE


def listed():
    return [
        # the smallest drop-in call: one Q8_0 attention projection of SmolLM2-360M for one token
        {"name": "gemv_q8_0_960", "kind": "gemv", "code": "q8_0", "n_out": 960, "n_in": 960},
        # a serving loop's FFN GEMV on device pointers: 8B-class gate / up matrix, one token
        {"name": "q8k_gemv_14336x4096", "kind": "q8k", "code": "q4_k", "n_out": 14336, "n_in": 4096, "nvec": 1},
        # one projection of a ragged prompt chunk through the prefill driver's per-format entry
        {"name": "gemm_q8_0_61x2560x960", "kind": "gemm", "code": "q8_0", "T": 61, "n_out": 2560, "n_in": 960},
        # the K-quant one: the down projection of a full 256-token chunk
        {"name": "gemm_q6_k_256x2048x8192", "kind": "gemm", "code": "q6_k", "T": 256, "n_out": 2048, "n_in": 8192},
        # a short chat turn of the small Q8_0 model: 32-token prompt, 64 greedy tokens
        {"name": "smol_turn_32_64", "kind": "llama_turn", "shape": "smollm2-360m", "n_layer": 32, "vocab": 49152,
         "ctx": 0, "n_prompt": 32, "n_gen": 64},
        # decode at long context, the flagship: 1B Q4_K_M, 960 cached rows, 32 greedy tokens
        {"name": "llama_decode_ctx960", "kind": "llama_turn", "shape": "llama-3.2-1b", "n_layer": 16,
         "vocab": 128256, "ctx": 960, "n_prompt": 1, "n_gen": 32},
        # a long prompt (chunked prefill) up to its logits, four layers of the 1B shape
        {"name": "llama_prefill_960", "kind": "llama_prefill", "shape": "llama-3.2-1b", "n_layer": 4,
         "vocab": 32768, "ctx": 0, "n_prompt": 960, "snapshot": False},
        # a ragged follow-up message over a cached prefix in the Q5_K_M mix, then the session snapshot
        {"name": "q5_followup_75_ctx200", "kind": "llama_prefill", "shape": "llama-3.2-1b-q5", "n_layer": 2,
         "vocab": 32768, "ctx": 200, "n_prompt": 75, "snapshot": True},
        # a chat turn of the MoE model (two layers, 128 experts, top 8): prompt and decode
        {"name": "moe_turn_192_32", "kind": "moe_turn", "n_layer": 2, "vocab": 32768, "n_prompt": 192, "n_gen": 32},
        # the prefill driver's token-batched expert FFN on one chunk
        {"name": "moe_tok_128", "kind": "moe_tok", "T": 128, "n_exp": 128, "n_used": 8},
        # a chat turn of the hybrid model from a reset session: 2000-token prompt, 32 tokens,
        # four layers (3 GDN, 1 full attention)
        {"name": "qwen_turn_2000_32", "kind": "qwen_turn", "n_layer": 4, "vocab": 32768, "ffn": 0, "n_prompt": 2000,
         "n_gen": 32},
        # the prefill driver's GDN scan on one 64-token chunk, its state handed in and out
        {"name": "gdn_scan_64", "kind": "gdn_scan", "T": 64, "n_vh": 32},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "q8k", "gemm", "gemm", "llama_turn", "llama_prefill", "llama_prefill", "moe_turn",
                       "moe_tok", "qwen_turn", "gdn_scan"])
    if kind == "gemv":
        code = rng.choice(sorted(CODE))
        unit = BLOCK[CODE[code]][0]
        return {"kind": kind, "code": code, "n_out": _log(rng, 100, 14336), "n_in": unit * _log(rng, 512 // unit, 8192 // unit)}
    if kind == "q8k":
        return {"kind": kind, "code": rng.choice(["q4_k", "q6_k"]), "n_out": _log(rng, 500, 14336),
                "n_in": 256 * _log(rng, 4, 32), "nvec": rng.choice([1, 4, 8])}
    if kind == "gemm":
        code = rng.choice(sorted(CODE))
        unit = BLOCK[CODE[code]][0]
        return {"kind": kind, "code": code, "T": _log(rng, 2, 256), "n_out": _log(rng, 320, 8192),
                "n_in": unit * _log(rng, 768 // unit, 4096 // unit)}
    if kind == "llama_turn":
        return {"kind": kind, "shape": rng.choice(sorted(DENSE)), "n_layer": rng.randint(2, 6), "vocab": 32768,
                "ctx": rng.choice([0, _log(rng, 20, 900)]), "n_prompt": _log(rng, 2, 120), "n_gen": _log(rng, 4, 40)}
    if kind == "llama_prefill":
        return {"kind": kind, "shape": rng.choice(sorted(DENSE)), "n_layer": rng.randint(1, 4), "vocab": 32768,
                "ctx": rng.choice([0, _log(rng, 16, 700)]), "n_prompt": _log(rng, 8, 900),
                "snapshot": rng.random() < 0.25}
    if kind == "moe_turn":
        return {"kind": kind, "n_layer": 1, "vocab": 32768, "n_prompt": _log(rng, 2, 200), "n_gen": _log(rng, 4, 40)}
    if kind == "moe_tok":
        return {"kind": kind, "T": _log(rng, 2, 256), "n_exp": rng.choice([32, 64, 128]), "n_used": rng.choice([4, 8])}
    if kind == "qwen_turn":
        return {"kind": kind, "n_layer": 4, "vocab": 32768, "ffn": rng.choice([0, 512]), "n_prompt": _log(rng, 8, 1500),
                "n_gen": _log(rng, 4, 40)}
    return {"kind": kind, "T": _log(rng, 1, 256), "n_vh": rng.choice([16, 32])}


# ---- weights: GGUF blocks on the device, and their values in 64 bits ------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))


def _halves(x):
    return x.to(torch.float16).view(torch.uint8).reshape(x.shape[0], 2)


def _blocks(gen, code, n_rows, n_in, std=0.02):
    """n_rows rows of random GGUF blocks [blocks][block bytes], on the device."""
    vals, size = BLOCK[code]
    n = n_rows * (n_in // vals)
    blk = torch.randint(0, 256, (n, size), generator=gen, dtype=torch.uint8, device="cuda")
    jit = 0.75 + 0.5 * torch.rand(n, generator=gen, device="cuda")
    if code == Q8_0:
        blk[:, 0:2] = _halves(jit * (std / 74.0))
    elif code == Q6_K:
        blk[:, 208:210] = _halves(jit * (std / 1367.0))
    else:
        d = (jit * (std / (255.0 if code == Q4_K else 520.0))).to(torch.float16).float()
        blk[:, 0:2] = _halves(d)
        blk[:, 2:4] = _halves(d * (7.5 if code == Q4_K else 15.5))
    return blk


def _host(blk):
    return blk.reshape(-1).cpu().numpy()


def _f16(blk, at):
    return blk[:, at:at + 2].contiguous().view(torch.float16).double()


def _values(blk, code, n_in):
    """The blocks' values in 64 bits, [rows][n_in] (the GGUF formats)."""
    if code == Q8_0:
        v = blk[:, 2:].contiguous().view(torch.int8).double() * _f16(blk, 0)
    elif code == Q6_K:
        b = blk.int()
        ql, qh = b[:, 0:128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
        q = torch.stack([(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                         (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 1] >> 4) | ((qh >> 6) << 4)], 2)
        sc = blk[:, 192:208].contiguous().view(torch.int8).double() * _f16(blk, 208)
        v = (q.reshape(-1, 16, 16).double() - 32) * sc[:, :, None]
    else:
        b = blk.int()
        s = b[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, -128:].reshape(-1, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
        if code == Q5_K:
            qh = b[:, 16:48]
            q = q + 16 * ((qh[:, None, :] >> torch.arange(8, device=b.device)[None, :, None]) & 1)
        v = q.double() * (sc * _f16(blk, 0))[:, :, None] - (mn * _f16(blk, 2))[:, :, None]
    return v.reshape(-1, n_in)


def _normal(gen, *shape, scale=1.0):
    return torch.randn(*shape, generator=gen, device="cuda") * scale


def _np(t):
    return np.ascontiguousarray(t.cpu().numpy())


class _Session:
    """What a program keeps for one model or matrix; the library's device
    copies of its host buffers are dropped with it."""

    def __init__(self, **kw):
        self.__dict__.update(kw)
        self.registered = []

    def hold(self, *arrays):
        self.registered += [a.ctypes.data for a in arrays]
        return arrays[0]

    def __del__(self):
        try:
            L = _lib.load()
            for p in self.registered:
                L.draco_forget(ct.c_void_p(p))
        except Exception:
            pass


# ---- one matrix: m5_gemv, m5_gemm_*, draco_gemv_q8k_f32_noalloc ------------

_streams = []


def _stream():
    """The serving loop's one stream (calls of the allocation-free GEMV on one GPU must not overlap)."""
    if not _streams:
        _streams.append(torch.cuda.Stream())
    return _streams[0]


def _matrix(case, seed):
    code = CODE[case["code"]]
    g = _gen(seed)
    blk = _blocks(g, code, case["n_out"], case["n_in"])
    T = case.get("T", case.get("nvec", 1))
    return code, blk, _normal(g, T, case["n_in"])


def _prepare_matrix(case, seed):
    code, blk, x = _matrix(case, seed)
    s = _Session(case=case, code=code, n_out=case["n_out"], n_in=case["n_in"], lib=_lib.load())
    W = _host(blk)
    T = x.shape[0]
    if case["kind"] == "q8k":
        L = s.lib
        dev = np.zeros(L.draco_layout_query(code, s.n_out, s.n_in, (ct.c_size_t * 4)()), np.uint8)
        _lib.check(L.draco_repack(code, _lib.pu8(W), s.n_out, s.n_in, _lib.pu8(dev)), "draco_repack")
        s.W, s.x = torch.from_numpy(dev).cuda(), x.contiguous()
        s.y = torch.zeros(T, s.n_out, device="cuda")
        _stream().wait_stream(torch.cuda.current_stream())
    else:
        s.W, s.x = s.hold(W), _np(x)
        s.y = np.zeros((T, s.n_out), np.float32)
    _run_matrix(s)  # the weights become resident
    return s


def _run_matrix(s):
    c, L = s.case, s.lib
    if c["kind"] == "gemv":
        _lib.check(L.m5_gemv(s.code, _lib.pf(s.x), _lib.pu8(s.W), s.n_out, s.n_in, _lib.pf(s.y)), "m5_gemv")
    elif c["kind"] == "gemm":
        getattr(L, GEMM_ENTRY[c["code"]])(_lib.pf(s.x), _lib.pu8(s.W), c["T"], s.n_out, s.n_in, _lib.pf(s.y))
    else:
        _lib.check(L.draco_gemv_q8k_f32_noalloc(
            s.code, s.x.data_ptr(), c["nvec"], s.W.data_ptr(), s.n_out, s.n_in, s.y.data_ptr(),
            _stream().cuda_stream), "draco_gemv_q8k_f32_noalloc")
    return s.y


def _q8k_values(x):
    """x after the Q8_K activation format's rounding (its definition, in fp32)."""
    b = x.reshape(-1, 256)
    mx = b.gather(1, b.abs().argmax(1, keepdim=True))
    isc = -127.0 / mx
    q = torch.clamp(torch.round(isc * b), max=127)
    return (q.double() * (1.0 / isc).double()).reshape(x.shape)


def _exact_matrix(case, seed):
    code, blk, x = _matrix(case, seed)
    x = _q8k_values(x) if case["kind"] == "q8k" else x.double()
    return x @ _values(blk, code, case["n_in"]).T


# ---- llama-family models (dense and MoE) ----------------------------------

def _llama_cfg(case):
    if case["kind"] == "moe_turn":
        b, codes = MOE, MOE.codes
    else:
        b, codes = DENSE[case["shape"]]["base"], DENSE[case["shape"]]["codes"]
    need = case.get("ctx", 0) + case["n_prompt"] + case.get("n_gen", 0)
    return _models.LlamaConfig(
        name=case["kind"], hidden=b.hidden, n_layer=case["n_layer"], n_head=b.n_head, n_kv=b.n_kv,
        head_dim=b.head_dim, n_ff=b.n_ff, vocab=case["vocab"], eps=b.eps, rope_base=b.rope_base, codes=codes,
        tied=b.tied, max_t=max(64, 64 * -(-need // 64)), n_exp=b.n_exp, n_used=b.n_used, exp_ff=b.exp_ff)


def _llama_tensors(cfg, gen):
    """(name, code, rows, n_in, blocks or fp32 values) of every matrix, then (name, fp32) of every norm."""
    H, QD, KD, c = cfg.hidden, cfg.n_head * cfg.head_dim, cfg.n_kv * cfg.head_dim, cfg.codes
    yield "token_embd.weight", c["emb"], cfg.vocab, H, _blocks(gen, c["emb"], cfg.vocab, H)
    for il in range(cfg.n_layer):
        p = "blk.%d." % il
        for nm, k, rows, n_in in (("attn_q", "q", QD, H), ("attn_k", "k", KD, H), ("attn_v", "v", KD, H),
                                  ("attn_output", "o", H, QD)):
            yield p + nm + ".weight", c[k], rows, n_in, _blocks(gen, c[k], rows, n_in)
        if cfg.moe:
            E, F = cfg.n_exp, cfg.exp_ff
            yield p + "ffn_gate_inp.weight", F32, E, H, _normal(gen, E, H, scale=0.02)
            shapes = (("ffn_gate_exps", "gate", E * F, H), ("ffn_up_exps", "up", E * F, H), ("ffn_down_exps", "down", E * H, F))
        else:
            shapes = (("ffn_gate", "gate", cfg.n_ff, H), ("ffn_up", "up", cfg.n_ff, H), ("ffn_down", "down", H, cfg.n_ff))
        for nm, k, rows, n_in in shapes:
            yield p + nm + ".weight", c[k], rows, n_in, _blocks(gen, c[k], rows, n_in)
    if not cfg.tied:
        yield "output.weight", c["out"], cfg.vocab, H, _blocks(gen, c["out"], cfg.vocab, H)


def _llama_norms(cfg, gen):
    for il in range(cfg.n_layer):
        for nm in ("attn_norm", "ffn_norm"):
            yield "blk.%d.%s.weight" % (il, nm), 1.0 + 0.1 * torch.randn(cfg.hidden, generator=gen, device="cuda")
    yield "output_norm.weight", 1.0 + 0.1 * torch.randn(cfg.hidden, generator=gen, device="cuda")


def _prompts(case, seed):
    r = np.random.default_rng(seed + 1000)
    return (r.integers(0, case["vocab"], case.get("ctx", 0)).astype(np.int32),
            r.integers(0, case["vocab"], case["n_prompt"]).astype(np.int32))


def _prepare_llama(case, seed):
    cfg, gen = _llama_cfg(case), _gen(seed)
    s = _Session(case=case)
    m = _models.LlamaModel(cfg=cfg, seed=int(seed))
    for name, code, rows, n_in, v in _llama_tensors(cfg, gen):
        a = _np(v).view(np.uint8).reshape(-1) if code == F32 else _host(v)
        m.tensors[name] = (a, code, rows, n_in)
        if name.endswith("_exps.weight"):
            per = a.nbytes // cfg.n_exp
            s.registered += [a.ctypes.data + e * per for e in range(cfg.n_exp)]
        else:
            s.hold(a)
    for name, v in _llama_norms(cfg, gen):
        m.norms[name] = s.hold(_np(v))
    s.drv = d = _driver.LlamaDriver(m, _driver.hip_engine_lib(), max_t=cfg.max_t)
    s.hold(*d.kc, *d.vc)
    ctx, s.prompt = _prompts(case, seed)
    # the model becomes resident (one token), then the session's earlier turns
    d.prefill_chunk(s.prompt[:1], 0)
    _rewind(d, 0)
    if len(ctx):
        d.prefill_chunk(ctx, 0)
    return s


def _rewind(d, rows):
    for t in d.tl:
        t[0] = rows


def _run_llama(s):
    c, d = s.case, s.drv
    ctx = c.get("ctx", 0)
    _rewind(d, ctx)  # the session at the start of this turn
    if c["kind"] == "llama_prefill":
        logits = d.prefill_chunk(s.prompt, ctx)
        out = {"hidden": d.x, "logits": logits}
        if c["snapshot"]:  # the server's session slot
            _lib.check(_lib.load().draco_state_pull(ct.cast(d.descs, ct.c_void_p), d.NL), "draco_state_pull")
            n = (ctx + c["n_prompt"]) * d.cfg.n_kv * d.cfg.head_dim
            out["k"] = [a[:n] for a in d.kc]
            out["v"] = [a[:n] for a in d.vc]
        return out
    toks, hidden, _ = d.generate_device(s.prompt, c["n_gen"])
    return {"hidden": hidden, "logits": d.logits_of_x(), "tokens": np.asarray(toks, np.int32)}


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _silu(x):
    return x / (1 + torch.exp(-x))


def _causal(q, k, v, pos):
    """q [T][NH][D] over k, v [rows][NKV][D]: query t sees rows 0 .. pos + t."""
    rep = q.shape[1] // k.shape[1]
    s = torch.einsum("tgrd,kgd->grtk", q.reshape(q.shape[0], k.shape[1], rep, -1), k) / math.sqrt(q.shape[2])
    at = torch.arange(k.shape[0], device=q.device)[None, :] > pos + torch.arange(q.shape[0], device=q.device)[:, None]
    p = torch.softmax(s.masked_fill(at, -math.inf), -1)
    return torch.einsum("grtk,kgd->tgrd", p, v).reshape(q.shape[0], -1)


class _ExactLlama:
    """The llama family's forward in 64 bits (src/m6_engine.c:31-517), with the
    rope angles rounded to fp32 as the model defines them."""

    def __init__(self, case, seed):
        self.cfg, gen = _llama_cfg(case), _gen(seed)
        self.blk = {n: (b, code, n_in) for n, code, _, n_in, b in _llama_tensors(self.cfg, gen)}
        self.norm = {n: v.double() for n, v in _llama_norms(self.cfg, gen)}
        self.w = {n: self._dense(n) for n in self.blk if "_exps" not in n and n != "token_embd.weight"}
        if self.cfg.tied:
            self.w["output.weight"] = self._dense("token_embd.weight")
        self.k = [None] * self.cfg.n_layer
        self.v = [None] * self.cfg.n_layer

    def _dense(self, n, part=slice(None)):
        b, code, n_in = self.blk[n]
        return b.double() if code == F32 else _values(b[part], code, n_in)

    def _rope(self, x, pos):
        c = self.cfg
        e = (np.float32(-2.0) * np.arange(c.rot // 2, dtype=np.float32) / np.float32(c.rot)).astype(np.float64)
        f = np.power(float(np.float32(c.rope_base)), e).astype(np.float32)
        a = np.arange(pos, pos + x.shape[0], dtype=np.float32)[:, None] * f
        a = torch.from_numpy(a.astype(np.float64)).to(x.device)[:, None, :]
        e, o = x[..., 0::2], x[..., 1::2]
        return torch.stack([e * a.cos() - o * a.sin(), e * a.sin() + o * a.cos()], -1).reshape(x.shape)

    def _moe(self, x, p):
        c = self.cfg
        prob = torch.softmax(x @ self.w[p + "ffn_gate_inp.weight"].T, -1)
        wt, idx = torch.topk(prob, c.n_used, -1)
        wt = wt / wt.sum(-1, keepdim=True).clamp_min(6.103515625e-5)
        out = torch.zeros_like(x)
        for e in idx.unique().tolist():
            t, j = torch.nonzero(idx == e, as_tuple=True)
            m = []
            for nm in ("gate", "up", "down"):
                per = self.blk[p + "ffn_%s_exps.weight" % nm][0].shape[0] // c.n_exp
                m.append(self._dense(p + "ffn_%s_exps.weight" % nm, slice(e * per, (e + 1) * per)))
            out.index_add_(0, t, wt[t, j][:, None] * ((_silu(x[t] @ m[0].T) * (x[t] @ m[1].T)) @ m[2].T))
        return out

    def forward(self, ids):
        c, w = self.cfg, self.w
        pos = 0 if self.k[0] is None else self.k[0].shape[0]
        b, code, n_in = self.blk["token_embd.weight"]
        nb = n_in // BLOCK[code][0]
        ids = torch.as_tensor(np.asarray(ids, np.int64)).cuda()
        x = _values(b.reshape(-1, nb, b.shape[1])[ids].reshape(-1, b.shape[1]), code, n_in)
        T = x.shape[0]
        for il in range(c.n_layer):
            p = "blk.%d." % il
            xn = _rms(x, self.norm[p + "attn_norm.weight"], c.eps)
            q = self._rope((xn @ w[p + "attn_q.weight"].T).reshape(T, c.n_head, c.head_dim), pos)
            k = self._rope((xn @ w[p + "attn_k.weight"].T).reshape(T, c.n_kv, c.head_dim), pos)
            v = (xn @ w[p + "attn_v.weight"].T).reshape(T, c.n_kv, c.head_dim)
            self.k[il] = k if pos == 0 else torch.cat([self.k[il], k])
            self.v[il] = v if pos == 0 else torch.cat([self.v[il], v])
            x = x + _causal(q, self.k[il], self.v[il], pos) @ w[p + "attn_output.weight"].T
            xn = _rms(x, self.norm[p + "ffn_norm.weight"], c.eps)
            if c.moe:
                x = x + self._moe(xn, p)
            else:
                x = x + (_silu(xn @ w[p + "ffn_gate.weight"].T) * (xn @ w[p + "ffn_up.weight"].T)) @ w[p + "ffn_down.weight"].T
        return x[-1]

    def logits(self, x):
        return self.w["output.weight"] @ _rms(x, self.norm["output_norm.weight"], self.cfg.eps)


def _exact_llama(case, seed):
    m = _ExactLlama(case, seed)
    ctx, prompt = _prompts(case, seed)
    if len(ctx):
        m.forward(ctx)
    x = m.forward(prompt)
    if case["kind"] == "llama_prefill":
        out = {"hidden": x, "logits": m.logits(x)}
        if case["snapshot"]:
            out["k"] = [a.reshape(-1) for a in m.k]
            out["v"] = [a.reshape(-1) for a in m.v]
        return out
    toks = [int(m.logits(x).argmax())]
    for _ in range(case["n_gen"] - 1):
        x = m.forward(toks[-1:])
        toks.append(int(m.logits(x).argmax()))
    return {"hidden": x, "logits": m.logits(x), "tokens": None}


# ---- the hybrid (GDN + full attention) stack ------------------------------

QH, NKH, SV, NH, HD, NKV = _qwen.H, _qwen.NKH, _qwen.SV, 16, _qwen.HD_A, _qwen.NKV_A


def _qwen_cfg(case):
    need = case["n_prompt"] + case["n_gen"]
    return _qwen.QwenStackConfig(name="turn", n_layer=case["n_layer"], vocab=case["vocab"], max_t=64 * -(-need // 64),
                                 ffn=_qwen.FFN_DENSE if case["ffn"] else _qwen.FFN_NONE, n_ff=case["ffn"])


def _qwen_tensors(cfg, gen):
    """Per layer its named arrays: (code, rows, n_in, blocks) or an fp32 tensor."""
    def mat(code, rows, n_in):
        return code, rows, n_in, _blocks(gen, code, rows, n_in)

    def norm(n):
        return 1.0 + 0.1 * torch.randn(n, generator=gen, device="cuda")

    top = {"emb": mat(cfg.emb_code, cfg.vocab, QH), "head": mat(cfg.out_code, cfg.vocab, QH), "onorm": norm(QH)}
    layers = []
    for il in range(cfg.n_layer):
        if (il + 1) % cfg.interval == 0:
            c = cfg.full_codes
            a = {"attn_norm": norm(QH), "q": mat(c[0], NH * 2 * HD, QH), "k": mat(c[1], NKV * HD, QH),
                 "v": mat(c[2], NKV * HD, QH), "o": mat(c[3], QH, NH * HD), "q_norm": norm(HD), "k_norm": norm(HD),
                 "post_norm": norm(QH)}
        else:
            c, nv = cfg.gdn_codes, cfg.n_vh
            nq = 2 * NKH * SV + nv * SV
            a = {"attn_norm": norm(QH), "qkv": mat(c[0], nq, QH), "gate": mat(c[1], nv * SV, QH),
                 "ssm_out": mat(c[2], QH, nv * SV), "beta_wt": _normal(gen, QH, nv, scale=0.02),
                 "alpha_wt": _normal(gen, QH, nv, scale=0.02), "ssm_a": -torch.exp(_normal(gen, nv, scale=0.3)),
                 "ssm_dt": _normal(gen, nv, scale=0.3), "conv": _normal(gen, nq, 4, scale=0.5), "ssm_norm": norm(SV),
                 "post_norm": norm(QH)}
        if cfg.ffn:
            c = cfg.ffn_codes
            a.update(g=mat(c[0], cfg.n_ff, QH), u=mat(c[1], cfg.n_ff, QH), d=mat(c[2], QH, cfg.n_ff))
        layers.append(a)
    return top, layers


def _prepare_qwen(case, seed):
    cfg = _qwen_cfg(case)
    top, tens = _qwen_tensors(cfg, _gen(seed))
    s = _Session(case=case)

    def host(v):
        return s.hold(_host(v[3]) if isinstance(v, tuple) else _np(v))

    st = _qwen.QwenStack(cfg=cfg, seed=int(seed), emb=host(top["emb"]), head=host(top["head"]), onorm=host(top["onorm"]))
    for a in tens:
        h = {k: host(v) for k, v in a.items()}
        full = "q_norm" in h
        w = _qwen.FullW() if full else _qwen.GdnW()
        for k in ("attn_norm", "post_norm") + (("q_norm", "k_norm") if full else
                                               ("beta_wt", "alpha_wt", "ssm_a", "ssm_dt", "conv", "ssm_norm")):
            setattr(w, k, _lib.pf(h[k]))
        for k in ("q", "k", "v", "o") if full else ("qkv", "gate", "ssm_out"):
            setattr(w, k + "_buf", h[k].ctypes.data)
            setattr(w, k + "_code", a[k][0])
        if full:
            h["rope_inv"] = _qwen.rope_inv()
            w.rope_inv, w.nh = _lib.pf(h["rope_inv"]), NH
            st.layers.append(_qwen.FullLayer(nh=NH, codes=cfg.full_codes, arrays=h, w=w))
        else:
            w.n_qkv, w.n_vh, w.d_in = a["qkv"][1], cfg.n_vh, cfg.n_vh * SV
            L = _qwen.GdnLayer(n_vh=cfg.n_vh, codes=cfg.gdn_codes, arrays=h, w=w)
            L.ssm, L.tail = np.zeros(cfg.n_vh * SV * SV, np.float32), np.zeros(w.n_qkv * 3, np.float32)
            s.hold(L.ssm, L.tail)
            st.layers.append(L)
        st.ffn.append({k: h[k] for k in "gud"} if cfg.ffn else None)
    s.drv = d = _qwen.QwenStackDriver(st, _qwen.hip_ops(_lib.load()), _lib.load())
    s.hold(*d.kr.values(), *d.vc.values())
    s.prompt = _prompts(case, seed)[1]
    d.generate_device(s.prompt[:1], 1)  # the model becomes resident
    return s


def _run_qwen(s):
    d = s.drv
    # a new session: the zeroed recurrent states to the device (cached rows need none: only rows below the
    # position are read)
    _lib.check(d.lib.draco_qwen_state_push(ct.cast(d.descs, ct.c_void_p), d.cfg.n_layer, 0), "draco_qwen_state_push")
    toks, hidden, _ = d.generate_device(s.prompt, s.case["n_gen"])
    return {"hidden": hidden, "logits": d.logits_of_x(), "tokens": np.asarray(toks, np.int32)}


def _l2(x):
    return x / torch.sqrt((x * x).sum(-1, keepdim=True)).clamp_min(1e-6)


def _gdn_tokens(qkv, z, beta, dec, conv, norm, tail, S):
    """The GDN recurrence over T tokens in 64 bits (src/m6_gdn_scan.c:18-93):
    returns the gated output rows, the new tail [n_qkv][3] and state."""
    T, nv = beta.shape
    x = torch.cat([tail.T, qkv])
    c = _silu(sum(x[j:j + T] * conv[:, j] for j in range(4)))
    nh = (c.shape[1] // SV - nv) // 2
    c = c.reshape(T, -1, SV)
    q, k, v = _l2(c[:, :nh]), _l2(c[:, nh:2 * nh]), c[:, 2 * nh:]
    head = torch.arange(nv, device=S.device) % nh
    q, k = q[:, head], k[:, head]
    out = torch.empty_like(v)
    S = S.clone()
    for t in range(T):
        S *= dec[t][:, None, None]
        delta = (v[t] - torch.einsum("hkv,hk->hv", S, k[t])) * beta[t][:, None]
        S += k[t][:, :, None] * delta[:, None, :]
        out[t] = torch.einsum("hkv,hk->hv", S, q[t])
    out = _rms(out / math.sqrt(SV), norm, 1e-6) * _silu(z.reshape(T, nv, SV))
    return out.reshape(T, -1), x[T:].T.contiguous(), S


class _ExactQwen:
    def __init__(self, case, seed):
        self.cfg = _qwen_cfg(case)
        top, layers = _qwen_tensors(self.cfg, _gen(seed))
        self.emb = top["emb"]
        self.head, self.onorm = _values(top["head"][3], top["head"][0], QH), top["onorm"].double()
        self.L = [{k: (_values(v[3], v[0], v[2]) if isinstance(v, tuple) else v.double()) for k, v in a.items()} for a in layers]
        for a in self.L:
            if "q_norm" in a:
                a["K"] = a["V"] = torch.zeros(0, NKV, HD, dtype=torch.float64, device="cuda")
            else:
                a["S"] = torch.zeros(self.cfg.n_vh, SV, SV, dtype=torch.float64, device="cuda")
                a["tail"] = torch.zeros(a["conv"].shape[0], 3, dtype=torch.float64, device="cuda")
        self.pos = 0

    def _rope(self, x):
        ang = np.arange(self.pos, self.pos + x.shape[0], dtype=np.float32)[:, None] * _qwen.rope_inv()
        ang = torch.from_numpy(ang.astype(np.float64)).to(x.device)[:, None, :]
        a, b = x[..., :32], x[..., 32:64]
        return torch.cat([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos(), x[..., 64:]], -1)

    def forward(self, ids):
        code, _, n_in, b = self.emb
        ids = torch.as_tensor(np.asarray(ids, np.int64)).cuda()
        x = _values(b.reshape(self.cfg.vocab, -1, b.shape[1])[ids].reshape(-1, b.shape[1]), code, n_in)
        T = x.shape[0]
        for a in self.L:
            xn = _rms(x, a["attn_norm"], 1e-6)
            if "q_norm" in a:
                qg = (xn @ a["q"].T).reshape(T, NH, 2, HD)
                q = self._rope(_rms(qg[:, :, 0], a["q_norm"], 1e-6))
                a["K"] = torch.cat([a["K"], self._rope(_rms((xn @ a["k"].T).reshape(T, NKV, HD), a["k_norm"], 1e-6))])
                a["V"] = torch.cat([a["V"], (xn @ a["v"].T).reshape(T, NKV, HD)])
                o = _causal(q, a["K"], a["V"], self.pos) * torch.sigmoid(qg[:, :, 1].reshape(T, -1))
                x = x + o @ a["o"].T
            else:
                sp = torch.nn.functional.softplus(xn @ a["alpha_wt"] + a["ssm_dt"], threshold=1e9)
                o, a["tail"], a["S"] = _gdn_tokens(xn @ a["qkv"].T, xn @ a["gate"].T, torch.sigmoid(xn @ a["beta_wt"]),
                                                   torch.exp(sp * a["ssm_a"]), a["conv"], a["ssm_norm"], a["tail"], a["S"])
                x = x + o @ a["ssm_out"].T
            if "g" in a:
                xn = _rms(x, a["post_norm"], 1e-6)
                x = x + (_silu(xn @ a["g"].T) * (xn @ a["u"].T)) @ a["d"].T
        self.pos += T
        return x[-1]

    def logits(self, x):
        return self.head @ _rms(x, self.onorm, self.cfg.eps)


def _exact_qwen(case, seed):
    m = _ExactQwen(case, seed)
    x = m.forward(_prompts(case, seed)[1])
    toks = [int(m.logits(x).argmax())]
    for _ in range(case["n_gen"] - 1):
        x = m.forward(toks[-1:])
        toks.append(int(m.logits(x).argmax()))
    return {"hidden": x, "logits": m.logits(x), "tokens": None}


# ---- the prefill driver's two ops on host buffers -------------------------

def _scan_inputs(case, seed):
    T, nv, g = case["T"], case["n_vh"], _gen(seed)
    nq = 2 * NKH * SV + nv * SV
    sp = torch.nn.functional.softplus
    return {"QKV": _normal(g, T, nq), "Z": _normal(g, T, nv * SV), "B": torch.sigmoid(_normal(g, T, nv)),
            "G": torch.exp(-sp(_normal(g, T, nv))), "conv": _normal(g, nq, 4, scale=0.5),
            "norm": 1.0 + 0.1 * torch.randn(SV, generator=g, device="cuda"), "tail": _normal(g, nq, 3),
            "S": _normal(g, nv, SV, SV, scale=0.05)}


def _prepare_scan(case, seed):
    a = {k: _np(v) for k, v in _scan_inputs(case, seed).items()}
    s = _Session(case=case, lib=_lib.load(), a=a, tail0=a["tail"].copy(), S0=a["S"].copy(),
                 ON=np.zeros((case["T"], case["n_vh"] * SV), np.float32), work=np.zeros(a["QKV"].shape[1], np.float32))
    s.hold(a["S"], a["tail"])
    return s


def _run_scan(s):
    a, c, pf = s.a, s.case, _lib.pf
    a["tail"][...], a["S"][...] = s.tail0, s.S0  # the session's state before this chunk
    s.lib.m6_gdn_scan(pf(a["QKV"]), pf(a["Z"]), pf(a["B"]), pf(a["G"]), pf(a["conv"]), pf(a["norm"]), pf(a["tail"]),
                      pf(a["S"]), c["T"], a["QKV"].shape[1], c["n_vh"], pf(s.ON), pf(s.work))
    return {"out": s.ON, "tail": a["tail"], "S": a["S"]}


def _exact_scan(case, seed):
    a = {k: v.double() for k, v in _scan_inputs(case, seed).items()}
    o, tail, S = _gdn_tokens(a["QKV"], a["Z"], a["B"], a["G"], a["conv"], a["norm"], a["tail"], a["S"])
    return {"out": o, "tail": tail, "S": S}


def _tok_inputs(case, seed):
    g, E, F, H, T = _gen(seed), case["n_exp"], MOE.exp_ff, MOE.hidden, case["T"]
    w = [_blocks(g, Q4_K, E * F, H), _blocks(g, Q4_K, E * F, H), _blocks(g, Q4_K, E * H, F)]
    wt, order = torch.topk(torch.softmax(_normal(g, T, E), -1), case["n_used"], -1)
    return w, _normal(g, T, H), (wt / wt.sum(-1, keepdim=True)).float(), order


def _prepare_tok(case, seed):
    w, x, wt, order = _tok_inputs(case, seed)
    E = case["n_exp"]
    s = _Session(case=case, lib=_lib.load(), w=[_host(b) for b in w], x=_np(x), wt=_np(wt),
                 order=_np(order.int()), ep=np.zeros(3 * E, np.uint64), ec=np.full(3 * E, Q4_K, np.int32),
                 out=np.zeros((case["T"], MOE.hidden), np.float32), work=np.zeros(64, np.float32),
                 iwork=np.zeros(64, np.int32))
    for k, a in enumerate(s.w):
        at = a.ctypes.data + (a.nbytes // E) * np.arange(E, dtype=np.uint64)
        s.ep[k::3] = at
        s.registered += [int(p) for p in at]
    _run_tok(s)  # the experts become resident
    return s


def _run_tok(s):
    c, pf, pi = s.case, _lib.pf, _lib.pi32
    s.lib.m6_moe_tok(None, None, pf(s.work), pf(s.x), pi(s.order), pf(s.wt), _lib.vp(s.ep), pi(s.ec), c["T"], c["n_used"],
                     MOE.exp_ff, MOE.hidden, MOE.hidden, c["n_exp"], pf(s.out), pf(s.work), pi(s.iwork))
    return s.out


def _exact_tok(case, seed):
    w, x, wt, order = _tok_inputs(case, seed)
    x, wt, out = x.double(), wt.double(), torch.zeros_like(x, dtype=torch.float64)
    per = [b.shape[0] // case["n_exp"] for b in w]
    for e in order.unique().tolist():
        t, j = torch.nonzero(order == e, as_tuple=True)
        g, u, d = (_values(b[e * p:(e + 1) * p], Q4_K, n) for b, p, n in zip(w, per, (MOE.hidden, MOE.hidden, MOE.exp_ff)))
        out.index_add_(0, t, wt[t, j][:, None] * ((_silu(x[t] @ g.T) * (x[t] @ u.T)) @ d.T))
    return out


# ---- the interface ---------------------------------------------------------

_KINDS = {"gemv": (_prepare_matrix, _run_matrix, _exact_matrix), "q8k": (_prepare_matrix, _run_matrix, _exact_matrix),
          "gemm": (_prepare_matrix, _run_matrix, _exact_matrix), "llama_turn": (_prepare_llama, _run_llama, _exact_llama),
          "llama_prefill": (_prepare_llama, _run_llama, _exact_llama),
          "moe_turn": (_prepare_llama, _run_llama, _exact_llama), "qwen_turn": (_prepare_qwen, _run_qwen, _exact_qwen),
          "gdn_scan": (_prepare_scan, _run_scan, _exact_scan), "moe_tok": (_prepare_tok, _run_tok, _exact_tok)}


def prepare(case, seed):
    return _KINDS[case["kind"]][0](case, seed)


def run(state):
    return _KINDS[state.case["kind"]][1](state)


def exact(case, seed):
    return _KINDS[case["kind"]][2](case, seed)


def _mat_bytes(code, rows, n_in):
    vals, size = BLOCK[code]
    return rows * n_in // vals * size


def _turn_work(layer_bytes, layer_macs, head_bytes, head_macs, row_bytes, attn_macs, ctx, n_prompt, n_gen, n_layer):
    """A prompt in one pass over the weights, then one pass a token; each
    cached row read once a pass and written once.  attn_macs: multiply-adds of one query and one cached row,
    over all layers; row_bytes: one cached row's K and V, over all layers."""
    steps = max(0, n_gen - 1)
    n = ctx + n_prompt
    b = layer_bytes * n_layer * (1 + steps) + head_bytes * max(1, n_gen)
    b += row_bytes * (n + sum(n + i for i in range(steps)) + n_prompt + steps)
    f = 2 * layer_macs * n_layer * (n_prompt + steps) + 2 * head_macs * max(1, n_gen)
    f += 2 * attn_macs * (sum(ctx + i + 1 for i in range(n_prompt)) + sum(n + i + 1 for i in range(steps)))
    return {"bytes": b, "flops": f}


def work(case):
    k = case["kind"]
    if k in ("gemv", "gemm", "q8k"):
        T, o, i = case.get("T", case.get("nvec", 1)), case["n_out"], case["n_in"]
        return {"bytes": _mat_bytes(CODE[case["code"]], o, i) + 4 * T * (o + i), "flops": 2 * T * o * i}
    if k in ("llama_turn", "llama_prefill", "moe_turn"):
        c = _llama_cfg(case)
        H, QD, KD, co = c.hidden, c.n_head * c.head_dim, c.n_kv * c.head_dim, c.codes
        mats = [(co["q"], QD, H), (co["k"], KD, H), (co["v"], KD, H), (co["o"], H, QD)]
        n_prompt = case["n_prompt"]
        if c.moe:
            # a token reads n_used experts; the prompt's tokens together read each expert they touch once
            ex = _mat_bytes(co["gate"], c.exp_ff, H) * 2 + _mat_bytes(co["down"], H, c.exp_ff)
            macs = sum(r * n for _, r, n in mats) + c.n_exp * H + c.n_used * 3 * c.exp_ff * H
            lb = sum(_mat_bytes(*m) for m in mats) + 4 * c.n_exp * H + c.n_used * ex
            extra = c.n_layer * ex * (c.n_exp * (1 - (1 - c.n_used / c.n_exp) ** n_prompt) - c.n_used)
        else:
            mats += [(co["gate"], c.n_ff, H), (co["up"], c.n_ff, H), (co["down"], H, c.n_ff)]
            macs, lb, extra = sum(r * n for _, r, n in mats), sum(_mat_bytes(*m) for m in mats), 0
        w = _turn_work(lb, macs, _mat_bytes(co["out"], c.vocab, H), c.vocab * H, 8 * KD * c.n_layer, 2 * QD * c.n_layer,
                       case.get("ctx", 0), n_prompt, case.get("n_gen", 0), c.n_layer)
        w["bytes"] += extra + (8 * KD * c.n_layer * (case["ctx"] + n_prompt) if case.get("snapshot") else 0)
        return w
    if k == "qwen_turn":
        c = _qwen_cfg(case)
        nf = c.n_layer // c.interval
        ng = c.n_layer - nf
        nq = 2 * NKH * SV + c.n_vh * SV
        gd = [(Q4_K, nq, QH), (Q4_K, c.n_vh * SV, QH), (Q4_K, QH, c.n_vh * SV)]
        fu = [(Q4_K, NH * 2 * HD, QH), (Q4_K, NKV * HD, QH), (Q4_K, NKV * HD, QH), (Q4_K, QH, NH * HD)]
        ff = [(Q4_K, c.n_ff, QH), (Q4_K, c.n_ff, QH), (Q6_K, QH, c.n_ff)] if c.ffn else []
        mats = gd * ng + fu * nf + ff * c.n_layer
        state = c.n_vh * SV * SV
        lb = sum(_mat_bytes(*m) for m in mats) + ng * (8 * state + 8 * QH * c.n_vh)
        macs = sum(r * n for _, r, n in mats) + ng * (4 * state + 2 * QH * c.n_vh)
        return _turn_work(lb, macs, _mat_bytes(c.out_code, c.vocab, QH), c.vocab * QH, 8 * NKV * HD * nf, 2 * NH * HD * nf,
                          0, case["n_prompt"], case["n_gen"], 1)
    if k == "gdn_scan":
        T, nv = case["T"], case["n_vh"]
        nq = 2 * NKH * SV + nv * SV
        return {"bytes": 4 * (T * (nq + 2 * nv * SV + 2 * nv) + 10 * nq + SV + 2 * nv * SV * SV), "flops": 8 * T * nv * SV * SV}
    T, H, F = case["T"], MOE.hidden, MOE.exp_ff
    touched = case["n_exp"] * (1 - (1 - case["n_used"] / case["n_exp"]) ** T)
    return {"bytes": touched * 3 * _mat_bytes(Q4_K, F, H) + 8 * T * H, "flops": 6 * T * case["n_used"] * F * H}


def tolerance(case):
    """About four times the error against 64 bits that the engine's fp32
    arithmetic shows over the listed and drawn cases (single products and ops
    2e-7; 1 to 16 layers of the 1B shape 8e-7 to 6e-6, rounding growing from
    layer to layer; the other stacks 3e-7 to 9e-7).  The largest difference is
    left to its usual multiple of these."""
    return {"gemv": {"rel": 1e-6}, "q8k": {"rel": 1e-6}, "gemm": {"rel": 1e-6}, "moe_tok": {"rel": 1e-6},
            "gdn_scan": {"rel": 1e-6}, "llama_prefill": {"rel": 1.2e-5}, "llama_turn": {"rel": 2.5e-5},
            "moe_turn": {"rel": 4e-6}, "qwen_turn": {"rel": 3e-6}}[case["kind"]]
