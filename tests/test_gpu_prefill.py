"""Chunked prefill of the llama family (draco_llama_prefill, and the prompt of
draco_llama_generate) against token-serial decoding.

The contract is the reference's forward_chunk (src/qwen35_prefill.py:209-210,
src/draco_engine_server.py:836-842): afterwards the engine state is the one
forward(ids[i], pos0 + i) leaves when run token by token, and the call returns
the last position's logits.  Checked here against the compiled-reference
oracle's token-serial run (logits, KV caches), against this library's own
token-serial device path, across chunk boundaries (ragged chunks, a second
call at pos0 > 0), at head dims 64 and 128 and GQA ratios 1-5, and through the
goldens of whole greedy decodes (the device-generate tests, whose prompts go
through the chunked prefill by default).

Bars: logits 1e-4 normwise (every layer's products are reordered fp32 sums,
as in the per-token deep-layer KV bar); KV rows 1e-5 for layer 0 (one GEMM +
rope from the input) and 1e-4 deeper; greedy continuations identical.
"""
import ctypes as ct
import dataclasses

import numpy as np
import pytest

from helpers import golden, rel_err
from dracohip import lib, models
from dracohip.driver import LlamaDriver, hip_engine_lib

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _restore_chunk():
    L = lib.load()
    old = L.draco_set_prefill_chunk(-1)
    yield
    L.draco_set_prefill_chunk(old)


def _pair(cfg, oracle):
    from tests_oracle_engine import oracle_engine
    model = models.build_llama(cfg, 0)
    lib.load().draco_reset()
    return model, LlamaDriver(model, hip_engine_lib()), LlamaDriver(model, oracle_engine(oracle))


def _serial_logits(drv, ids, pos0):
    for i, t in enumerate(ids):
        drv.forward(int(t), pos0 + i)
    return drv.logits_of_x().copy()


@pytest.mark.parametrize("chunk", [256, 7, 1])
@pytest.mark.parametrize("cfgname", ["tiny-kquant", "tiny-q8_0"])
def test_prefill_matches_oracle_serial(oracle, cfgname, chunk):
    """40 tokens in one call (chunks of `chunk` tokens, the last one ragged)
    against the oracle's token-serial run: logits, every layer's KV rows,
    tlen, and 6 greedy continuation tokens."""
    cfg = dataclasses.replace(models.CONFIGS[cfgname], max_t=64)
    model, drv, ref = _pair(cfg, oracle)
    L = lib.load()
    L.draco_set_prefill_chunk(chunk)
    ids = np.random.default_rng(7).integers(0, cfg.vocab, 40).astype(np.int32)
    print(f"[prefill] {cfgname} chunk {chunk}", flush=True)
    lg = drv.prefill_chunk(ids, 0).copy()
    lr = _serial_logits(ref, ids, 0)
    assert rel_err(lg, lr) <= 1e-4
    assert drv.tl[0][0] == ref.tl[0][0] == len(ids)
    assert L.draco_state_pull(ct.cast(drv.descs, ct.c_void_p), drv.NL) == 0
    n = len(ids) * cfg.n_kv * cfg.head_dim
    for l in range(cfg.n_layer):
        tol = 1e-5 if l == 0 else 1e-4
        assert rel_err(drv.kc[l][:n], ref.kc[l][:n]) <= tol
        assert rel_err(drv.vc[l][:n], ref.vc[l][:n]) <= tol
    # greedy continuation from the prefilled state, token by token on both
    a, b = [int(np.argmax(lg))], [int(np.argmax(lr))]
    assert a == b
    for s in range(5):
        pos = len(ids) + s
        drv.forward(a[-1], pos)
        ref.forward(b[-1], pos)
        a.append(int(np.argmax(drv.logits_of_x())))
        b.append(int(np.argmax(ref.logits_of_x())))
    assert a == b


def test_prefill_second_call_at_offset(oracle):
    """Two calls (20 tokens, then 17 at pos0 = 20, chunk 8): the second
    chunk's queries attend the first call's cache rows."""
    cfg = dataclasses.replace(models.TINY_K, max_t=64)
    model, drv, ref = _pair(cfg, oracle)
    lib.load().draco_set_prefill_chunk(8)
    ids = np.random.default_rng(11).integers(0, cfg.vocab, 37).astype(np.int32)
    drv.prefill_chunk(ids[:20], 0)
    lg = drv.prefill_chunk(ids[20:], 20).copy()
    lr = _serial_logits(ref, ids, 0)
    assert rel_err(lg, lr) <= 1e-4
    assert drv.tl[-1][0] == 37


@pytest.mark.parametrize("hd,nh,nkv", [(128, 3, 1), (128, 2, 2), (64, 5, 1), (64, 8, 1)])
def test_prefill_head_shapes(oracle, hd, nh, nkv):
    """Head dim 128 and GQA ratios 1, 2(rep 1), 5 and 8 through the chunk
    attention kernel, 48 tokens in chunks of 16 against the oracle."""
    cfg = dataclasses.replace(models.TINY_Q8, name=f"pf-{hd}-{nh}-{nkv}", head_dim=hd, n_head=nh, n_kv=nkv,
                              max_t=128)
    model, drv, ref = _pair(cfg, oracle)
    lib.load().draco_set_prefill_chunk(16)
    ids = np.random.default_rng(13).integers(0, cfg.vocab, 48).astype(np.int32)
    print(f"[prefill] hd {hd} nh {nh} nkv {nkv}", flush=True)
    lg = drv.prefill_chunk(ids, 0).copy()
    lr = _serial_logits(ref, ids, 0)
    assert rel_err(lg, lr) <= 1e-4


@pytest.mark.parametrize("hd,nh,nkv", [(64, 2, 2), (64, 4, 2), (64, 6, 2), (128, 7, 1)])
def test_prefill_attention_tile_edges(oracle, hd, nh, nkv):
    """The attention's 16-query and 32-key tiles at their edges: chunks of 33,
    33 and 5 tokens, with blocks of one q head and four query tiles, two and
    two, three and two (six waves) and seven heads (the logits depend on every
    position's attention through the second layer's K / V rows)."""
    cfg = dataclasses.replace(models.TINY_Q8, name=f"pfe-{hd}-{nh}-{nkv}", head_dim=hd, n_head=nh, n_kv=nkv,
                              max_t=128)
    model, drv, ref = _pair(cfg, oracle)
    lib.load().draco_set_prefill_chunk(33)
    ids = np.random.default_rng(17).integers(0, cfg.vocab, 71).astype(np.int32)
    lg = drv.prefill_chunk(ids, 0).copy()
    lr = _serial_logits(ref, ids, 0)
    assert rel_err(lg, lr) <= 1e-4


@pytest.mark.parametrize("chunk", [1, 4, 5, 33])
@pytest.mark.parametrize("n_used", [1, 3])
def test_moe_prefill_matches_oracle_serial(oracle, chunk, n_used):
    """A MoE model's prompt in chunks (the router, top-k and expert grouping
    of all rows on the device) against the oracle's token-serial run, at chunk
    lengths around the router's four tokens a block and the experts' 32-token
    tiles."""
    cfg = dataclasses.replace(models.MOE_TINY, name=f"moe-pf-{n_used}", hidden=1024, n_head=8, n_kv=2,
                              n_exp=16, n_used=n_used, exp_ff=512, vocab=512, max_t=64, wscale=0.05)
    model, drv, ref = _pair(cfg, oracle)
    lib.load().draco_set_prefill_chunk(chunk)
    ids = np.random.default_rng(19).integers(0, cfg.vocab, 38).astype(np.int32)
    lg = drv.prefill_chunk(ids, 0).copy()
    lr = _serial_logits(ref, ids, 0)
    assert rel_err(lg, lr) <= 1e-4


@pytest.mark.parametrize("n", [1, 2, 3])
def test_moe_prefill_of_few_tokens_is_token_serial(n):
    """Up to three tokens of a MoE model go through the decode layers (a chunk
    takes more launches and reads as many experts): the hidden row and the
    generation after them are those of the tokens one by one, bit for bit."""
    cfg = dataclasses.replace(models.MOE_TINY, name="moe-pf-few", n_exp=16, n_used=3, exp_ff=256, vocab=256, max_t=16,
                              wscale=0.05)
    model = models.build_llama(cfg, 0)
    ids = np.random.default_rng(41).integers(0, cfg.vocab, n).astype(np.int32)
    lib.load().draco_reset()
    one, many = LlamaDriver(model, hip_engine_lib()), LlamaDriver(model, hip_engine_lib())
    lr = _serial_logits(one, ids, 0)
    assert np.array_equal(many.prefill_chunk(ids, 0), lr) and np.array_equal(many.x, one.x)


def test_moe_prefill_wider_than_the_chunk_norms(oracle):
    """A MoE model of hidden rows beyond the chunk's norms (4096): its prompt
    goes token by token through the decode layers."""
    cfg = dataclasses.replace(models.MOE_TINY, name="moe-pf-wide", hidden=4352, n_layer=1, n_head=4, n_kv=2,
                              head_dim=64, n_exp=8, n_used=2, exp_ff=256, vocab=256, max_t=16, wscale=0.05)
    model, drv, ref = _pair(cfg, oracle)
    ids = np.random.default_rng(23).integers(0, cfg.vocab, 5).astype(np.int32)
    lg = drv.prefill_chunk(ids, 0).copy()
    lr = _serial_logits(ref, ids, 0)
    assert rel_err(lg, lr) <= 1e-4


@pytest.mark.parametrize("base", ["TINY_K", "TINY_Q8"])
def test_dense_prefill_wider_than_the_chunk_norms(oracle, base):
    """A dense model of hidden rows beyond the chunk's norms (4096) and an
    attention shape that the chunk serves: its prompt goes token by token, also
    inside a generate call."""
    cfg = dataclasses.replace(getattr(models, base), name="pf-wide-" + base, hidden=4352, n_layer=1, n_head=4, n_kv=2,
                              head_dim=64, n_ff=512, vocab=256, max_t=16)
    model, drv, ref = _pair(cfg, oracle)
    ids = np.random.default_rng(29).integers(0, cfg.vocab, 5).astype(np.int32)
    lg = drv.prefill_chunk(ids, 0).copy()
    lr = _serial_logits(ref, ids, 0)
    assert rel_err(lg, lr) <= 1e-4
    drv.reset()
    lib.load().draco_reset()
    _, hidden, _ = drv.generate_device(ids, 1)
    assert rel_err(hidden, ref.x) <= 1e-4


@pytest.mark.parametrize("qk,v,ff,hidden", [(5, 4, 5, 1024), (3, 4, 3, 1024), (4, 4, 4, 768), (0, 0, 0, 960)])
def test_prefill_two_stream_launches(oracle, qk, v, ff, hidden):
    """Rows of at most four super-blocks and 1024 or more (row, token) tiles:
    q, k and v (mixed formats: Q4_K or Q5_K with Q6_K) and the gate / up pair
    run in the GEMM's two-stream form, the pair over an odd number of row tiles
    (129), so that a block's second stream ends past the matrix.  Every token's
    K / V rows of the second layer see the first layer's whole output."""
    cfg = dataclasses.replace(models.TINY_K, name=f"pf2s-{qk}-{ff}", hidden=hidden, n_layer=2, n_head=32, n_kv=8,
                              head_dim=128, n_ff=4128, vocab=256, max_t=256, wscale=0.05,
                              codes=dict(models.TINY_K.codes, q=qk, k=qk, v=v, gate=ff, up=ff, down=0, emb=0, out=0))
    model, drv, ref = _pair(cfg, oracle)
    lib.load().draco_set_prefill_chunk(256)
    ids = np.random.default_rng(37).integers(0, cfg.vocab, 230).astype(np.int32)
    lg = drv.prefill_chunk(ids, 0).copy()
    lr = _serial_logits(ref, ids, 0)
    assert rel_err(lg, lr) <= 1e-4
    assert lib.load().draco_state_pull(ct.cast(drv.descs, ct.c_void_p), drv.NL) == 0
    n = len(ids) * cfg.n_kv * cfg.head_dim
    for l in range(cfg.n_layer):
        assert rel_err(drv.kc[l][:n], ref.kc[l][:n]) <= (1e-5 if l == 0 else 1e-4)
        assert rel_err(drv.vc[l][:n], ref.vc[l][:n]) <= (1e-5 if l == 0 else 1e-4)


@pytest.mark.parametrize("cfgname,fname", [("tiny-kquant", "llama_tiny_k.npz"), ("tiny-q8_0", "llama_tiny_q8.npz")])
def test_generate_token_serial_prompt(cfgname, fname):
    """draco_llama_generate with the chunked prefill switched off feeds the
    prompt token by token (graph-replayed steps): still the golden tokens."""
    g = golden(fname)
    cfg = models.CONFIGS[cfgname]
    model = models.build_llama(cfg, 0)
    L = lib.load()
    L.draco_reset()
    L.draco_set_prefill_chunk(0)
    drv = LlamaDriver(model, hip_engine_lib())
    toks, hidden, _ = drv.generate_device(model.prompt(), cfg.n_gen, use_graph=True)
    assert toks == list(g["tokens"])


def test_llama1b_chunked_matches_serial_device():
    """the 960-token prompt through 256-token chunks against the
    same prompt through token-serial device steps: identical greedy tokens,
    final hidden states within 1e-3."""
    cfg = models.LLAMA1B
    model = models.build_llama(cfg, 0)
    L = lib.load()
    L.draco_reset()
    out = {}
    for chunk in (256, 0):
        L.draco_set_prefill_chunk(chunk)
        drv = LlamaDriver(model, hip_engine_lib())
        drv.reset()
        L.draco_state_push(ct.cast(drv.descs, ct.c_void_p), drv.NL)
        toks, hidden, st = drv.generate_device(model.prompt(), 16, use_graph=True)
        print(f"[prefill] llama1b chunk {chunk}: prefill {st[1]:.1f} ms", flush=True)
        out[chunk] = (toks, hidden.copy())
    assert out[256][0] == out[0][0]
    assert np.max(np.abs(out[256][1] - out[0][1])) <= 1e-3
