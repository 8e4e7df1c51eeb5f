"""The batched GEMV (plh_matmul_batch) on the matrix cores, bit for bit against
the oracle's vec_dot per (row, token): every waves-per-row-tile form (chosen by
the number of 16 x 16 tiles: to 256 eight waves where rows are of 1024 or more,
below 1024 four, below 2048 two, else one),
rows and tokens that leave partial tiles, rows of one unit, of one chunk, of an
odd number of blocks (Q8_0's half unit), and the shapes that stay on the VALU
kernel.  Subnormal and huge activations, and infinities and NaNs that must stay
in their token."""
import ctypes as C

import numpy as np
import pytest

from attn_check import FWD_TOL_FAST, KV_TOL
from picolm_amd import gemv as G
from picolm_amd import synth as S

pytestmark = pytest.mark.gpu

Q4, Q6, Q8 = G.TYPE_Q4_K, G.TYPE_Q6_K, G.TYPE_Q8_0


def batch(P, W, X):
    dx, out = P.DeviceBuffer.from_numpy(X), P.DeviceBuffer(4 * X.shape[0] * W.d)
    P.check(P.lib.plh_matmul_batch(W.qtype, W.n, W.d, C.c_void_p(W.ptr), C.c_void_p(dx.ptr),
                                   X.shape[0], C.c_void_p(out.ptr)), "plh_matmul_batch")
    got = out.download(np.float32, (X.shape[0], W.d))
    dx.free()
    out.free()
    return got


def assert_bits(got, want, what):
    bad = np.flatnonzero(got.view(np.uint32) != want.view(np.uint32))
    # a NaN's payload is not part of the contract
    bad = bad[~(np.isnan(got.ravel()[bad]) & np.isnan(want.ravel()[bad]))]
    assert bad.size == 0, (what, bad[:8], got.ravel()[bad[:4]], want.ravel()[bad[:4]])


@pytest.mark.parametrize("qtype,n,d,tokens", [
    (Q4, 256, 1, 16), (Q4, 256, 77, 33), (Q4, 512, 16, 15), (Q4, 768, 65, 17), (Q4, 2048, 200, 5),
    (Q6, 256, 3, 19), (Q6, 512, 33, 16), (Q6, 1280, 130, 31), (Q6, 2048, 64, 6),
    (Q8, 32, 5, 20), (Q8, 64, 16, 16), (Q8, 96, 100, 37), (Q8, 288, 17, 18), (Q8, 1056, 64, 33),
    (Q4, 1280, 64, 17), (Q4, 1536, 40, 16), (Q6, 1024, 50, 16), (Q6, 2304, 33, 31),  # eight
    (Q8, 1184, 48, 33), (Q8, 2080, 17, 16), (Q4, 2048, 2048, 32), (Q4, 2048, 2049, 32),
    (Q4, 256, 8200, 32), (Q6, 256, 8200, 32), (Q8, 160, 8200, 32),     # two waves a tile
    (Q4, 512, 16400, 31), (Q6, 256, 16400, 32), (Q8, 96, 16400, 32),   # one (Q8_0 two)
    (Q4, 11008, 65, 5), (Q6, 11008, 20, 3), (Q8, 11008, 33, 4)])       # the VALU kernel
def test_matmul_batch_tiles(gpu, oracle_mod, qtype, n, d, tokens):
    P, O = gpu, oracle_mod
    print(f"[case] batch type {qtype} n {n} d {d} tokens {tokens}", flush=True)
    rng = np.random.default_rng([qtype, n, d, tokens])
    rows = S.random_weights(rng, qtype, n, d, S.unit_scale_exp(qtype, n))
    W = G.QMatrix(qtype, n, d, rows)
    X = rng.standard_normal((tokens, n)).astype(np.float32)
    got = batch(P, W, X)
    for t in range(tokens):
        assert_bits(got[t], O.matmul(rows, X[t], n, d, qtype), t)
    W.free()


@pytest.mark.parametrize("qtype", [Q4, Q6, Q8])
def test_matmul_batch_special_values(gpu, oracle_mod, qtype):
    """Tokens of subnormal, huge, mixed and zero activations, one with an
    infinity and one with a NaN (whose rows alone are not finite), and rows
    with zero scales."""
    P, O = gpu, oracle_mod
    n, d, tokens = 512, 40, 24
    rng = np.random.default_rng(77 + qtype)
    rows = S.random_weights(rng, qtype, n, d, S.unit_scale_exp(qtype, n))
    at = {Q4: slice(0, 4), Q6: slice(208, 210), Q8: slice(0, 2)}[qtype]
    rows.reshape(d, -1, G.BLOCK[qtype][1])[::5, :, at] = 0
    X = rng.standard_normal((tokens, n)).astype(np.float32)
    X[1] *= 1e-39
    X[2] *= 1e-43
    X[3] *= 1e30
    X[4] = 0.0
    X[5] *= np.exp2(rng.integers(-60, 60, n)).astype(np.float32)
    X[6] = -0.0
    X[7, 100] = np.inf
    X[8, 200] = np.nan
    W = G.QMatrix(qtype, n, d, rows)
    got = batch(P, W, X)
    for t in range(tokens):
        with np.errstate(all="ignore"):
            want = O.matmul(rows, X[t], n, d, qtype)
        assert_bits(got[t], want, t)
    assert np.isfinite(got[[0, 4, 9, 23]]).all() and not np.isfinite(got[7:9]).all()
    W.free()


def test_matmul_batch_more_outputs_than_a_launch(gpu, oracle_mod):
    """131072 rows of one block and 65600 tokens: 2^33 outputs and some, past
    what one launch of 16 x 16 tiles can hold (2^32 threads), not past the VALU
    kernel's.  Some tokens' rows bit for bit, the last ones among them."""
    P, O = gpu, oracle_mod
    n, d, tokens = 32, 131072, 65600
    rng = np.random.default_rng(33)
    rows = S.random_weights(rng, Q8, n, d, S.unit_scale_exp(Q8, n))
    W = G.QMatrix(Q8, n, d, rows)
    X = rng.standard_normal((tokens, n)).astype(np.float32)
    dx, out = P.DeviceBuffer.from_numpy(X), P.DeviceBuffer(4 * tokens * d)
    P.check(P.lib.plh_matmul_batch(Q8, n, d, C.c_void_p(W.ptr), C.c_void_p(dx.ptr), tokens,
                                   C.c_void_p(out.ptr)), "plh_matmul_batch")
    got = np.empty(d, np.float32)
    for t in (0, 40000, 65535, 65536, tokens - 1):
        P.check(P.lib.plh_memcpy_dtoh(got.ctypes.data, out.ptr + 4 * t * d, 4 * d), "dtoh")
        assert_bits(got, O.matmul(rows, X[t], n, d, Q8), t)
    for b in (dx, out):
        b.free()
    W.free()


def layer0_rows_exact(P, O, n_tok, **kw):
    """A prompt's layer-0 cached rows (exact order, nothing transcendental)
    against the oracle's, bit for bit."""
    cfg = dict(n_layers=1, n_ffn=256, n_heads=4, n_kv_heads=2, head_dim=64, vocab_size=64,
               max_seq_len=n_tok + 3, rope_type=0, rope_base=1e4, eps=1e-5, **kw)
    h = S.SynthModel(**cfg, seed=cfg["n_embd"])
    dm, orc = P.DeviceModel(h), O.OracleForward(h)
    toks = np.arange(n_tok, dtype=np.int32) % 64
    try:
        dm.prefill(toks, 1)
        P.synchronize()
        orc.prefill(toks, 1, n_threads=8)
        for a, b in zip(dm.fetch_cache(), (orc.kc, orc.vc)):
            assert np.array_equal(a, b)
    finally:
        dm.free()


@pytest.mark.parametrize("n_embd", [96, 544, 4096, 4128, 8448, 12288])
def test_prompt_norm_rows(gpu, oracle_mod, n_embd):
    """rmsnorm rows from short of one piece a thread to several batches of
    registers."""
    kinds = ("embd", "output", "q", "k", "v", "o", "gate", "up", "down")
    layer0_rows_exact(gpu, oracle_mod, 5, n_embd=n_embd, types={k: Q8 for k in kinds})


@pytest.mark.parametrize("q,k,v", [(Q4, Q4, Q6), (Q6, Q6, Q4), (Q8, Q8, Q8), (Q4, Q8, Q6),
                                   (Q8, Q4, Q4)])
@pytest.mark.parametrize("n_tok", [17, 120])
def test_prompt_qkv_launches(gpu, oracle_mod, q, k, v, n_tok):
    """q, k and v of a prompt: K quants or Q8_0 in one launch, mixed in three."""
    types = dict(embd=Q8, output=Q8, q=q, k=k, v=v, o=Q4, gate=Q4, up=Q4, down=Q4)
    layer0_rows_exact(gpu, oracle_mod, n_tok, n_embd=768, types=types)


@pytest.mark.parametrize("n_embd,gate", [(1280, Q4), (1536, Q6), (1312, Q8)])
@pytest.mark.parametrize("n_tok", [17, 60])
def test_prompt_long_rows_few_tiles(gpu, oracle_mod, n_embd, gate, n_tok):
    """A layer's q/k/v launch and gate/up pair of few tiles and long rows: the
    residual and the logits (the fast order) against the oracle."""
    types = dict(embd=Q8, output=Q8, q=Q8, k=Q8, v=Q8, o=Q8, gate=gate, up=gate, down=Q8)
    cfg = dict(n_layers=1, n_embd=n_embd, n_ffn=512, n_heads=4, n_kv_heads=2, head_dim=64,
               vocab_size=64, max_seq_len=80, rope_type=0, rope_base=1e4, eps=1e-5, types=types)
    h = S.SynthModel(**cfg, seed=n_tok)
    dm, orc = gpu.DeviceModel(h), oracle_mod.OracleForward(h)
    toks = np.arange(n_tok, dtype=np.int32)
    try:
        dm.prefill(toks, 0)
        gpu.synchronize()
        for got, want in zip((dm.fetch_logits(), dm.fetch_x()), orc.prefill(toks, 0, n_threads=8)):
            assert np.max(np.abs(got - want)) <= FWD_TOL_FAST * np.max(np.abs(want))
        for a, b in zip(dm.fetch_cache(), (orc.kc, orc.vc)):
            assert np.array_equal(a, b)
    finally:
        dm.free()


def prompt_rows_two_layers(P, O, n_tok, **kw):
    """A prompt's cached rows against the oracle's: layer 0's bit for bit (exact
    order), layer 1's, which every token's q, attention, o, gate/up pair and
    down products of layer 0 reach, within one fp16 step and KV_TOL (silu's
    expf and the softmax round apart)."""
    cfg = dict(n_layers=2, vocab_size=64, max_seq_len=n_tok + 1, rope_type=0, rope_base=1e4,
               eps=1e-5, **kw)
    h = S.SynthModel(**cfg, seed=cfg["n_ffn"] + n_tok)
    dm, orc = P.DeviceModel(h), O.OracleForward(h)
    toks = np.arange(n_tok, dtype=np.int32) * 7 % 64
    try:
        dm.prefill(toks, 0)
        P.synchronize()
        orc.prefill(toks, 0, n_threads=8)
        for a, b in zip(dm.fetch_cache(), (orc.kc, orc.vc)):
            half = a.size // 2
            assert np.array_equal(a[:half], b[:half])
            x, y = O.f16_to_f32(a[half:]), O.f16_to_f32(b[half:])
            step = np.spacing(np.maximum(np.abs(x), np.abs(y)).astype(np.float16))
            bad = np.abs(x - y) > step.astype(np.float32) + KV_TOL * np.max(np.abs(y))
            assert not bad.any(), np.flatnonzero(bad)[:8]
    finally:
        dm.free()


@pytest.mark.parametrize("gate", [Q4, Q6, Q8])
@pytest.mark.parametrize("n_ffn", [2080, 4128])
def test_prompt_pair_many_tiles(gpu, oracle_mod, gate, n_ffn):
    """The gate/up pair from 4 x 256 tiles (two waves a row tile) and, K quants,
    from 8 x 256 (one wave, the last workgroup's rows half there)."""
    types = dict(embd=Q8, output=Q8, q=Q8, k=Q8, v=Q8, o=Q8, gate=gate, up=gate, down=Q8)
    prompt_rows_two_layers(gpu, oracle_mod, 120, n_embd=256, n_ffn=n_ffn, n_heads=4,
                           n_kv_heads=2, head_dim=64, types=types)


@pytest.mark.parametrize("q,k,v", [(Q4, Q4, Q6), (Q6, Q4, Q4), (Q8, Q8, Q8)])
@pytest.mark.parametrize("n_embd,heads,n_tok", [(256, 42, 120), (256, 84, 119), (1024, 6, 17)])
def test_prompt_qkv_waves(gpu, oracle_mod, q, k, v, n_embd, heads, n_tok):
    """The joint q/k/v launch with two, one (Q8_0 two) and eight waves a row
    tile; k's and v's rows end inside a workgroup's."""
    types = dict(embd=Q8, output=Q8, q=q, k=k, v=v, o=Q8, gate=Q8, up=Q8, down=Q8)
    prompt_rows_two_layers(gpu, oracle_mod, n_tok, n_embd=n_embd, n_ffn=128, n_heads=heads,
                           n_kv_heads=3, head_dim=48, types=types)
