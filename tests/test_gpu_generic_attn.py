"""The generic attention kernels (attn_generic.hip) where their tiles can go
wrong, against the oracle: every built number of 16-wide d tiles and head dims
between them (also ones that are not multiples of 4, whose rows are not 8-byte
aligned), one key to several tiles per wave, key ranges split over workgroups,
GQA groups that leave partial column tiles or fill several.  Rows after a
token's own must not reach it whatever they hold; the allocation-free entry
point and a first call under graph capture work as with the tuned kernels."""
import numpy as np
import pytest

import test_gpu_decode as TD
import test_gpu_decode_rows as TR
import test_gpu_prefill as TP
import test_gpu_qknorm as TQ
from attn_check import assert_attn_close, filled_cache, normal_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [4, 16, 34, 48, 50, 72, 80, 100, 112, 130, 160, 176, 192, 208, 256])
@pytest.mark.parametrize("pos", [15, 64, 777])
def test_decode_head_dims(gpu, oracle_mod, D, pos):
    cfg = gpu.AttnConfig(2, 6, 2, D, 800, 1e4, D // 2 % 2)
    TD.run_decode(gpu, oracle_mod, cfg, pos, seed=D + pos, poison=True)


@pytest.mark.parametrize("heads", [(7, 1), (40, 2), (32, 32), (20, 20)])
@pytest.mark.parametrize("pos", [16, 63, 1023, 2500])
def test_decode_groups_and_splits(gpu, oracle_mod, heads, pos):
    cfg = gpu.AttnConfig(3, heads[0], heads[1], 80, 2600, 1e4, 0)
    TD.run_decode(gpu, oracle_mod, cfg, pos, seed=pos, check_layers=[1], per_layer=pos == 1023)


@pytest.mark.parametrize("case", [  # n_heads, n_kv_heads, head_dim, start, n
    (4, 4, 20, 0, 16), (4, 4, 48, 0, 17), (14, 2, 80, 5, 33), (8, 2, 96, 700, 3),
    (6, 6, 112, 64, 65), (8, 8, 144, 0, 40), (2, 1, 176, 31, 50), (2, 2, 250, 0, 70),
    (2, 2, 250, 60, 70), (2, 1, 256, 0, 150),
    (8, 8, 80, 1200, 20)])
def test_prefill_tiles(gpu, oracle_mod, case):
    Hq, Hkv, D, start, n = case
    cfg = gpu.AttnConfig(2, Hq, Hkv, D, start + n + 3, 1e4, 1)
    TP.run_prefill(gpu, oracle_mod, cfg, start, n, seed=D + n)


@pytest.mark.parametrize("keys", [128, 129, 256, 257, 385])
@pytest.mark.parametrize("D", [80, 96])
def test_key_splits(gpu, oracle_mod, D, keys):
    """Launches of few workgroups split their keys from 257 on: one token and a
    prompt that end at each edge."""
    cfg = gpu.AttnConfig(2, 6, 2, D, keys, 1e4, 0)
    TD.run_decode(gpu, oracle_mod, cfg, keys - 1, seed=keys)
    TP.run_prefill(gpu, oracle_mod, cfg, keys - 20, 20, seed=keys)


@pytest.mark.parametrize("case", [  # layers, n_heads, n_kv_heads, head_dim, start, n: keys
    (1, 4, 4, 256, 63, 1), (1, 4, 4, 256, 64, 1),          # 64 of one token, 65 tiles
    (12, 32, 32, 160, 84, 1), (12, 32, 32, 160, 85, 1),    # 32768 with 384 rows, more
    (6, 48, 48, 208, 226, 1), (6, 48, 48, 208, 227, 1),    # 65536 with 288, more
    (1, 6, 2, 224, 172, 20), (1, 6, 2, 224, 173, 20),      # 192 of a prompt, 193
    (3, 6, 2, 224, 108, 20), (3, 6, 2, 224, 109, 20),      # 128 with 360 rows, 129
    (1, 8, 2, 192, 0, 32), (1, 8, 2, 192, 0, 33),          # 32, 33
    (1, 8, 8, 100, 172, 20), (1, 8, 8, 100, 173, 20),      # 192 with 160 rows, 193
    (1, 16, 2, 66, 0, 16), (1, 17, 1, 66, 0, 16),          # 256 rows, 272
    (1, 8, 8, 160, 0, 16), (1, 8, 4, 160, 0, 17)])         # 16, 17
def test_few_keys_of_wide_heads(gpu, oracle_mod, case):
    """Either side of the rule that runs one workgroup per token and q head."""
    L, Hq, Hkv, D, start, n = case
    cfg = gpu.AttnConfig(L, Hq, Hkv, D, start + n + 1, 1e4, D // 4 % 2)
    TP.run_prefill(gpu, oracle_mod, cfg, start, n, seed=start + n, check_layers=[0, L - 1])
    if n == 1:
        TD.run_decode(gpu, oracle_mod, cfg, start, seed=start, check_layers=[0, L - 1], poison=True)


def test_few_keys_qknorm_and_rows(gpu, oracle_mod):
    """The same with QK-norm, two prompt chunks and a token after them, and with
    the appended rows mirrored."""
    TQ.test_prefill_qknorm_chunks_then_decode(gpu, oracle_mod, (1, 6, 2, 256, 512, 1e4, 1))
    TQ.test_decode_qknorm(gpu, oracle_mod, (2, 8, 4, 248, 64, 1e4, 0), 20)
    TR.test_decode_rows_match_plain_decode(gpu, (2, 8, 2, 256, 300, 1, 0, 2, 20, True), False)


@pytest.mark.parametrize("D,n", [(66, 20), (72, 33), (80, 48), (96, 63), (112, 17), (120, 65)])
def test_prefill_two_tiles_a_workgroup(gpu, oracle_mod, D, n):
    """From 4 x 256 column tiles in a launch a workgroup takes two of them:
    the last one's second tile full, partial or missing."""
    cfg = gpu.AttnConfig(11, 48, 48, D, n + 2, 1e4, D // 8 % 2)
    TP.run_prefill(gpu, oracle_mod, cfg, 0, n, seed=D + n, check_layers=[0, 10])


@pytest.mark.parametrize("D,n,rope", [(80, 33, 0), (112, 49, 1)])
def test_two_tiles_a_workgroup_qknorm(gpu, oracle_mod, D, n, rope):
    """The same with QK-norm: the first and the last layer's outputs and rows."""
    P, O = gpu, oracle_mod
    L, H, S = 11, 48, n + 4
    cfg = P.AttnConfig(L, H, H, D, S, 1e4, rope)
    rng = np.random.default_rng(D + n)
    q, k, v = (normal_f32(rng, (L, n, H * D), 3.0) for _ in "qkv")
    qw, kw = (rng.uniform(0.5, 1.5, (L, D)).astype(np.float32) for _ in "qk")
    d = [P.DeviceBuffer.from_numpy(x) for x in (q, k, v, qw, kw)]
    cache, out = P.KVCache(cfg), P.DeviceBuffer(4 * L * n * H * D)
    P.prefill(cache, 0, 0, n, d[0].ptr, d[1].ptr, d[2].ptr, out.ptr, None, L, q_norm=d[3].ptr,
              k_norm=d[4].ptr, norm_eps=1e-5)
    P.synchronize()
    got = out.download(np.float32, (L, n, H * D))
    rows = [c.reshape(L, S, H * D) for c in cache.fetch()]
    cache.free()
    shp = O.Shape(L, H, H, D, S, 1e4, rope)
    cos_t, sin_t = O.rope_tables(S, D, 1e4)
    want = [np.zeros(cfg.cache_elems, np.uint16) for _ in "kv"]
    for l in (0, L - 1):
        ref = O.attn_prefill(shp, l, 0, n, q[l].copy(), k[l].copy(), v[l], *want, cos_t, sin_t,
                             q_norm=qw[l], k_norm=kw[l], eps=1e-5)
        assert_attn_close(got[l], ref, D, what=f"two tiles, QK-norm, layer {l}")
        for a, b in zip(rows, want):
            assert np.array_equal(a[l], b.reshape(L, S, H * D)[l])


def test_decode_unaligned_caches(gpu):
    """Caches that start 2 elements past a 16-byte boundary (4-byte loads): the
    same bits as aligned ones."""
    P = gpu
    S, D, Hkv, pos = 300, 80, 2, 250
    rng = np.random.default_rng(5)
    kc, vc = (normal_f32(rng, (S * Hkv * D,)).astype(np.float16) for _ in "kv")
    q, k, v = (normal_f32(rng, (h * D,)) for h in (6, Hkv, Hkv))
    ang = rng.uniform(0, 6, (S, D // 2)).astype(np.float32)
    d = [P.DeviceBuffer.from_numpy(x) for x in (q, k, v, np.cos(ang), np.sin(ang))]
    outs = []
    for off in (0, 2):
        pad = [np.concatenate([np.zeros(off, np.float16), x]) for x in (kc, vc)]
        c = [P.DeviceBuffer.from_numpy(x) for x in pad]
        out = P.DeviceBuffer(4 * 6 * D)
        P.check(P.lib.plh_attn_decode(1, 6, Hkv, D, S, 0, 0, 1, pos, d[0].ptr, d[1].ptr, d[2].ptr,
                                      c[0].ptr + 2 * off, c[1].ptr + 2 * off, d[3].ptr, d[4].ptr,
                                      out.ptr), "plh_attn_decode")
        P.synchronize()
        outs.append(out.download(np.uint32, (6 * D,)))
        row = slice(off + pos * Hkv * D, off + (pos + 1) * Hkv * D)
        assert np.array_equal(c[1].download(np.float16, pad[1].shape)[row], v.astype(np.float16))
    assert np.array_equal(outs[0], outs[1])


FEW = [  # n_layers, n_heads, n_kv_heads, head_dim, rope_type, qk_norm, start, n, stride pad
    (3, 32, 4, 64, 0, False, 0, 1, 0), (2, 8, 4, 128, 1, True, 900, 1, 4),
    (1, 14, 2, 64, 0, True, 300, 1, 0), (1, 32, 4, 64, 1, False, 0, 65, 4),
    (1, 14, 2, 64, 1, True, 200, 100, 0), (1, 16, 8, 128, 1, True, 0, 509, 0),
    (1, 28, 4, 128, 0, False, 17, 80, 8), (22, 12, 4, 64, 0, False, 260, 10, 0),
    (9, 16, 8, 128, 1, True, 400, 16, 0),
    (16, 8, 8, 128, 0, False, 300, 16, 0), (3, 16, 8, 128, 1, True, 300, 10, 4),
    (1, 128, 1, 64, 0, False, 90, 6, 0)]


@pytest.mark.parametrize("case", FEW)
def test_small_prefill_launches_match_units(gpu, case):
    """Head dims 64 and 128: the 16-column tiles of small launches against the
    32-column units (plh_set_tuning key 5 at -1) on the same inputs.  The same
    appended rows bit for bit, outputs within the units' hi/lo precision."""
    L, Hq, Hkv, D, rope, norm, start, n, pad = case
    P = gpu
    cfg = P.AttnConfig(L, Hq, Hkv, D, start + n + 1, 1e4, rope)
    rng = np.random.default_rng(start + n)
    rows = cfg.max_seq_len * L * cfg.kv_dim
    kc, vc = (normal_f32(rng, (rows,)).astype(np.float16).view(np.uint16) for _ in "kv")
    ins = [normal_f32(rng, (L, n, w)) for w in (cfg.q_dim, cfg.kv_dim, cfg.kv_dim)]
    ins += [rng.uniform(0.5, 1.5, (L, D)).astype(np.float32) for _ in "qk"]
    d = [P.DeviceBuffer.from_numpy(x) for x in ins]
    kw = dict(q_norm=d[3].ptr, k_norm=d[4].ptr, norm_eps=1e-5) if norm else {}
    got = []
    for key5 in (0, -1):
        cache = P.KVCache(cfg)
        cache.load(kc, vc)
        out = P.DeviceBuffer(4 * L * n * (cfg.q_dim + pad))
        out.zero()
        P.check(P.lib.plh_set_tuning(5, key5), "plh_set_tuning")
        try:
            P.prefill(cache, 0, start, n, d[0].ptr, d[1].ptr, d[2].ptr, out.ptr,
                      cfg.q_dim + pad, L, **kw)
            P.synchronize()
        finally:
            P.lib.plh_set_tuning(5, 0)
        got.append((out.download(np.float32, (L * n, cfg.q_dim + pad)), *cache.fetch()))
        cache.free()
    for a, b in zip(got[0][1:], got[1][1:]):
        assert np.array_equal(a, b)
    assert not got[0][0][:, cfg.q_dim:].any()
    assert_attn_close(got[0][0][:, :cfg.q_dim], got[1][0][:, :cfg.q_dim], D, what="few")


@pytest.mark.parametrize("case", [  # layers, n_heads, n_kv_heads, head_dim, start
    (1, 48, 1, 64, 300), (2, 71, 1, 128, 900), (3, 40, 2, 128, 70),  # 16-column tiles
    (16, 96, 2, 128, 2100), (20, 71, 1, 64, 6000)])                   # units
def test_one_token_wide_groups(gpu, oracle_mod, case):
    """plh_attn_prefill of a single token with more than 16 q heads per kv head,
    on either side of the rule for many tiles over long contexts."""
    L, Hq, Hkv, D, start = case
    cfg = gpu.AttnConfig(L, Hq, Hkv, D, start + 2, 1e4, 0)
    TP.run_prefill(gpu, oracle_mod, cfg, start, 1, seed=start, check_layers=[0, L - 1])


def test_prefill_later_rows_do_not_matter(gpu):
    """Tokens 0..19 give the same bits whatever finite rows tokens 20..39 hold;
    with infinities and NaNs among them (whose tiles are taken again in fp32)
    the same to fp32 rounding: 40 terms of 2^-24 of the largest."""
    P = gpu
    cfg = P.AttnConfig(1, 6, 2, 80, 64, 1e4, 0)
    rng = np.random.default_rng(3)
    n, outs = 40, []
    q, k, v = (normal_f32(rng, (n, d)) for d in (cfg.q_dim, cfg.kv_dim, cfg.kv_dim))
    for bad in (None, 1.0, np.inf, np.nan):
        if bad is not None:
            k[20:], v[20:] = normal_f32(rng, k[20:].shape), normal_f32(rng, v[20:].shape)
            k[21, ::7], v[20:30, ::5] = bad, bad
        cache = P.KVCache(cfg)
        d = [P.DeviceBuffer.from_numpy(x) for x in (q, k, v)]
        out = P.DeviceBuffer(4 * n * cfg.q_dim)
        P.prefill(cache, 0, 0, n, d[0].ptr, d[1].ptr, d[2].ptr, out.ptr)
        P.synchronize()
        outs.append(out.download(np.float32, (n, cfg.q_dim)))
        cache.free()
    assert np.isfinite(outs[0]).all()
    assert np.array_equal(outs[1][:20].view(np.uint32), outs[0][:20].view(np.uint32))
    for o in outs[2:]:
        assert np.max(np.abs(o[:20] - outs[0][:20])) <= 40 * 2.0 ** -24 * np.abs(outs[0]).max()
    assert np.isnan(outs[3][21:]).any()


@pytest.mark.parametrize("kind", ["k_inf", "v_inf"])
def test_decode_infinite_cached_rows(gpu, oracle_mod, kind):
    """fp16 infinities in the cache (a k or v beyond 65504 rounds to one): a key
    whose score is minus infinity has no weight, an infinite v reaches its own
    d alone, as in the reference's fp32 arithmetic."""
    P, O = gpu, oracle_mod
    cfg = P.AttnConfig(1, 4, 2, 48, 256, 1e4, 0)
    pos, rng = 200, np.random.default_rng(11)
    kc, vc = filled_cache(O, cfg, pos, rng)
    k3, v3 = kc.reshape(256, 2, 48), vc.reshape(256, 2, 48)
    q = np.abs(normal_f32(rng, (cfg.q_dim,))) + np.float32(0.1)
    k, v = normal_f32(rng, (cfg.kv_dim,)), normal_f32(rng, (cfg.kv_dim,))
    cos_t, sin_t = O.rope_tables(256, 48, 1e4)
    cos_t[pos], sin_t[pos] = 1.0, 0.0      # no rotation: q stays positive
    if kind == "k_inf":
        k3[40, :, 7] = 0xFC00
    else:
        v3[40, :, 7] = 0x7C00
    cache = P.KVCache(cfg)
    cache.load(kc, vc)
    cache.cos.upload(cos_t)
    cache.sin.upload(sin_t)
    d = [P.DeviceBuffer.from_numpy(x) for x in (q, k, v)]
    out = P.DeviceBuffer(4 * cfg.q_dim)
    P.decode(cache, 0, pos, d[0].ptr, d[1].ptr, d[2].ptr, out.ptr)
    P.synchronize()
    got = out.download(np.float32, (4, 48))
    shp = O.Shape(1, 4, 2, 48, 256, 1e4, 0)
    ref = O.attn_decode(shp, 0, pos, q.copy(), k.copy(), v, kc, vc, cos_t, sin_t).reshape(4, 48)
    inf = np.zeros(48, bool)
    inf[7] = kind == "v_inf"
    assert np.isinf(ref[:, inf]).all() and np.array_equal(got[:, inf], ref[:, inf])
    assert_attn_close(got[:, ~inf].copy(), ref[:, ~inf].copy(), 48 - inf.sum(), what=kind)
    cache.free()


def attend64(q, k, v, group):
    """Causal attention of the last len(q) rows in 64 bits: q [n, Hq, D], k and
    v [rows, Hkv, D] (no rotation)."""
    n, hq, d = q.shape
    out = np.zeros((n, hq, d))
    for t in range(n):
        rows = len(k) - n + t + 1
        for h in range(hq):
            s = k[:rows, h // group].astype(np.float64) @ q[t, h].astype(np.float64) / np.sqrt(d)
            w = np.exp(s - s.max())
            out[t, h] = (w / w.sum()) @ v[:rows, h // group].astype(np.float64)
    return out


@pytest.mark.parametrize("D,n", [(80, 1), (48, 1), (50, 1), (96, 5), (34, 17), (64, 1), (128, 40)])
@pytest.mark.parametrize("kind", ["w30", "w45", "w30_alone", "w80_alone", "v_zero", "q_wide"])
def test_wide_ranges(gpu, D, n, kind):
    """q and the softmax weights count at fp32's precision over fp32's range.
    wB: one key's weight is 2^-B of the others' and its v 6e4 among values of
    1e-4 (w30), the smallest fp16 (w45) or zero (alone: it is the whole
    output); q_wide: a q element 2^30 times the others meets a channel of K
    that is zero.  Against 64 bits, each head's 2-norm: a score of B ln 2 goes
    through three roundings (its sum, its scale, the maximum's subtraction),
    and a result through one per row."""
    P = gpu
    Hq, Hkv, start, at = 4, 2, 200, 57
    cfg = P.AttnConfig(1, Hq, Hkv, D, start + n, 1e4, 0)
    rng = np.random.default_rng(D + n)
    rows = start + n
    q = np.zeros((n, Hq, D), np.float32)
    k, v = (np.zeros((rows, Hkv, D), np.float32) for _ in "kv")
    bits = 4
    if kind == "q_wide":
        q, k, v = (normal_f32(rng, x.shape).astype(np.float16).astype(np.float32)
                   for x in (q, k, v))
        q[..., 3], k[..., 3] = 2.0 ** 30, 0.0
    elif kind != "v_zero":
        bits = int(kind[1:3])
        q[..., 0] = np.sqrt(np.float32(D))
        k[at, :, 0] = -bits * np.log(2.0)
        k = k.astype(np.float16).astype(np.float32)
        v[:] = {"w30": 1e-4, "w45": 2.0 ** -24}.get(kind, 0.0)
        v[at] = 6e4 * rng.choice([-1.0, 1.0], (Hkv, D))
        v = v.astype(np.float16).astype(np.float32)
    cos, sin = (np.full((rows, D // 2), x, np.float32) for x in (1.0, 0.0))
    cache = P.KVCache(cfg)
    full = [np.zeros((rows, Hkv, D), np.uint16) for _ in "kv"]
    for f, x in zip(full, (k, v)):
        f[:start] = x[:start].astype(np.float16).view(np.uint16)
    cache.load(*(f.reshape(-1) for f in full))
    cache.cos.upload(cos)
    cache.sin.upload(sin)
    d = [P.DeviceBuffer.from_numpy(np.ascontiguousarray(x)) for x in (q, k[start:], v[start:])]
    out = P.DeviceBuffer(4 * n * Hq * D)
    P.prefill(cache, 0, start, n, d[0].ptr, d[1].ptr, d[2].ptr, out.ptr)
    P.synchronize()
    got = out.download(np.float32, (n, Hq, D)).astype(np.float64)
    want = attend64(q, k, v, Hq // Hkv)
    cache.free()
    if kind == "v_zero":
        assert not got.any()
        return
    err = np.linalg.norm(got - want, axis=-1) / np.linalg.norm(want, axis=-1)
    tol = (3 * bits * np.log(2.0) + rows) * 2.0 ** -24
    print(f"[wide] {kind} D {D} n {n}: {err.max():.2e} of {tol:.2e}", flush=True)
    assert err.max() <= tol, (kind, err.max(), tol)


@pytest.mark.parametrize("heads,n", [(256, 1 << 24), (512, 1 << 23), (300, 1 << 23)])
def test_sizes_past_one_launch_are_refused(gpu, heads, n):
    """More (token, q head) pairs than a launch has workgroups, their product 0
    modulo 2^32 or past 2^31: -1 with a message, nothing read."""
    P = gpu
    p = P.DeviceBuffer(256).ptr
    rc = P.lib.plh_attn_prefill(1, heads, 1, 80, n, 0, 0, 1, 0, n, p, p, p, p, p, p, p, p,
                                heads * 80)
    assert rc == -1 and b"exceed one launch" in P.lib.plh_last_error()
    P.synchronize()


def test_decode_capture_and_noalloc(gpu, oracle_mod):
    """A split launch captured at its first call and replayed, and the
    allocation-free entry point: the eager call's bits each time."""
    P, O = gpu, oracle_mod
    cfg = P.AttnConfig(2, 8, 4, 96, 1100, 1e4, 0)
    pos, rng = 1000, np.random.default_rng(9)
    kc, vc = filled_cache(O, cfg, pos, rng)
    q, k, v = (normal_f32(rng, (2, d)) for d in (cfg.q_dim, cfg.kv_dim, cfg.kv_dim))
    d = [P.DeviceBuffer.from_numpy(x) for x in (q, k, v)]
    outs = [P.DeviceBuffer(4 * 2 * cfg.q_dim) for _ in range(3)]
    caches = [P.KVCache(cfg) for _ in range(3)]
    for c in caches:
        c.load(kc, vc)
    with P.Graph() as gr:
        P.decode(caches[0], 0, pos, d[0].ptr, d[1].ptr, d[2].ptr, outs[0].ptr, 2)
    P.decode(caches[1], 0, pos, d[0].ptr, d[1].ptr, d[2].ptr, outs[1].ptr, 2)
    P.synchronize()
    eager = outs[1].download(np.float32, (2, cfg.q_dim))
    c = caches[2]
    P.check(P.lib.plh_attn_decode_noalloc(2, 8, 4, 96, 1100, 0, 0, 2, pos, d[0].ptr, d[1].ptr,
                                          d[2].ptr, c.key.ptr, c.val.ptr, c.cos.ptr, c.sin.ptr,
                                          outs[2].ptr), "plh_attn_decode_noalloc")
    P.synchronize()
    assert np.array_equal(outs[2].download(np.float32, eager.shape), eager)
    for _ in range(3):
        outs[0].zero()
        gr.launch()
        P.synchronize()
        assert np.array_equal(outs[0].download(np.float32, eager.shape), eager)
        P.decode(caches[1], 0, pos, d[0].ptr, d[1].ptr, d[2].ptr, outs[1].ptr, 2)
        P.synchronize()
    shp = O.Shape(2, 8, 4, 96, 1100, 1e4, 0)
    cos_t, sin_t = O.rope_tables(1100, 96, 1e4)
    ref = O.attn_decode(shp, 1, pos, q[1].copy(), k[1].copy(), v[1], kc, vc, cos_t, sin_t)
    assert_attn_close(eager[1], ref, 96, what="layer 1")
