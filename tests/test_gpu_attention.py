"""GPU parity of the attention around the Q4 linears (ForwardPass::attention,
forward.cc:376-508) and the KV cache writes (LocalKvCache / GlobalKvCache append,
kv_cache.h:33,143): hyp_attention against the oracle's fp64 restatement
(oracle/q4_oracle.c orc_attention_f64, pinned on the CPU against dense numpy attention and
closed forms), hyp_kv_cache_write against the slot rule p % capacity.

Bar (written per test): every output within 2^-8 |ref| + 2^-9 max|v| of the fp64 truth
(the output's bf16 rounding, plus the P.V products' bf16 P), and sig_rel <= 1e-2. MLX's
own SDPA bits are parity unpinned (no reference vectors).
"""
import ctypes
import sys

import numpy as np
import pytest

import hyperion_amd as hy
import oracle as O
from hyperion_amd import synthetic as syn

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def dev(a, stream):
    return hy.DeviceArray.from_host(a, stream)


def _fill_cache(cache, ck, cv, stream):
    kp, vp = cache.buffers()
    for ptr, host in ((kp, ck), (vp, cv)):
        hy.call("hyp_memcpy_htod", ptr, host.ctypes.data_as(ctypes.c_void_p), host.nbytes, stream.handle)
    stream.synchronize()


def _check(got_bits, ref, v_all, what):
    got = syn.bf16_to_f32(got_bits).astype(np.float64)
    vmax = float(np.max(np.abs(syn.bf16_to_f32(v_all)))) if v_all.size else 0.0
    bound = 2.0**-8 * np.abs(ref) + 2.0**-9 * vmax
    err = np.abs(got - ref)
    worst = float(np.max(err / bound))
    rel = syn.sig_rel(got, ref)
    say(f"  {what}: worst {worst:.3f} of the bound, sig_rel {rel:.2e}")
    assert np.all(err <= bound), what
    assert rel <= 1e-2, what


CASES = [
    # L, H, KVH, D, cap, offset, prefix, window, q scale
    (1, 16, 8, 256, 1032, 0, 0, 1024, 0.25),        # sliding decode, first token
    (1, 16, 8, 256, 1032, 700, 700, 1024, 0.25),    # sliding decode inside the window
    (1, 16, 8, 256, 1032, 5000, 1024, 1024, 0.25),  # sliding decode, ring wrapped
    (4, 16, 8, 256, 1032, 3000, 1024, 1024, 0.25),  # batch-4-token decode
    (1, 16, 1, 512, 8192, 4000, 4000, 0, 0.18),     # global decode (K = V layers)
    (4, 16, 1, 512, 8192, 100, 100, 0, 0.18),
    (300, 16, 8, 256, 1032, 0, 0, 1024, 0.25),      # prefill chunk
    (300, 16, 8, 256, 1032, 2000, 1024, 1024, 0.25),   # continuation prefill over the ring
    (2048, 16, 8, 256, 2048, 0, 0, 1024, 0.25),     # a full prefill chunk, window inside it
    (300, 16, 1, 512, 4096, 0, 0, 0, 0.18),         # global prefill
    (257, 16, 1, 512, 4096, 1000, 1000, 0, 0.18),
    (10, 4, 2, 64, 16, 0, 0, 8, 0.5),               # the tiny fixture's shapes
    (1, 4, 2, 64, 16, 20, 8, 8, 0.5),
    (5, 4, 1, 128, 64, 30, 30, 0, 0.4),
]


@pytest.mark.parametrize("L,H,KVH,D,cap,offset,prefix,window,qs", CASES)
def test_attention_matches_oracle(stream, L, H, KVH, D, cap, offset, prefix, window, qs):
    say(f"attention L={L} H={H} KVH={KVH} D={D} cap={cap} offset={offset} prefix={prefix} window={window}")
    rng = np.random.default_rng(L * 7919 + offset * 13 + D)
    b = lambda scale, *shape: syn.bf16_bits((rng.standard_normal(shape) * scale).astype(np.float32))  # noqa: E731
    q, k, v = b(qs, L, H, D), b(1.0, L, KVH, D), b(1.0, L, KVH, D)
    ck, cv = b(1.0, cap, KVH, D), b(1.0, cap, KVH, D)
    cache = hy.KvCache(cap, KVH, D)
    _fill_cache(cache, ck, cv, stream)
    qd, kd, vd = dev(q, stream), dev(k, stream), dev(v, stream)
    out = hy.DeviceArray((L, H, D), np.uint16)
    hy.attention(qd, kd, vd, L, H, cache, offset, prefix, window, out, stream)
    ref = O.attention_f64(q, k, v, ck, cv, offset, prefix, window)
    _check(out.to_host(stream), ref, np.concatenate([v.reshape(-1), cv.reshape(-1)]), f"L={L} D={D} offset={offset}")
    for a in (qd, kd, vd, out):
        a.close()
    cache.close()


CHUNK_CASES = [
    # L, H, KVH, D, cap, offset, prefix, window, chunk in the cache
    (17, 4, 4, 64, 64, 5, 5, 0, True),            # one row per token, one more than the decode form takes
    (33, 4, 1, 64, 64, 20, 20, 24, True),         # 132 rows: 4 past a row tile; window edges in a block
    (32, 8, 2, 128, 40, 101, 8, 8, True),         # 128 rows exactly; the ring wraps inside a block
    (31, 8, 2, 128, 40, 77, 9, 10, False),        # chunk beside a wrapped prefix
    (129, 2, 2, 256, 300, 1000, 171, 172, True),  # one row past a tile, prefix + chunk fill the ring
    (5, 16, 1, 512, 700, 650, 650, 0, True),      # many key splits of one partial tile
    (70, 16, 1, 512, 2200, 2100, 2100, 0, True),  # splits whose causal end is inside the last block
    (64, 16, 1, 512, 16, 33, 16, 0, False),       # a ring of half a key block
    # the decode form with more than 64 splits: fewer in use than in the grid; the first ones
    # wholly behind the window
    (1, 4, 1, 64, 9000, 8700, 8700, 0, True),
    (2, 16, 2, 128, 9000, 9990, 8500, 300, True),
]


@pytest.mark.parametrize("L,H,KVH,D,cap,offset,prefix,window,cached", CHUNK_CASES)
def test_chunk_kernel_edges(stream, L, H, KVH, D, cap, offset, prefix, window, cached):
    """The chunk kernel at the edges of its row tiles, key blocks, splits and rings. One cached
    K row is NaN: its scores count as masked. Slots no position maps to hold NaN and must not
    reach a result. Bar as above."""
    say(f"chunk attention L={L} KVH={KVH} D={D} cap={cap} offset={offset} prefix={prefix} window={window}")
    rng = np.random.default_rng(L * 31 + D + cap)
    b = lambda scale, *shape: syn.bf16_bits((rng.standard_normal(shape) * scale).astype(np.float32))  # noqa: E731
    nan = np.uint16(0x7FC0)
    q, k, v = b(D ** -0.5 * 2.0, L, H, D), b(1.0, L, KVH, D), b(1.0, L, KVH, D)
    ck, cv = np.full((cap, KVH, D), nan), np.full((cap, KVH, D), nan)
    for p in range(offset - prefix, offset):
        ck[p % cap], cv[p % cap] = b(1.0, KVH, D), b(1.0, KVH, D)
    dead = prefix // 2                      # index of the NaN key, in the oracle a very negative one
    ckr, cvr = ck.copy(), cv.copy()
    ckr[ck == nan], cvr[cv == nan] = 0, 0
    slot = (offset - prefix + dead) % cap
    ck[slot] = nan
    q[:, :, 0] = syn.bf16_bits(-np.maximum(np.abs(syn.bf16_to_f32(q[:, :, 0])), 0.01).astype(np.float32))
    ckr[slot] = 0
    ckr[slot, :, 0] = syn.bf16_bits(np.full((KVH,), 1e6, np.float32))   # score <= -1e4: weight 0
    ref = O.attention_f64(q, k, v, ckr, cvr, offset, prefix, window)
    cache = hy.KvCache(cap, KVH, D)
    if cached:
        for t in range(L):
            ck[(offset + t) % cap], cv[(offset + t) % cap] = k[t], v[t]
    _fill_cache(cache, ck, cv, stream)
    qd, kd, vd = dev(q, stream), dev(k, stream), dev(v, stream)
    out = hy.DeviceArray((L, H, D), np.uint16)
    hy.call("hyp_attention", qd.ptr, None if cached else kd.ptr, None if cached else vd.ptr, L, H, cache.handle, offset,
            prefix, window, out.ptr, stream.handle)
    _check(out.to_host(stream), ref, np.concatenate([v.reshape(-1), cvr.reshape(-1)]), f"L={L} D={D}")
    for a in (qd, kd, vd, out):
        a.close()
    cache.close()


def _running_max_f32(q, k, v, prefix):
    """Attention of one kv head as the online softmax with an exact running maximum gives it:
    probabilities against the row's maximum, rounded to bf16 for P V, their sum unrounded."""
    L, H, D = q.shape
    s = np.einsum("thd,jd->thj", q.astype(np.float64), k.astype(np.float64)) * np.log2(np.e)
    s = np.where(np.arange(k.shape[0]) <= prefix + np.arange(L)[:, None, None], s, -np.inf)
    p = np.exp2(s - s.max(-1, keepdims=True)).astype(np.float32)
    o = syn.bf16_to_f32(syn.bf16_bits(p)).astype(np.float64) @ v.astype(np.float64)
    return syn.bf16_bits((o / p.astype(np.float64).sum(-1, keepdims=True)).astype(np.float32))


@pytest.mark.parametrize("place", [64 + 5, 64 + 21])
def test_chunk_dominant_key_precision(stream, place):
    """A key that outgrows the maximum of the keys before it by 4 to 8 octaves, in either half
    of a key block, at head_dim 512 (where the output is not rescaled for it): the error against
    fp64 stays that of the running-maximum form, whose largest probability is an exact 1. The
    bar is 3% above that form's own error, measured over the 65536 outputs (whose relative
    standard error is 1 / sqrt(2 x 65536) = 0.3%)."""
    L, H, D, prefix = 8, 16, 512, 120
    T = prefix + L
    rng = np.random.default_rng(place)
    f = lambda a: syn.bf16_to_f32(syn.bf16_bits(a.astype(np.float32)))  # noqa: E731
    q, k, v = f(rng.standard_normal((L, H, D)) * 0.02), f(rng.standard_normal((T, D)) * 0.2), f(rng.standard_normal((T, D)))
    k[:, 0] = 0.0
    q[:, :, 0] = f(rng.uniform(4.0, 8.0, (L, H)) / np.log2(np.e))
    k[place] = 0.0
    k[place, 0] = 1.0
    say(f"dominant key at {place}")
    qb, kb, vb = (syn.bf16_bits(a) for a in (q, k, v))
    ref = O.attention_f64(qb, kb[prefix:, None], vb[prefix:, None], kb[:, None], vb[:, None], prefix, prefix, 0)
    cache = hy.KvCache(T, 1, D)
    _fill_cache(cache, kb, vb, stream)
    qd, out = dev(qb, stream), hy.DeviceArray((L, H, D), np.uint16)
    hy.call("hyp_attention", qd.ptr, None, None, L, H, cache.handle, prefix, prefix, 0, out.ptr, stream.handle)
    rel = lambda bits: np.linalg.norm(syn.bf16_to_f32(bits) - ref) / np.linalg.norm(ref)  # noqa: E731
    got, bar = rel(out.to_host(stream)), rel(_running_max_f32(q, k, v, prefix))
    say(f"  error {got:.3e}, running-maximum form {bar:.3e}")
    assert got <= 1.03 * bar
    for a in (qd, out):
        a.close()
    cache.close()


def test_chunks_overlap_on_one_cache(stream):
    """Chunks that split their keys, on two streams over one cache at once (both only read it):
    each gives the bits of the call alone. 4 tokens (64 query rows per kv head), then 150."""
    H, KVH, D, prefix, cap = 16, 1, 512, 3000, 3200
    rng = np.random.default_rng(77)
    b = lambda scale, *shape: syn.bf16_bits((rng.standard_normal(shape) * scale).astype(np.float32))  # noqa: E731
    cache = hy.KvCache(cap, KVH, D)
    _fill_cache(cache, b(1.0, cap, KVH, D), b(1.0, cap, KVH, D), stream)
    streams = [hy.Stream(), hy.Stream()]
    for L in (4, 150):
        say(f"overlapping chunks L={L}")
        qs = [dev(b(0.1, L, H, D), stream) for _ in streams]
        outs = [[hy.DeviceArray((L, H, D), np.uint16) for _ in range(6)] for _ in streams]
        stream.synchronize()
        call = lambda i, out: hy.call("hyp_attention", qs[i].ptr, None, None, L, H, cache.handle, prefix, prefix,  # noqa: E731
                                      0, out.ptr, streams[i].handle)
        alone = []
        for i, s in enumerate(streams):
            call(i, outs[i][0])
            s.synchronize()
            alone.append(outs[i][0].to_host(s))
        for n in range(6):
            for i in range(2):
                call(i, outs[i][n])
        for i, s in enumerate(streams):
            for n in range(6):
                np.testing.assert_array_equal(outs[i][n].to_host(s), alone[i], err_msg=f"L={L} stream {i} call {n}")
        for a in (*qs, *outs[0], *outs[1]):
            a.close()
    for s in streams:
        s.synchronize()
        s.close()
    cache.close()


@pytest.mark.parametrize("L", [4, 150])
def test_chunk_recorded_into_a_graph(stream, L):
    """A chunk that splits its keys outside a capture, recorded: in the handle's workspace (64
    query rows per kv head) or unsplit. Every replay, with eager work between, meets the bar."""
    H, KVH, D, prefix, cap = 16, 1, 512, 1200, 1400
    rng = np.random.default_rng(L)
    b = lambda scale, *shape: syn.bf16_bits((rng.standard_normal(shape) * scale).astype(np.float32))  # noqa: E731
    q, k, v = b(0.1, L, H, D), b(1.0, L, KVH, D), b(1.0, L, KVH, D)
    ck, cv = b(1.0, cap, KVH, D), b(1.0, cap, KVH, D)
    ref = O.attention_f64(q, k, v, ck, cv, prefix, prefix, 0)
    ck[prefix:prefix + L], cv[prefix:prefix + L] = k, v
    cache = hy.KvCache(cap, KVH, D)
    _fill_cache(cache, ck, cv, stream)
    qd, out, other = dev(q, stream), hy.DeviceArray((L, H, D), np.uint16), hy.DeviceArray((L, H, D), np.uint16)
    call = lambda o: hy.call("hyp_attention", qd.ptr, None, None, L, H, cache.handle, prefix, prefix, 0, o.ptr,  # noqa: E731
                             stream.handle)
    call(other)
    stream.synchronize()
    with hy.Graph.capture(stream) as graph:
        call(out)
    for rep in range(3):
        call(other)
        stream.synchronize()
        out.upload(np.zeros((L, H, D), np.uint16), stream)
        graph.launch(stream)
        _check(out.to_host(stream), ref, np.concatenate([v.reshape(-1), cv.reshape(-1)]), f"L={L} replay {rep}")
    graph.close()
    for a in (qd, out, other):
        a.close()
    cache.close()


def _free_bytes():
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_cache_handle_memory_follows_its_capacity(stream):
    """A cache handle holds its K and V and a split workspace for its capacity: 64 caches of 256
    tokens (0.5 MiB of K and V and 0.3 MiB of workspace each) in 192 MiB, allocation granules
    included; one of 20000 tokens in its K and V and at most 4096 rows."""
    stream.synchronize()
    for cap, count, bound in ((256, 64, 192 << 20), (20000, 4, 4 * (2 * 20000 * 1024 + 4096 * 2056 + (8 << 20)))):
        before = _free_bytes()
        caches = [hy.KvCache(cap, 1, 512) for _ in range(count)]
        used = before - _free_bytes()
        say(f"{count} caches of {cap} tokens: {used / 2**20:.1f} MiB")
        assert used <= bound
        for c in caches:
            c.close()


def test_decode_form_fills_its_workspace(stream):
    """The most rows and splits that a small cache's workspace has to hold: 16 tokens of one
    head beside a full prefix, for capacities around a key block."""
    for cap in (1, 15, 16, 17, 48, 49):
        say(f"decode form, full cache of {cap}")
        rng = np.random.default_rng(cap)
        b = lambda scale, *shape: syn.bf16_bits((rng.standard_normal(shape) * scale).astype(np.float32))  # noqa: E731
        q, k, v, ck, cv = b(0.3, 16, 2, 64), b(1.0, 16, 2, 64), b(1.0, 16, 2, 64), b(1.0, cap, 2, 64), b(1.0, cap, 2, 64)
        cache = hy.KvCache(cap, 2, 64)
        _fill_cache(cache, ck, cv, stream)
        qd, kd, vd, out = dev(q, stream), dev(k, stream), dev(v, stream), hy.DeviceArray((16, 2, 64), np.uint16)
        hy.attention(qd, kd, vd, 16, 2, cache, cap, cap, 0, out, stream)
        ref = O.attention_f64(q, k, v, ck, cv, cap, cap, 0)
        _check(out.to_host(stream), ref, np.concatenate([v.reshape(-1), cv.reshape(-1)]), f"cap={cap}")
        for a in (qd, kd, vd, out):
            a.close()
        cache.close()


@pytest.mark.parametrize("L,H,KVH,D,prefix,window,cached", [
    (8, 16, 1, 512, 40, 0, True),        # one row tile; 2 tokens a wave
    (3, 16, 1, 512, 8, 0, False),        # rows past the end repeat the last
    (5, 16, 1, 512, 650, 0, True),       # key splits
    (64, 4, 2, 256, 33, 0, True),        # 16 tokens a wave, whole waves before the key
    (70, 4, 2, 128, 50, 20, True),       # a window's edges in the same waves
    (40, 2, 2, 64, 16, 16, False),
])
def test_chunk_values_that_are_not_finite(stream, L, H, KVH, D, prefix, window, cached):
    """An infinite or NaN value of V reaches the rows that see its key and no others: V of the
    last token (which no earlier token sees) and of a key that a window shows the first tokens
    only. Everything else meets the bar against V without them."""
    say(f"not finite L={L} KVH={KVH} D={D} prefix={prefix} window={window}")
    T = prefix + L
    rng = np.random.default_rng(D + L)
    b = lambda scale, *shape: syn.bf16_bits((rng.standard_normal(shape) * scale).astype(np.float32))  # noqa: E731
    q, k, v = b(D ** -0.5, L, H, D), b(1.0, T, KVH, D), b(1.0, T, KVH, D)
    bad = [(T - 1, 3, 0x7F80), (T - 1, D - 9, 0x7FC0)]
    if window:
        bad += [(prefix - window + 3, 17, 0xFF80)]      # visible to tokens 0 .. 2
    vb = v.copy()
    for j, d, bits in bad:
        v[j, :, d], vb[j, :, d] = 0, bits
    cache = hy.KvCache(T, KVH, D)
    _fill_cache(cache, k, vb, stream)
    qd, out = dev(q, stream), hy.DeviceArray((L, H, D), np.uint16)
    kd, vd = dev(k[prefix:], stream), dev(vb[prefix:], stream)
    hy.call("hyp_attention", qd.ptr, None if cached else kd.ptr, None if cached else vd.ptr, L, H, cache.handle, prefix,
            prefix, window, out.ptr, stream.handle)
    got = out.to_host(stream)
    ref = O.attention_f64(q, k[prefix:], v[prefix:], k, v, prefix, prefix, window)
    for j, d, bits in bad:
        t = np.arange(L)
        sees = (j <= prefix + t) & ((j > prefix + t - window) if window else True)
        assert np.all(np.isnan(syn.bf16_to_f32(got[sees, :, d])) if bits == 0x7FC0 else got[sees, :, d] == bits), (j, d)
        got[sees, :, d] = syn.bf16_bits(ref[sees, :, d].astype(np.float32))   # (leaves the bar to the others)
    _check(got, ref, v, f"L={L} D={D}")
    for a in (qd, kd, vd, out):
        a.close()
    cache.close()


def test_kv_cache_write_slots_and_ring_overwrite(stream):
    """Tokens land in slot p % capacity; a write longer than the ring keeps its last
    `capacity` tokens; attention over the written prefix equals attention over the same
    rows uploaded directly."""
    cap, KVH, D = 24, 2, 64
    rng = np.random.default_rng(3)
    cache = hy.KvCache(cap, KVH, D)
    kp, vp = cache.buffers()
    expect_k = np.zeros((cap, KVH, D), np.uint16)
    expect_v = np.zeros((cap, KVH, D), np.uint16)
    _fill_cache(cache, expect_k, expect_v, stream)
    pos = 0
    for n in (5, 1, 30, 7, 3):      # 30 > cap wraps past a whole ring
        k = syn.bf16_bits(rng.standard_normal((n, KVH, D)).astype(np.float32))
        v = syn.bf16_bits(rng.standard_normal((n, KVH, D)).astype(np.float32))
        kd, vd = dev(k, stream), dev(v, stream)
        cache.write(kd, vd, n, pos, stream)
        for t in range(n):
            expect_k[(pos + t) % cap] = k[t]
            expect_v[(pos + t) % cap] = v[t]
        pos += n
        kd.close()
        vd.close()
    stream.synchronize()
    got_k = np.zeros_like(expect_k)
    got_v = np.zeros_like(expect_v)
    for ptr, host in ((kp, got_k), (vp, got_v)):
        hy.call("hyp_memcpy_dtoh", host.ctypes.data_as(ctypes.c_void_p), ptr, host.nbytes, stream.handle)
    stream.synchronize()
    np.testing.assert_array_equal(got_k, expect_k)
    np.testing.assert_array_equal(got_v, expect_v)
    # decode one token over the last 20 written positions
    q = syn.bf16_bits((rng.standard_normal((1, 4, D)) * 0.5).astype(np.float32))
    k1 = syn.bf16_bits(rng.standard_normal((1, KVH, D)).astype(np.float32))
    v1 = syn.bf16_bits(rng.standard_normal((1, KVH, D)).astype(np.float32))
    qd, kd, vd = dev(q, stream), dev(k1, stream), dev(v1, stream)
    out = hy.DeviceArray((1, 4, D), np.uint16)
    hy.attention(qd, kd, vd, 1, 4, cache, pos, 20, 21, out, stream)
    ref = O.attention_f64(q, k1, v1, expect_k, expect_v, pos, 20, 21)
    _check(out.to_host(stream), ref, np.concatenate([v1.reshape(-1), expect_v.reshape(-1)]), "after writes")
    for a in (qd, kd, vd, out):
        a.close()
    cache.close()


def test_attention_rejects_bad_arguments(stream):
    cache = hy.KvCache(16, 2, 64)
    x = hy.DeviceArray((4, 4, 64), np.uint16)
    for args, what in (((x, x, x, 1, 3, cache, 5, 5, 0, x), "heads"),       # 3 heads over 2 kv heads
                       ((x, x, x, 1, 4, cache, 5, 6, 0, x), "prefix"),      # prefix beyond offset
                       ((x, x, x, 1, 4, cache, 50, 17, 0, x), "capacity")):  # prefix beyond capacity
        with pytest.raises(hy.HypError) as e:
            hy.attention(*args, stream)
        assert e.value.status_name == "INVALID_ARGUMENT", what
    x.close()
    cache.close()
