"""GPU parity: paged-attention decode vs the float64 brute-force oracle.  The reference tree
has no attention operator (parity unpinned by the reference); tolerance is the north-star
1e-3 relative error, taken against the largest magnitude of each output row."""
import numpy as np
import pytest

from nncase_amd import kernels as K
from nncase_amd import runtime as rt
from oracle import oracle as O

pytestmark = pytest.mark.gpu
RTOL = 1e-3


def make_case(rng, bsz, hq, hkv, d, blk, max_ctx, ctx_lens=None):
    max_blocks = -(-max_ctx // blk)
    nb = bsz * max_blocks + 3
    q = rng.standard_normal((bsz, hq, d)).astype(np.float16)
    kc = rng.standard_normal((nb, hkv, blk, d)).astype(np.float16)
    vc = rng.standard_normal((nb, hkv, blk, d)).astype(np.float16)
    perm = rng.permutation(nb)[: bsz * max_blocks].reshape(bsz, max_blocks).astype(np.int32)  # scattered physical blocks
    cl = np.asarray(ctx_lens if ctx_lens is not None else rng.integers(1, max_ctx + 1, bsz), np.int32)
    return q, kc, vc, perm, cl


def check(hip_ctx, q, kc, vc, bt, cl, scale, out_dtype=np.float32):
    """vc is token-major [blocks, Hkv, block, D] (easy to index in the expectations); the kernel and
    the oracle both take the d-major cache layout."""
    vt = K.v_cache_from_token_major(vc)
    got = K.paged_attention_decode(q, kc, vt, bt, cl, scale, out_dtype, ctx=hip_ctx).astype(np.float64)
    want = O.paged_attention_decode(q.view(np.uint16), kc.view(np.uint16), vt.view(np.uint16), bt, cl, scale)
    tol = RTOL * np.abs(want).max(axis=-1, keepdims=True) + (1e-3 if out_dtype == np.float16 else 1e-6)
    assert (np.abs(got - want) <= tol).all(), f"max err {np.abs(got - want).max()}"
    return got


@pytest.mark.parametrize("bsz,hq,hkv,d,blk,max_ctx", [
    (2, 14, 2, 64, 16, 700),     # Qwen2-0.5B head geometry, two splits
    (3, 4, 4, 64, 16, 100),      # MHA
    (2, 8, 1, 64, 32, 1100),     # MQA, 8 query heads on one kv head, block 32, three splits
    (2, 8, 2, 128, 16, 600),     # head_dim 128
    (1, 2, 2, 64, 64, 64),
    (2, 16, 1, 64, 48, 500),     # 16 query heads on one kv head; block size not a power of two
    (2, 32, 2, 128, 16, 300),    # 16 per kv head at head_dim 128
    (3, 1, 1, 128, 32, 257),     # a single head
])
def test_random_cases(hip_ctx, bsz, hq, hkv, d, blk, max_ctx):
    rng = np.random.default_rng(bsz * 1000 + hq)
    case = make_case(rng, bsz, hq, hkv, d, blk, max_ctx)
    check(hip_ctx, *case, 1.0 / np.sqrt(d))
    check(hip_ctx, *case, 1.0 / np.sqrt(d), np.float16)


def test_edge_context_lengths(hip_ctx):
    rng = np.random.default_rng(7)
    lens = [0, 1, 15, 16, 17, 511, 512, 513, 1024]
    q, kc, vc, bt, cl = make_case(rng, len(lens), 14, 2, 64, 16, 1024, lens)
    got = check(hip_ctx, q, kc, vc, bt, cl, 0.125)
    assert (got[0] == 0).all()                                  # empty context -> zeros
    for h in range(14):                                         # ctx == 1 -> that token's V row
        assert np.array_equal(got[1, h], vc[bt[1, 0], h // 7, 0].astype(np.float64))


def test_closed_forms(hip_ctx):
    rng = np.random.default_rng(11)
    q, kc, vc, bt, cl = make_case(rng, 2, 14, 2, 64, 16, 900, [900, 333])
    base = check(hip_ctx, q, kc, vc, bt, cl, 0.125)
    # uniform keys -> plain mean of the cached values
    ku = np.ones_like(kc)
    got = K.paged_attention_decode(q, ku, K.v_cache_from_token_major(vc), bt, cl, 0.125, ctx=hip_ctx)
    for b in range(2):
        toks = [(bt[b, t // 16], t % 16) for t in range(cl[b])]
        for kvh in range(2):
            mean = np.mean([vc[p, kvh, o].astype(np.float64) for p, o in toks], axis=0)
            np.testing.assert_allclose(got[b, kvh * 7 + 3], mean, rtol=RTOL, atol=1e-4)
    # relabelling physical blocks leaves the output bit-identical
    perm = rng.permutation(kc.shape[0])
    inv = np.argsort(perm).astype(np.int32)
    again = K.paged_attention_decode(q, kc[perm], K.v_cache_from_token_major(vc[perm]), inv[bt], cl, 0.125, ctx=hip_ctx)
    assert np.array_equal(again.astype(np.float64), base)
    # large logits do not overflow the softmax; a negative scale is honoured
    check(hip_ctx, (q * 30).astype(np.float16), kc, vc, bt, cl, 1.0)
    check(hip_ctx, q, kc, vc, bt, cl, -0.125)


def test_slots_past_the_context_are_ignored(hip_ctx):
    """Cache slots of the last block beyond ctx_len (and blocks the table lists past it) may hold
    anything, NaN and Inf included, without touching the result."""
    rng = np.random.default_rng(13)
    lens = [5, 16, 37, 600]
    q, kc, vc, bt, cl = make_case(rng, len(lens), 14, 2, 64, 16, 640, lens)
    base = check(hip_ctx, q, kc, vc, bt, cl, 0.125)
    kc2, vc2 = kc.copy(), vc.copy()
    poison = np.array([np.nan, np.inf, -np.inf, 65504.0], np.float16)
    for b, n in enumerate(lens):
        for t in range(n, bt.shape[1] * 16):
            kc2[bt[b, t // 16], :, t % 16, :] = poison[t % 4]
            vc2[bt[b, t // 16], :, t % 16, :] = poison[(t + 1) % 4]
    vt2 = K.v_cache_from_token_major(vc2)
    again = K.paged_attention_decode(q, kc2, vt2, bt, cl, 0.125, ctx=hip_ctx).astype(np.float64)
    assert np.array_equal(again, base)


def test_config5_shape(hip_ctx):
    """BASELINE config 5 attention geometry: batch 32, 14 q / 2 kv heads, d 64, block 16, ctx U[512, 4096]."""
    rng = np.random.default_rng(5)
    q, kc, vc, bt, cl = make_case(rng, 32, 14, 2, 64, 16, 4096, rng.integers(512, 4097, 32))
    check(hip_ctx, q, kc, vc, bt, cl, 0.125, np.float16)


def test_long_runs_per_wave(hip_ctx):
    """Enough sequences that the kernel takes its longest per-wave runs (8 tiles of 16 tokens at head_dim 64,
    4 at head_dim 128), with ragged lengths around the split boundaries."""
    rng = np.random.default_rng(17)
    lens = np.concatenate([[1, 511, 512, 513, 1023, 1025, 2048], rng.integers(1, 2049, 89)])
    q, kc, vc, bt, cl = make_case(rng, len(lens), 8, 4, 64, 16, 2048, lens)
    check(hip_ctx, q, kc, vc, bt, cl, 0.125)
    lens = np.concatenate([[1, 255, 256, 257, 1024], rng.integers(1, 1025, 91)])
    q, kc, vc, bt, cl = make_case(rng, len(lens), 8, 8, 128, 16, 1024, lens)
    check(hip_ctx, q, kc, vc, bt, cl, 0.09)


def test_repeated_calls_reuse_the_workspace(hip_ctx):
    """The completion counters return to zero after every call: different shapes back to back."""
    rng = np.random.default_rng(19)
    for bsz, hq, hkv, d, max_ctx in [(4, 14, 2, 64, 2000), (2, 8, 8, 128, 700), (4, 14, 2, 64, 2000), (1, 4, 1, 64, 90)]:
        case = make_case(rng, bsz, hq, hkv, d, 16, max_ctx)
        check(hip_ctx, *case, 0.125)
        check(hip_ctx, *case, 0.125)


def test_error_paths(hip_ctx):
    from nncase_amd import runtime as rt
    rng = np.random.default_rng(1)
    q, kc, vc, bt, cl = make_case(rng, 1, 3, 2, 64, 16, 32)   # 3 query heads on 2 kv heads
    with pytest.raises(rt.HipError) as e:
        K.paged_attention_decode(q, kc, K.v_cache_from_token_major(vc), bt, cl, 0.125, ctx=hip_ctx)
    assert e.value.code == -rt.ERR_SHAPE_MISMATCH
    q, kc, vc, bt, cl = make_case(rng, 1, 2, 2, 32, 16, 32)   # unsupported head_dim
    with pytest.raises(rt.HipError) as e:
        K.paged_attention_decode(q, kc, K.v_cache_from_token_major(vc), bt, cl, 0.125, ctx=hip_ctx)
    assert e.value.code == -rt.ERR_SHAPE_MISMATCH
    q, kc, vc, bt, cl = make_case(rng, 1, 2, 2, 64, 8, 32)    # block size not a multiple of 16
    with pytest.raises(rt.HipError) as e:
        K.paged_attention_decode(q, kc, K.v_cache_from_token_major(vc), bt, cl, 0.125, ctx=hip_ctx)
    assert e.value.code == -rt.ERR_SHAPE_MISMATCH
    q, kc, vc, bt, cl = make_case(rng, 1, 17, 1, 64, 16, 32)  # 17 query heads on one kv head
    with pytest.raises(rt.HipError) as e:
        K.paged_attention_decode(q, kc, K.v_cache_from_token_major(vc), bt, cl, 0.125, ctx=hip_ctx)
    assert e.value.code == -rt.ERR_SHAPE_MISMATCH


def test_capture_without_a_warm_up_and_pinned_workspace(hip_ctx):
    """Recording the operator sizes the context's split workspace, so a capture needs no eager call first;
    while the captured function lives, a call that would have to move the workspace is refused (-EBUSY)
    instead of freeing memory the graph still addresses."""
    import errno
    from nncase_amd import runtime as rt
    from nncase_amd.runtime import Context, Function
    ctx = Context(0)  # a context of its own: its workspace starts empty
    try:
        rng = np.random.default_rng(99)
        q, kc, vc, bt, cl = make_case(rng, 3, 14, 2, 64, 16, 2048, [2048, 700, 33])
        vt = K.v_cache_from_token_major(vc)
        dq, dk, dv, dbt, dcl = (ctx.to_device(t) for t in (q, kc, vt, bt, cl))
        dout = ctx.alloc(q.size * 4)
        args = rt.PagedAttnArgs(3, 14, 2, 64, 16, bt.shape[1], kc.shape[0], 0.125, rt.DT_F32)
        fn = Function(ctx)
        fn.add_paged_attention_decode(dq, dk, dv, dbt, dcl, dout, args)
        fn.capture()                       # no eager call came before
        want = O.paged_attention_decode(q.view(np.uint16), kc.view(np.uint16), vt.view(np.uint16), bt, cl, 0.125)
        first = None
        for _ in range(3):
            dout.fill(0)
            fn.invoke()
            ctx.sync()
            got = dout.download(q.shape, np.float32)
            assert (np.abs(got - want) <= RTOL * np.abs(want).max(axis=-1, keepdims=True) + 1e-6).all()
            first = got if first is None else first
            assert np.array_equal(got, first)
        # a larger geometry on the same context would move the workspace under the graph
        q2, kc2, vc2, bt2, cl2 = make_case(rng, 16, 14, 2, 64, 16, 4096)
        big = rt.PagedAttnArgs(16, 14, 2, 64, 16, bt2.shape[1], kc2.shape[0], 0.125, rt.DT_F32)
        d2 = [ctx.to_device(t) for t in (q2, kc2, K.v_cache_from_token_major(vc2), bt2, cl2)]
        dout2 = ctx.alloc(q2.size * 4)
        with pytest.raises(rt.HipError) as e:
            ctx.paged_attention_decode(*d2, dout2, big)
        assert e.value.code == -errno.EBUSY
        fn.invoke()                        # the graph still replays on intact memory
        ctx.sync()
        assert np.array_equal(dout.download(q.shape, np.float32), first)
        fn.destroy()                       # nothing refers to the workspace any more: growth is allowed again
        ctx.paged_attention_decode(*d2, dout2, big)
        ctx.sync()
        want2 = O.paged_attention_decode(q2.view(np.uint16), kc2.view(np.uint16), d2 and K.v_cache_from_token_major(vc2).view(np.uint16), bt2, cl2, 0.125)
        got2 = dout2.download(q2.shape, np.float32)
        assert (np.abs(got2 - want2) <= RTOL * np.abs(want2).max(axis=-1, keepdims=True) + 1e-6).all()
    finally:
        ctx.close()


@pytest.mark.parametrize("hq,hkv,d", [(14, 2, 64), (4, 1, 128), (16, 1, 128)])
@pytest.mark.parametrize("capacity", [128, 144, 256, 272, 1024, 1040, 2064, 4096, 8208])
def test_every_split_of_the_capacity(hip_ctx, hq, hkv, d, capacity):
    """Both sides of every capacity at which the tokens per block change, contexts that end inside the first, a middle and the
    last block, more splits than one run of the merge takes."""
    rng = np.random.default_rng(capacity + d)
    lens = [1, capacity // 3 + 1, capacity]
    case = make_case(rng, len(lens), hq, hkv, d, 16, capacity, lens)
    check(hip_ctx, *case, 1.0 / np.sqrt(d))


@pytest.mark.parametrize("b,hq,hkv,d,capacity", [(33, 14, 2, 64, 3216), (20, 16, 16, 64, 208), (2, 12, 12, 64, 6512), (4, 32, 8, 128, 2064), (1, 16, 8, 128, 10016),
                                                 (33, 32, 8, 128, 160), (64, 16, 4, 128, 1040)])
def test_block_shapes_by_the_launch(hip_ctx, b, hq, hkv, d, capacity):
    """Capacities at which the number of sequences and kv heads decides the tokens per block, on both sides."""
    rng = np.random.default_rng(capacity + d)
    lens = ([1, capacity // 3 + 1, capacity, capacity - 15] * b)[-b:]
    check(hip_ctx, *make_case(rng, b, hq, hkv, d, 16, capacity, lens), 1.0 / np.sqrt(d))


def test_a_workspace_that_cannot_grow_takes_longer_runs(hip_ctx):
    """While a captured graph holds the workspace, a call whose usual split needs more of it runs with fewer splits instead."""
    rng = np.random.default_rng(3)
    ctx = rt.Context(0)
    try:
        def device(case, out):
            q, kc, vc, bt, cl = case
            bufs = [ctx.to_device(t) for t in (q, kc, K.v_cache_from_token_major(vc), bt, cl)]
            args = rt.PagedAttnArgs(q.shape[0], q.shape[1], kc.shape[1], q.shape[2], 16, bt.shape[1], kc.shape[0], 0.125, rt.DT_F32)
            return bufs, ctx.alloc(q.size * 4), args
        first = make_case(rng, 32, 14, 2, 64, 16, 512, [500] * 32)       # four splits
        fn = rt.Function(ctx)
        bufs, out, args = device(first, np.float32)
        fn.add_paged_attention_decode(*bufs, out, args)
        fn.capture()
        second = make_case(rng, 32, 14, 2, 64, 16, 1024, [1000] * 32)    # eight
        bufs2, out2, args2 = device(second, np.float32)
        ctx.paged_attention_decode(*bufs2, out2, args2)
        got = out2.download((32, 14, 64), np.float32)
        q, kc, vc, bt, cl = second
        vt = K.v_cache_from_token_major(vc)
        want = O.paged_attention_decode(q.view(np.uint16), kc.view(np.uint16), vt.view(np.uint16), bt, cl, 0.125)
        assert np.abs(got - want).max() <= RTOL * np.abs(want).max()
        fn.invoke()
        ctx.sync()
    finally:
        ctx.close()


@pytest.mark.parametrize("b,hq,hkv,d,blk,capacity", [
    (2, 32, 8, 128, 16, 6144), (16, 16, 1, 128, 48, 6144), (38, 8, 8, 128, 32, 704), (26, 28, 4, 128, 64, 1024), (33, 8, 8, 128, 16, 384),
    (9, 32, 32, 128, 16, 1040), (16, 64, 64, 128, 16, 1024), (64, 16, 16, 128, 16, 1040),
    (12, 14, 2, 64, 16, 272), (24, 16, 1, 64, 64, 320), (3, 12, 12, 64, 48, 480), (40, 24, 24, 64, 16, 512)])
def test_a_split_gone_through_in_steps(hip_ctx, b, hq, hkv, d, blk, capacity):
    """Launches of the kernel that goes through a split 128 tokens at a time (few splits, one split, 512 and 1024 tokens each, values
    past the caches): contexts that end around a wave's 32 tokens, a step and the splits.  Slots past a context hold NaN."""
    rng = np.random.default_rng(b * 1000 + capacity)
    edges = [1, 31, 32, 33, 127, 128, 129, 255, 257, 383, 385, 511, 513, 1023, 1025, capacity - 1, capacity]
    lens = np.asarray([n for n in edges if n <= capacity] + [0], np.int32)
    cl = np.resize(np.roll(lens, 1 + b % 5), b)
    cl[0] = capacity
    blocks, nb = capacity // blk, 40     # (entries of the table repeat: the caches stay small)
    q = rng.standard_normal((b, hq, d)).astype(np.float16)
    kc, vc = (rng.standard_normal((nb + b, hkv, blk, d)).astype(np.float16) for _ in range(2))
    bt = rng.integers(0, nb, (b, blocks)).astype(np.int32)
    for i, n in enumerate(cl):           # a sequence's last, partly filled block is its own
        if n % blk:
            bt[i, n // blk] = nb + i
            kc[nb + i, :, n % blk:], vc[nb + i, :, n % blk:] = np.nan, np.nan
    vt = K.v_cache_from_token_major(vc)
    got = K.paged_attention_decode(q, kc, vt, bt, cl, d ** -0.5, np.float32, ctx=hip_ctx).astype(np.float64)
    want = O.paged_attention_decode(q.view(np.uint16), np.nan_to_num(kc).view(np.uint16), np.nan_to_num(vt).view(np.uint16), bt, cl, d ** -0.5)
    # of the exponent's rounding (at most 2^-23 of a logit of about 8 / ln 2), the float32 sums' and the final division's: 1e-5
    assert (np.abs(got - want) <= 1e-5 * np.abs(want).max(axis=-1, keepdims=True)).all(), f"max err {np.abs(got - want).max()}"


def test_infinite_and_very_large_logits_in_steps(hip_ctx):
    """Whole steps of keys at -inf have no weight, whatever comes before and after them; logits whose float32 neighbours are thousands
    apart choose one key."""
    rng = np.random.default_rng(23)
    b, hq, hkv, d, blk, capacity = 2, 16, 8, 128, 16, 6144
    q = rng.uniform(0.5, 1, (b, hq, d)).astype(np.float16)
    kc, vc = (rng.standard_normal((b * capacity // blk, hkv, blk, d)).astype(np.float16) for _ in range(2))
    bt = np.arange(b * capacity // blk, dtype=np.int32).reshape(b, -1)
    dead = kc.copy()
    dead[:8], dead[24:32], dead[100:104], dead[384:400] = -np.inf, -np.inf, -np.inf, -np.inf
    vt = K.v_cache_from_token_major(vc)
    cl = np.asarray([capacity, 700], np.int32)
    got = K.paged_attention_decode(q, dead, vt, bt, cl, d ** -0.5, np.float32, ctx=hip_ctx).astype(np.float64)
    want = O.paged_attention_decode(q.view(np.uint16), np.maximum(dead, np.float16(-60000)).view(np.uint16), vt.view(np.uint16), bt, cl, d ** -0.5)
    assert (np.abs(got - want) <= 1e-5 * np.abs(want).max(axis=-1, keepdims=True)).all()
    big = (kc * 8000).clip(-60000, 60000).astype(np.float16)
    got = K.paged_attention_decode((q * 60000).astype(np.float16), big, vt, bt, cl, 1.0, np.float32, ctx=hip_ctx)
    for i in range(b):
        for h in range(hq):
            keys = big[bt[i], h // 2].reshape(-1, d)[: cl[i]].astype(np.float64)
            at = np.argmax(keys @ (q[i, h] * 60000).astype(np.float16).astype(np.float64))
            assert np.array_equal(got[i, h], vc[bt[i], h // 2].reshape(-1, d)[at].astype(np.float32))


@pytest.mark.parametrize("b,hq,hkv,capacity,split", [(2, 16, 8, 6144, 384), (16, 64, 8, 2048, 1024)])
def test_a_split_of_infinite_logits(hip_ctx, b, hq, hkv, capacity, split):
    """Splits whose keys are all at -inf, the first and a later one of a context, have no weight beside the others."""
    rng = np.random.default_rng(29)
    d, blk = 128, 16
    q = rng.uniform(0.5, 1, (b, hq, d)).astype(np.float16)
    kc, vc = (rng.standard_normal((b * capacity // blk, hkv, blk, d)).astype(np.float16) for _ in range(2))
    bt = np.arange(b * capacity // blk, dtype=np.int32).reshape(b, -1)
    dead = kc.copy()
    n = capacity // blk
    dead[:split // blk] = -np.inf
    dead[2 * n - split // blk:2 * n] = -np.inf
    vt = K.v_cache_from_token_major(vc)
    cl = np.full(b, capacity, np.int32)
    got = K.paged_attention_decode(q, dead, vt, bt, cl, d ** -0.5, np.float32, ctx=hip_ctx).astype(np.float64)
    want = O.paged_attention_decode(q.view(np.uint16), np.maximum(dead, np.float16(-60000)).view(np.uint16), vt.view(np.uint16), bt, cl, d ** -0.5)
    # (the bound of the launches above)
    assert (np.abs(got - want) <= 1e-5 * np.abs(want).max(axis=-1, keepdims=True)).all(), f"max err {np.abs(got - want).max()}"


@pytest.mark.parametrize("b,hkv,capacity,lens", [
    (4, 8, 16384, [300]), (4, 8, 16384, [385, 1000, 0, 1]), (32, 1, 16384, [400]), (16, 8, 4096, [129, 256, 257, 0, 511]), (10, 8, 3008, [2049, 2047, 1]),
    (70, 3, 2048, [640, 33, 0]), (256, 1, 2048, [512, 513, 64]), (130, 1, 4096, [384, 383]), (16, 3, 8192, [0]), (2, 8, 32768, [8001, 7])])
@pytest.mark.parametrize("one_fills_it", [False, True])
def test_contexts_shorter_than_the_cache(hip_ctx, b, hkv, capacity, lens, one_fills_it):
    """Splits as the launch's lengths have it: short contexts in a large cache, with and without a sequence that fills it, more sequences
    than a wave has lanes, empty ones among them and alone."""
    rng = np.random.default_rng(b * 1000 + capacity)
    cl = np.resize(np.asarray(lens, np.int32), b)
    if one_fills_it: cl[b // 2] = capacity
    d, blk, nb, hq = 128, 16, 40, hkv * 2
    q = rng.standard_normal((b, hq, d)).astype(np.float16)
    kc, vc = (rng.standard_normal((nb, hkv, blk, d)).astype(np.float16) for _ in range(2))
    bt = rng.integers(0, nb, (b, capacity // blk)).astype(np.int32)
    vt = K.v_cache_from_token_major(vc)
    want = O.paged_attention_decode(q.view(np.uint16), kc.view(np.uint16), vt.view(np.uint16), bt, cl, d ** -0.5)
    for _ in range(2):                                                       # (the second finds the counters as the first left them)
        got = K.paged_attention_decode(q, kc, vt, bt, cl, d ** -0.5, np.float32, ctx=hip_ctx).astype(np.float64)
        # (the bound of the launches above)
        assert (np.abs(got - want) <= 1e-5 * np.abs(want).max(axis=-1, keepdims=True)).all(), f"max err {np.abs(got - want).max()}"


@pytest.mark.parametrize("b,hkv,capacity,n", [(4, 8, 3072, 200), (16, 1, 6400, 700), (4, 8, 16384, 900)])
def test_short_contexts_beside_a_products_weights(hip_ctx, b, hkv, capacity, n):
    """Recorded with a product behind it (whose weights the launch brings along) and replayed as a graph: the same bits as the call alone."""
    rng = np.random.default_rng(b + capacity)
    d, blk, nb, hq = 128, 16, 40, hkv * 2
    q, kc, vt = (rng.standard_normal(s).astype(np.float16) for s in ((b, hq, d), (nb, hkv, blk, d), (nb, hkv, d, blk)))
    bt = rng.integers(0, nb, (b, capacity // blk)).astype(np.int32)
    bufs = [hip_ctx.to_device(t) for t in (q, kc, vt, bt, np.resize(np.asarray([n, n // 2, 1], np.int32), b))]
    out, y, alone, y_alone = (hip_ctx.alloc(x) for x in (b * hq * d * 2, b * 256 * 2, b * hq * d * 2, b * 256 * 2))
    args = rt.PagedAttnArgs(b, hq, hkv, d, blk, capacity // blk, nb, d ** -0.5, rt.DT_F16)
    w = hip_ctx.prepack_w8a16(rng.integers(-127, 128, (256, hq * d), dtype=np.int8), np.full(256, 1e-3, np.float32))
    fn = rt.Function(hip_ctx)
    fn.add_paged_attention_decode(*bufs, out, args)
    fn.add_w8a16_gemm(out, w, y, b)
    fn.capture()
    hip_ctx.paged_attention_decode(*bufs, alone, args)
    hip_ctx.w8a16_gemm(alone, w, y_alone, b)
    want = alone.download((b, hq, d), np.uint16), y_alone.download((b, 256), np.uint16)
    for _ in range(3):
        fn.invoke()
        hip_ctx.sync()
        assert np.array_equal(out.download((b, hq, d), np.uint16), want[0]) and np.array_equal(y.download((b, 256), np.uint16), want[1])
