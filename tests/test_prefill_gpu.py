"""The batched prefill (generate's prompt tokens before the last) against the
decode path token by token (forward), which the oracle tests pin.

Both add the same exact fp64 products and round each output once; only the
order of the additions differs, which can move an output across an fp32
rounding boundary about once in 10^8 (2^-52 * a few roundings against 2^-24),
and with it, once in 10^4 of those, a cached fp16 value.  So the caches are
compared bit by bit with one part in 1000 allowed to differ by one fp16 ulp
(a moved value travels through the layers after it), the picks with a tie's
worth of room."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BASE = dict(n_layers=2, dim=4096, ffn_dim=4096, n_heads=32, n_kv_heads=8, head_dim=128, vocab=512, max_ctx=128,
            rope_theta=10000.0, norm_eps=1e-5)


def make(iam, ctx, **kw):
    m = iam.Model(ctx, iam.ModelConfig(**dict(BASE, **kw)))
    m.synthesize(3)
    return m


def state(m, cfg, n):
    kv = (cfg["n_layers"], cfg["max_ctx"], cfg["n_kv_heads"], 128)
    k, v = (m.read_tensor(t, np.uint16).view(np.float16).reshape(kv)[:, :n] for t in ("kcache", "vcache"))
    return k, v, m.read_tensor("history", np.int32)[1:n + 1], m.read_tensor("logits", np.float32)


def ulp16(a, b):
    """Distance in fp16 steps."""
    def order(x):
        i = x.view(np.int16).astype(np.int32)
        return np.where(i < 0, -(i & 0x7FFF), i)
    return np.abs(order(a) - order(b))


def check(O, ctx, m, cfg, n, effort, seed=5, after=None):
    """after: called once the prompt has been fed."""
    prompt = O.gen_tokens(0, seed, n, cfg["vocab"])
    m.reset_caches()
    ctx.walk_counters(reset=True)
    first = m.generate(prompt, 1, effort)
    if after:
        after()
    counted = ctx.walk_counters(reset=True)
    k, v, hist, logits = state(m, cfg, n)
    m.reset_caches()
    log = ctx.empty(cfg["vocab"], np.float32)
    picks = []
    for pos, tok in enumerate(prompt):
        m.forward(int(tok), pos, effort, log)
        picks.append(O.argmax(log.read()))
    wanted = ctx.walk_counters(reset=True)
    wk, wv, _, _ = state(m, cfg, n)
    want = log.read()
    log.free()
    for got, ref in ((k, wk), (v, wv)):
        d = ulp16(got, ref)
        assert np.mean(d != 0) < 1e-3 and d.max() <= 1, (n, effort, np.mean(d != 0), d.max())
    assert np.mean(hist != np.array(picks)) <= 0.02
    assert first[0] == hist[-1]
    assert np.linalg.norm(logits - want) <= 1e-5 * np.linalg.norm(want)
    # rows, bytes and matrices counted as the steps count them
    assert counted[2] == wanted[2]
    assert abs(counted[1] - wanted[1]) <= 1e-5 * wanted[1] and abs(counted[0] - wanted[0]) <= 1e-5 * wanted[0]


@pytest.fixture(scope="module")
def model(iam, ctx):
    m = make(iam, ctx)
    yield m
    m.close()


# too few tokens; one token group (part of one, all of it, and one or six
# tokens more), two, three (the workgroups of four groups) and six groups,
# whole and with a remainder the steps take or the batch takes
@pytest.mark.parametrize("n,effort", [(5, 0.25), (16, 0.25), (10, 1.0), (17, 0.5), (18, 0.05), (23, 0.05), (33, 1.0),
                                      (40, 0.25), (97, 0.125), (108, 0.25)])
def test_token_groups(O, ctx, model, n, effort):
    check(O, ctx, model, BASE, n, effort)


# the tokens past a multiple of 64: all in the batch, or the ones past the last
# full group, or all of them by steps (which of these, the effort decides)
@pytest.mark.parametrize("n", [66, 68, 75, 82, 98, 122])
@pytest.mark.parametrize("effort", [0.05, 1.0])
def test_tokens_past_a_row(O, ctx, model, n, effort):
    check(O, ctx, model, BASE, n, effort)


@pytest.mark.parametrize("kw,n", [(dict(ffn_dim=4112, vocab=528), 40),                 # 257 and 33 bucket columns
                                  (dict(dim=5120, n_heads=40, n_kv_heads=8, n_layers=1), 20),   # the norm apart
                                  (dict(ffn_dim=5008, n_kv_heads=4, vocab=16, n_layers=1), 70)])
def test_ragged_shapes(O, iam, ctx, kw, n):
    cfg = dict(BASE, **kw)
    m = make(iam, ctx, **kw)
    try:
        check(O, ctx, m, cfg, n, 0.25)
    finally:
        m.close()


# (two layers: the second one's cache depends on the first one's attention)
LONG = dict(BASE, n_kv_heads=32, max_ctx=1152)


@pytest.fixture(scope="module")
def long_model(iam, ctx):
    """One query head per KV head (attention's one-head form) and room for
    prompts of more than two chunks of 512."""
    m = make(iam, ctx, n_kv_heads=32, max_ctx=1152)
    yield m
    m.close()


# one chunk past 64 and past 128 positions; a second chunk the steps take (4
# tokens), a batch takes (47, part of a group), in part (70); three chunks; the
# whole KV capacity
@pytest.mark.parametrize("n,effort", [(100, 0.25), (200, 0.05), (517, 0.25), (560, 0.25), (583, 0.05), (1050, 1.0),
                                      (1151, 0.25)])
def test_prompts_of_several_chunks(O, ctx, long_model, n, effort):
    check(O, ctx, long_model, LONG, n, effort)


def test_several_chunks_pair_heads_and_batches(O, iam, ctx):
    """Two heads per workgroup, and the number of batches that run."""
    cfg = dict(BASE, max_ctx=640)
    m = make(iam, ctx, max_ctx=640)
    try:
        names = []

        def batches():
            ctx.sync()
            ctx.profiling(False)
            names.append(ctx.kernel_stat("prefill.pick")[1])

        ctx.kernel_stats_reset()
        ctx.profiling(True)
        check(O, ctx, m, cfg, 560, 0.25, after=batches)
        assert names == [2]
    finally:
        ctx.profiling(False)
        m.close()


def test_several_chunks_dense_head(O, iam, ctx, long_model):
    """The dense head's picks and the cache of a prompt of two chunks."""
    head = ctx.upload(O.gen_f16(0, 21, 512 * 4096, 0.0, 0.02))
    n = 600
    prompt = O.gen_tokens(0, 8, n, 512)
    long_model.set_lm_dense(head)
    try:
        long_model.reset_caches()
        got = long_model.generate(prompt, 1, 0.25)
        k, v, hist, _ = state(long_model, LONG, n)
        long_model.reset_caches()
        log = ctx.empty(512, np.float32)
        picks = []
        for pos, tok in enumerate(prompt):
            long_model.forward(int(tok), pos, 0.25, log)
            picks.append(O.argmax(log.read()))
        wk, wv, _, _ = state(long_model, LONG, n)
        log.free()
        for a, b in ((k, wk), (v, wv)):
            d = ulp16(a, b)
            assert np.mean(d != 0) < 1e-3 and d.max() <= 1
        assert np.mean(hist != np.array(picks)) <= 0.02
        assert got[0] == hist[-1]
    finally:
        long_model.set_lm_dense(None)
        head.free()


def test_weights_no_converter_writes(O, iam, ctx):
    """Stats that rise with the rank (the selected ranks are not the first
    ones), buckets with a position twice, and an embedding scale."""
    m = make(iam, ctx)
    try:
        for name in ("layer0.wq", "layer1.w1", "layer1.w2"):
            st = m.read_tensor(f"{name}.stats3", np.uint16).reshape(-1, 16)
            st[::7] = st[::7, ::-1]
            m.write_tensor(f"{name}.stats3", np.ascontiguousarray(st))
        for name in ("layer0.wk", "layer0.w1", "lm_head"):
            b = m.read_tensor(f"{name}.buckets", np.uint16)
            b[::1009] = (b[::1009] & 0xFFF0) | 3
            m.write_tensor(f"{name}.buckets", b)
        m.set_embed_scale(np.linspace(0.5, 2.0, 4096).astype(np.float32))
        check(O, ctx, m, BASE, 50, 0.25)
    finally:
        m.close()


@pytest.mark.parametrize("block", [2, 16])
def test_block_selection(O, ctx, model, block):
    ctx.set_selection_block(block, 2.0)
    try:
        check(O, ctx, model, BASE, 20, 0.25)
    finally:
        ctx.set_selection_block(1, 2.0)


def test_dense_head_and_continuation(O, iam, ctx, model):
    """The dense LM head's picks, and tokens decoded after the prompt equal to
    those after a prompt fed by steps."""
    head = ctx.upload(O.gen_f16(0, 21, 512 * 4096, 0.0, 0.02))
    prompt = O.gen_tokens(0, 6, 18, 512)
    model.set_lm_dense(head)
    try:
        model.reset_caches()
        got = model.generate(prompt, 6, 0.25)
        hist = model.read_tensor("history", np.int32)[1:24]
        model.reset_caches()
        log = ctx.empty(512, np.float32)
        seq = list(prompt)
        for pos in range(23):
            model.forward(int(seq[pos]), pos, 0.25, log)
            pick = O.argmax(log.read())
            assert hist[pos] == pick, pos
            if pos >= 17:
                seq.append(pick)
        assert list(got) == seq[18:24]
        log.free()
    finally:
        model.set_lm_dense(None)
        head.free()


def test_buffers_hold_the_bucket_head_after_the_dense_one(O, iam, ctx):
    """The prefill buffers, first allocated under the dense head, hold the
    bucket-layout head's partial sums, the widest here, afterwards."""
    cfg = dict(BASE, n_layers=1, vocab=32000)
    m = make(iam, ctx, n_layers=1, vocab=32000)
    head = ctx.upload(O.gen_f16(0, 22, 32000 * 4096, 0.0, 0.02))
    try:
        m.set_lm_dense(head)
        m.generate(O.gen_tokens(0, 7, 100, 32000), 1, 0.25)
        m.set_lm_dense(None)
        before = ctx.mem_status()[0]
        check(O, ctx, m, cfg, 100, 0.25)
        assert ctx.mem_status()[0] == before
    finally:
        m.close()
        head.free()


class Budget:
    """The context's memory budget set to a number of bytes.  There is no call
    for that: the field (after the device, the stream and the total) is written
    in place, and mem_status has to read it back."""

    def __init__(self, ctx):
        self.ctx = ctx
        self.field = ctypes.c_size_t.from_address(ctx.h.value + 24)
        self.usable = ctx.mem_status()[1]
        assert self.field.value == self.usable

    def set(self, n):
        self.field.value = n
        assert self.ctx.mem_status()[1] == n

    def __enter__(self):
        return self

    def __exit__(self, *a):
        self.set(self.usable)


def test_prefill_buffers_make_room(O, iam):
    """What a context without prefill buffers can allocate, it can allocate
    with them too (they are freed), and a prompt after that is as before."""
    with iam.Ctx(0) as ctx, Budget(ctx) as budget:
        m = make(iam, ctx, n_layers=1)
        bare = ctx.mem_status()[0]
        check(O, ctx, m, dict(BASE, n_layers=1), 60, 0.25)
        kept = ctx.mem_status()[0]
        assert kept > bare
        budget.set(kept + 4096)
        buf = ctx.alloc(kept - bare)
        assert ctx.mem_status()[0] == kept
        # no room now: by steps
        check(O, ctx, m, dict(BASE, n_layers=1), 60, 0.25)
        assert ctx.mem_status()[0] == kept
        buf.free()
        check(O, ctx, m, dict(BASE, n_layers=1), 60, 0.25)
        assert ctx.mem_status()[0] == kept
        m.close()
        assert ctx.mem_status()[0] < kept


@pytest.mark.parametrize("n", [65, 97])
def test_prefill_in_chunks_that_fit(O, iam, n):
    """Where the buffers of the whole prompt find no room, the prompt goes in
    smaller batches, and smaller buffers that are there already stay in use."""
    cfg = dict(BASE, n_layers=1)
    with iam.Ctx(0) as ctx, Budget(ctx) as budget:
        m = make(iam, ctx, n_layers=1)
        check(O, ctx, m, cfg, 33, 0.25)                     # buffers of two groups
        two = ctx.mem_status()[0]
        names = []

        def batched():
            ctx.profiling(False)
            names.append(ctx.kernel_stat("prefill.products")[1])

        budget.set(two + 4096)
        ctx.kernel_stats_reset()
        ctx.profiling(True)
        check(O, ctx, m, cfg, n, 0.25, after=lambda: (ctx.sync(), batched()))
        assert ctx.mem_status()[0] == two
        # a layer's four products and the head's, per batch of 32 tokens
        assert names[0] == 5 * ((n - 1) // 32)
        m.close()
