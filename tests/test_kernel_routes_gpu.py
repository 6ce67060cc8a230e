"""GPU tests (-m gpu) of kernels and dispatch rules at the sizes where they change hands: edges of tiles, remainders, the smallest and largest of a
route's range, against the oracle or against the general path of the same operation."""
import ctypes as C

import numpy as np
import pytest

import nvr_import
import oracle
from oracle import model_oracle as mo

nvr = nvr_import.load()
pytestmark = pytest.mark.gpu

F16 = np.float16


def dev(a):
    return nvr.DeviceBuffer.from_numpy(np.ascontiguousarray(a))


def _small(dtype, batch, **kw):
    m = mo.small()
    model = nvr.ModelConfig(vocab_size=m.vocab_size, hidden_size=m.hidden_size, intermediate_size=m.intermediate_size, num_hidden_layers=m.num_hidden_layers,
                            num_attention_heads=m.num_attention_heads, num_key_value_heads=m.num_key_value_heads, head_dim=m.head_dim,
                            max_position_embeddings=m.max_position_embeddings, rms_norm_eps=m.rms_norm_eps, rope_theta=m.rope_theta,
                            tie_word_embeddings=m.tie_word_embeddings, init_std=m.init_std, seed=m.seed)
    cfg = nvr.Config(skip_block_size_check=1, max_num_seqs=batch, max_num_batched_tokens=batch * 24, max_model_len=64, kvcache_block_size=16,
                     num_kvcache_blocks=4 * batch, dtype=dtype, **kw)
    return cfg, model, m.vocab_size


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("batch", [1, 33])
def test_execute_model_stores_the_logits_with_the_step_as_on_demand(dtype, batch):
    """execute_model of a greedy batch writes the f32 logits in the step's own LM head; an engine's step leaves them to a second launch on demand: same
    bits, same tokens, prefill and decode steps (eager and replayed), one row block and more."""
    cfg, model, vocab = _small(dtype, batch)
    prompts = [nvr.synthetic_tokens(3 + i % 17, 5, i, vocab) for i in range(batch)]
    sp = nvr.SamplingParams(temperature=0.0, max_tokens=6, ignore_eos=True)
    nvr.lib().nvr_seq_reset_id_counter()
    eng = nvr.LLMEngine(cfg, model)
    for p in prompts:
        eng.add_request(p, sp)
    want = []
    while not eng.is_finished():
        rec = eng.step()
        want.append((rec["tokens"], eng.model_runner.logits(batch).copy()))
    runner = nvr.ModelRunner(cfg, model)
    bm = nvr.BlockManager(4 * batch, 16)
    seqs = [nvr.Sequence(p, sp, 16) for p in prompts]
    for s in seqs:
        bm.allocate(s)
    for i, (tokens, logits) in enumerate(want):
        runner.execute_model(seqs, i == 0)
        assert runner.sample_tokens(seqs) == tokens, i
        assert np.array_equal(runner.logits(batch), logits), i
        for s, t in zip(seqs, tokens):
            s.append_token(t)
            bm.may_append(s)


@pytest.mark.parametrize("T,H,KVH,D,shift", [(1, 2, 2, 64, 0), (27, 16, 8, 128, 0), (65, 32, 8, 128, 0), (3, 3, 1, 256, 0), (5, 1, 1, 64, 0),    # the wide form: less than a round of lanes, several
                                             (7, 4, 2, 96, 0), (7, 4, 2, 32, 0), (27, 16, 8, 128, 1)])                                         # the general form: other heads, unaligned weights
def test_qk_norm_forms(T, H, KVH, D, shift):
    """nvr_qk_norm_rope_store_kv on both of its kernels (16-byte pieces of a head by neighbouring lanes; a wave per head) against the oracle's ops with
    their fp16 roundings: one rounding of each of n, the two products' difference and the store (3 ulps, as the operation's other test); slots, values."""
    rng = np.random.default_rng(T + D)
    N = (H + 2 * KVH) * D
    xb = (rng.standard_normal((T, N)) * 1.5).astype(F16)
    qw, kw = (1 + 0.3 * rng.standard_normal(D)).astype(F16), (1 + 0.3 * rng.standard_normal(D)).astype(F16)
    pos = rng.integers(0, 400, T).astype(np.int64)
    nslots = 2 * T + 4
    slots = rng.permutation(nslots)[:T].astype(np.int32)
    if T > 2:
        slots[2] = -1
    cos, sin = oracle.rope_table(D, 512, 1e6)
    d_x, d_pos, d_slots, d_cos, d_sin = dev(xb), dev(pos), dev(slots), dev(cos), dev(sin)
    d_qw, d_kw = dev(np.concatenate([np.zeros(shift, F16), qw])), dev(np.concatenate([np.zeros(shift, F16), kw]))
    d_kc, d_vc = nvr.DeviceBuffer(nslots * KVH * D * 2), nvr.DeviceBuffer(nslots * KVH * D * 2)
    d_kc.zero(); d_vc.zero()
    nvr.check(nvr.lib().nvr_qk_norm_rope_store_kv(d_x.ptr, d_pos.ptr, d_slots.ptr, T, H, KVH, D, d_cos.ptr, d_sin.ptr, d_qw.ptr + 2 * shift, d_kw.ptr + 2 * shift, 1e-6,
                                                  d_kc.ptr, d_vc.ptr, None))
    nvr.check(nvr.lib().nvr_device_synchronize())
    got = d_x.to_numpy((T, N), F16)
    x = xb.astype(np.float32)
    heads = []
    for w, a, n in ((qw, 0, H), (kw, H, KVH)):
        y = oracle.round_f16(oracle.rmsnorm(x[:, a * D:(a + n) * D].reshape(T * n, D), w.astype(np.float32), 1e-6)).reshape(T, n, D)
        heads.append(oracle.round_f16(oracle.rope_apply(y, pos, cos, sin)).reshape(T, n * D))
    ref = np.concatenate(heads + [x[:, (H + KVH) * D:]], 1)
    assert np.all(np.abs(got.astype(np.float32) - ref) <= 2e-3 + 3 * 2.0 ** -10 * np.abs(ref))
    kc, vc = d_kc.to_numpy((nslots, KVH * D), np.uint16), d_vc.to_numpy((nslots, KVH * D), np.uint16)
    bits = got.view(np.uint16)
    assert np.array_equal(bits[:, (H + KVH) * D:], xb.view(np.uint16)[:, (H + KVH) * D:])
    seen = np.zeros(nslots, bool)
    for t in range(T):
        if slots[t] >= 0:
            assert np.array_equal(kc[slots[t]], bits[t, H * D:(H + KVH) * D]) and np.array_equal(vc[slots[t]], bits[t, (H + KVH) * D:])
            seen[slots[t]] = True
    assert not kc[~seen].any() and not vc[~seen].any()


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("T,K,H,KVH", [(65, 1024, 16, 8), (97, 256, 16, 4), (200, 512, 8, 4), (509, 1024, 16, 8), (1000, 128, 16, 8), (1100, 1024, 5, 3), (2304, 256, 16, 8), (3062, 1024, 32, 8)])
def test_qkv_product_with_head_norms(T, K, H, KVH, dtype):
    """nvr_linear_qkv_norm_rope_store has the bits of nvr_linear_tiled with nvr_qk_norm_rope_store_kv behind it: tiles of 32, 64 and 128 rows, 256-row tiles, both in one product, ragged last
    tiles, a tile of q and k heads; rows without a slot, of zeros, with an infinity, of the largest numbers; k and v rows in the caches alone leave their columns of qkv as they were."""
    D, N, bf = 128, (H + 2 * KVH) * 128, dtype == "bfloat16"
    rng = np.random.default_rng(T * 7 + K)

    def bits(a):
        a = np.ascontiguousarray(a, np.float32)
        if not bf:
            return a.astype(F16).view(np.uint16)
        u = a.view(np.uint32)
        return ((u + 0x7fff + ((u >> 16) & 1)) >> 16).astype(np.uint16)
    x = rng.standard_normal((T, K)).astype(np.float32)
    x[3] = 0
    x[5, 0] = np.inf
    x[7] *= 1e4 if bf else 30.0
    x[T - 1] *= 1e-3
    xb, Wb = bits(x), bits(rng.standard_normal((N, K)) * K ** -0.5)
    qw, kw = bits(1 + 0.3 * rng.standard_normal(D)), bits(1 + 0.3 * rng.standard_normal(D))
    pos = rng.integers(0, 400, T).astype(np.int64)
    slots = rng.permutation(2 * T)[:T].astype(np.int32)
    slots[[2, T - 2]] = -1
    cos, sin = oracle.rope_table(D, 512, 1e6)
    l = nvr.lib()
    d_x, d_W, d_qw, d_kw, d_pos, d_slots, d_cos, d_sin = (dev(a) for a in (xb, Wb, qw, kw, pos, slots, cos, sin))
    d_Wt = nvr.DeviceBuffer(N * K * 2)
    nvr.check(l.nvr_ops_set_dtype(dtype.encode()))
    try:
        nvr.check(l.nvr_retile_weight(d_W.ptr, d_Wt.ptr, N, K, 0, H, KVH, D, None))
        out = []
        for form in range(4):                                              # two launches; one; one from W alone; one with k and v in the caches alone
            y, kc, vc = dev(np.full((T, N), 0x7b7b, np.uint16)), nvr.DeviceBuffer(2 * T * KVH * D * 2), nvr.DeviceBuffer(2 * T * KVH * D * 2)
            kc.zero(); vc.zero()
            if form == 0:
                nvr.check(l.nvr_linear_tiled(d_x.ptr, K, d_W.ptr, d_Wt.ptr, T, K, N, y.ptr, 0, None))
                nvr.check(l.nvr_qk_norm_rope_store_kv(y.ptr, d_pos.ptr, d_slots.ptr, T, H, KVH, D, d_cos.ptr, d_sin.ptr, d_qw.ptr, d_kw.ptr, 1e-6, kc.ptr, vc.ptr, None))
            else:
                nvr.check(l.nvr_linear_qkv_norm_rope_store(d_x.ptr, K, d_W.ptr, None if form == 2 else d_Wt.ptr, T, K, H, KVH, D, d_pos.ptr, d_slots.ptr, d_cos.ptr, d_sin.ptr, d_qw.ptr, d_kw.ptr, 1e-6,
                                                           y.ptr, kc.ptr, vc.ptr, int(form == 3), None))
            nvr.check(l.nvr_device_synchronize())
            out.append((y.to_numpy((T, N), np.uint16), kc.to_numpy((2 * T, KVH * D), np.uint16), vc.to_numpy((2 * T, KVH * D), np.uint16)))
        assert l.nvr_linear_qkv_norm_rope_store(d_x.ptr, K, d_W.ptr, None, 32, K, H, KVH, D, d_pos.ptr, d_slots.ptr, d_cos.ptr, d_sin.ptr, d_qw.ptr, d_kw.ptr, 1e-6, y.ptr, kc.ptr, vc.ptr, 0, None) == -10
    finally:
        nvr.check(l.nvr_ops_set_dtype(b"float16"))
    want = out[0]
    nan = 0x7f80 if bf else 0x7c00                                         # (a NaN is a NaN, whatever its bits)
    canon = [[np.where((a & 0x7fff) > nan, 0x7fff, a) for a in o] for o in out]
    for form in (1, 2):
        for a, b in zip(canon[form], canon[0]):
            assert np.array_equal(a, b), form
    assert np.array_equal(canon[3][0][:, :H * D], canon[0][0][:, :H * D]) and (out[3][0][:, H * D:] == 0x7b7b).all()
    assert np.array_equal(canon[3][1], canon[0][1]) and np.array_equal(canon[3][2], canon[0][2])
    assert (want[1].any(1) | want[2].any(1)).sum() <= T - 2 and np.isfinite(x).sum() == x.size - 1


@pytest.mark.parametrize("B,V", [(1, 65536), (1, 65535), (3, 151936), (1, 65539), (128, 65540), (129, 65540), (300, 64)])
def test_greedy_rows_cut_into_parts(B, V):
    """The greedy choice of f32 logits rows: cut into parts over the grid (few long rows) or one workgroup per row (short rows, or many of them), through a
    float32 runner whose LM head leaves no arg-max partials — compared with the first maximum of the logits it returns, with ties planted by a zero head."""
    for std in (0.02, 0.0):                                                # (0: every logit of a row is equal, the lowest index wins)
        model = nvr.ModelConfig(vocab_size=V, hidden_size=64, intermediate_size=64, num_hidden_layers=1, num_attention_heads=1, num_key_value_heads=1, head_dim=64,
                                max_position_embeddings=64, tie_word_embeddings=0, init_std=std, seed=3)
        runner = nvr.ModelRunner(nvr.Config(skip_block_size_check=1, max_num_seqs=B, max_num_batched_tokens=4 * B, max_model_len=16, kvcache_block_size=16,
                                            num_kvcache_blocks=B, dtype="float32"), model)
        bm = nvr.BlockManager(B, 16)
        seqs = [nvr.Sequence([(7 * i) % 64, i % 61], nvr.SamplingParams(temperature=0.0, ignore_eos=True), 16) for i in range(B)]
        for s in seqs:
            bm.allocate(s)
        runner.execute_model(seqs, True)
        tokens = runner.sample_tokens(seqs)
        assert tokens == runner.logits(B).argmax(1).tolist()


def _attn_meta(ctx, tables=None, max_blocks=0):
    m = nvr.AttnMetaC()
    d_ctx = dev(np.asarray(ctx, np.int32))
    m.context_lens, m.batch, m.max_context_len, m.max_blocks = d_ctx.ptr, len(ctx), max(ctx), max_blocks
    d_bt = None
    if tables is not None:
        d_bt = dev(np.asarray(tables, np.int32))
        m.block_tables = d_bt.ptr
    return m, (d_ctx, d_bt)


@pytest.mark.parametrize("H,KVH,D,ctx", [(2, 1, 64, [1, 127, 128, 129, 513]), (4, 4, 128, [1, 2, 128, 129, 256, 257, 700]), (2, 2, 192, [65, 64, 1]), (2, 1, 256, [63, 129, 300]),
                                         (4, 2, 128, [5, 300] * 70),                                    # four waves per row: the rows fill the chip
                                         (2, 1, 96, [1, 130])])                                         # the general form
def test_float32_decode_attention_forms(H, KVH, D, ctx):
    """The float32 paged decode attention at the edges of its rounds (4 keys x 32 or 16 groups, two rounds in flight) and in its general form, against the
    oracle's softmax in float64; shuffled blocks, stale table entries behind a context."""
    bs, B = 16, len(ctx)
    rng = np.random.default_rng(D + B)
    mb = max(-(-c // bs) for c in ctx) + 2
    nb = B * mb
    perm = rng.permutation(nb)
    tables = perm.reshape(B, mb).astype(np.int32)
    q = rng.standard_normal((B, H * D)).astype(np.float32)
    k, v = rng.standard_normal((nb, bs, KVH, D)).astype(np.float32), rng.standard_normal((nb, bs, KVH, D)).astype(np.float32)
    nvr.check(nvr.lib().nvr_ops_set_dtype(b"float32"))
    try:
        meta, keep = _attn_meta(ctx, tables, mb)
        d_q, d_k, d_v, out = dev(q), dev(k), dev(v), nvr.DeviceBuffer(B * H * D * 4)
        ws = nvr.DeviceBuffer(max(16, nvr.lib().nvr_paged_attn_workspace_bytes(B, H, D, max(ctx))))
        scale = float(D ** -0.5)
        nvr.check(nvr.lib().nvr_paged_attn_decode(d_q.ptr, H * D, d_k.ptr, d_v.ptr, C.byref(meta), H, KVH, D, bs, scale, out.ptr, ws.ptr, None))
        nvr.check(nvr.lib().nvr_device_synchronize())
        got = out.to_numpy((B, H, D), np.float32)
    finally:
        nvr.check(nvr.lib().nvr_ops_set_dtype(b"float16"))
    for b in range(B):
        kk = k[tables[b]].reshape(-1, KVH, D)[:ctx[b]].astype(np.float64)
        vv = v[tables[b]].reshape(-1, KVH, D)[:ctx[b]].astype(np.float64)
        for h in range(H):
            g = h // (H // KVH)
            s = kk[:, g] @ q[b, h * D:(h + 1) * D].astype(np.float64) * scale
            p = np.exp(s - s.max())
            ref = p @ vv[:, g] / p.sum()
            # a score is a sum of D products (error about sqrt(D) eps |q||k| scale), a weight moves by that much of itself, and the output by the weights' shares of |v|
            assert np.abs(got[b, h] - ref).max() <= 2e-5, (b, h)


@pytest.mark.parametrize("T", [9, 64, 65, 128, 200])
@pytest.mark.parametrize("hidden,inter", [(256, 512), (1024, 3072), (96, 160)])
def test_float32_prompt_products_cut_along_k(T, hidden, inter):
    """Prompts of the float32 path, whose o / down products are cut along k when their output tiles are few, against the oracle (f32): remainders of the
    K-tiles a step requests ahead (160 = 5 of 32), tiles of one and more rows, one layer."""
    heads = 1 if hidden == 96 else 2
    m = mo.ModelConfig(vocab_size=256, hidden_size=hidden, intermediate_size=inter, num_hidden_layers=1, num_attention_heads=heads, num_key_value_heads=heads,
                       head_dim=hidden // heads if hidden == 96 else 64, max_position_embeddings=256, rms_norm_eps=1e-6, rope_theta=1e4, tie_word_embeddings=True, init_std=0.05, seed=9)
    from oracle import engine_oracle as eo
    eo.reset_sequence_counter(); nvr.lib().nvr_seq_reset_id_counter()
    ecfg = dict(max_num_seqs=1, max_num_batched_tokens=256, max_model_len=256, kvcache_block_size=16, num_kvcache_blocks=16)
    model = nvr.ModelConfig(vocab_size=256, hidden_size=hidden, intermediate_size=inter, num_hidden_layers=1, num_attention_heads=heads, num_key_value_heads=heads,
                            head_dim=m.head_dim, max_position_embeddings=256, rms_norm_eps=1e-6, rope_theta=1e4, tie_word_embeddings=1, init_std=0.05, seed=9)
    o = mo.OracleEngine(m, eo.Config(**ecfg), fp16=False, bf16=False, max_pos=256)
    p = nvr.LLMEngine(nvr.Config(skip_block_size_check=1, dtype="float32", **ecfg), model)
    prompt = nvr.synthetic_tokens(T, 3, 1, 256).tolist()
    o.add_request(prompt, eo.SamplingParams(temperature=0.0, max_tokens=1, ignore_eos=True))
    p.add_request(prompt, nvr.SamplingParams(temperature=0.0, max_tokens=1, ignore_eos=True))
    rec = p.step()
    orec = o.step(forced_tokens=rec["tokens"])
    assert np.abs(p.model_runner.logits(1) - orec["logits"]).max() < 2e-4


@pytest.mark.parametrize("hidden,inter,heads,kv,dim", [(1024, 3072, 16, 8, 128),       # o / down in 8 segments of k
                                                       (512, 1024, 4, 2, 64),          # in 1 and 4
                                                       (768, 2560, 4, 1, 192)])        # in 2 and 4; heads of three pieces
def test_float32_prompt_rows_have_the_same_bits_in_every_step(hidden, inter, heads, kv, dim):
    """A float32 prompt alone, in portions, beside another prompt and in engines of other sizes: steps of few and many rows, whose products' segments run apart or one after the other and whose
    rows' keys are shared by eight waves or four.  The last row's logits have the same bits (portions of more than 8 rows: fewer run the decode step's products)."""
    model = nvr.ModelConfig(vocab_size=256, hidden_size=hidden, intermediate_size=inter, num_hidden_layers=2, num_attention_heads=heads, num_key_value_heads=kv, head_dim=dim,
                            max_position_embeddings=2048, rms_norm_eps=1e-6, rope_theta=1e4, tie_word_embeddings=0, init_std=hidden ** -0.5, seed=5)
    sp = nvr.SamplingParams(temperature=0.0, ignore_eos=True)

    def last_row(lengths, cuts=(), budget=4096, seqs=2):
        r = nvr.ModelRunner(nvr.Config(skip_block_size_check=1, max_num_seqs=seqs, max_num_batched_tokens=budget, max_model_len=2048, kvcache_block_size=16, num_kvcache_blocks=256,
                                       dtype="float32", enable_chunked_prefill=1), model)
        bm = nvr.BlockManager(256, 16)
        group = [nvr.Sequence(nvr.synthetic_tokens(L, 6, i, 256), sp, 16) for i, L in enumerate(lengths)]
        for s in group:
            bm.allocate(s)
        done = 0
        for c in cuts:                                                       # portions of the first prompt, alone
            group[0].set_chunk(done, c - done)
            r.execute_model(group[:1], True)
            done = c
        if cuts:
            group[0].set_chunk(done, lengths[0] - done)
        r.execute_model(group, True)
        return r.logits(len(group))[0].copy()
    for T in (33, 200, 700):
        whole = last_row([T])
        assert np.isfinite(whole).all() and whole.std() > 0
        for other in (dict(lengths=[T], cuts=[9]), dict(lengths=[T], cuts=[T - 20]), dict(lengths=[T], cuts=[T // 3, 2 * T // 3]), dict(lengths=[T, 300]), dict(lengths=[T, 900], cuts=[T - 9]),
                      dict(lengths=[T], budget=max(T, 64), seqs=1)):
            assert np.array_equal(last_row(**other), whole), (T, other)


@pytest.mark.parametrize("W,taps,heads,kv,dim,lengths", [(64, 1, 4, 2, 64, [1, 31, 32]), (1024, 4, 2, 1, 64, [33, 127]), (1040, 4, 4, 1, 128, [30, 255, 256]), (2080, 8, 4, 4, 64, [3, 129]),
                                                         (4160, 3, 4, 2, 64, [5]), (96, 9, 2, 2, 64, [40, 7]), (256, 4, 4, 2, 64, [20] * 64), (256, 4, 4, 2, 64, [20] * 66)])
def test_layer_list_decode_steps(W, taps, heads, kv, dim, lengths):
    """Decode steps of the distance-penalty design in bfloat16: the output product cut along k, the join with the next norm and convolution in one launch (widths of one piece per thread to
    four, one tap to eight) or apart (beyond), attention with the penalty table over few query rows at the edges of its chunks, batches of the parts' rows and above them — against the float64 restatement; every row is looked at."""
    import rugudra_util as u
    cfg = u.make_config([u.attention_layer(heads, kv, dim, dim, ff=256), u.retention_layer(2, 32, 32, ff=None), u.attention_layer(heads, kv, dim, dim, ff=64)], width=W, taps=taps)
    w = u.make_weights(cfg, seed=W + taps)
    n = len(lengths)
    d = u.Driver(cfg, w, dtype="bfloat16", slots=n, pages=n * 20, max_tokens=max(512, sum(lengths)), max_len=512)
    rng = np.random.default_rng(taps)
    base = [rng.integers(0, 97, L + 3) for L in lengths[:3]]
    tokens = [base[i % 3] for i in range(n)]
    d.step([("s%d" % i, t[:L]) for i, (t, L) in enumerate(zip(tokens, lengths))])
    got = [d.step([("s%d" % i, t[L + k:L + k + 1]) for i, (t, L) in enumerate(zip(tokens, lengths))]) for k in range(3)]
    _compare_layer_rows(cfg, w, "bfloat16", base, [np.concatenate([g["s%d" % i] for g in got]) for i in range(n)])


def _compare_layer_rows(cfg, w, dtype, base, rows):
    """rows[i]: a request's last logits, its tokens base[i % 3].  The first three against the float64 restatement, row by row; every further row has the bits of the request it repeats (a row's
    sums do not depend on its place in the batch).  bfloat16: a row may be three times as far off as the worst of four draws in which every weight moves by a rounding of its own size — where a
    retention head's output nearly cancels, its norm magnifies both alike (measured: 0.5 of it in the middle, 1.07 at the worst; a wrong key, row or part is off at the order of 1)."""
    import rugudra_util as u
    for i, t in enumerate(base):
        n = len(rows[i])
        want = u.expected_logits(cfg, w, t)
        err = u.row_errors(rows[i], want[-n:])
        bound = u.TOL["float32"] / 2
        if dtype == "bfloat16":
            moved = []
            for seed in range(4):
                rng = np.random.default_rng(100 + seed)
                v = {k: np.asarray(x, np.float64) * (1 + 2.0 ** -9 * rng.standard_normal(np.shape(x))) for k, x in w.items()}
                moved.append(u.row_errors(u.expected_logits(cfg, v, t)[-n:], want[-n:]))
            bound = 3 * np.max(moved, axis=0)
        assert np.all(err < bound), (i, err, bound)
    for i in range(3, len(rows)):
        assert np.array_equal(rows[i], rows[i % 3]), i


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("hidden,inter,heads,kv,dim,qk_norm", [(256, 512, 4, 2, 64, 0), (1024, 1024, 8, 8, 128, 1), (2048, 512, 8, 4, 128, 0), (256, 512, 4, 1, 128, 1), (384, 512, 4, 2, 64, 0)])
def test_decode_steps_of_one_and_two_rows_against_more(dtype, hidden, inter, heads, kv, dim, qk_norm):
    """One or two sequences (add + norm inside the products behind them, where the width is a multiple of 256) give the logits that the same sequences give in a batch of three (launches of
    their own): sums in another order, so within the 16-bit rounding of three layers; contexts on both sides of the 256 keys a single workgroup takes."""
    model = nvr.ModelConfig(vocab_size=192, hidden_size=hidden, intermediate_size=inter, num_hidden_layers=3, num_attention_heads=heads, num_key_value_heads=kv, head_dim=dim,
                            max_position_embeddings=512, rms_norm_eps=1e-6, rope_theta=1e4, tie_word_embeddings=0, init_std=hidden ** -0.5, seed=11, qk_norm=qk_norm)
    sp = nvr.SamplingParams(temperature=0.0, ignore_eos=True)
    lengths = [16, 127, 300]
    prompts = [nvr.synthetic_tokens(L + 4, 4, i, 192) for i, L in enumerate(lengths)]

    def steps(which):
        r = nvr.ModelRunner(nvr.Config(skip_block_size_check=1, max_num_seqs=3, max_num_batched_tokens=512, max_model_len=512, kvcache_block_size=16, num_kvcache_blocks=64, dtype=dtype), model)
        bm = nvr.BlockManager(64, 16)
        seqs = [nvr.Sequence(prompts[i][:lengths[i]], sp, 16) for i in which]
        for s in seqs:
            bm.allocate(s)
        r.execute_model(seqs, True)
        out = []
        for k in range(4):
            for i, s in zip(which, seqs):
                s.append_token(int(prompts[i][lengths[i] + k]))
                bm.may_append(s)
            r.execute_model(seqs, False)
            out.append(r.logits(len(which)).copy())
        return np.stack(out, 1)                                            # [sequence, step, vocabulary]
    full = steps([0, 1, 2])
    # a sum in another order crosses a rounding of half an ulp here and there, eight places a layer on the residual stream: sqrt(24) * 2^-12 / sqrt(3) relative (float16) if all of them did;
    # three times that for a row's norm, and for its largest of 192 logits four times its norm (measured, float16: 0.0012 and 0.0038; bfloat16, eight times as coarse: 0.0094 and 0.030)
    row = 3 * 24 ** 0.5 * 2.0 ** (-12 if dtype == "float16" else -9) / 3 ** 0.5
    rms = np.sqrt((full ** 2).mean(-1, keepdims=True))
    for which in ([0], [1], [2], [0, 1], [1, 2]):
        d = (steps(which) - full[which]) / rms[which]
        assert np.sqrt((d ** 2).mean(-1)).max() < row and np.abs(d).max() < 4 * row, which


@pytest.mark.parametrize("B,G,KVH,D,bs,ctx", [
    (40, 2, 8, 128, 256, [1 + (577 * i) % 1900 for i in range(40)]),                       # ragged: many queries to a share, long ones cut
    (300, 1, 1, 64, 8, [1, 63, 64, 65, 300] * 60),                                         # one kv head, the smallest block, shares of one or two units
    (130, 8, 2, 64, 16, [1 + 2 * i for i in range(130)]),                                  # the widest group
    (90, 4, 3, 128, 64, [0 if i % 7 == 3 else 1 + (311 * i) % 700 for i in range(90)]),    # 3 kv heads do not divide the CUs; queries without keys
    (33, 2, 8, 128, 16, [5000] + [1] * 32),                                                # one long query: shares that end inside the charge of a short one
])
def test_work_balanced_attention_against_the_per_pair_form(B, G, KVH, D, bs, ctx):
    """Equal shares of all queries' keys (each query charged two units for its start) against a workgroup per pair, over the same cache: both keep f32 scores,
    weights and sums and round once, so their outputs differ by one rounding of the result and the order of f32 sums of up to 5000 terms — 2 ulps of float16."""
    _work_balanced_against_per_pair(B, G, KVH, D, bs, ctx, max(ctx), 1)


@pytest.mark.parametrize("B,G,KVH,D,bs,ctx", [
    (300, 2, 1, 64, 8, [128 if i % 30 == 0 else 0 for i in range(300)]),                   # 40 units, 256 shares: a cut query's units lay in shares 19 and 25
    (300, 1, 1, 128, 16, [[0, 256, 1, 129, 192][i % 97 % 5] if i % 97 < 5 else 0 for i in range(300)]),
    (270, 4, 1, 64, 16, [0] * 269 + [256]),                                                # one query: all units are its own
    (100, 2, 3, 64, 8, [65 if i == 50 else 0 for i in range(100)]),
    (260, 2, 1, 64, 8, [0] * 260),
])
def test_work_balanced_attention_of_few_queries_with_keys(B, G, KVH, D, bs, ctx):
    """Fewer units of keys than shares: every cut query is merged by its last share and its counter returns to zero, so that a second launch over the same counters does the same."""
    _work_balanced_against_per_pair(B, G, KVH, D, bs, ctx, 256, 2)


def _work_balanced_against_per_pair(B, G, KVH, D, bs, ctx, bound, launches):
    l = nvr.lib()
    rng = np.random.default_rng(B + D)
    H, blocks = G * KVH, [(c + bs - 1) // bs for c in ctx]
    mb, nb, o = max(blocks) + 1, max(sum(blocks), 1), 0
    perm = rng.permutation(nb)
    bt = np.full((B, mb), -1, np.int32)
    for b, n in enumerate(blocks):
        bt[b, :n] = perm[o:o + n]; o += n
    k, v = (dev(rng.standard_normal((nb, bs, KVH, D)).astype(F16).view(np.uint16)) for _ in range(2))
    q = dev(rng.standard_normal((B, H, D)).astype(F16).view(np.uint16))
    d_ctx, d_bt, tickets = dev(np.asarray(ctx, np.int32)), dev(bt), dev(np.zeros(B * KVH, np.uint32))
    meta = nvr.AttnMetaC()
    meta.context_lens, meta.block_tables, meta.max_blocks, meta.batch, meta.max_context_len = d_ctx.ptr, d_bt.ptr, mb, B, bound
    ws = nvr.DeviceBuffer(l.nvr_paged_attn_workspace_bytes(B, H, D, bound))
    ref, got = nvr.DeviceBuffer(B * H * D * 2), nvr.DeviceBuffer(B * H * D * 2)
    args = (q.ptr, H * D, k.ptr, v.ptr, C.byref(meta), H, KVH, D, bs, D ** -0.5)
    nvr.check(l.nvr_paged_attn_decode(*args, ref.ptr, ws.ptr, None))
    a = ref.to_numpy((B, H, D), F16).astype(np.float32)
    for _ in range(launches):
        nvr.check(l.nvr_fill_const(got.ptr, B * H * D, C.c_float(float("nan")), None))
        nvr.check(l.nvr_paged_attn_decode_fused(*args, got.ptr, ws.ptr, tickets.ptr, None))
        b = got.to_numpy((B, H, D), F16).astype(np.float32)
        assert np.all(np.abs(a - b) <= 2 * np.maximum(np.spacing(np.abs(a).astype(F16)).astype(np.float32), 2.0 ** -14 / 8)), np.abs(a - b).max()
        assert not tickets.to_numpy((B * KVH,), np.uint32).any()


@pytest.mark.parametrize("B,G,KVH,D,bs,ctx,bound", [
    (1, 2, 8, 128, 256, [136], 136),
    (5, 1, 2, 64, 16, [1, 15, 128, 129, 136], 136),
    (6, 4, 2, 128, 24, [127, 24, 136, 130, 48, 2], 136),                                   # blocks that are no multiple of a chunk's 16 keys
    (9, 2, 3, 64, 5, [136, 7, 129, 128, 64, 65, 10, 113, 1], 136),
    (16, 2, 8, 128, 48, [100 + i for i in range(16)], 130),                                # the most pairs of a round's contexts
    (17, 2, 8, 128, 16, [240 + i % 17 for i in range(17)], 256),                           # from here on whole buckets
    (23, 8, 8, 64, 24, [1 + 11 * i for i in range(23)], 256),
    (191, 8, 1, 128, 32, [1 + (37 * i) % 256 for i in range(191)], 256),
    (16, 2, 8, 128, 16, [137 + i for i in range(16)], 256),                                # beside the rule: longer contexts of few pairs, groups of 8, more pairs
    (2, 8, 2, 64, 16, [100, 136], 136),
    (24, 1, 8, 64, 16, [130] * 24, 136),
])
def test_brief_decode_attention_against_partitions(B, G, KVH, D, bs, ctx, bound):
    """Contexts that one workgroup per pair takes without partitions, and their neighbours, against the same call with a bound that cuts them into partitions: f32 sums in another order and one
    rounding, 2 ulps of float16 as above."""
    l = nvr.lib()
    rng = np.random.default_rng(B + D)
    H, blocks = G * KVH, [(c + bs - 1) // bs for c in ctx]
    mb, perm, o = max(blocks) + 1, rng.permutation(sum(blocks)), 0
    bt = np.full((B, mb), -1, np.int32)
    for b, n in enumerate(blocks):
        bt[b, :n] = perm[o:o + n]; o += n
    k, v = (dev(rng.standard_normal((sum(blocks), bs, KVH, D)).astype(F16).view(np.uint16)) for _ in range(2))
    q = dev(rng.standard_normal((B, H, D)).astype(F16).view(np.uint16))
    d_ctx, d_bt, tickets = dev(np.asarray(ctx, np.int32)), dev(bt), dev(np.zeros(B * KVH, np.uint32))
    out = []
    for most in (bound, 2048):
        meta = nvr.AttnMetaC()
        meta.context_lens, meta.block_tables, meta.max_blocks, meta.batch, meta.max_context_len = d_ctx.ptr, d_bt.ptr, mb, B, most
        ws, got = nvr.DeviceBuffer(l.nvr_paged_attn_workspace_bytes(B, H, D, most)), nvr.DeviceBuffer(B * H * D * 2)
        nvr.check(l.nvr_fill_const(got.ptr, B * H * D, C.c_float(float("nan")), None))
        nvr.check(l.nvr_paged_attn_decode_fused(q.ptr, H * D, k.ptr, v.ptr, C.byref(meta), H, KVH, D, bs, D ** -0.5, got.ptr, ws.ptr, tickets.ptr, None))
        out.append(got.to_numpy((B, H, D), F16).astype(np.float32))
        assert not tickets.to_numpy((B * KVH,), np.uint32).any()
    a, b = out
    assert np.all(np.abs(a - b) <= 2 * np.maximum(np.spacing(np.abs(b).astype(F16)).astype(np.float32), 2.0 ** -14 / 8)), np.abs(a - b).max()


@pytest.mark.parametrize("B,G,KVH,bs,P,own", [
    (3, 2, 8, 64, 1, [4300, 10, 0]),                                                       # own blocks past the 64 a wave holds; one sequence a workgroup, waves without a chunk of the prefix
    (32, 1, 8, 128, 3, [(5 * i) % 40 for i in range(32)]),
    (33, 2, 8, 256, 2, [1 + 8 * i for i in range(33)]),                                     # two sequences a workgroup, the last one alone
    (65, 4, 8, 64, 7, [(17 * i) % 150 for i in range(65)]),                                 # four, 16 rows
    (101, 4, 8, 128, 12, [3] * 101),                                                       # the longest prefix of the one launch
    (131, 2, 8, 64, 5, [(29 * i) % 90 for i in range(131)]),                                # eight
    (256, 1, 8, 64, 24, [64 + i % 3 for i in range(256)]),
    (2047, 2, 1, 64, 1, [i % 7 for i in range(2047)]),                                     # one kv head
    (129, 4, 8, 64, 2, [40] * 129), (40, 2, 8, 64, 25, [9] * 40),                           # beside the rule: more workgroups than CUs, a longer prefix
    (2, 2, 8, 64, 4, [256, 0]), (2, 2, 8, 64, 4, [257, 1]), (12, 4, 8, 128, 4, [384] + [5] * 11), (12, 4, 8, 128, 4, [385] + [5] * 11),     # both sides of the rule: one sequence a workgroup
    (33, 2, 8, 64, 8, [192] + [31] * 32), (64, 4, 8, 64, 16, [1 + (3 * i) % 96 for i in range(64)]), (64, 1, 8, 64, 16, [97] * 64),          # two
    (65, 4, 8, 64, 7, [(17 * i) % 97 for i in range(65)]), (127, 2, 8, 256, 4, [48] * 127), (66, 2, 8, 64, 2, [97] * 66),                   # four
    (131, 2, 8, 64, 5, [(29 * i) % 65 for i in range(131)]), (255, 1, 8, 64, 16, [32] * 255), (255, 1, 8, 64, 16, [33] * 255),              # eight
])
def test_shared_prefix_decode_attention_in_one_launch(B, G, KVH, bs, P, own):
    """Shared and own keys of a batch in one launch (1, 2, 4 and 8 sequences a workgroup, groups of 1, 2 and 4) against the plain kernel on the same inputs: f32 sums in another order, the prefix's
    weights rounded to float16, one rounding (3 ulps, as the two launches' test)."""
    l, D, H = nvr.lib(), 128, G * KVH
    rng = np.random.default_rng(B + P)
    S, blocks = P * bs, [(o + bs - 1) // bs for o in own]
    mb, pool = P + max(blocks) + 1, P + sum(blocks)
    perm, at = rng.permutation(pool), P
    bt = np.full((B, mb), -1, np.int32)
    for b in range(B):
        bt[b, :P] = perm[:P]
        bt[b, P:P + blocks[b]] = perm[at:at + blocks[b]]
        at += blocks[b]
    q = rng.standard_normal((B, H, D)).astype(F16)
    k, v = (rng.standard_normal((pool, bs, KVH, D)).astype(F16) for _ in range(2))
    k[perm[P - 1], -1] = 3 * q[0].reshape(KVH, G, D)[:, 0]                 # a prefix whose last key outweighs the rest for some rows
    d_q, d_k, d_v, d_bt, d_ctx = dev(q), dev(k), dev(v), dev(bt), dev(np.asarray([S + o for o in own], np.int32))
    meta = nvr.AttnMetaC()
    meta.context_lens, meta.block_tables, meta.max_blocks, meta.batch, meta.max_context_len = d_ctx.ptr, d_bt.ptr, mb, B, S + max(own)
    ws = nvr.DeviceBuffer(l.nvr_paged_attn_workspace_bytes(B, H, D, S + max(own) + bs))
    a, b = nvr.DeviceBuffer(B * H * D * 2), nvr.DeviceBuffer(B * H * D * 2)
    nvr.check(l.nvr_fill_const(b.ptr, B * H * D, C.c_float(float("nan")), None))
    nvr.check(l.nvr_paged_attn_decode(d_q.ptr, H * D, d_k.ptr, d_v.ptr, C.byref(meta), H, KVH, D, bs, D ** -0.5, a.ptr, ws.ptr, None))
    nvr.check(l.nvr_paged_attn_decode_shared(d_q.ptr, H * D, d_k.ptr, d_v.ptr, C.byref(meta), H, KVH, D, bs, D ** -0.5, S, None, None, None, b.ptr, ws.ptr, None))
    x, y = a.to_numpy((B, H, D), F16).astype(np.float32), b.to_numpy((B, H, D), F16).astype(np.float32)
    assert np.all(np.abs(x - y) <= 1e-3 + 3 * 2.0 ** -10 * np.abs(x)), np.abs(x - y).max()


@pytest.mark.parametrize("B,G,KVH,P", [(33, 2, 8, 5), (64, 4, 8, 9), (40, 1, 8, 4), (150, 2, 8, 8)])
@pytest.mark.parametrize("masked", ["first", "one_wave", "prefix", "everything", "nan_query"])
def test_shared_prefix_decode_attention_with_infinities(B, G, KVH, P, masked):
    """Keys of score -inf among the shared ones (the first 32, all of one wave's chunks, the whole prefix; everything: zeros, as the other decode kernels leave), and a query of NaN (zeros) beside others
    that must not notice: against 64 bits, with the bound of the test above for the rounding of the prefix's weights and of the result."""
    l, D, H, bs = nvr.lib(), 128, G * KVH, 64
    rng = np.random.default_rng(B + P)
    S, own = P * bs, [(7 * i) % 60 + 1 for i in range(B)]
    pool = P + B
    bt = np.zeros((B, P + 1), np.int32)
    bt[:, :P], bt[:, P] = np.arange(P), P + np.arange(B)
    q = rng.standard_normal((B, H, D)).astype(F16)
    q[..., 0] = 1
    k, v = (rng.standard_normal((pool, bs, KVH, D)).astype(F16) for _ in range(2))
    keys = k.reshape(pool * bs, KVH, D)
    if masked == "first":
        keys[:32, :, 0] = -np.inf
    elif masked == "one_wave":
        for x in range(3, S // 32, 8):
            keys[x * 32:x * 32 + 32, :, 0] = -np.inf
    elif masked == "prefix":
        keys[:S, :, 0] = -np.inf
    elif masked == "everything":
        keys[..., 0] = -np.inf
    want = np.zeros((B, H, D))
    for b in range(B):
        rows = np.concatenate([np.arange(S), (P + b) * bs + np.arange(own[b])])
        kb, vb = keys[rows].astype(np.float64), v.reshape(pool * bs, KVH, D)[rows].astype(np.float64)
        for g in range(KVH):
            sc = q[b, g * G:(g + 1) * G].astype(np.float64) @ kb[:, g].T * D ** -0.5
            m = sc.max(1, keepdims=True)
            if np.isfinite(m).all():
                w = np.exp(sc - m)
                want[b, g * G:(g + 1) * G] = w / w.sum(1, keepdims=True) @ vb[:, g]
    if masked == "nan_query":
        q[1, 0] = np.nan
        want[1, 0] = 0
    d_q, d_k, d_v, d_bt, d_ctx = dev(q), dev(k), dev(v), dev(bt), dev(np.asarray([S + o for o in own], np.int32))
    meta = nvr.AttnMetaC()
    meta.context_lens, meta.block_tables, meta.max_blocks, meta.batch, meta.max_context_len = d_ctx.ptr, d_bt.ptr, P + 1, B, S + max(own)
    ws = nvr.DeviceBuffer(l.nvr_paged_attn_workspace_bytes(B, H, D, S + bs))
    out = nvr.DeviceBuffer(B * H * D * 2)
    nvr.check(l.nvr_fill_const(out.ptr, B * H * D, C.c_float(float("nan")), None))
    nvr.check(l.nvr_paged_attn_decode_shared(d_q.ptr, H * D, d_k.ptr, d_v.ptr, C.byref(meta), H, KVH, D, bs, D ** -0.5, S, None, None, None, out.ptr, ws.ptr, None))
    got = out.to_numpy((B, H, D), F16).astype(np.float64)
    assert np.all(np.abs(got - want) <= 1e-3 + 3 * 2.0 ** -10 * np.abs(want)), np.nanmax(np.abs(got - want))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads,vdim,ff,batch", [(1, 30, 48, 1), (3, 32, 48, 16), (5, 4, 64, 17), (2, 64, 2064, 32), (4, 96, 40, 33)])
def test_layer_list_gated_head_norm_and_clamped_unit(dtype, heads, vdim, ff, batch):
    """A retention layer's gated head norm by a wave per head (head widths that are multiples of 4, head counts that leave waves without a head) and by the general form, and the clamped unit in
    its product's epilogue (up to 32 rows: one and two blocks of 16, few and many column tiles) or behind it, against the float64 restatement; every row is looked at."""
    import rugudra_util as u
    cfg = u.make_config([u.retention_layer(heads, 32, vdim, ff=ff), u.attention_layer(2, 1, 64, 64, ff=ff)], width=64, taps=4)
    w = u.make_weights(cfg, seed=heads + vdim)
    d = u.Driver(cfg, w, dtype=dtype, slots=batch, pages=batch * 2, max_tokens=max(64, 9 * batch), max_len=64)
    rng = np.random.default_rng(ff)
    base = [rng.integers(0, 97, 8 + i) for i in range(min(batch, 3))]
    tokens = [base[i % 3] for i in range(batch)]
    d.step([("s%d" % i, t[:-2]) for i, t in enumerate(tokens)])
    got = [d.step([("s%d" % i, t[len(t) - 2 + k:len(t) - 1 + k]) for i, t in enumerate(tokens)]) for k in range(2)]
    _compare_layer_rows(cfg, w, dtype, base, [np.concatenate([g["s%d" % i] for g in got]) for i in range(batch)])


@pytest.mark.parametrize("width,ff,batch,tokens", [(64, 2112, 3, 24), (64, 2112, 9, 34), (128, 2176, 5, 140), (1024, 3072, 24, 96)])
def test_layer_list_clamped_unit_on_tiles(width, ff, batch, tokens):
    """The clamped unit in the epilogue of 32-, 64-, 128- and 256-row tiles, against the float64 restatement: prompts of slightly different lengths in one step, every row of it."""
    import rugudra_util as u
    cfg = u.make_config([u.retention_layer(2, 32, 32, ff=ff), u.attention_layer(2, 1, 64, 64, ff=ff)], width=width, taps=4)
    w = u.make_weights(cfg, seed=ff + width)
    d = u.Driver(cfg, w, dtype="bfloat16", slots=batch, pages=batch * (tokens // 16 + 2), max_tokens=batch * (tokens + 2), max_len=256)
    rng = np.random.default_rng(batch)
    base = [rng.integers(0, 97, tokens + i) for i in range(3)]
    got = d.step([("s%d" % i, base[i % 3]) for i in range(batch)])
    _compare_layer_rows(cfg, w, "bfloat16", base, [got["s%d" % i] for i in range(batch)])


@pytest.mark.parametrize("width,ff,batch,tokens", [(64, 2112, 9, 34), (256, 2176, 3, 300), (1024, 3072, 40, 100), (256, 2176, 22, 303)])      # (the last two: 384 and 459 tiles of 256 rows)
def test_layer_list_clamped_unit_does_not_depend_on_the_step(width, ff, batch, tokens):
    """A row's clamped unit in a prompt step (on 32- to 256-row tiles, one and several of them a workgroup) and in portions of up to 32 rows: bit for bit.  Every product of the model has one term (the mixer's output none), so that the
    order of its sums does not matter; half of the stream's columns hold the token's embedding, the others the unit and nothing else, scaled until its smallest values (gates down to -12) count."""
    import rugudra_util as u
    half, limit = width // 2, 7.0
    cfg = u.make_config([u.retention_layer(2, 32, 32, ff=ff, limit=limit)], width=width, taps=2, embedding_scale=1.0, residual_mult=1.0)
    w = u.make_weights(cfg, seed=width)
    rng = np.random.default_rng(ff)
    w["embed"][:, half:] = 0
    w["l0.mix.o"][:] = 0
    for name, scale in (("l0.mlp.gate", 4.0), ("l0.mlp.up", 2.0)):
        w[name][:] = 0
        w[name][np.arange(ff), rng.integers(0, half, ff)] = scale * rng.choice([-1.0, 1.0], ff)
    w["l0.mlp.down"][:] = 0
    w["l0.mlp.down"][np.arange(half, width), rng.permutation(ff)[:half]] = 2.0 ** 20
    w["head"][:] = 0
    w["head"][np.arange(97), half + np.arange(97) * 7 % half] = 1
    base = [rng.integers(0, 97, tokens) for _ in range(batch)]
    rows = []
    for portion in (tokens, 32):
        d = u.Driver(cfg, w, dtype="bfloat16", slots=batch, pages=batch * (tokens // 16 + 2), max_tokens=batch * tokens, max_len=512)
        if portion == tokens:
            got = d.step([("s%d" % i, t) for i, t in enumerate(base)])
            rows.append(np.concatenate([got["s%d" % i] for i in range(batch)]))
        else:
            rows.append(np.concatenate([d.run_alone(t, cuts=[portion]) for t in base]))
    assert np.abs(rows[0]).max() > 0 and np.array_equal(rows[0].view(np.uint32), rows[1].view(np.uint32)), (rows[0] != rows[1]).mean()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("taps,width,batch", [(2, 64, 130), (3, 1028, 3), (4, 64, 130), (4, 1088, 9), (5, 64, 130)])
def test_layer_list_norm_and_convolution_rows(dtype, taps, width, batch):
    """Norm and convolution of chunks of many rows by 16, 4 and one row per workgroup, with the rows behind kept in registers (2 to 4 taps) and not: sequences that begin, end and go on in the
    middle of a workgroup's rows, chunks shorter than the taps, a second chunk behind the history of the first; against the float64 restatement."""
    import rugudra_util as u
    cfg = u.make_config([u.retention_layer(3, 32, 36, ff=48)], width=width, taps=taps)
    w = u.make_weights(cfg, seed=taps + width)
    d = u.Driver(cfg, w, dtype=dtype, slots=batch, pages=batch * 6, max_tokens=batch * 48, max_len=128)
    rng = np.random.default_rng(taps)
    base = [rng.integers(0, 97, n) for n in (33, 46, 37)]
    cuts = [(0, c, len(t)) for c, t in zip((32, 1, 34), base)]
    got = [[], []]
    for k in range(2):
        got[k] = d.step([("s%d" % i, base[i % 3][cuts[i % 3][k]:cuts[i % 3][k + 1]]) for i in range(batch)])
    _compare_layer_rows(cfg, w, dtype, base, [np.concatenate([g["s%d" % i] for g in got]) for i in range(batch)])


@pytest.mark.parametrize("batch", [1, 16, 17, 32, 33, 130])
@pytest.mark.parametrize("vocab", [112, 100, 4112])
def test_layer_list_head_and_greedy_choice(vocab, batch):
    """Logits and greedy choice of a layer list whose head runs on the dense graph's (widths and vocabularies it takes, 1 .. 130 rows) or as a plain product (a vocabulary of 100), first step and
    replays: logits against the float64 restatement, tokens the first maximum of the logits."""
    import rugudra_util as u
    cfg = u.make_config([u.retention_layer(2, 32, 32, ff=64)], width=256, taps=2)
    cfg["vocab"] = vocab
    w = u.make_weights(cfg, seed=vocab)
    d = u.Driver(cfg, w, dtype="bfloat16", slots=batch, pages=batch * 2, max_tokens=max(64, 9 * batch), max_len=64)
    rng = np.random.default_rng(vocab)
    base = [rng.integers(0, vocab, 6 + i) for i in range(min(batch, 3))]
    names = ["s%d" % i for i in range(batch)]
    d.step([(n, base[i % 3][:-3]) for i, n in enumerate(names)])
    rows = [[] for _ in names]
    for k in range(3):
        logits = d.step([(n, base[i % 3][len(base[i % 3]) - 3 + k:][:1]) for i, n in enumerate(names)])
        seqs = [d.live[n] for n in names]
        tokens = d.runner.sample_tokens(seqs)
        for i, n in enumerate(names):
            assert tokens[i] == int(np.argmax(logits[n][-1])), (i, k)
            rows[i].append(logits[n])
    _compare_layer_rows(cfg, w, "bfloat16", base, [np.concatenate(r) for r in rows])


def _bits(rng, shape, std):
    """float16 numbers of a deviation."""
    return (rng.standard_normal(shape) * std).astype(F16)


def _copy_of(d_W, N, K, mode=0, H=0, KVH=0, D=0):
    d_T = nvr.DeviceBuffer(N * K * 2)
    nvr.check(nvr.lib().nvr_retile_weight(d_W.ptr, d_T.ptr, N, K, mode, H, KVH, D, None))
    return d_T


def _product_bound(x, W):
    """|x . W^T rounded to float16 - exact|: K roundings to 24 bits of a sum of products, and one to 11 bits."""
    ref = x.astype(np.float64) @ W.astype(np.float64).T
    room = x.shape[1] * 2.0 ** -24 * (np.abs(x.astype(np.float64)) @ np.abs(W.astype(np.float64)).T)
    return ref, np.abs(ref) * 2.0 ** -11 + room + 2.0 ** -25


@pytest.mark.parametrize("T,K,N", [(97, 64, 4112), (129, 128, 4112), (255, 192, 2064), (200, 320, 4112), (301, 576, 4112), (700, 256, 1040), (1030, 1088, 4112)])
def test_tile_products_of_few_k_tiles_and_ragged_edges(T, K, N):
    """Products on 32-, 64- and 128-token tiles with fewer K-tiles than the ring holds, a column tile that is mostly past the edge and tiles that do not fill the XCDs' shares evenly: against
    64 bits, and the tiled copy of the weights against the weights, bit for bit."""
    rng, l = np.random.default_rng(T + K), nvr.lib()
    x, W = _bits(rng, (T, K), 0.5), _bits(rng, (N, K), 0.1)
    d_x, d_W = dev(x), dev(W)
    d_T, ya, yb = _copy_of(d_W, N, K), nvr.DeviceBuffer(T * N * 2), nvr.DeviceBuffer(T * N * 2)
    nvr.check(l.nvr_linear(d_x.ptr, K, d_W.ptr, T, K, N, ya.ptr, 0, None))
    nvr.check(l.nvr_linear_tiled(d_x.ptr, K, d_W.ptr, d_T.ptr, T, K, N, yb.ptr, 0, None))
    a, b = ya.to_numpy((T, N), F16), yb.to_numpy((T, N), F16)
    assert np.array_equal(a.view(np.uint16), b.view(np.uint16))
    ref, bound = _product_bound(x, W)
    assert np.all(np.abs(a - ref) <= bound)
    S = 2
    if K % (64 * S) == 0:
        sa, sb = nvr.DeviceBuffer(S * T * N * 4), nvr.DeviceBuffer(S * T * N * 4)
        nvr.check(l.nvr_linear_splitk(d_x.ptr, K, d_W.ptr, T, K, N, S, sa.ptr, None))
        nvr.check(l.nvr_linear_splitk_tiled(d_x.ptr, K, d_W.ptr, d_T.ptr, T, K, N, S, sb.ptr, None))
        s = sa.to_numpy((S, T, N), np.float32)
        assert np.array_equal(s, sb.to_numpy((S, T, N), np.float32))
        assert np.all(np.abs(s.astype(np.float64).sum(0) - ref) <= bound)


@pytest.mark.parametrize("T,K,N,S", [(20, 1024, 16384, 4), (3, 1056, 12288, 1), (32, 2592, 6144, 1), (17, 3616, 4096, 1), (1, 6144, 4096, 2),
                                     (20, 1024, 12288, 8), (4, 1152, 12288, 9), (7, 128, 98304, 1), (32, 96, 131072, 3),
                                     (16, 4096, 4096, 4), (31, 3072, 4096, 2), (2, 2048, 8192, 1), (32, 5120, 4096, 2), (17, 3584, 4096, 1), (5, 4096, 3200, 1)])
def test_split_products_of_large_weights(T, K, N, S):
    """Slabs of weights of 24 MiB and more, no step to 16 steps of a wave (slices of 32 to 224 columns, odd steps, waves of one step less than others; two to eight whole sets of two), one and two row tiles:
    against 64 bits, and the tiled copy's bits."""
    rng, l = np.random.default_rng(T + K), nvr.lib()
    x, W = _bits(rng, (T, K), 0.5), _bits(rng, (N, K), 0.1)
    d_x, d_W = dev(x), dev(W)
    d_T, sa, sb = _copy_of(d_W, N, K), nvr.DeviceBuffer(S * T * N * 4), nvr.DeviceBuffer(S * T * N * 4)
    nvr.check(l.nvr_linear_splitk(d_x.ptr, K, d_W.ptr, T, K, N, S, sa.ptr, None))
    nvr.check(l.nvr_linear_splitk_tiled(d_x.ptr, K, d_W.ptr, d_T.ptr, T, K, N, S, sb.ptr, None))
    s = sa.to_numpy((S, T, N), np.float32)
    assert np.array_equal(s, sb.to_numpy((S, T, N), np.float32))
    ref, bound = _product_bound(x, W)
    assert np.all(np.abs(s.astype(np.float64).sum(0) - ref) <= bound)


@pytest.mark.parametrize("T,kslice,N,S", [(3, 1024, 12288, 1), (20, 1536, 4096, 2), (32, 3072, 4096, 1), (16, 2048, 8192, 1)])
def test_split_products_have_one_order_of_sums(T, kslice, N, S):
    """Slices that linear_slab_kernel takes, and the same with 32 columns of zeros in x behind each, which it leaves to linear_skinny_kernel: bit for bit (the first wave adds zeros to its sums)."""
    rng, l = np.random.default_rng(T + kslice), nvr.lib()
    out = []
    x, W = _bits(rng, (T, S, kslice), 0.5), _bits(rng, (N, S, kslice), 0.1)
    for pad in (0, 32):
        K = S * (kslice + pad)
        xp = np.concatenate([x, np.zeros((T, S, pad), F16)], 2).reshape(T, K)
        Wp = np.concatenate([W, np.ones((N, S, pad), F16)], 2).reshape(N, K)
        d_x, d_W, d_s = dev(xp), dev(Wp), nvr.DeviceBuffer(S * T * N * 4)
        nvr.check(l.nvr_linear_splitk(d_x.ptr, K, d_W.ptr, T, K, N, S, d_s.ptr, None))
        out.append(d_s.to_numpy((S, T, N), np.float32))
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("T,K,N", [(33, 1536, 768), (48, 2048, 1040), (64, 512, 784), (64, 3072, 2048)])
def test_products_of_33_to_64_rows_in_eight_slices(T, K, N):
    """The o / down products of such steps on the tiles, eight slices of one to six K-tiles: the slabs' sum against 64 bits, the tiled copy's bits, and the residual add + norm over eight slabs."""
    rng, l, S = np.random.default_rng(T + K), nvr.lib(), 8
    x, W, h, w = _bits(rng, (T, K), 0.5), _bits(rng, (N, K), 0.1), _bits(rng, (T, N), 1.0), _bits(rng, (N,), 0.1) + F16(1)
    d_x, d_W = dev(x), dev(W)
    d_T, sa, sb = _copy_of(d_W, N, K), nvr.DeviceBuffer(S * T * N * 4), nvr.DeviceBuffer(S * T * N * 4)
    nvr.check(l.nvr_linear_splitk(d_x.ptr, K, d_W.ptr, T, K, N, S, sa.ptr, None))
    nvr.check(l.nvr_linear_splitk_tiled(d_x.ptr, K, d_W.ptr, d_T.ptr, T, K, N, S, sb.ptr, None))
    s = sa.to_numpy((S, T, N), np.float32)
    assert np.array_equal(s, sb.to_numpy((S, T, N), np.float32))
    ref, bound = _product_bound(x, W)
    assert np.all(np.abs(s.astype(np.float64).sum(0) - ref) <= bound)
    d_h, d_w, d_o = dev(h), dev(w), nvr.DeviceBuffer(T * N * 2)
    nvr.check(l.nvr_add_rmsnorm_slabs(d_h.ptr, sa.ptr, S, d_w.ptr, 1e-6, T, N, d_o.ptr, None))
    total = s[0]
    for z in range(1, S):
        total = total + s[z]
    want = (h.astype(np.float32) + total.astype(F16).astype(np.float32)).astype(F16)
    assert np.array_equal(d_h.to_numpy((T, N), np.uint16), want.view(np.uint16))
    v = want.astype(np.float64)
    norm = (v / np.sqrt((v * v).mean(1, keepdims=True) + 1e-6)) * w.astype(np.float64)
    assert np.all(np.abs(d_o.to_numpy((T, N), F16) - norm) <= np.abs(norm) * 1.01 * 2.0 ** -11 + 2.0 ** -25)


@pytest.mark.parametrize("T,K,I", [(97, 128, 3072), (200, 64, 4160), (509, 1024, 3072), (384, 192, 3072), (700, 320, 2112)])
def test_tile_gate_up_forms(T, K, I):
    """gate_up + SiLU on the tiles (128-row and 96-row ones): the tiled copy's bits, and every element within two roundings of the unit of the rounded products."""
    rng, l = np.random.default_rng(T + I), nvr.lib()
    x, W = _bits(rng, (T, K), 0.5), _bits(rng, (2 * I, K), 0.1)
    d_x, d_W = dev(x), dev(W)
    d_T, oa, ob, d_y = _copy_of(d_W, 2 * I, K), nvr.DeviceBuffer(T * I * 2), nvr.DeviceBuffer(T * I * 2), nvr.DeviceBuffer(T * 2 * I * 2)
    nvr.check(l.nvr_linear_silu_mul(d_x.ptr, K, d_W.ptr, T, K, I, oa.ptr, None))
    nvr.check(l.nvr_linear_silu_mul_tiled(d_x.ptr, K, d_W.ptr, d_T.ptr, T, K, I, ob.ptr, None))
    nvr.check(l.nvr_linear(d_x.ptr, K, d_W.ptr, T, K, 2 * I, d_y.ptr, 0, None))           # the unfused product: the same sums
    a = oa.to_numpy((T, I), F16)
    assert np.array_equal(a.view(np.uint16), ob.to_numpy((T, I), F16).view(np.uint16))
    y = d_y.to_numpy((T, 2 * I), F16).astype(np.float64)
    want = y[:, :I] / (1 + np.exp(-y[:, :I])) * y[:, I:]
    assert np.all(np.abs(a - want) <= np.abs(want) * 2.0 ** -10 + 2.0 ** -24)


@pytest.mark.parametrize("T,K,H,KVH,D", [(200, 128, 30, 3, 64), (129, 64, 20, 6, 128), (333, 256, 41, 5, 32), (260, 64, 66, 3, 16), (700, 320, 8, 4, 128)])
def test_tile_qkv_rope_store_forms(T, K, H, KVH, D):
    """qkv + RoPE + store on the tiles: heads of 16..128 whose boundaries lie inside a wave's columns, tokens without a slot; the rotation of the product's own rounded values with every
    operation rounded apart is exact, and so are the cache rows and the tiled copy."""
    rng, l = np.random.default_rng(T + D), nvr.lib()
    N, heads = (H + 2 * KVH) * D, H + KVH
    x, W = _bits(rng, (T, K), 0.5), _bits(rng, (N, K), 0.1)
    d_x, d_W = dev(x), dev(W)
    d_T, d_y = _copy_of(d_W, N, K, 1, H, KVH, D), nvr.DeviceBuffer(T * N * 2)
    nvr.check(l.nvr_linear(d_x.ptr, K, d_W.ptr, T, K, N, d_y.ptr, 0, None))
    pos = rng.integers(0, 512, T).astype(np.int64)
    slots = rng.permutation(1024)[:T].astype(np.int32)
    slots[::7] = -1
    cos, sin = oracle.rope_table(D, 512, 1e6)
    d_pos, d_slots, d_cos, d_sin = dev(pos), dev(slots), dev(cos), dev(sin)
    y = d_y.to_numpy((T, N), F16).reshape(T, H + 2 * KVH, D)
    u, v = y[:, :heads, :D // 2].astype(np.float32), y[:, :heads, D // 2:].astype(np.float32)
    c, s = np.asarray(cos, np.float32)[pos][:, None], np.asarray(sin, np.float32)[pos][:, None]
    want = y.copy()
    want[:, :heads, :D // 2], want[:, :heads, D // 2:] = (u * c - v * s).astype(F16), (v * c + u * s).astype(F16)
    kept = slots >= 0
    for fn, extra in ((l.nvr_linear_qkv_rope_store, ()), (l.nvr_linear_qkv_rope_store_tiled, (d_T.ptr,))):
        q, kc, vc = nvr.DeviceBuffer(T * N * 2), dev(np.zeros((1024, KVH, D), F16)), dev(np.zeros((1024, KVH, D), F16))
        nvr.check(fn(d_x.ptr, K, d_W.ptr, *extra, T, K, H, KVH, D, d_pos.ptr, d_slots.ptr, d_cos.ptr, d_sin.ptr, q.ptr, kc.ptr, vc.ptr, None))
        assert np.array_equal(q.to_numpy((T, N), np.uint16), want.reshape(T, N).view(np.uint16))
        for cache, first in ((kc, H), (vc, H + KVH)):
            full = np.zeros((1024, KVH, D), F16)
            full[slots[kept]] = want[kept, first:first + KVH]
            assert np.array_equal(cache.to_numpy((1024, KVH, D), np.uint16), full.view(np.uint16))


def _prefill(q, ctx, nq, k, v, tables, H, KVH, D, bs):
    """nvr_attn_prefill_paged of sequences of ctx tokens whose last nq are queries."""
    T, B = int(sum(nq)), len(nq)
    cu = np.concatenate([[0], np.cumsum(nq)]).astype(np.int32)
    bt = np.zeros((B, max(len(t) for t in tables)), np.int32)
    for b, t in enumerate(tables):
        bt[b, :len(t)] = t
    d_cu, d_ctx, d_bt, d_out, d_q, d_k, d_v = dev(cu), dev(np.asarray(ctx, np.int32)), dev(bt), nvr.DeviceBuffer(T * H * D * 2), dev(q), dev(k), dev(v)
    meta = nvr.AttnMetaC()
    meta.is_prefill, meta.cu_seqlens_q, meta.context_lens, meta.block_tables = 1, d_cu.ptr, d_ctx.ptr, d_bt.ptr
    meta.max_blocks, meta.batch, meta.max_context_len = bt.shape[1], B, int(max(ctx))
    nvr.check(nvr.lib().nvr_attn_prefill_paged(d_q.ptr, H * D, d_k.ptr, d_v.ptr, C.byref(meta), T, H, KVH, D, bs, float(D ** -0.5), d_out.ptr, None))
    return d_out.to_numpy((T, H, D), F16)


@pytest.mark.parametrize("G,KVH,bs,ctx,growth", [
    (2, 2, 64, [1, 63, 64, 65, 129], 0.0), (1, 3, 128, [127, 128, 200], 0.0), (4, 1, 64, [33, 97, 320], 0.0),
    (2, 1, 64, [700], 9.0), (1, 2, 48, [391, 70], 9.0), (4, 2, 256, [513], -9.0),      # scores that outgrow the running maximum again and again, and that fall off; a block size without a power of two
    (2, 1, 64, [4400], 3.0),                                                          # more blocks than the register copy of a table holds
])
def test_prompt_attention_of_heads_of_128(G, KVH, bs, ctx, growth):
    """The plain prompt attention against 64 bits at the edges of its tiles and steps, and the bits of a prompt in portions against the prompt whole."""
    rng, D, H = np.random.default_rng(sum(ctx)), 128, G * KVH
    NB = sum(-(-c // bs) for c in ctx)
    order, tables, at = rng.permutation(NB), [], 0
    k, v = np.zeros((NB * bs, KVH, D), F16), _bits(rng, (NB * bs, KVH, D), 1.0)
    q, want, spread, square = [], [], [], []
    for c in ctx:
        t = order[at:at + -(-c // bs)]
        at += len(t)
        rows = (t[:, None] * bs + np.arange(bs)[None]).reshape(-1)[:c]
        ramp = np.linspace(0.1, abs(growth), c)[::1 if growth > 0 else -1] if growth else np.ones(c)
        qs = _bits(rng, (c, H, D), 1.0)
        if growth:                                                                    # keys near one direction that every query has: the score follows the ramp
            axis = np.ones(D) / np.sqrt(D)
            k[rows] = (rng.standard_normal((c, KVH, D)) * 0.3 + axis * ramp[:, None, None] * 4).astype(F16)
            qs = (qs.astype(np.float64) + axis * 4).astype(F16)
        else:
            k[rows] = _bits(rng, (c, KVH, D), 1.0)
        tables.append(t.astype(np.int32))
        q.append(qs)
        kk, vv, qq = (np.repeat(a[rows].astype(np.float64), G, 1) if a is not None else qs.astype(np.float64) for a in (k, v, None))
        s = np.matmul(qq.transpose(1, 0, 2), kk.transpose(1, 2, 0)) * D ** -0.5
        s[:, np.arange(c)[None, :] > np.arange(c)[:, None]] = -np.inf
        p = np.exp(s - s.max(2, keepdims=True))
        p /= p.sum(2, keepdims=True)
        w = np.matmul(p, vv.transpose(1, 0, 2)).transpose(1, 0, 2)
        want.append(w)
        sums = [np.matmul(a, b.transpose(1, 0, 2)) for a, b in ((p, vv * vv), (p * p, vv * vv), (p * p, vv))]
        wh = w.transpose(1, 0, 2)
        spread.append(np.sqrt(np.maximum(sums[0] - wh * wh, 0)).transpose(1, 0, 2))   # at least the sum of weight x |value - result| (weights add up to 1)
        square.append(np.maximum(sums[1] - 2 * wh * sums[2] + wh * wh * np.sum(p * p, 2, keepdims=True), 0).transpose(1, 0, 2))      # the sum of (weight x (value - result))^2
    whole = _prefill(np.concatenate(q), ctx, ctx, k, v, tables, H, KVH, D, bs)
    # the result is rounded to 11 bits, and so is every weight before it meets its value and joins the row's sum: at most 2^-11 of |result| and of the sum of weight x |value - result|, and a
    # twentieth for the 24 bits of scores and sums
    w, spread, square, got = (np.concatenate(a).astype(np.float64).reshape(-1, D) for a in (want, spread, square, [whole]))
    assert np.all(np.abs(got - w) <= 1.05 * 2.0 ** -11 * (np.abs(w) + spread) + 2.0 ** -25)
    # a row's sum that is off moves the whole row by a factor.  Roundings are as often up as down: a deviation of at most 2^-11 / sqrt(3) each, those of the weights one for all columns of a row;
    # the factor of all rows together within five deviations (and the 24 bits of a sum)
    moved = np.sum((got - w) * w) / np.sum(w * w)
    deviation = 2.0 ** -11 / np.sqrt(3) * np.sqrt(np.sum(np.sum(np.abs(w) * np.sqrt(square), 1) ** 2) + np.sum(w ** 4)) / np.sum(w * w)
    assert abs(moved) <= 5 * deviation + 2.0 ** -20, (moved, deviation)
    at = 0
    for i, c in enumerate(ctx):
        for n in {1, min(c, 17), min(c, 70), c}:                                      # its last n tokens alone
            part = _prefill(q[i][c - n:], [c], [n], k, v, [tables[i]], H, KVH, D, bs)
            assert np.array_equal(part.view(np.uint16), whole[at + c - n:at + c].view(np.uint16)), (c, n)
        at += c


@pytest.mark.parametrize("kind,T,K,N", [("plain", 4200, 1024, 4096), ("silu", 3062, 1024, 3072), ("rope", 4300, 1024, 4096)])
def test_products_whose_rows_are_split_over_two_kernels(kind, T, K, N):
    """Prompt products whose last rows go to smaller tiles: the rows around the line have the bits of the same rows in a call of their own."""
    rng, l = np.random.default_rng(T), nvr.lib()
    rows, H, KVH, D = (2 * N if kind == "silu" else N), 16, 8, 128
    x, W = _bits(rng, (T, K), 0.5), _bits(rng, (rows, K), 0.1)
    d_W, pos = dev(W), rng.integers(0, 512, T).astype(np.int64)
    slots = np.arange(T, dtype=np.int32)
    cos, sin = oracle.rope_table(D, 512, 1e6)
    d_cos, d_sin = dev(cos), dev(sin)

    def run(a, b):
        n, d_x, y = b - a, dev(x[a:b]), nvr.DeviceBuffer((b - a) * N * 2)
        if kind == "plain":
            nvr.check(l.nvr_linear(d_x.ptr, K, d_W.ptr, n, K, N, y.ptr, 0, None))
        elif kind == "silu":
            nvr.check(l.nvr_linear_silu_mul(d_x.ptr, K, d_W.ptr, n, K, N, y.ptr, None))
        else:
            kc, vc, d_pos, d_slots = dev(np.zeros((n, KVH, D), F16)), dev(np.zeros((n, KVH, D), F16)), dev(pos[a:b]), dev(slots[:n])
            nvr.check(l.nvr_linear_qkv_rope_store(d_x.ptr, K, d_W.ptr, n, K, H, KVH, D, d_pos.ptr, d_slots.ptr, d_cos.ptr, d_sin.ptr, y.ptr, kc.ptr, vc.ptr, None))
            out = y.to_numpy((n, N), np.uint16)
            assert np.array_equal(kc.to_numpy((n, KVH * D), np.uint16), out[:, H * D:(H + KVH) * D]) and np.array_equal(vc.to_numpy((n, KVH * D), np.uint16), out[:, (H + KVH) * D:])
            return out
        return y.to_numpy((n, N), np.uint16)
    whole = run(0, T)
    for a, b in ((0, 130), (2500, 2700), (4030, 4160), (T - 140, T)):
        if b <= T:
            assert np.array_equal(run(a, b), whole[a:b]), (a, b)


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("tokens", [2200, 3300, 4400])
def test_prompt_steps_add_products_to_the_residual_rows_in_place(dtype, tokens):
    """Steps whose o / down products are added where the residual rows lie (tiles of both kernels, a last tile that is partly past the end): the logits of a prompt of more tokens than split-k
    slabs hold against the same prompt in portions of 1100 tokens, which take other tiles, bit for bit."""
    model = nvr.ModelConfig(vocab_size=512, hidden_size=1024, intermediate_size=1536, num_hidden_layers=2, num_attention_heads=8, num_key_value_heads=4, head_dim=128,
                            max_position_embeddings=8192, tie_word_embeddings=1, seed=7)
    prompt, got = nvr.synthetic_tokens(tokens, 3, 0, 512), []
    sp = nvr.SamplingParams(temperature=0.0, max_tokens=1, ignore_eos=True)
    for kw in (dict(max_num_batched_tokens=tokens + 64), dict(max_num_batched_tokens=1100, enable_chunked_prefill=1)):
        eng = nvr.LLMEngine(nvr.Config(max_num_seqs=1, max_model_len=tokens + 8, kvcache_block_size=256, num_kvcache_blocks=tokens // 256 + 2, dtype=dtype, **kw), model)
        eng.add_request(prompt, sp)
        while not eng.is_finished():
            rec = eng.step()
        got.append(eng.model_runner.logits(1).copy())
    assert np.array_equal(got[0], got[1])                                             # (portions of more than 1024 tokens: none sums k in slices)


@pytest.mark.parametrize("dim,vdim", [(64, 64), (64, 192), (128, 64), (128, 128)])
@pytest.mark.parametrize("lens", [(16, 1, 17), (31, 33, 15), (48, 50, 3)])
def test_retention_prompts_in_chunks_of_16_tokens(dim, vdim, lens):
    """The prompt form of retention (key sizes 64 and 128, bfloat16): whole chunks, one token over and one short, sequences of less than a chunk beside longer ones, a second portion that starts from
    the state the first one left, then two single tokens through the recurrence; quick, slow and nearly no decay.  Row by row against the float64 restatement."""
    import rugudra_util as u
    cfg = u.make_config([u.retention_layer(3, dim, vdim, decay=[0.3, 0.95, 0.9995], ff=None)], width=128, taps=3)
    w = u.make_weights(cfg, seed=dim + vdim)
    d = u.Driver(cfg, w, dtype="bfloat16", slots=3, pages=48, max_tokens=256, max_len=256)
    rng = np.random.default_rng(lens[0])
    toks = [rng.integers(0, 97, n + 2 * lens[0] + 2) for n in lens]
    at, rows = [0, 0, 0], [[], [], []]
    for step in (lens, (lens[0], lens[0] + 1, lens[0] - 1), (1, 1, 1), (1, 1, 1)):
        out = d.step([("s%d" % i, toks[i][at[i]:at[i] + n]) for i, n in enumerate(step)])
        for i, n in enumerate(step):
            at[i] += n
            rows[i].append(out["s%d" % i])
    for i in range(3):
        _compare_layer_rows(cfg, w, "bfloat16", [toks[i][:at[i]]], [np.concatenate(rows[i])])


@pytest.mark.parametrize("rows,width,ff", [(190, 256, 1024), (94, 512, 2048)])
def test_products_with_gelu_in_their_epilogue_beside_a_few_more_rows(rows, width, ff):
    """GELU of the unrounded product, in its epilogue, up to 384 Ki outputs: a prompt on either side of 192 Ki, where products without it change to the tiles (which would round before a GELU of
    its own), has the same bits alone and beside a prompt of ten tokens."""
    import kiduvik_util as k
    import rugudra_util as u
    cfg = k.make_config([k.diff(heads=4, kv_heads=2, dim=32, vdim=64, rot=16, mlp=k.dense(ff)) for _ in range(2)], width=width, vocab=96, side=0)
    d = u.Driver(cfg, k.make_weights(cfg, seed=rows), dtype="bfloat16", page=64, pages=8, slots=2, max_tokens=256, max_len=256)
    toks = np.random.default_rng(rows).integers(0, 96, rows + 10)
    assert rows * ff <= 192 * 1024 < (rows + 10) * ff
    alone = d.step([("a", toks[:rows])])["a"]
    d.end("a")
    beside = d.step([("a", toks[:rows]), ("b", toks[rows:])])["a"]
    assert np.array_equal(alone.view(np.uint32), beside.view(np.uint32))


@pytest.mark.parametrize("dim,vdim", [(64, 128), (128, 64)])
@pytest.mark.parametrize("n", [1, 7, 15])
def test_retention_of_a_short_portion_does_not_depend_on_its_neighbours(dim, vdim, n):
    """A sequence of less than a chunk of rows, in a step of the same size beside one long portion and beside several short ones, first and behind other tokens: the bits of its logits, and of
    those of the single token behind it (its state)."""
    import rugudra_util as u
    cfg = u.make_config([u.retention_layer(3, dim, vdim, decay=[0.3, 0.95, 0.9995], ff=None)], width=128, taps=3)
    w = u.make_weights(cfg, seed=n)
    d = u.Driver(cfg, w, dtype="bfloat16", slots=8, pages=48, max_tokens=256, max_len=256)
    rng = np.random.default_rng(n)
    toks, other = rng.integers(0, 97, 2 * n + 2), rng.integers(0, 97, 45)
    got = []
    for parts in ((45,), (15, 15, 15), (30, 15)):
        rows = []
        for a, b in ((0, n), (n, 2 * n)):
            rows.append(d.step([("s", toks[a:b])] + [("o%d" % i, other[:k]) for i, k in enumerate(parts)])["s"])
            for i in range(len(parts)):
                d.end("o%d" % i)
        rows += [d.step([("s", toks[k:k + 1])])["s"] for k in (2 * n, 2 * n + 1)]
        d.end("s")
        got.append(np.concatenate(rows).view(np.uint32))
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])


@pytest.mark.parametrize("dim,vdim", [(64, 64), (128, 128)])
@pytest.mark.parametrize("at", [1, 9, 15, 16, 30])
def test_retention_values_that_are_not_finite_reach_no_earlier_token(dim, vdim, at):
    """A token whose values overflow, inside a chunk and at its ends: every row in front of it has the bits that it has with an ordinary token in that place, every row from it on holds what the
    recurrence has there too, no number."""
    import rugudra_util as u
    cfg = u.make_config([u.retention_layer(2, dim, vdim, decay=[0.9, 0.999], ff=None)], width=128, taps=3)
    w = u.make_weights(cfg, seed=at)
    w["embed"][:, 5], w["l0.canon1"][5], w["l0.mix.v"][:, 5] = 0.0, 0.0, 0.0
    w["embed"][96, 5], w["l0.mix.v"][3, 5] = 8.0, 3e38                                # token 96 alone has a channel that takes one value column beyond the largest number
    d = u.Driver(cfg, w, dtype="bfloat16", slots=1, pages=8, max_tokens=64, max_len=64)
    toks = np.random.default_rng(at).integers(0, 96, 37)
    want = d.run_alone(toks)
    toks[at] = 96
    got = d.run_alone(toks)
    assert np.all(np.isfinite(want)) and np.array_equal(got[:at].view(np.uint32), want[:at].view(np.uint32))
    assert not np.any(np.isfinite(got[at:]).all(axis=1))


@pytest.mark.parametrize("taps", [2, 3, 4, 5])
@pytest.mark.parametrize("dim,width", [(64, 132), (128, 1028)])
def test_layer_list_single_tokens_across_pages(taps, dim, width):
    """Single tokens of a layer-list model: the norm and convolution with their weights in registers (2 to 4 taps, one of several 4-column pieces of a row left over) and read one by one (5), the
    decode attention that puts the step's own key and value rows into the pages itself — first and last row of a page, a page just begun — with chunks of keys that end at, before and behind the
    position.  Against the float64 restatement, row by row."""
    import rugudra_util as u
    cfg = u.make_config([u.attention_layer(4, 2, dim, dim, ff=None), u.attention_layer(2, 1, dim, dim, ff=None)], width=width, taps=taps)
    w = u.make_weights(cfg, seed=taps)
    d = u.Driver(cfg, w, dtype="bfloat16", slots=3, pages=24, max_tokens=128, max_len=96)
    rng = np.random.default_rng(dim)
    toks = [rng.integers(0, 97, n) for n in (20, 36, 70)]
    first = [n - 6 for n in (20, 36, 70)]                                    # positions 14 .. 19, 30 .. 35 and 64 .. 69 of pages of 16
    d.step([("s%d" % i, t[:f]) for i, (t, f) in enumerate(zip(toks, first))])
    out = [d.step([("s%d" % i, t[f + k:f + k + 1]) for i, (t, f) in enumerate(zip(toks, first))]) for k in range(6)]
    _compare_layer_rows(cfg, w, "bfloat16", toks, [np.concatenate([o["s%d" % i] for o in out]) for i in range(3)])


@pytest.mark.parametrize("hidden", [72, 1020, 1284, 3072])
def test_float32_decode_rows_form_their_norm_from_columns_in_registers(hidden):
    """float32 decode steps of 5, 2 and 1 rows whose add + norm rides in the consuming products: rows of less than a thread's first four columns, a few short of them, and beyond them (ragged and
    whole) — the logits of the runner that keeps the launches apart, bit for bit; pages of 24 tokens (no power of two) beside pages of 16."""
    import os
    model = nvr.ModelConfig(vocab_size=400, hidden_size=hidden, intermediate_size=96, num_hidden_layers=2, num_attention_heads=2, num_key_value_heads=1, head_dim=64, max_position_embeddings=128,
                            tie_word_embeddings=1, seed=hidden)
    prompts = [nvr.synthetic_tokens(11 + 9 * i, 5, i, 400) for i in range(5)]
    got = []
    for fused, page in (("0", 16), ("1", 16), ("1", 24)):
        os.environ["NVR_F32_FUSED_NORM"] = fused
        try:
            eng = nvr.LLMEngine(nvr.Config(skip_block_size_check=1, dtype="float32", max_num_seqs=5, max_num_batched_tokens=256, max_model_len=96, kvcache_block_size=page, num_kvcache_blocks=40), model)
        finally:
            os.environ.pop("NVR_F32_FUSED_NORM", None)
        for i, p in enumerate(prompts):
            eng.add_request(p, nvr.SamplingParams(temperature=0.0, max_tokens=(9, 6, 3, 3, 3)[i], ignore_eos=True))
        out, rows = [], set()
        while not eng.is_finished():
            rec = eng.step()
            rows.add(rec["num_seqs"])
            out.append((rec["tokens"], eng.model_runner.logits(rec["num_seqs"]).copy().view(np.uint32)))
        assert {1, 2, 5} <= rows
        got.append(out)
    for other in got[1:]:
        assert len(other) == len(got[0])
        for (ta, la), (tb, lb) in zip(got[0], other):
            assert ta == tb and np.array_equal(la, lb)


@pytest.mark.parametrize("hidden,inter,kv,dim,rows,length", [(16, 20, 1, 64, 1, 9), (28, 36, 1, 128, 3, 9),      # less than one run of four rows per XCD, and seven or nine of them
                                                             (64, 30, 1, 64, 8, 5),                            # columns that are no multiple of four
                                                             (1024, 3072, 4, 128, 1, 40), (1024, 1028, 2, 192, 7, 20),
                                                             (2048, 4096, 1, 256, 2, 12),                      # the gate half does not fit beside the output product's rows
                                                             (64, 64, 2, 256, 6, 420)])                        # keys and values that leave the caches no room
def test_float32_decode_attention_brings_weights_into_the_caches(hidden, inter, kv, dim, rows, length):
    """float32 decode steps whose attention launch holds workgroups that request the next products' weights: the runner that keeps the launches apart, which brings nothing, bit for bit (the requests
    leave nothing behind), with and without graphs."""
    import os
    model = nvr.ModelConfig(vocab_size=400, hidden_size=hidden, intermediate_size=inter, num_hidden_layers=2, num_attention_heads=2 * kv, num_key_value_heads=kv, head_dim=dim,
                            max_position_embeddings=512, tie_word_embeddings=1, seed=hidden)
    got = []
    for fused, eager in (("0", 0), ("1", 0), ("1", 1)):
        os.environ["NVR_F32_FUSED_NORM"] = fused
        try:
            eng = nvr.LLMEngine(nvr.Config(skip_block_size_check=1, dtype="float32", enforce_eager=eager, max_num_seqs=rows, max_num_batched_tokens=4096, max_model_len=480, kvcache_block_size=16,
                                           num_kvcache_blocks=30 * rows), model)
        finally:
            os.environ.pop("NVR_F32_FUSED_NORM", None)
        for i in range(rows):
            eng.add_request(nvr.synthetic_tokens(length + i, 5, i, 400), nvr.SamplingParams(temperature=0.0, max_tokens=4, ignore_eos=True))
        out = []
        while not eng.is_finished():
            rec = eng.step()
            out.append((rec["tokens"], eng.model_runner.logits(rec["num_seqs"]).copy().view(np.uint32)))
        got.append(out)
    for other in got[1:]:
        assert len(other) == len(got[0]) >= 4
        for (ta, la), (tb, lb) in zip(got[0], other):
            assert ta == tb and np.array_equal(la, lb)


# Prompts whose attention brings the gated unit's weights, 256 columns: an eighth of them to an XCD, or 48 rows of them in turn for tiles of 96 rows (what tests/test_weights_ahead.py looks at)
AHEAD_PROMPTS = [(3072, [65]), (3072, [330]), (2304, [512]), (2112, [130, 7]),     # (2112: columns in no eighths, which bring nothing)
                 (512, [200]), (3072, [1216]), (3072, [1217]), (3072, [1281])]     # 152 workgroups of attention, 160, and 168, which bring nothing
AHEAD_96_ROWS = {(sum(lengths), inter): sum(lengths) in (330, 512) for inter, lengths in AHEAD_PROMPTS}


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("inter,lengths", AHEAD_PROMPTS)
def test_prompt_attention_brings_weights_into_the_caches(inter, lengths, dtype):
    """Prompt steps whose attention launch holds workgroups that request the gated unit's weights, at the ends of the rule: the prompts' logits and those of the token behind them against the oracle, at the
    engine's tolerance for the type."""
    from oracle import model_oracle as mo
    from test_engine_gpu import _run_pair
    mcfg = mo.small(hidden_size=256, num_hidden_layers=2, intermediate_size=inter, head_dim=128, num_attention_heads=16, num_key_value_heads=8, max_position_embeddings=2048, seed=inter, init_std=0.02)
    ecfg = dict(max_num_seqs=2, max_num_batched_tokens=1344, max_model_len=1344, kvcache_block_size=16, num_kvcache_blocks=160)
    prompts = [oracle.fill_tokens(n, 3, i, mcfg.vocab_size).tolist() for i, n in enumerate(lengths)]
    _run_pair(mcfg, ecfg, prompts, [dict(temperature=0.0, max_tokens=2, ignore_eos=True) for _ in lengths], dtype=dtype)


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("hidden,qk_norm", [(256, False), (768, True), (1024, False), (1280, False)])
def test_decode_steps_of_one_to_five_rows(hidden, qk_norm, dtype):
    """A batch that shrinks from five rows to one: the add + norm formed by the consuming products (up to four rows of 1024 numbers, three of 1280; a wave count of row pieces that is and is not a
    multiple of four) and by its own launch, the rotation's sines requested behind the first weights (key heads, value heads, with and without q / k norms) — logits against the oracle, step by
    step, at the engine's tolerance for the type."""
    from oracle import model_oracle as mo
    from test_engine_gpu import _run_pair
    mcfg = mo.small(hidden_size=hidden, num_hidden_layers=2, intermediate_size=512, head_dim=128, num_attention_heads=4, num_key_value_heads=2, qk_norm=qk_norm, seed=hidden, init_std=0.02)
    ecfg = dict(max_num_seqs=5, max_num_batched_tokens=256, max_model_len=128, kvcache_block_size=16, num_kvcache_blocks=40)
    prompts = [oracle.fill_tokens(6 + 5 * i, 3, i, mcfg.vocab_size).tolist() for i in range(5)]
    sps = [dict(temperature=0.0, max_tokens=3 + 2 * i, ignore_eos=True) for i in range(5)]
    r = _run_pair(mcfg, ecfg, prompts, sps, dtype=dtype)
    assert r["decode_steps"] >= 10


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("heads,kv", [(2, 2), (4, 2), (4, 1)])
def test_decode_attention_forms_norms_and_stores_its_own_rows(heads, kv, dtype):
    """Models with q / k norms on heads of 128: a decode step whose attention norms, rotates and stores the step's rows itself (pages of 16 tokens; four and eight waves, one workgroup
    per sequence and head, and several with a last one that merges) against the same step with that launch in front (pages of 20 tokens, no whole chunks): logits bit for bit, step by step, over contexts that end at, before and behind
    a round of keys and a page, and as graph replays and eagerly."""
    model = nvr.ModelConfig(vocab_size=512, hidden_size=256, intermediate_size=256, num_hidden_layers=2, num_attention_heads=heads, num_key_value_heads=kv, head_dim=128,
                            max_position_embeddings=1024, tie_word_embeddings=1, seed=heads, qk_norm=1)
    for lens in ([126, 30, 5, 8], [700], [255, 120, 640], [640, 7, 321, 64] * 5, [260] * (97 if heads == kv else 1)):
        got = []
        for page, eager in ((20, 1), (16, 1), (16, 0)):
            eng = nvr.LLMEngine(nvr.Config(skip_block_size_check=1, max_num_seqs=len(lens), max_num_batched_tokens=2048, max_model_len=960, kvcache_block_size=page, num_kvcache_blocks=2000, dtype=dtype,
                                           enforce_eager=eager), model)
            for i, n in enumerate(lens):
                eng.add_request(nvr.synthetic_tokens(n, 9, i, 512), nvr.SamplingParams(temperature=0.0, max_tokens=6, ignore_eos=True))
            out = []
            while not eng.is_finished():
                rec = eng.step()
                out.append((rec["tokens"], eng.model_runner.logits(rec["num_seqs"]).copy().view(np.uint32)))
            got.append(out)
        for other in got[1:]:
            assert len(other) == len(got[0])
            for (ta, la), (tb, lb) in zip(got[0], other):
                assert ta == tb and np.array_equal(la, lb), lens


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("heads", [8, 16])
def test_work_balanced_decode_attention_forms_its_own_rows(heads, dtype):
    """The work-balanced decode attention (34 sequences of 8 kv heads) where it norms, rotates and stores the step's rows itself: segments that hold a query's last key and segments that do not,
    queries cut by shares — logits against the oracle step by step, at the engine's tolerance for the type."""
    from oracle import model_oracle as mo
    from test_engine_gpu import _run_pair
    mcfg = mo.small(hidden_size=256, num_hidden_layers=1, intermediate_size=256, head_dim=128, num_attention_heads=heads, num_key_value_heads=8, qk_norm=True, seed=heads, init_std=0.02)
    ecfg = dict(max_num_seqs=34, max_num_batched_tokens=8192, max_model_len=512, kvcache_block_size=16, num_kvcache_blocks=700)
    prompts = [oracle.fill_tokens(250 + i if i % 3 else 12 + 7 * i, 3, i, mcfg.vocab_size).tolist() for i in range(34)]
    r = _run_pair(mcfg, ecfg, prompts, [dict(temperature=0.0, max_tokens=4, ignore_eos=True)] * 34, dtype=dtype)
    assert r["decode_steps"] >= 3


@pytest.mark.parametrize("hidden,heads,kv,dim,qk_norm,dtype", [(256, 4, 4, 64, False, "float16"), (512, 8, 2, 64, False, "bfloat16"), (512, 16, 8, 128, False, "float16"), (512, 8, 8, 128, True, "bfloat16"),
                                                               (256, 8, 2, 128, True, "float16"), (1024, 16, 8, 128, False, "float16"), (1024, 8, 8, 128, True, "bfloat16")])
@pytest.mark.parametrize("page", [16, 20])
def test_decode_attention_takes_the_output_product_along(hidden, heads, kv, dim, qk_norm, dtype, page):
    """One to four sequences (64 and 128 rows of the product a workgroup) whose attention multiplies its heads with the output product's columns itself: groups of one, two and four heads, slabs of two, four and eight kv heads, pages of whole
    chunks of keys and others, contexts on both sides of a round of keys (128) and of the 256 beyond which the product is a launch of its own — logits against the oracle, step by step."""
    from oracle import model_oracle as mo
    from test_engine_gpu import _run_pair
    mcfg = mo.small(hidden_size=hidden, num_hidden_layers=2, intermediate_size=512, head_dim=dim, num_attention_heads=heads, num_key_value_heads=kv, qk_norm=qk_norm, seed=heads, init_std=0.02)
    ecfg = dict(max_num_seqs=4, max_num_batched_tokens=512, max_model_len=300, kvcache_block_size=page, num_kvcache_blocks=64)
    for lengths in ([122], [251], [1, 126]) + (([30, 121, 1, 9], [5, 124, 17]) if hidden == 1024 else ()):
        prompts = [oracle.fill_tokens(n, 3, i, mcfg.vocab_size).tolist() for i, n in enumerate(lengths)]
        sps = [dict(temperature=0.0, max_tokens=9, ignore_eos=True)] * len(lengths)
        assert _run_pair(mcfg, ecfg, prompts, sps, dtype=dtype)["decode_steps"] >= 8


@pytest.mark.parametrize("eager", [False, True])
def test_decode_of_four_sequences_whose_output_product_leaves_the_attention(eager):
    """Four sequences whose longest context passes the 136 keys up to which their attention multiplies its heads with the output product's columns, replayed steps and eager ones — logits against the
    oracle, step by step."""
    from oracle import model_oracle as mo
    from test_engine_gpu import _run_pair
    mcfg = mo.small(hidden_size=1024, num_hidden_layers=2, intermediate_size=512, head_dim=128, num_attention_heads=16, num_key_value_heads=8, seed=4, init_std=0.02)
    ecfg = dict(max_num_seqs=4, max_num_batched_tokens=512, max_model_len=300, kvcache_block_size=64, num_kvcache_blocks=32)
    prompts = [oracle.fill_tokens(n, 3, i, mcfg.vocab_size).tolist() for i, n in enumerate((130, 5, 60, 1))]
    r = _run_pair(mcfg, ecfg, prompts, [dict(temperature=0.0, max_tokens=12, ignore_eos=True)] * 4, **(dict(enforce_eager=True) if eager else {}))
    assert r["decode_steps"] >= 11


@pytest.mark.parametrize("eager", [False, True])
def test_decode_behind_a_shared_prefix_while_own_contexts_grow(eager):
    """Three requests behind 512 tokens whose longest passes 128 tokens of its own on the way: one launch before, two behind it, each form a captured step of its own — logits against the oracle, step
    by step."""
    from oracle import model_oracle as mo
    from test_engine_gpu import _run_pair
    mcfg = mo.small(seed=9, hidden_size=512, num_attention_heads=4, num_key_value_heads=2, head_dim=128, intermediate_size=768, num_hidden_layers=2)
    ecfg = dict(max_num_seqs=4, max_num_batched_tokens=2048, max_model_len=768, kvcache_block_size=64, num_kvcache_blocks=60)
    system = oracle.fill_tokens(512, 4, 7, mcfg.vocab_size).tolist()
    prompts = [system + oracle.fill_tokens(n, 4, 100 + n, mcfg.vocab_size).tolist() for n in (120, 3, 60)]
    r = _run_pair(mcfg, ecfg, prompts, [dict(temperature=0.0, max_tokens=20, ignore_eos=True)] * 3, product_kw=dict(shared_prefix_min_seqs=2), **(dict(enforce_eager=True) if eager else {}))
    assert r["decode_steps"] >= 19 and r["near_ties"] <= 2, r


@pytest.mark.parametrize("width,heads,ff,batch", [(64, 2, 80, 1), (256, 2, 96, 16), (256, 2, 96, 17), (1024, 2, 208, 32), (64, 16, 2064, 17), (1024, 16, 2048, 32)])
def test_layer_list_decode_steps_of_two_products_in_one_launch(width, heads, ff, batch):
    """Decode steps of a layer list whose mixer's product and clamped unit share a launch: four and eight waves, one and two row tiles to a workgroup, last tiles of one row and full ones, in both kinds
    of layers — a first step and replays, against the float64 restatement."""
    import rugudra_util as u
    cfg = u.make_config([u.retention_layer(heads, 32, 32, ff=ff), u.attention_layer(heads, 1 if heads < 16 else heads, 64, 64, ff=ff)], width=width, taps=2)
    w = u.make_weights(cfg, seed=ff + width)
    d = u.Driver(cfg, w, dtype="bfloat16", slots=batch, pages=batch * 2, max_tokens=9 * batch, max_len=64)
    rng = np.random.default_rng(width)
    base = [rng.integers(0, 97, 6 + i) for i in range(min(batch, 3))]
    names = ["s%d" % i for i in range(batch)]
    d.step([(n, base[i % 3][:-3]) for i, n in enumerate(names)])
    steps = [d.step([(n, base[i % 3][len(base[i % 3]) - 3 + k:][:1]) for i, n in enumerate(names)]) for k in range(3)]
    _compare_layer_rows(cfg, w, "bfloat16", base, [np.concatenate([s[n] for s in steps]) for n in names])


@pytest.mark.parametrize("width,ff", [(256, 208), (1024, 1024)])
def test_layer_list_two_products_in_one_launch_have_the_bits_of_two(width, ff):
    """Decode steps of 16 sequences, whose two first products share a launch, and of 32 (a wide mixer beside a narrow feed-forward: two launches, of two and one row tiles to a workgroup): the 16
    sequences that both hold come out bit for bit."""
    import rugudra_util as u
    cfg = u.make_config([u.retention_layer(16, 32, 32, ff=ff), u.retention_layer(16, 32, 32, ff=ff)], width=width, taps=2)
    w = u.make_weights(cfg, seed=ff + width)
    toks = np.random.default_rng(width).integers(0, 97, (32, 6))
    got = []
    for batch in (16, 32):
        d = u.Driver(cfg, w, dtype="bfloat16", slots=batch, pages=2 * batch, max_tokens=4 * batch, max_len=64)
        for first in range(0, batch, 16):                                  # (the prompts in steps of the same size)
            d.step([("s%d" % i, toks[i][:3]) for i in range(first, first + 16)])
        steps = [d.step([("s%d" % i, toks[i][k:k + 1]) for i in range(batch)]) for k in range(3, 6)]
        got.append(np.concatenate([s["s%d" % i] for s in steps for i in range(16)]).view(np.uint32))
    assert np.array_equal(got[0], got[1]), (got[0] != got[1]).mean()


@pytest.mark.parametrize("dim,vdim", [(64, 64), (64, 128), (128, 64), (128, 128)])
def test_retention_of_single_tokens_norms_and_gates_its_heads(dim, vdim):
    """Steps of one token per sequence, whose retention norms and gates its heads itself, against the same tokens in steps beside a portion of several rows (launches of their own): bit for bit, from a
    sequence's first token (no state yet, in a slot that another sequence left) on, first steps and replays."""
    import rugudra_util as u
    cfg = u.make_config([u.retention_layer(3, dim, vdim, decay=[0.3, 0.95, 0.9995], ff=None)], width=128, taps=3)
    w = u.make_weights(cfg, seed=dim + vdim)
    d = u.Driver(cfg, w, dtype="bfloat16", slots=3, pages=24, max_tokens=64, max_len=64)
    rng = np.random.default_rng(vdim)
    toks, other = [rng.integers(0, 97, 6) for _ in range(2)], rng.integers(0, 97, 3)
    got = []
    for beside in (False, True):
        rows = []
        for k in range(6):
            step = d.step([("s%d" % i, toks[i][k:k + 1]) for i in range(2)] + ([("o", other)] if beside else []))
            rows += [step["s0"], step["s1"]]
            if beside:
                d.end("o")
        for i in range(2):
            d.end("s%d" % i)
        got.append(np.concatenate(rows).view(np.uint32))
    assert np.array_equal(got[0], got[1])
