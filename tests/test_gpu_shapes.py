"""Model shapes outside the batched decode kernels, against the CPU oracle.

The reference decodes any shape ModelConfig::new accepts (src/config.rs:15-30;
its CPU decode kernels take any head size, src/shaders/cpu.rs:144-178) and its
FLASH_ATTENTION any head_dim up to 128 (src/nn/ops/emit.rs:564-572).  The
batched decode kernels need a head size that is a multiple of 4, a dim that
is a multiple of 32 (at most 4096) and an ffn_hidden that is a multiple of 32;
other shapes decode on the generic kernels (decode_generic.hip).  Each case:
ragged prefill and greedy decode steps of a batch, sequences checked against
the oracle (identical tokens, logits within 1e-3), also with the bfloat16 KV
cache (within 2e-2) and through generate's sampler.
"""

import ctypes
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-3


def _model(pkg, backend, dim, heads, layers, ffn, seed):
    cfg = dataclasses.replace(pkg.ModelConfig.new(173, dim, heads, layers, 40), ffn_hidden=ffn)
    w = pkg.synthetic_weights(cfg, seed=seed)
    model = pkg.hip.Model(backend, cfg)
    model.upload(w)
    return cfg, w, model


# (dim, heads, ffn): head sizes 50, 6 and 34 (not multiples of 4; dim 102
# is not even a multiple of 4), dim 48 and 100 (not multiples of 32), an
# ffn_hidden of 200 (not a multiple of 32), head size 2.
SHAPES = [(100, 2, 400), (24, 4, 96), (102, 3, 408), (48, 4, 192), (100, 1, 200), (8, 4, 32)]


@pytest.mark.parametrize("dim,heads,ffn", SHAPES)
@pytest.mark.parametrize("batch", [3, 33])
def test_generic_shape_session_matches_oracle(backend, pkg, ora, dim, heads, ffn, batch):
    layers, ctx, steps = 2, 40, 4
    case = f"dim {dim} heads {heads} (hd {dim // heads}) ffn {ffn} batch {batch}"
    print(case, flush=True)
    cfg, w, model = _model(pkg, backend, dim, heads, layers, ffn, seed=dim + heads)
    r = np.random.default_rng(dim * 7 + batch)
    lens = [int(x) for x in r.integers(1, ctx - steps - 4, size=batch)]
    prompts = [r.integers(0, cfg.vocab_size, size=n).astype(np.uint32) for n in lens]
    s = pkg.hip.Session(model, ctx, batch)
    logits, nxt = s.prefill(prompts)
    got = [(logits, nxt)] + [s.decode_step(None) for _ in range(steps)]
    assert list(s.cur_len()) == [n + steps for n in lens], case
    for b in sorted({0, batch // 2, batch - 1}):
        o = ora.OracleSession(cfg, w, ctx)
        ref = o.prefill(prompts[b])
        for i in range(steps + 1):
            if i:
                ref = o.decode_step(ora.argmax(ref))
            assert np.abs(got[i][0][b] - ref).max() < TOL, f"{case}, sequence {b} step {i}"
            assert int(got[i][1][b]) == ora.argmax(ref), f"{case}, sequence {b} step {i}"
        # The cache rows the decode steps appended equal the oracle's.
        for layer in range(layers):
            n = lens[b] + steps
            kc = s.cache(layer, b, 0)[:n]
            assert np.abs(kc - o.k_cache(layer)[:n]).max() < 1e-4, f"{case}, K cache {layer}"
        o.close()
    # Greedy decode_greedy replays (a captured graph) continue the same way.
    toks = s.decode_greedy(3)
    o = ora.OracleSession(cfg, w, ctx)
    ref = o.prefill(prompts[0])
    for i in range(steps):
        ref = o.decode_step(ora.argmax(ref))
    for i in range(3):
        ref = o.decode_step(ora.argmax(ref))
        assert int(toks[i][0]) == ora.argmax(ref), f"{case}, replayed step {i}"
    o.close()
    s.close()
    model.close()


@pytest.mark.parametrize("kv16", [False, True])
def test_generic_shape_long_context(backend, pkg, ora, kv16):
    # The generic attention holds 1024 scores per pass over the keys: a
    # 1500-token prompt and decode steps past it take two passes, the
    # running maximum and sum rescaled between them.  Against the oracle
    # (logits within 1e-3, or 2e-2 with the bfloat16 cache).
    cfg, w, model = _model(pkg, backend, 100, 2, 2, 400, seed=17)
    r = np.random.default_rng(18)
    prompt = r.integers(0, cfg.vocab_size, size=(2, 1500)).astype(np.uint32)
    s = pkg.hip.Session(model, 1600, 2)
    if kv16:
        s.set_kv_bf16(True)
    logits, nxt = s.prefill(prompt)
    got = [(logits, nxt)] + [s.decode_step(None) for _ in range(3)]
    tol = 2e-2 if kv16 else TOL
    for b in range(2):
        o = ora.OracleSession(cfg, w, 1600)
        ref = o.prefill(prompt[b])
        for i in range(4):
            if i:
                ref = o.decode_step(int(got[i - 1][1][b]))
            assert np.abs(got[i][0][b] - ref).max() < tol, f"sequence {b} step {i}"
            if not kv16:
                assert int(got[i][1][b]) == ora.argmax(ref), f"sequence {b} step {i}"
        o.close()
    s.close()
    model.close()


@pytest.mark.parametrize("dim,heads,ffn", [(100, 2, 400), (102, 3, 408)])
def test_generic_shape_bf16_kv_cache(backend, pkg, ora, dim, heads, ffn):
    # The bfloat16 KV cache on the generic kernels: logits within 2e-2 of
    # the oracle's fp32 decode.
    layers, ctx, steps, batch = 2, 40, 3, 4
    cfg, w, model = _model(pkg, backend, dim, heads, layers, ffn, seed=dim)
    r = np.random.default_rng(dim)
    prompt = r.integers(0, cfg.vocab_size, size=(batch, 20)).astype(np.uint32)
    s = pkg.hip.Session(model, ctx, batch)
    s.set_kv_bf16(True)
    logits, _ = s.prefill(prompt)
    got = [logits]
    o = ora.OracleSession(cfg, w, ctx)
    ref = [o.prefill(prompt[0])]
    for _ in range(steps):
        t = ora.argmax(ref[-1])
        got.append(s.decode_step(np.full(batch, t, np.uint32))[0])
        ref.append(o.decode_step(t))
    for i in range(steps + 1):
        assert np.abs(got[i][0] - ref[i]).max() < 2e-2, f"step {i}"
    o.close()
    s.close()
    model.close()


def test_generic_shape_generate_and_errors(backend, pkg, ora):
    # generate (greedy, eos / length stops) on the generic kernels equals the
    # oracle's greedy loop; the timing entry points of the batched kernels
    # refuse such a session.
    cfg, w, model = _model(pkg, backend, 100, 2, 2, 400, seed=5)
    r = np.random.default_rng(6)
    prompt = r.integers(0, cfg.vocab_size, size=(2, 9)).astype(np.uint32)
    s = pkg.hip.Session(model, 40, 2)
    outs = s.generate(prompt, 6)
    for b in range(2):
        o = ora.OracleSession(cfg, w, 40)
        ref = o.prefill(prompt[b])
        want = []
        for _ in range(6):
            t = ora.argmax(ref)
            want.append(t)
            if t == cfg.eos_token:
                break
            ref = o.decode_step(t)
        o.close()
        assert list(outs[b]) == want, b
    with pytest.raises(pkg.hip.InvalidArgument):
        s.time_decode_kernel(1, 4)
    with pytest.raises(pkg.hip.InvalidArgument):
        s.set_fused_norm(True)
    s.close()
    model.close()


# One to four sequences decode on GEMVs that norm their own rows: the narrowest
# row, one that leaves threads and the last K range partly idle, ffn widths of
# one K range and of more k than a pass holds, the widest row, and the first
# that is too wide (the batched kernels); ragged prompts, so positions differ.
@pytest.mark.parametrize("batch,dim,heads,ffn", [
    (1, 32, 2, 32), (2, 96, 3, 224), (3, 320, 5, 1280), (4, 768, 12, 3072), (1, 768, 6, 4128),
    (2, 1024, 8, 96), (1, 1056, 11, 2080), (5, 96, 3, 224),
])
def test_few_sequences_decode_matches_oracle(backend, pkg, ora, batch, dim, heads, ffn):
    cfg = dataclasses.replace(pkg.ModelConfig.new(173, dim, heads, 2, 40), ffn_hidden=ffn)
    w = pkg.synthetic_weights(cfg, seed=91, std=0.05)
    model = pkg.hip.Model(backend, cfg)
    model.upload(w)
    s = pkg.hip.Session(model, 40, batch)
    few = batch <= 4 and dim <= 1024
    assert s.decode_launches() == (5 * 2 + 3 if few else 7 * 2 + 3)
    prompts = [pkg.synthetic_tokens(3 + 7 * b, 173, seed=92 + b) for b in range(batch)]
    logits, nxt = s.prefill(prompts)
    refs = [ora.OracleSession(cfg, w, 40) for _ in range(batch)]
    want = [r.prefill(p) for r, p in zip(refs, prompts)]
    for step in range(4):
        for b in range(batch):
            assert np.abs(logits[b] - want[b]).max() < 1e-3, (step, b)
            assert int(nxt[b]) == ora.argmax(want[b]), (step, b)
        want = [r.decode_step(int(t)) for r, t in zip(refs, nxt)]
        logits, nxt = s.decode_step(None)
    # The same steps replayed several to a graph.
    s.truncate(3)
    greedy = s.decode_greedy(9)
    s.truncate(3)
    assert np.array_equal(greedy, np.stack([s.decode_step(None)[1] for _ in range(9)]))
    s.close()


# Feed-forwards too long for those GEMVs decode on the batched kernels, with the
# sequences at which that begins: the last that one to three take, the first
# that none takes, one whose rows would not fit a block's LDS.
@pytest.mark.parametrize("batch,dim,ffn,few", [
    (3, 32, 8192, True), (4, 32, 8192, False), (1, 64, 12288, False), (4, 32, 131072, False),
])
def test_few_sequences_long_ffn_matches_oracle(backend, pkg, ora, batch, dim, ffn, few):
    cfg = dataclasses.replace(pkg.ModelConfig.new(173, dim, 2, 2, 24), ffn_hidden=ffn)
    w = pkg.synthetic_weights(cfg, seed=93, std=0.02)
    model = pkg.hip.Model(backend, cfg)
    model.upload(w)
    s = pkg.hip.Session(model, 24, batch)
    assert s.decode_launches() == (5 * 2 + 3 if few else 7 * 2 + 3)
    prompts = [pkg.synthetic_tokens(3 + 2 * b, 173, seed=94 + b) for b in range(batch)]
    logits, nxt = s.prefill(prompts)
    refs = [ora.OracleSession(cfg, w, 24) for _ in range(batch)]
    want = [r.prefill(p) for r, p in zip(refs, prompts)]
    for step in range(3):
        for b in range(batch):
            assert np.abs(logits[b] - want[b]).max() < 1e-3, (step, b)
            assert int(nxt[b]) == ora.argmax(want[b]), (step, b)
        want = [r.decode_step(int(t)) for r, t in zip(refs, nxt)]
        logits, nxt = s.decode_step(None)
    s.close()


def test_prefill_memory_is_what_its_rows_need(backend, pkg):
    # 64 rows of dim 36 (no split kernels) and of dim 64 (eight K ranges of 64 x 64
    # sums, 128 KB): a fixed 16 MB buffer of partial sums shows in either.
    rt = ctypes.CDLL("libamdhip64.so")

    def free():
        backend.synchronize()
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert rt.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    for dim in (36, 64):
        cfg = pkg.ModelConfig.new(97, dim, 1, 2, 64)
        model = pkg.hip.Model(backend, cfg)
        model.upload(pkg.synthetic_weights(cfg, seed=3))
        sessions = [pkg.hip.Session(model, 64, 1) for _ in range(4)]
        t = pkg.synthetic_tokens(64, 97, seed=4).reshape(1, -1)
        sessions[0].prefill(t)
        before = free()
        for s in sessions[1:]:
            s.prefill(t)
        assert before - free() < 3 * (16 << 20), dim
        for s in sessions:
            s.close()
        model.close()


def test_few_sequences_scores_at_minus_infinity(backend, pkg):
    # A first token whose one score overflows to -inf (q columns 1e20, k columns
    # -1e20 times the same sum): no weight remains and the attention adds nothing,
    # on the few-sequence and on the batched kernels alike.
    cfg = pkg.ModelConfig.new(97, 64, 2, 1, 16)
    w = pkg.synthetic_weights(cfg, seed=31)
    w[2][:, :64] = 1e20
    w[2][:, 64:128] = -1e20
    model = pkg.hip.Model(backend, cfg)
    model.upload(w)
    out = []
    for batch in (1, 5):
        s = pkg.hip.Session(model, 16, batch)
        logits, _ = s.decode_step(np.full(batch, 11, np.uint32))
        out.append(logits[0].copy())
        s.close()
    assert np.isfinite(out[1]).all()
    np.testing.assert_allclose(out[0], out[1], atol=1e-5)
    model.close()
