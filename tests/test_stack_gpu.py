"""Layer-list models (Ralasun) on the GPU against the plain float64 implementation in oracle/stack_oracle.py.

Every test builds its own small configuration and random weights (synth.build_stack). The product path is libtlhip.so
(operators, engine, decode graph) and, for generation, the C++ host (Session over a checkpoint folder). Exact mode
(three-term chunk GEMMs, FP32 GEMVs) is compared at FP32 tolerances; the bf16-activation mode at bf16 tolerances, and its
GEMM operator exactly against a product with bf16-rounded activations."""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FP32_TOL = 3e-5   # relative RMS per row, exact mode (observed ~1e-6)
BF16_TOL = 8e-2   # the same with bf16-rounded activations in the chunk GEMMs


def rel_rms(got, want):
    got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
    d = got - want
    return float(np.sqrt((d * d).mean(-1)).max() / max(1e-12, np.sqrt((want * want).mean())))


@pytest.fixture(scope="module")
def env(pkg):
    from tinyllama_cpp_amd import capi, engine, synth
    from oracle import stack_oracle
    engine.init(0)
    return {"capi": capi, "engine": engine, "synth": synth, "oracle": stack_oracle}


def small_config(synth, variant="mixed"):
    L = synth.stack_layer
    if variant == "mixed":  # unequal layers: windows 9 / 5 / none / 17, a layer without feed-forward, one without mixing
        layers = [L(4, 2, 24, 12, 9, v_mix=True, experts=4, top=2, ff=24, shared_ff=40),
                  L(6, 3, 20, 8, 5, v_mix=False, experts=3, top=1, ff=16, shared_ff=0, limit=0.7),
                  L(4, 2, 24, 12, None, v_mix=True, mlp=False),
                  L(2, 2, 36, 12, 17, v_mix=True, experts=5, top=5, ff=8, shared_ff=24, shared_limit=2.0)]
        return synth.stack_config(72, 101, layers)
    if variant == "odd":  # nothing divisible by 4: every scalar fallback path
        layers = [L(3, 1, 10, 6, 4, v_mix=True, experts=2, top=1, ff=5, shared_ff=7),
                  L(3, 3, 10, 2, 3, v_mix=True, experts=1, top=1, ff=9, shared_ff=0)]
        return synth.stack_config(37, 53, layers, eps=1e-3)
    if variant == "equal":  # values a model may happen to make equal or 1
        layers = [L(2, 2, 16, 16, 1, v_mix=False, experts=2, top=2, ff=16, shared_ff=16),
                  L(1, 1, 32, 32, 64, v_mix=True, experts=2, top=1, ff=16, shared_ff=16, scale=1.0)]
        return synth.stack_config(32, 64, layers)
    if variant == "wide":  # several 64-wide tiles in every product, window longer than a key piece of the kernel
        layers = [L(4, 2, 64, 32, 150, v_mix=True, experts=8, top=3, ff=96, shared_ff=160) for _ in range(2)]
        return synth.stack_config(256, 300, layers)
    raise ValueError(variant)


def make(env, cfg, seed=1, max_pos=512, exact=True, **environ):
    old = {k: os.environ.get(k) for k in environ}
    os.environ.update({k: str(v) for k, v in environ.items()})
    try:
        tensors = env["synth"].build_stack(cfg, seed)
        m = env["engine"].StackModel(cfg, max_pos).load(tensors)
    finally:
        for k, v in old.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v
    m.set_prefill(3 if exact else 1, 1)
    return m, tensors, env["oracle"].StackOracle(cfg, tensors)


# ---- each mechanism alone ---------------------------------------------------------------------------------------------
def dev(env, a):
    return env["engine"].DeviceBuffer.from_numpy(np.ascontiguousarray(a))


@pytest.mark.parametrize("rows,cols,T", [(64, 64, 64), (70, 40, 3), (129, 72, 130), (33, 37, 65), (256, 512, 200), (330, 100, 259)])
def test_dense_matmul(env, rows, cols, T):
    synth, capi = env["synth"], env["capi"]
    rng = np.random.default_rng(rows + cols + T)
    w = synth.to_bf16(rng.standard_normal((rows, cols)).astype(np.float32))
    x = (rng.standard_normal((T, cols)) * np.exp(rng.uniform(-6, 6, (T, cols)))).astype(np.float32)
    wd, xd = dev(env, w), dev(env, x)
    yd = env["engine"].DeviceBuffer(4 * T * rows)
    wf = synth.from_bf16(w).astype(np.float64)
    for terms, tile in ((3, "64"), (1, "64"), (3, "128"), (1, "128"), (3, None)):  # both tile shapes, then the launcher's pick
        if tile is None:
            os.environ.pop("TL_DENSE_TILE", None)
        else:
            os.environ["TL_DENSE_TILE"] = tile
        try:
            capi.check(capi.lib().tl_dense_matmul(wd.ptr, rows, cols, xd.ptr, yd.ptr, T, terms, None), "tl_dense_matmul")
        finally:
            os.environ.pop("TL_DENSE_TILE", None)
        capi.check(capi.lib().tl_device_sync(), "sync")
        got = yd.to_numpy(np.float32, (T, rows))
        xin = x if terms == 3 else synth.from_bf16(synth.to_bf16(x))  # terms 1: exactly the bf16-rounded activations
        want = xin.astype(np.float64) @ wf.T
        mag = np.abs(xin).astype(np.float64) @ np.abs(wf).T
        assert np.all(np.abs(got - want) <= 4e-6 * mag + 1e-30), (terms, float(np.abs(got - want).max()))
    capi.check(capi.lib().tl_dense_matmul(wd.ptr, rows, cols, xd.ptr, yd.ptr, 1, 0, None), "tl_dense_matmul gemv")
    capi.check(capi.lib().tl_device_sync(), "sync")
    got = yd.to_numpy(np.float32, (1, rows))[0]
    want = x[0].astype(np.float64) @ wf.T
    assert np.all(np.abs(got - want) <= 4e-6 * (np.abs(x[0]).astype(np.float64) @ np.abs(wf).T))


def run_swa(env, q, k, v, start, heads, kv_heads, dim, vdim, window, scale):
    capi = env["capi"]
    T = q.shape[0]
    qd, kd, vd = dev(env, q), dev(env, k), dev(env, v)
    od = env["engine"].DeviceBuffer(4 * T * heads * vdim)
    capi.check(capi.lib().tl_swa_attention(qd.ptr, kd.ptr, vd.ptr, od.ptr, T, start, heads, kv_heads, dim, vdim, window,
                                           scale, None), "tl_swa_attention")
    capi.check(capi.lib().tl_device_sync(), "sync")
    return od.to_numpy(np.float32, (T, heads * vdim))


@pytest.mark.parametrize("heads,kv_heads,dim,vdim,window", [(4, 2, 24, 12, 9), (3, 1, 10, 6, 70), (2, 2, 64, 80, 300),
                                                            (2, 1, 32, 16, 0), (1, 1, 8, 8, 1)])
def test_window_attention_prompt_and_decode(env, heads, kv_heads, dim, vdim, window):
    rng = np.random.default_rng(window + dim)
    n = 420
    k = rng.standard_normal((n, kv_heads * dim)).astype(np.float32)
    v = rng.standard_normal((n, kv_heads * vdim)).astype(np.float32)
    qall = rng.standard_normal((n, heads * dim)).astype(np.float32)
    scale = 0.37
    want = env["oracle"].window_attention(qall.astype(np.float64), k.astype(np.float64), v.astype(np.float64), heads, kv_heads,
                                          dim, vdim, window, scale, np.arange(n), np.arange(n))
    # what lies ahead of a position and what the window has left behind must not be read: poison it per call
    for start, T in ((0, n), (0, 3), (5, 64), (131, 200), (n - 1, 1), (window, 1), (max(window - 1, 1), 1), (257, 1)):
        kp, vp = k.copy(), v.copy()
        kp[start + T:], vp[start + T:] = 1e30, np.nan
        lo = start - window + 1 if window > 0 else 0
        if lo > 0:
            kp[:lo], vp[:lo] = 1e30, np.nan
        got = run_swa(env, qall[start:start + T], kp, vp, start, heads, kv_heads, dim, vdim, window, scale)
        assert rel_rms(got, want[start:start + T]) < 1e-5, (start, T)


def test_window_edge_key_stands_out(env):
    """One key is made to dominate the softmax: at distance window - 1 the output is its value row, at distance window it must
    not be seen at all. In a prompt portion and in a single decoded token; across the 64-key pieces of the kernel."""
    heads, kv_heads, dim, vdim, scale = 2, 1, 16, 8, 1.0
    rng = np.random.default_rng(3)
    for window in (5, 64, 65, 200):
        n = window + 80
        for i in (window + 3, n - 1):  # the query position
            for dist, seen in ((window - 1, True), (window, False), (0, True), (1, True)):
                k = (0.1 * rng.standard_normal((n, dim))).astype(np.float32)
                v = rng.standard_normal((n, vdim)).astype(np.float32)
                q = (0.1 * rng.standard_normal((n, heads * dim))).astype(np.float32)
                j = i - dist
                direction = rng.standard_normal(dim).astype(np.float32)
                direction /= np.linalg.norm(direction)
                k[j] = 30.0 * direction
                q[i] = np.tile(30.0 * direction, heads)  # score 900 against everything else at ~0
                v[j] = 7.0
                for start, T in ((i, 1), (i - 2, 5 if i + 3 <= n else n - i + 2)):
                    got = run_swa(env, q[start:start + T], k, v, start, heads, kv_heads, dim, vdim, window, scale)[i - start]
                    if seen:
                        assert np.allclose(got, 7.0, atol=1e-4), (window, i, dist, T)
                    else:
                        assert np.abs(got).max() < 6.0, (window, i, dist, T)


def test_router_top_choice_and_weights(env):
    capi, synth = env["capi"], env["synth"]
    rng = np.random.default_rng(5)
    for width, experts, top in ((72, 8, 4), (37, 3, 3), (64, 70, 5), (16, 1, 1)):
        T = 33
        x = rng.standard_normal((T, width)).astype(np.float32)
        w = synth.to_bf16((rng.standard_normal((experts, width)) / np.sqrt(width)).astype(np.float32))
        b = rng.standard_normal(experts).astype(np.float32)
        xd, wd, bd = dev(env, x), dev(env, w), dev(env, b)
        idd, wtd = env["engine"].DeviceBuffer(4 * T * top), env["engine"].DeviceBuffer(4 * T * top)
        capi.check(capi.lib().tl_moe_route(xd.ptr, T, width, wd.ptr, bd.ptr, experts, top, idd.ptr, wtd.ptr, None), "tl_moe_route")
        capi.check(capi.lib().tl_device_sync(), "sync")
        ids, wts = idd.to_numpy(np.int32, (T, top)), wtd.to_numpy(np.float32, (T, top))
        want_ids, want_w = env["oracle"].route(x.astype(np.float64), synth.from_bf16(w).astype(np.float64), b.astype(np.float64), top)
        assert np.array_equal(ids, want_ids)
        assert np.allclose(wts, want_w, rtol=1e-5, atol=1e-7)
        assert np.allclose(wts.sum(1), 1.0, atol=1e-5)


def test_clamped_gate_hits_its_limits(env):
    capi = env["capi"]
    rng = np.random.default_rng(7)
    rows, ff = 9, 21
    gu = (3.0 * rng.standard_normal((rows, 2 * ff))).astype(np.float32)  # well beyond the limits on both sides
    for limit, alpha in ((1.0, 1.702), (0.25, 1.0), (7.0, 1.702)):
        gd = dev(env, gu)
        od = env["engine"].DeviceBuffer(4 * rows * ff)
        capi.check(capi.lib().tl_glu_clamp(gd.ptr, rows, ff, limit, alpha, od.ptr, None), "tl_glu_clamp")
        capi.check(capi.lib().tl_device_sync(), "sync")
        g = np.minimum(gu[:, :ff].astype(np.float64), limit)
        u = np.clip(gu[:, ff:].astype(np.float64), -limit, limit)
        want = g / (1 + np.exp(-alpha * g)) * (u + 1)
        assert np.allclose(od.to_numpy(np.float32, (rows, ff)), want, rtol=2e-6, atol=1e-6)


def test_residual_output_norm(env):
    capi = env["capi"]
    rng = np.random.default_rng(9)
    for T, width, eps in ((5, 72, 1e-5), (3, 37, 1e-2), (2, 1024, 1e-6)):
        x = rng.standard_normal((T, width)).astype(np.float32)
        y = (rng.standard_normal((T, width)) * 1e-2).astype(np.float32)  # small: eps matters
        w = (0.1 * rng.standard_normal(width)).astype(np.float32)
        xd, yd, wd = dev(env, x), dev(env, y), dev(env, w)
        capi.check(capi.lib().tl_resid_rmsnorm(xd.ptr, yd.ptr, wd.ptr, T, width, eps, None), "tl_resid_rmsnorm")
        capi.check(capi.lib().tl_device_sync(), "sync")
        want = x + env["oracle"].rms_norm(y.astype(np.float64), w.astype(np.float64), eps, True)
        assert np.allclose(xd.to_numpy(np.float32, (T, width)), want, rtol=1e-5, atol=1e-6)


# ---- the whole model ----------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("variant", ["mixed", "odd", "equal", "wide"])
def test_layers_and_logits_of_a_prompt(env, variant):
    cfg = small_config(env["synth"], variant)
    m, _, orc = make(env, cfg, seed=11, TL_NO_GRAPH=1)
    rng = np.random.default_rng(1)
    toks = rng.integers(0, cfg["vocab"], 77).astype(np.int32)
    want_layers = []
    want = orc.forward(list(toks), want_layers)
    got_layers = m.capture_layers(lambda: m.prefill_rows(toks, 0))
    assert [l for l, _ in got_layers] == list(range(len(cfg["layers"])))
    for (l, a), w in zip(got_layers, want_layers):
        assert rel_rms(a, w) < FP32_TOL, f"residual stream after layer {l}"
    m.reset_kv()
    assert rel_rms(m.prefill_rows(toks, 0), want) < FP32_TOL
    # the first tokens of a sequence on their own, and chosen rows only
    m.reset_kv()
    assert rel_rms(m.prefill_rows(toks[:3], 0), want[:3]) < FP32_TOL
    m.reset_kv()
    rows = np.array([0, 1, 40, 76], np.int32)
    assert rel_rms(m.prefill_rows(toks, 0, rows), want[rows]) < FP32_TOL
    m.set_prefill(1, 1)  # bf16 activations in the chunk products
    m.reset_kv()
    assert rel_rms(m.prefill_rows(toks, 0), want) < BF16_TOL
    m.free()


@pytest.mark.parametrize("variant,gemv", [("mixed", 1), ("mixed", 0), ("odd", 1), ("equal", 1), ("wide", 1)])
def test_prompt_against_token_by_token_decoding(env, variant, gemv):
    """Every position decoded alone through the captured step (replayed once per token, prefill work in between) equals the
    prompt pass; positions run far beyond every window of the configuration."""
    cfg = small_config(env["synth"], variant)
    m, _, orc = make(env, cfg, seed=13, TL_STACK_GEMV=gemv, TL_STACK_FUSE_ROUTER=gemv)  # 0: also the router as its own launch
    assert m.graph_captured()
    rng = np.random.default_rng(2)
    n = 330 if variant == "wide" else 90
    toks = rng.integers(0, cfg["vocab"], n).astype(np.int32)
    want = orc.forward(list(toks))
    got = np.stack([m.decode(int(t), i)[0] for i, t in enumerate(toks)])
    assert rel_rms(got, want) < FP32_TOL
    # a prompt first, then decoding on top of its cache
    m.reset_kv()
    cut = n // 2 + 3
    head = m.prefill_rows(toks[:cut], 0)
    tail = np.stack([m.decode(int(toks[i]), i)[0] for i in range(cut, n)])
    assert rel_rms(np.concatenate([head, tail]), want) < FP32_TOL
    m.free()


@pytest.mark.parametrize("variant,chunk", [("mixed", 512), ("mixed", 16), ("wide", 64), ("odd", 5)])
def test_portions_of_any_size(env, variant, chunk):
    """A prompt cut into portions (down to two tokens and one) gives the logits of the uncut prompt; `chunk` also cuts long
    portions inside the engine, so window and piece edges fall everywhere."""
    cfg = small_config(env["synth"], variant)
    m, _, orc = make(env, cfg, seed=17, TL_STACK_CHUNK=chunk)
    rng = np.random.default_rng(3)
    n = 400 if variant == "wide" else 120
    toks = rng.integers(0, cfg["vocab"], n).astype(np.int32)
    want = orc.forward(list(toks))
    for sizes in ([7, 2, 13, 1, 20, 2, 5, 64, 3], [2] * 20, [n]):
        m.reset_kv()
        outs, p = [], 0
        for s in sizes + [n]:
            s = min(s, n - p)
            if s <= 0:
                break
            outs.append(m.prefill_rows(toks[p:p + s], p))
            p += s
        assert rel_rms(np.concatenate(outs), want) < FP32_TOL, sizes[:4]
    m.free()


def test_cache_given_back_and_used_again(env):
    """A second request after reset_kv equals the same request on a fresh model, also when the first one was longer."""
    cfg = small_config(env["synth"], "mixed")
    m, tensors, orc = make(env, cfg, seed=19)
    rng = np.random.default_rng(4)
    a = rng.integers(0, cfg["vocab"], 150).astype(np.int32)
    b = rng.integers(0, cfg["vocab"], 40).astype(np.int32)
    m.prefill_rows(a, 0)
    for i in range(5):
        m.decode(int(a[i]), 150 + i)
    m.reset_kv()
    got = m.prefill_rows(b[:30], 0)
    tail = np.stack([m.decode(int(b[i]), i)[0] for i in range(30, 40)])
    want = orc.forward(list(b))
    assert rel_rms(np.concatenate([got, tail]), want) < FP32_TOL
    m.free()


def test_far_key_decides_the_logits(env):
    """The query/key weights of a layer with no window are scaled up so that attention is nearly one-hot: a fault in a far
    key then moves the logits by far more than the tolerance. Prompt pass and decode against the oracle."""
    synth = env["synth"]
    cfg = synth.stack_config(64, 97, [synth.stack_layer(2, 1, 32, 16, None, v_mix=True, experts=2, top=1, ff=16, shared_ff=0),
                                      synth.stack_layer(2, 1, 32, 16, 40, v_mix=True, experts=2, top=1, ff=16, shared_ff=16)])
    tensors = synth.build_stack(cfg, 23)
    for name in ("l0.mix.q.norm", "l1.mix.q.norm"):
        tensors[name] = synth.to_bf16(synth.from_bf16(tensors[name]) * 8.0)  # sharp softmax
    m = env["engine"].StackModel(cfg, 512).load(tensors)
    m.set_prefill(3, 1)
    orc = env["oracle"].StackOracle(cfg, tensors)
    rng = np.random.default_rng(5)
    toks = rng.integers(0, 97, 300).astype(np.int32)
    want = orc.forward(list(toks))
    assert rel_rms(m.prefill_rows(toks, 0), want) < 2e-4
    m.reset_kv()
    m.prefill_rows(toks[:250], 0, np.array([249], np.int32))
    tail = np.stack([m.decode(int(toks[i]), i)[0] for i in range(250, 300)])
    assert rel_rms(tail, want[250:]) < 2e-4
    m.free()


def test_long_decoding_and_device_loops(env):
    """Greedy generation on the device (graph replays back to back) for several windows' worth of tokens equals the oracle's
    token-by-token arg-max; the sampled loop is reproducible by seed and stays inside the vocabulary."""
    cfg = small_config(env["synth"], "mixed")
    m, _, orc = make(env, cfg, seed=29)
    prompt = np.array([3, 14, 15, 92, 65, 35], np.int32)
    want = orc.generate_greedy(list(prompt), 70)
    last = m.prefill_rows(prompt, 0, np.array([len(prompt) - 1], np.int32))[0]
    first = int(np.argmax(last))
    more = m.generate_greedy(first, len(prompt), 69)
    assert [first] + list(more) == want
    m.reset_kv()
    m.prefill_rows(prompt, 0, np.array([len(prompt) - 1], np.int32))
    s1 = m.generate_sampled(first, len(prompt), 30, temperature=0.9, top_k=20, top_p=0.95, seed=7)
    m.reset_kv()
    m.prefill_rows(prompt, 0, np.array([len(prompt) - 1], np.int32))
    s2 = m.generate_sampled(first, len(prompt), 30, temperature=0.9, top_k=20, top_p=0.95, seed=7)
    assert list(s1) == list(s2) and all(0 <= t < cfg["vocab"] for t in s1)
    m.free()


def test_generation_through_the_host_session(env, tmp_path):
    """The framework's own entry point: a checkpoint folder opened by tlhost::Session (model registry, config.json reader,
    safetensors loader), greedy generate() for a short (token-by-token) and a long (batched prefill) prompt, generate_batch
    prompt by prompt, and the step function the trace runner uses."""
    from tinyllama_cpp_amd import hostapi
    synth = env["synth"]
    cfg = small_config(synth, "mixed")
    tensors = synth.build_stack(cfg, 31)
    synth.write_stack_dir(str(tmp_path / "ckpt"), cfg, tensors)
    orc = env["oracle"].StackOracle(cfg, tensors)
    s = hostapi.Session(str(tmp_path / "ckpt"), 0, 256)
    info = s.info()
    assert info["architecture"] == "Ralasun" and info["vocab"] == cfg["vocab"] and info["max_pos"] == 256
    s.set_repetition_penalty(1.0)
    s.set_exact(True)
    rng = np.random.default_rng(6)
    for n in (5, 45):
        prompt = rng.integers(0, cfg["vocab"], n).astype(np.int32)
        assert list(s.generate(prompt, steps=24, temperature=0.0)) == orc.generate_greedy(list(prompt), 24)
    prompts = [rng.integers(0, cfg["vocab"], n).astype(np.int32) for n in (3, 40, 11)]
    s.set_max_batch(3)
    outs = s.generate_batch(prompts, steps=10, temperature=0.0)
    for p, o in zip(prompts, outs):
        assert list(o) == orc.generate_greedy(list(p), 10)
    toks = rng.integers(0, cfg["vocab"], 60).astype(np.int32)
    orc.reset()
    want = orc.forward(list(toks))
    s.reset()
    got = [s.forward(toks[:37], 0, [0, 5, 36]), s.forward(toks[37:39], 37, [1])]
    got += [s.forward(toks[i:i + 1], i, [0]) for i in range(39, 60)]
    rows = [0, 5, 36, 38] + list(range(39, 60))
    assert rel_rms(np.concatenate(got), want[rows]) < FP32_TOL
    s.close()
    # a checkpoint that names an unknown design is refused with the names this build has
    bad = dict(cfg, architecture="NoSuchDesign")
    synth.write_stack_dir(str(tmp_path / "bad"), bad, tensors)
    with pytest.raises(hostapi.TlHostError, match="Ralasun"):
        hostapi.Session(str(tmp_path / "bad"), 0, 64)


@pytest.mark.parametrize("family", ["windows", "sink", "latent", "chunk"])
def test_half_attention_routes(pkg, monkeypatch, family):
    """The two-part f16 attention of a chunk against the FP32 matrix kernel (TL_HATTN=0): windows that end inside a tile and head
    sizes 64, 128 and 128 over 64, a sink with unequal groups, expanded latent rows of 96 under a window with gated heads, and
    chunked masks; a prompt that is walked whole and one that is continued, lengths off every tile. Three-term products: only the
    attention differs, by 32-bit rounding (2^-21 of a score of a few units, halved on average over independent errors): 3e-5 of
    the logits' size holds three layers of it."""
    from tinyllama_cpp_amd import engine, synth
    engine.init(0)
    if family == "windows":
        cfg = synth.stack_config(128, 90, [synth.stack_layer(4, 2, 64, 64, 40), synth.stack_layer(2, 1, 128, 128, None),
                                           synth.stack_layer(6, 2, 128, 64, 33)])
        tensors = synth.build_stack(cfg, 3)
    elif family == "sink":
        cfg = synth.sogalix_config(128, 90, [synth.sogalix_layer("attention", synth.sogalix_attention(6, 2, 64, 64, q_temp=(0.5, 20)), ff=64),
                                             synth.sogalix_layer("attention", synth.sogalix_attention(1, 1, 128, 128), ff=64),
                                             synth.sogalix_layer("latent_attention", synth.sogalix_latent(3, 64, 32, 64, 48, 40), ff=64)])
        tensors = synth.build_sogalix(cfg, 3)
    elif family == "latent":
        cfg = synth.madudra_config(128, 90, [synth.madudra_layer("latent_attention", synth.madudra_latent(5, 64, 32, 64, 48, 40, w))
                                             for w in (50, 0, 129)])
        tensors = synth.build_madudra(cfg, 3)
    else:
        cfg = synth.ratuzen_config(128, 90, [synth.ratuzen_layer("parallel", synth.ratuzen_chunked(4, 1, 64, 64, c, 2, 16, 16, [0.5, 0.7]), ff=64)
                                             for c in (48, 100)])
        tensors = synth.build_ratuzen(cfg, 3)
    toks = np.random.default_rng(5).integers(0, 90, 420).astype(np.int32)
    m = engine.StackModel(cfg, 512, tensors).load(tensors)
    m.set_prefill(3, 1)
    got = []
    for route in ("0", "1"):
        monkeypatch.setenv("TL_HATTN", route)
        m.reset_kv()
        got.append(np.stack([np.array(m.prefill(toks[:a], 0) if a < 400 else m.prefill(toks[333:a], 333), np.float64) for a in (65, 333, 420)]))
    m.free()
    assert np.isfinite(got[1]).all() and not np.array_equal(got[0], got[1])
    assert np.linalg.norm(got[1] - got[0]) <= 3e-5 * np.linalg.norm(got[0]), np.linalg.norm(got[1] - got[0]) / np.linalg.norm(got[0])


@pytest.mark.parametrize("dim,vdim,spread", [(64, 64, "row"), (128, 128, "row"), (96, 64, "first row"), (128, 64, "tiles"),
                                             (64, 64, "steps"), (128, 128, "steps"), (64, 64, "none")])
def test_half_attention_value_range(env, dim, vdim, spread):
    """The two-part f16 attention holds one power of two per tile of 32 value rows and one for its running sum. A row 2^18 times
    the others' size, of negligible weight, must coarsen neither the tiles behind it nor those in front of it (its own tile's rows
    are held to 2^-39 of it: 2^-21), nor may tiles of values 2^-60 .. 2^60 apart, at random or rising and falling. As many heads as
    keep the keys of a row in one piece. Against float64, relative to the weights times the values' size: two parts hold 2^-23 of
    each factor, and errors of many keys average out, so 2^-22 bounds the L2 distance (FP32 kernel: 7e-8, this one 5e-8 to 1.3e-7)."""
    rng = np.random.default_rng(dim + vdim)
    heads, n, T = 128, 600, 512
    u = rng.standard_normal(dim)
    u /= np.linalg.norm(u)
    q = (rng.standard_normal((T, heads, dim)) + 8 * u).astype(np.float32)
    k = rng.standard_normal((n, heads, dim)).astype(np.float32)
    v = rng.standard_normal((n, heads, vdim)).astype(np.float32)
    tiles = -(-n // 32)
    if spread in ("row", "first row"):
        at = 70 if spread == "row" else 0
        k[at] = -5.0 * np.sqrt(dim) * u  # (a score of -40)
        v[at] *= 2.0 ** 18
    elif spread != "none":
        e = rng.integers(-60, 61, tiles) if spread == "tiles" else np.abs(np.arange(tiles) * 13 - 120) - 60
        v *= np.exp2(e).astype(np.float32).repeat(32)[:n, None, None]
    scale = dim ** -0.5
    f = lambda a: a.reshape(len(a), -1).astype(np.float64)
    args = (heads, heads, dim, vdim, 0, scale, np.arange(n - T, n), np.arange(n))
    want = env["oracle"].window_attention(f(q), f(k), f(v), *args)
    size = env["oracle"].window_attention(f(q), f(k), np.abs(f(v)), *args)
    qd, kd, vd, od = dev(env, q), dev(env, k), dev(env, v), env["engine"].DeviceBuffer(4 * T * heads * vdim)
    capi = env["capi"]
    capi.check(capi.lib().tl_debug_half_attention(qd.ptr, kd.ptr, vd.ptr, od.ptr, T, n - T, heads, heads, dim, vdim, 0, scale, None), "half attention")
    capi.check(capi.lib().tl_device_sync(), "sync")
    err = np.linalg.norm((od.to_numpy(np.float32, want.shape) - want) / size) / np.sqrt(want.size)
    assert err <= 2.0 ** -22, err


@pytest.mark.parametrize("scale", [0.0, -0.125, 2.0 ** -140, 0.125])
def test_attention_scale_of_any_sign_in_a_chunk(env, scale):
    """A layer's factor on the scores is a plain number of its configuration: zero (every visible key alike), negative, or too small
    for the powers of two of the two-part f16 kernel, which takes positive ones of ordinary size and leaves the rest to the FP32
    kernel. Chunks of 16 tokens and more, whole and continued, against the oracle."""
    L = env["synth"].stack_layer
    cfg = env["synth"].stack_config(128, 90, [L(4, 2, 64, 64, 40, scale=scale), L(2, 1, 128, 128, None, scale=scale)])
    m, _, oracle = make(env, cfg)
    toks = np.random.default_rng(4).integers(0, 90, 150).astype(np.int32)
    want = oracle.forward(toks)
    for parts in ((150,), (70, 80)):
        m.reset_kv()
        at, got = 0, []
        for n in parts:
            got.append(m.prefill_rows(toks[at:at + n], at))
            at += n
        assert rel_rms(np.concatenate(got), want) < FP32_TOL, parts
    m.free()


@pytest.mark.parametrize("rows,cols,T,terms", [(64, 64, 64, 1), (65, 72, 63, 1), (130, 200, 65, 3), (33, 8, 16, 1), (70, 130, 40, 1),
                                               (70, 131, 40, 3), (256, 192, 130, 1), (4096, 96, 1024, 1), (4100, 40, 1030, 1)])
def test_dense_gemm_steps(pkg, rows, cols, T, terms):
    """The pipelined steps of the dense GEMM: columns below, at and off one and two steps (zeros beyond the last), rows that are
    not 16 bytes apart (narrow loads), both tiles with remainders. Against float64 over the operands that the terms keep: a bf16
    activation exactly, three of them within 2^-24; a sum of cols products in FP32 is off by at most cols 2^-24 |w| . |x|."""
    from tinyllama_cpp_amd import capi, engine, synth
    engine.init(0)
    rng = np.random.default_rng(rows + cols + T)
    w = synth.to_bf16(rng.standard_normal((rows, cols)).astype(np.float32))
    x = rng.standard_normal((T, cols)).astype(np.float32)
    dev = engine.DeviceBuffer.from_numpy
    wd, xd, yd = dev(w), dev(x), engine.DeviceBuffer(4 * T * rows)
    capi.check(capi.lib().tl_dense_matmul(wd.ptr, rows, cols, xd.ptr, yd.ptr, T, terms, None), "tl_dense_matmul")
    capi.check(capi.lib().tl_device_sync(), "sync")
    W = synth.from_bf16(w).astype(np.float64)
    X = (synth.from_bf16(synth.to_bf16(x)) if terms == 1 else x).astype(np.float64)
    bound = (cols + 4) * 2.0 ** -24 * (np.abs(X) @ np.abs(W).T)
    assert (np.abs(yd.to_numpy(np.float32, (T, rows)) - X @ W.T) <= bound).all()


@pytest.mark.parametrize("rows,cols,T", [(257, 96, 129), (4096, 96, 1024), (4100, 40, 1030), (260, 130, 70)])
@pytest.mark.parametrize("terms", [1, 3])
def test_dense_gemm_tiles_give_the_same_bits(pkg, monkeypatch, rows, cols, T, terms):
    """The rule between small and large tiles looks at their number and at the columns only: each output is the same sum in the same
    order in either, with one row and one token beyond a tile too, so the choice changes no bit. Bound as above."""
    from tinyllama_cpp_amd import capi, engine, synth
    engine.init(0)
    rng = np.random.default_rng(rows + cols + T)
    w = synth.to_bf16(rng.standard_normal((rows, cols)).astype(np.float32))
    x = rng.standard_normal((T, cols)).astype(np.float32)
    dev, got = engine.DeviceBuffer.from_numpy, []
    wd, xd, yd = dev(w), dev(x), engine.DeviceBuffer(4 * T * rows)
    for tile in ("64", "128", None):
        monkeypatch.setenv("TL_DENSE_TILE", tile) if tile else monkeypatch.delenv("TL_DENSE_TILE")
        capi.check(capi.lib().tl_dense_matmul(wd.ptr, rows, cols, xd.ptr, yd.ptr, T, terms, None), "tl_dense_matmul")
        capi.check(capi.lib().tl_device_sync(), "sync")
        got.append(yd.to_numpy(np.float32, (T, rows)))
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    W = synth.from_bf16(w).astype(np.float64)
    X = (synth.from_bf16(synth.to_bf16(x)) if terms == 1 else x).astype(np.float64)
    assert (np.abs(got[0] - X @ W.T) <= (cols + 4) * 2.0 ** -24 * (np.abs(X) @ np.abs(W).T)).all()


@pytest.mark.parametrize("rows,cols,T,ld", [(1, 64, 1, 64), (257, 192, 129, 200), (130, 1088, 1050, 1088), (128, 128, 31, 132), (900, 64, 33, 64)])
@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("exact", [0, 1, 5, 31, 32])
def test_dense_plane_gemm_gives_the_same_bits(pkg, monkeypatch, rows, cols, T, ld, waves, exact):
    """The kernel that takes its items from a bf16 plane against the one that converts them itself: tiles with one row and one token
    more, fewer steps than it fetches ahead, item tiles beyond a panel of eight, rows apart, a plane that holds NaN before. The same
    sums in the same order, also where the first items have two terms (as the tile that is chosen has them). Against float64: with two
    terms 16 of 24 bits are kept (2^-16 of each product), for all of the first 32 items."""
    from tinyllama_cpp_amd import capi, engine, synth
    engine.init(0)
    rng = np.random.default_rng(rows + cols + T + waves)
    w = synth.to_bf16(rng.standard_normal((rows, cols)).astype(np.float32))
    x = np.full((T, ld), np.nan, np.float32)
    x[:, :cols] = rng.standard_normal((T, cols))
    dev = engine.DeviceBuffer.from_numpy
    wd, xd, yd = dev(w), dev(x), engine.DeviceBuffer(4 * T * rows)
    plane = engine.DeviceBuffer(2 * (T + 32) * cols)

    def run(at):
        capi.check(capi.lib().tl_memset(yd.ptr, 0xff, yd.nbytes, None))
        capi.check(capi.lib().tl_memset(plane.ptr, 0xff, plane.nbytes, None))
        capi.check(capi.lib().tl_debug_dense_plane(wd.ptr, rows, cols, xd.ptr, ld, yd.ptr, T, exact, waves, at, None), "tl_debug_dense_plane")
        capi.check(capi.lib().tl_device_sync(), "sync")
        return yd.to_numpy(np.float32, (T, rows))

    X, W = x[:32, :cols].astype(np.float64), synth.from_bf16(w).astype(np.float64)
    for tile in ("64", "128"):
        monkeypatch.setenv("TL_DENSE_TILE", tile)
        got = run(plane.ptr)
        if exact:
            assert (np.abs(got[:32] - X @ W.T) <= (2.0 ** -16 + (cols + 4) * 2.0 ** -24) * (np.abs(X) @ np.abs(W).T)).all()
        assert np.array_equal(got, run(None)), tile


def test_causal_conv_output_behind_the_last_row(pkg):
    """Channels at the end of wider rows, the output right behind the last row's: no overlap, whatever the row stride adds up to
    (buffers that the allocator places back to back); one float earlier it is one, and refused."""
    from tinyllama_cpp_amd import capi, engine, synth
    engine.init(0)
    rng = np.random.default_rng(2)
    T, C, taps, ld, off = 9, 8, 3, 24, 16
    x = rng.standard_normal(off + (T - 1) * ld + C + T * C).astype(np.float32)
    w = synth.to_bf16(rng.standard_normal((C, taps)).astype(np.float32))
    buf, wd = engine.DeviceBuffer.from_numpy(x), engine.DeviceBuffer.from_numpy(w)
    end = buf.ptr + 4 * (off + (T - 1) * ld + C)
    far, got = engine.DeviceBuffer(4 * T * C), []
    for out in (far.ptr, end):
        hist = engine.DeviceBuffer.from_numpy(np.zeros((taps - 1, C), np.float32))
        capi.check(capi.lib().tl_causal_conv(buf.ptr + 4 * off, ld, C, taps, T, None, wd.ptr, hist.ptr, 0, 0, out, C, None), "conv")
        capi.check(capi.lib().tl_device_sync(), "sync")
        got.append(far.to_numpy(np.float32, (T, C)) if out == far.ptr else buf.to_numpy(np.float32, (x.size,))[-T * C:].reshape(T, C))
    assert np.array_equal(got[0], got[1]) and np.abs(got[0]).max() > 0
    hist = engine.DeviceBuffer.from_numpy(np.zeros((taps - 1, C), np.float32))
    assert capi.lib().tl_causal_conv(buf.ptr + 4 * off, ld, C, taps, T, None, wd.ptr, hist.ptr, 0, 0, end - 4, C, None) != 0


@pytest.mark.parametrize("heads,kv_heads,dim,window", [(8, 2, 64, 300), (3, 3, 64, 0), (4, 1, 128, 259), (2, 2, 128, 64)])
def test_window_attention_over_wide_rows(env, heads, kv_heads, dim, window):
    """Rows of 64 and 128 numbers for keys and values: sixteen lanes a key, records merged in a second launch."""
    test_window_attention_prompt_and_decode(env, heads, kv_heads, dim, dim, window)


@pytest.mark.parametrize("dim,top,ff,shared_ff", [(64, 6, 1032, 40), (128, 4, 24, 0), (64, 10, 16, 1544), (128, 2, 776, 1536), (64, 1, 2048, 514)])
def test_decode_step_with_wide_rows_and_many_slots(env, dim, top, ff, shared_ff):
    """The captured decode step over heads of 64 and 128: positions across 256, 512 and the window (one split, several, the last of
    which merges), two to eleven expert slots of rows below, at and above 512 and 1024 columns, 16-byte pieces or not, and a norm row of two numbers a thread."""
    S = env["synth"]
    L = S.stack_layer
    cfg = S.stack_config(1040, 211, [L(4, 2, dim, dim, 600, v_mix=True, experts=12, top=top, ff=ff, shared_ff=shared_ff),
                                     L(2, 2, dim, dim, None, v_mix=True, experts=12, top=top, ff=ff, shared_ff=shared_ff)])
    m, _, orc = make(env, cfg, seed=5, max_pos=1024)
    toks = np.random.default_rng(dim).integers(0, cfg["vocab"], 640).astype(np.int32)
    want = orc.forward(list(toks))
    for lo, hi in ((0, 3), (252, 260), (508, 516), (596, 604), (636, 640)):
        m.reset_kv()
        if lo:
            m.prefill_rows(toks[:lo], 0, np.array([lo - 1], np.int32))
        got = np.stack([m.decode(int(toks[i]), i)[0] for i in range(lo, hi)])
        assert rel_rms(got, want[lo:hi]) < FP32_TOL, (lo, hi)
    m.free()


@pytest.mark.parametrize("heads,kv_heads,dim,n,window", [(4, 2, 64, 70, 0), (2, 2, 128, 300, 0), (2, 1, 64, 290, 130), (3, 3, 128, 9, 5)])
@pytest.mark.parametrize("T", [1, 3])
def test_an_infinite_value_stays_one(env, heads, kv_heads, dim, n, window, T):
    """The last key's value row has an infinity: that column is infinite for the token that sees it, not NaN, and all others are what
    they are without it (loads beyond the last key read its row again)."""
    rng = np.random.default_rng(n)
    k, v = (rng.standard_normal((n, kv_heads * dim)).astype(np.float32) for _ in range(2))
    q = rng.standard_normal((T, heads * dim)).astype(np.float32)
    col = (kv_heads - 1) * dim + 5
    v[-1, col] = np.inf
    got = run_swa(env, q, k, v, n - T, heads, kv_heads, dim, dim, window, 0.1).reshape(T, heads, dim)
    v[-1, col] = 0.0
    want = run_swa(env, q, k, v, n - T, heads, kv_heads, dim, dim, window, 0.1).reshape(T, heads, dim)
    sees = np.zeros((T, heads, dim), bool)
    sees[-1, heads - heads // kv_heads:, 5] = True
    assert (got[sees] == np.inf).all() and np.array_equal(got[~sees], want[~sees])


@pytest.mark.parametrize("T,width", [(1, 513), (8, 1024), (3, 1025), (1, 2048), (5, 4095), (2, 4097), (1, 8192), (9, 512), (20, 513), (9, 1024), (1025, 1023),
                                     (9, 2047), (1030, 2048), (10, 2049)])
def test_residual_output_norm_of_every_row_length(env, T, width):
    """One, two, four and eight numbers a thread and the loop, in workgroups of 1024 (up to 8 rows) and 256 threads."""
    rng = np.random.default_rng(width)
    x, y = (rng.standard_normal((T, width)).astype(np.float32) for _ in range(2))
    w = (0.1 * rng.standard_normal(width)).astype(np.float32)
    xd, yd, wd = dev(env, x), dev(env, y), dev(env, w)
    env["capi"].check(env["capi"].lib().tl_resid_rmsnorm(xd.ptr, yd.ptr, wd.ptr, T, width, 1e-6, None), "tl_resid_rmsnorm")
    env["capi"].check(env["capi"].lib().tl_device_sync(), "sync")
    want = x + env["oracle"].rms_norm(y.astype(np.float64), w.astype(np.float64), 1e-6, True)
    assert np.allclose(xd.to_numpy(np.float32, (T, width)), want, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("heads,dim,width", [(16, 64, 1024), (16, 128, 1000), (32, 128, 2048), (36, 128, 520)])
def test_projections_and_router_rows_of_every_length(env, heads, dim, width):
    """Queries of 1024, 2048, 4096 and more numbers, routers over rows of one to four pieces a lane: a short portion, a longer one and
    single tokens against the float64 oracle."""
    S = env["synth"]
    L = S.stack_layer
    cfg = S.stack_config(width, 211, [L(heads, 4, dim, dim, 50, v_mix=True, experts=20, top=3, ff=64, shared_ff=32) for _ in range(2)])
    m, _, orc = make(env, cfg, seed=9, max_pos=64)
    toks = np.random.default_rng(width).integers(0, cfg["vocab"], 40).astype(np.int32)
    want = orc.forward(list(toks))
    got = np.concatenate([m.prefill_rows(toks[:5], 0), m.prefill_rows(toks[5:37], 5), np.stack([m.decode(int(toks[i]), i)[0] for i in (37, 38, 39)])])
    assert rel_rms(got, want) < FP32_TOL
    m.free()


@pytest.mark.parametrize("width,heads,n_layers", [(1024, 5, 1), (1024, 16, 2), (2048, 9, 3), (4096, 40, 4), (1536, 4, 3)])
def test_residual_sum_in_front_of_the_next_product(env, width, heads, n_layers):
    """One token's residual norm carried by the next layer's product: none to three moves of the residual row (a layer without feed-forward
    among them), few rows and more rows than waves, single tokens from the captured step and as a portion of one, both against the float64 oracle
    and against the launches of their own."""
    S = env["synth"]
    L = S.stack_layer
    layers = [L(heads, 1, 64, 32, 50, v_mix=True, experts=4, top=2, ff=64, shared_ff=32, mlp=l != 1) for l in range(n_layers)]
    cfg = S.stack_config(width, 211, layers)
    toks = np.random.default_rng(width).integers(0, cfg["vocab"], 30).astype(np.int32)
    got = []
    for fuse in (1, 0):
        m, _, orc = make(env, cfg, seed=9, max_pos=64, TL_STACK_FUSE_RESID=fuse)
        got.append(np.concatenate([m.prefill_rows(toks[:20], 0), np.stack([m.decode(int(toks[i]), i)[0] for i in range(20, 25)]),
                                   m.prefill_rows(toks[25:26], 25), np.stack([m.decode(int(toks[i]), i)[0] for i in range(26, 30)])]))
        assert rel_rms(got[-1], orc.forward(list(toks))) < FP32_TOL
        m.free()
    assert rel_rms(got[0], got[1]) < FP32_TOL


@pytest.mark.parametrize("width,carried", [(512, 1), (520, 0), (1536, 1), (2560, 1), (3072, 1), (3584, 1), (4608, 1), (5120, 1), (5632, 0)])
def test_widths_whose_residual_sum_rides_in_the_next_product(env, width, carried):
    """Every width of one to ten whole 512-column pieces takes the product that carries the residual norm, others do not (the launches are
    counted): single tokens against the float64 oracle."""
    S, capi = env["synth"], env["capi"]
    layers = [S.stack_layer(6, 1, 64, 32, 50, v_mix=True, experts=4, top=2, ff=64, shared_ff=32) for _ in range(2)]
    cfg = S.stack_config(width, 211, layers)
    toks = np.random.default_rng(width).integers(0, cfg["vocab"], 12).astype(np.int32)
    count = ctypes.c_longlong()

    def carried_products():
        capi.check(capi.lib().tl_debug_resid_products(ctypes.byref(count)))
        return count.value

    before = carried_products()
    m, _, orc = make(env, cfg, seed=11, max_pos=32)  # (the step may be captured here)
    m.prefill_rows(toks[:4], 0, np.array([3], np.int32))
    got = np.stack([m.decode(int(toks[i]), i)[0] for i in range(4, 12)])
    assert (carried_products() > before) == bool(carried)
    assert rel_rms(got, orc.forward(list(toks))[4:]) < FP32_TOL
    m.free()


@pytest.mark.parametrize("experts", [1, 2, 15, 16, 17, 33, 64, 65, 130])
def test_router_choice_among_equals_and_without_numbers(env, experts):
    """Choices of a row of lanes, of a wave and of more: logits that are their biases, with equal ones (the lower index first),
    numbers that are none (never chosen while others are left) and as many choices as there are experts; softmax over the chosen in 64 bits
    (an exp's and a quotient's roundings: some 1e-6)."""
    capi, synth = env["capi"], env["synth"]
    rng = np.random.default_rng(experts)
    for kind in ("distinct", "equal", "none"):
        for top in sorted({1, min(4, experts), min(16, experts), experts}):
            b = rng.permutation(experts).astype(np.float32) / 8
            if kind == "equal":
                b = np.round(b).astype(np.float32)
            if kind == "none":
                if top > max(1, experts - 2) or experts < 2:
                    continue
                b[rng.integers(experts)] = np.nan
            xd, wd, bd = dev(env, np.ones((2, 16), np.float32)), dev(env, synth.to_bf16(np.zeros((experts, 16), np.float32))), dev(env, b)
            idd, wtd = env["engine"].DeviceBuffer(8 * top), env["engine"].DeviceBuffer(8 * top)
            capi.check(capi.lib().tl_moe_route(xd.ptr, 2, 16, wd.ptr, bd.ptr, experts, top, idd.ptr, wtd.ptr, None), "tl_moe_route")
            capi.check(capi.lib().tl_device_sync(), "sync")
            order = np.lexsort((np.arange(experts), -np.where(np.isnan(b), -np.inf, b).astype(np.float64)))[:top]
            z = b[order].astype(np.float64)
            p = np.exp(z - z[0])
            for t in range(2):
                assert np.array_equal(idd.to_numpy(np.int32, (2, top))[t], order), (kind, top)
                assert np.allclose(wtd.to_numpy(np.float32, (2, top))[t], p / p.sum(), rtol=4e-6, atol=1e-30), (kind, top)
