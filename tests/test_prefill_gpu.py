"""Batched prefill on the matrix cores (MI355X), through the C-ABI, against the CPU oracle.

Bars: the prefill GEMM with 6 bf16 MFMAs per FP32 product (the default) meets the decode tolerance
(|delta| <= 1e-4 * max(1, |ref|) vs the Kahan-double oracle); the reduced forms are opt-in and carry their own stated
tolerances (3 terms: 1e-3, 1 term = plain bf16: 5e-2 of the output scale). Prefill attention (FP32 MFMA): 2e-5 absolute.
Whole-model prefill (all logits, KV contents) at the decode tolerance, incl. prompts longer than one chunk, ragged
lengths and a prefill that continues an existing cache."""
import numpy as np
import pytest

from oracle.oracle import OracleModel, Q4_K, Q6_K, Q8_0, Q8_K

pytestmark = pytest.mark.gpu
TYPES = {"q4_k": Q4_K, "q6_k": Q6_K, "q8_0": Q8_0, "q8_k": Q8_K}
TOL = {6: 1e-4, 3: 1e-3, 1: 5e-2}


@pytest.fixture(scope="module")
def E(pkg):
    from tinyllama_cpp_amd import engine
    engine.init(0)
    yield engine
    from tinyllama_cpp_amd.capi import lib
    lib().tl_gemm_set_terms(6)


def close(a, b, tol):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return np.abs(a - b) <= tol * np.maximum(1.0, np.abs(b))


def _matmul(E, w, x):
    from tinyllama_cpp_amd.capi import lib, check
    xb = E.DeviceBuffer.from_numpy(np.ascontiguousarray(x, np.float32))
    yb = E.DeviceBuffer(4 * x.shape[0] * w.rows)
    check(lib().tl_matmul_q(w.h, xb.ptr, yb.ptr, x.shape[0], None))
    return yb.to_numpy(np.float32, (x.shape[0], w.rows))


@pytest.mark.parametrize("name,rows,cols,T", [
    ("q4_k", 512, 1024, 8), ("q4_k", 333, 512, 33), ("q4_k", 1024, 2048, 130), ("q6_k", 256, 1024, 200),
    ("q6_k", 100, 256, 64), ("q8_0", 192, 512, 129), ("q8_0", 64, 32, 16), ("q8_k", 128, 768, 40)])
def test_gemm_vs_oracle(E, pkg, oracle, name, rows, cols, T):
    from tinyllama_cpp_amd.capi import lib, check
    t, S = TYPES[name], pkg.synth
    rng = np.random.default_rng(rows + 3 * cols + T)
    blocks = S.random_blocks(t, rows * cols // S.BLOCK_ELEMS[t], rng, w_std=1.0 / np.sqrt(cols))
    x = rng.standard_normal((T, cols)).astype(np.float32)
    sc = np.ones((T, 1), np.float32)  # rows of very different scale share a tile; the bars scale with the row
    sc[0], sc[-1] = 2.0 ** -10, 64.0
    x *= sc
    want = oracle.matmul_q_batch(t, blocks, x, T, rows, cols)
    w = E.QWeight(t, blocks, rows, cols)
    for terms in (6, 3, 1):
        check(lib().tl_gemm_set_terms(terms))
        y = _matmul(E, w, x)
        if terms == 6:
            assert close(y / sc, want / sc, TOL[6]).all(), np.abs(y / sc - want / sc).max()
        else:  # reduced forms: relative to the scale of the token's output row
            rowmax = np.maximum(sc, np.abs(want).max(axis=1, keepdims=True))
            assert (np.abs(y - want) <= TOL[terms] * rowmax).all(), (terms, (np.abs(y - want) / rowmax).max())
    check(lib().tl_gemm_set_terms(6))
    # each token row only depends on its own input row: a batch of the same rows in another order gives the same rows
    perm = rng.permutation(T)
    assert np.array_equal(_matmul(E, w, x[perm]), _matmul(E, w, x)[perm])
    # fewer than 8 tokens: GEMV launches, bit-identical to the mat-vec
    y3 = _matmul(E, w, x[:3])
    assert np.array_equal(y3[1], w.matvec(x[1]))


@pytest.mark.parametrize("name,rows,cols,T", [
    ("q4_k", 333, 4096, 9), ("q4_k", 1024, 14336, 12), ("q6_k", 257, 1024, 32), ("q6_k", 4100, 4096, 40),
    ("q8_0", 100, 192, 17), ("q8_k", 130, 768, 20), ("q4_k", 96, 256, 64), ("q8_0", 2048, 2048, 50)])
def test_direct_small_token_gemm(E, pkg, oracle, monkeypatch, name, rows, cols, T):
    """The f16 form in tl_matmul_q (weights from global memory straight into the operands; launches of at most 32 tokens by
    default, 64 with TL_GEMM_DIRECT=64): every format, row counts off the 64- and 128-row tiles, K splits and a single
    super-block -- against the oracle at the GEMM bars, and against the integer-plane kernel it stands in for
    (TL_GEMM_DIRECT=0): both of the 32-bit grade, so FP32 rounding apart."""
    from tinyllama_cpp_amd.capi import lib, check
    t, S = TYPES[name], pkg.synth
    rng = np.random.default_rng(7 * rows + cols + T)
    blocks = S.random_blocks(t, rows * cols // S.BLOCK_ELEMS[t], rng, w_std=1.0 / np.sqrt(cols))
    x = rng.standard_normal((T, cols)).astype(np.float32)
    sc = np.ones((T, 1), np.float32)
    sc[0], sc[-1] = 2.0 ** -10, 64.0
    x *= sc
    want = oracle.matmul_q_batch(t, blocks, x, T, rows, cols)
    w = E.QWeight(t, blocks, rows, cols)
    rowmax = np.maximum(sc, np.abs(want).max(axis=1, keepdims=True))
    out = {}
    for direct in ("64", "0"):
        monkeypatch.setenv("TL_GEMM_DIRECT", direct)
        for terms in (6, 3):
            check(lib().tl_gemm_set_terms(terms))
            y = _matmul(E, w, x)
            out[direct, terms] = y
            if terms == 6:
                assert close(y / sc, want / sc, TOL[6]).all(), (direct, np.abs(y / sc - want / sc).max())
            else:
                assert (np.abs(y - want) <= TOL[3] * rowmax).all(), (direct, (np.abs(y - want) / rowmax).max())
    check(lib().tl_gemm_set_terms(6))
    assert (np.abs(out["64", 6] - out["0", 6]) <= 2e-5 * rowmax).all()
    monkeypatch.setenv("TL_GEMM_DIRECT", "64")
    perm = rng.permutation(T)
    assert np.array_equal(_matmul(E, w, x[perm]), out["64", 6][perm])
    if T <= 32:  # the default limit takes the same kernel as the explicit one
        monkeypatch.delenv("TL_GEMM_DIRECT")
        assert np.array_equal(_matmul(E, w, x), out["64", 6])


@pytest.mark.parametrize("name,rows,cols,T", [
    ("q4_k", 4096, 4096, 2), ("q4_k", 333, 1024, 3), ("q4_k", 1024, 14336, 5), ("q6_k", 257, 4096, 4),
    ("q6_k", 64, 14336, 7), ("q8_0", 1000, 2048, 6), ("q8_0", 33, 32, 2), ("q8_k", 128, 768, 3), ("q4_k", 1, 256, 7)])
def test_few_tokens_take_the_multi_vector_gemv(E, pkg, oracle, name, rows, cols, T):
    """2..7 tokens: one pass over the weights for up to four tokens (gemv_nv_kernel; 14336 columns only stage two
    vectors at a time; Q8_K falls back to one mat-vec per token). Every row is bit-identical to the single mat-vec
    (same chunk dots, same lane order) and within the GEMV tolerance of the oracle."""
    t, S = TYPES[name], pkg.synth
    rng = np.random.default_rng(rows + cols + T)
    blocks = S.random_blocks(t, rows * cols // S.BLOCK_ELEMS[t], rng, w_std=1.0 / np.sqrt(cols))
    x = rng.standard_normal((T, cols)).astype(np.float32)
    x[0] *= 1e-3
    x[-1] *= 50.0
    w = E.QWeight(t, blocks, rows, cols)
    y = _matmul(E, w, x)
    want = oracle.matmul_q_batch(t, blocks, x, T, rows, cols)
    sc = np.array([1e-3] + [1.0] * (T - 2) + [50.0], np.float32)[:, None]
    assert close(y / sc, want / sc, 1e-4).all(), np.abs(y / sc - want / sc).max()
    for i in range(T):
        assert np.array_equal(y[i], w.matvec(x[i])), i


@pytest.mark.parametrize("name,rows,cols,T", [
    ("q4_k", 512, 1024, 65), ("q4_k", 333, 512, 130), ("q4_k", 4096, 4096, 512), ("q4_k", 1024, 14336, 128),
    ("q6_k", 256, 1024, 200), ("q6_k", 4100, 4096, 257), ("q8_0", 192, 512, 129), ("q8_0", 2048, 2048, 384),
    ("q8_k", 128, 768, 140), ("q6_k", 1000, 256, 100), ("q4_k", 4096, 4096, 64), ("q4_k", 700, 14336, 40),
    ("q6_k", 1024, 4096, 50), ("q8_0", 300, 512, 33)])
def test_expanded_plane_gemm_is_bit_identical(E, pkg, oracle, monkeypatch, name, rows, cols, T):
    """tl_qweight_expand: the batched GEMM fed by LDS-DMA from the resident bf16 integer plane + scale words
    (gemm_px_kernel, 256-row tiles, producers that only issue DMAs) forms exactly the sums of the kernel that unpacks the
    quantized planes in every workgroup (gemm_qi_ws_kernel): every format, row counts off the 256-row tile, K splits (few
    tiles) and none (many), token counts off the 128-token tile, 3- and 6-term products -- bit for bit, and within the GEMM
    bar of the oracle."""
    from tinyllama_cpp_amd.capi import lib, check
    t, S = TYPES[name], pkg.synth
    rng = np.random.default_rng(11 * rows + cols + T)
    blocks = S.random_blocks(t, rows * cols // S.BLOCK_ELEMS[t], rng, w_std=1.0 / np.sqrt(cols))
    x = rng.standard_normal((T, cols)).astype(np.float32)
    sc = np.ones((T, 1), np.float32)
    sc[0], sc[-1] = 2.0 ** -10, 64.0
    x *= sc
    w = E.QWeight(t, blocks, rows, cols)
    before = {}
    for terms in (6, 3):
        check(lib().tl_gemm_set_terms(terms))
        before[terms] = _matmul(E, w, x)
    def px_launches():
        import ctypes as C
        n = C.c_longlong()
        check(lib().tl_debug_gemm_px_launches(C.byref(n)))
        return n.value

    monkeypatch.setenv("TL_GEMM_PX_SLICES", "0")  # the unpacking kernel's K slices: then the sums agree bit for bit
    n0 = px_launches()
    nbytes = w.expand()
    mt, nk = (rows + 255) // 256, cols // 32
    assert nbytes == mt * nk * (256 * 32 * 2 + 3 * 256 * 4)
    for terms in (6, 3):
        check(lib().tl_gemm_set_terms(terms))
        y = _matmul(E, w, x)
        assert np.array_equal(y, before[terms]), (terms, np.abs(y - before[terms]).max())
        n1 = px_launches()
        monkeypatch.setenv("TL_GEMM_PX", "0")  # the planes are there but ignored: the unpacking kernel again
        assert np.array_equal(_matmul(E, w, x), before[terms])
        monkeypatch.delenv("TL_GEMM_PX")
        assert px_launches() == n1
    assert n1 == n0 + 2  # (one launch per product: the expanded-plane kernel formed y)
    monkeypatch.setenv("TL_GEMM_PX_BM", "128")  # half a record per workgroup (the form taken for few row tiles): same sums
    assert np.array_equal(_matmul(E, w, x), before[3])
    monkeypatch.delenv("TL_GEMM_PX_BM")
    assert px_launches() == n1 + 1
    check(lib().tl_gemm_set_terms(6))
    # the kernel's own K slices (the default): other partial sums, FP32 rounding apart
    monkeypatch.delenv("TL_GEMM_PX_SLICES")
    y6 = _matmul(E, w, x)
    rowmax = np.maximum(sc, np.abs(before[6]).max(axis=1, keepdims=True))
    assert (np.abs(y6 - before[6]) <= 2e-5 * rowmax).all()
    if rows * cols * T <= 4096 * 4096 * 64:  # (the oracle's Kahan-double dots: seconds)
        want = oracle.matmul_q_batch(t, blocks, x, T, rows, cols)
        assert close(y / sc, want / sc, TOL[3]).all()
        assert close(y6 / sc, want / sc, TOL[6]).all()
    w.free()


def test_gemm_edge_scales(E, pkg, oracle):
    """fp16 sub-normal / zero / negative super-scales inside an MFMA tile."""
    from tinyllama_cpp_amd.capi import lib, check
    S = pkg.synth
    rng = np.random.default_rng(4)
    rows, cols, T = 64, 512, 24
    x = rng.standard_normal((T, cols)).astype(np.float32)
    check(lib().tl_gemm_set_terms(6))
    for t in (Q4_K, Q6_K, Q8_0, Q8_K):
        blocks = S.random_blocks(t, rows * cols // S.BLOCK_ELEMS[t], rng, w_std=0.02)
        edge = S.edge_blocks(t, rng)
        keep = [i for i, h in enumerate(S.EDGE_F16) if (h & 0x7c00) != 0x7c00 and (h & 0x7fff) < 0x7000]
        blocks[: len(keep)] = edge[keep]
        want = oracle.matmul_q_batch(t, blocks, x, T, rows, cols)
        y = _matmul(E, E.QWeight(t, blocks, rows, cols), x)
        assert np.isfinite(want).all()
        assert close(y, want, 1e-4 * max(1.0, np.abs(want).max())).all()


@pytest.mark.parametrize("nh,nkv,hd,T,start", [(4, 2, 64, 33, 0), (8, 2, 64, 100, 57), (32, 8, 128, 70, 0),
                                               (16, 4, 128, 45, 200), (8, 8, 128, 1, 31),
                                               # pairs of query tiles: an odd tile count (the middle tile alone), heads not
                                               # a multiple of 8, several key tiles per wave (the K prefetch), the bench shape
                                               (8, 2, 128, 160, 0), (12, 4, 128, 300, 100), (8, 2, 64, 257, 300),
                                               (32, 8, 128, 512, 0)])
def test_prefill_attention_vs_oracle(E, oracle, nh, nkv, hd, T, start):
    from tinyllama_cpp_amd.capi import lib, check
    rng = np.random.default_rng(nh * 100 + T)
    npos = start + T
    max_seq = npos + 3
    kc = np.zeros((max_seq, nkv * hd), np.float32)
    vc = np.zeros((max_seq, nkv * hd), np.float32)
    kc[:npos] = rng.standard_normal((npos, nkv * hd))
    vc[:npos] = rng.standard_normal((npos, nkv * hd))
    Q = rng.standard_normal((T, nh * hd)).astype(np.float32)
    dev = lambda a: E.DeviceBuffer.from_numpy(np.ascontiguousarray(a, np.float32))
    kb, vb, Qb, Ob = dev(kc), dev(vc), dev(Q), E.DeviceBuffer(Q.nbytes)
    scale = float(np.float32(1.0) / np.sqrt(np.float32(hd)))
    check(lib().tl_attention_batch_prefill(Qb.ptr, kb.ptr, vb.ptr, Ob.ptr, T, start, max_seq, nh, nkv, hd, scale, None))
    got = Ob.to_numpy(np.float32, Q.shape)
    want = oracle.attention_batch(Q, kc, vc, T, start, nh, nkv, hd)
    assert np.allclose(got, want, rtol=0, atol=2e-5), np.abs(got - want).max()


@pytest.mark.parametrize("shape,mix,T", [("tiny", "q4_k_m", 600), ("tiny-gqa", "q6_k", 129), ("tiny-gqa", "q8_0", 8),
                                         ("tiny-tp", "q4_k_m", 77)])
def test_model_prefill_batched_vs_oracle(E, pkg, oracle, shape, mix, T):
    cfg = dict(pkg.synth.SHAPES[shape], max_pos=max(640, T + 8) if T > 256 else pkg.synth.SHAPES[shape]["max_pos"])
    cfg, tensors = pkg.synth.build_model(cfg, mix, seed=8)
    m = E.Model(cfg).load(tensors)
    om = OracleModel(oracle, cfg, tensors)
    toks = np.random.default_rng(T).integers(0, cfg["vocab"], T).astype(np.int32)
    last, allb = m.prefill(toks, 0, all_logits=True)
    X = np.stack([om.lookup_embedding(t) for t in toks])
    _, lb = om.forward_batch(X, 0)
    assert close(allb, lb, TOL[6]).all(), np.abs(allb - lb).max()
    assert close(last, lb[-1], TOL[6]).all()
    for layer in (0, cfg["n_layers"] - 1):
        k, v = m.kv_cache(layer, T)
        assert close(k, om.kcache(layer, T), TOL[6]).all()
        assert close(v, om.vcache(layer, T), TOL[6]).all()
    # greedy continuation from the prefilled cache == the oracle's continuation from its own cache
    if T + 6 <= cfg["max_pos"]:
        first = int(np.argmax(lb[-1]))
        got = m.generate_greedy(first, T, 6, 1.0, history=[first])
        tok, want = first, []
        for i in range(6):
            _, lg = om.forward(om.lookup_embedding(tok), T + i)
            tok = int(np.argmax(lg))
            want.append(tok)
        assert got.tolist() == want
    m.free()
    om.close()


def test_model_prefill_continues_cache_and_reduced_terms(E, pkg, oracle):
    """A second prefill call appends to the cache (start_pos > 0); the token-by-token route (min_batch above the
    prompt length) and the batched route agree; the reduced-precision forms stay within their stated tolerances."""
    cfg, tensors = pkg.synth.build_model("tiny-gqa", "q4_k_m", seed=3)
    m = E.Model(cfg).load(tensors)
    om = OracleModel(oracle, cfg, tensors)
    toks = np.random.default_rng(6).integers(0, cfg["vocab"], 90).astype(np.int32)
    X = np.stack([om.lookup_embedding(t) for t in toks])
    _, lb = om.forward_batch(X, 0)
    m.prefill(toks[:50], 0)
    last = m.prefill(toks[50:], 50)
    assert close(last, lb[-1], TOL[6]).all(), np.abs(last - lb[-1]).max()
    m.reset_kv()
    m.set_prefill(terms=0, min_batch=1000)
    serial = m.prefill(toks, 0)
    assert close(serial, lb[-1], TOL[6]).all()
    for terms in (3, 1):
        m.reset_kv()
        m.set_prefill(terms=terms, min_batch=8)
        got = m.prefill(toks, 0)
        scale = max(1.0, np.abs(lb[-1]).max())
        assert (np.abs(got - lb[-1]) <= TOL[terms] * scale).all(), (terms, np.abs(got - lb[-1]).max())
    from tinyllama_cpp_amd.capi import TlError
    with pytest.raises(TlError):
        m.set_prefill(terms=2)
    with pytest.raises(TlError):
        m.prefill(toks, cfg["max_pos"] - 10)  # runs past the cache
    m.free()
    om.close()


# a model without the f16 form of the chunk products: Q8_0 rows (352 columns) that are not whole pairs of blocks
ODD_Q8 = dict(hidden=256, inter=352, n_heads=4, n_kv_heads=2, n_layers=2, vocab=64, max_pos=160, eps=1e-5, rope_theta=10000.0)


def _count(name):
    import ctypes as C
    from tinyllama_cpp_amd.capi import check, lib
    n = C.c_longlong()
    check(getattr(lib(), name)(C.byref(n)))
    return n.value


@pytest.mark.parametrize("shape,mix,n,every", [("tiny-gqa", "q4_k_m", 150, (1,)), ("tiny-tp", "q6_k", 77, (1,)), (ODD_Q8, "q8_0", 150, (6, 3, 1))])
def test_prefill_attention_writes_the_gemm_planes_bit_identically(E, pkg, monkeypatch, shape, mix, n, every):
    """The prefill attention kernel writes the bf16 planes of the attn_output GEMM itself (no split launch): every logit of an
    all-logits prefill -- one call, and a second call appending to the cache -- is bit for bit what TL_ATTN_PLANES=0 (attention ->
    float rows -> split launch) gives. With plain bf16 chunks, and, for a model whose matrices have no f16 form, with 6 and 3 MFMA
    terms. The split launches are counted: a layer of a chunk has three, and one more with TL_ATTN_PLANES=0."""
    rng = np.random.default_rng(12)
    cfg, tensors = pkg.synth.build_model(shape, mix, seed=4)
    toks = rng.integers(0, cfg["vocab"], n).astype(np.int32)
    m = E.Model(cfg).load(tensors)
    for terms in every:
        m.set_prefill(terms=terms, min_batch=8)
        got, splits = {}, {}
        for ap in ("0", "1"):
            monkeypatch.setenv("TL_ATTN_PLANES", ap)
            m.reset_kv()
            before = _count("tl_debug_split_launches")
            _, a = m.prefill(toks[:n - 40], 0, all_logits=True)
            _, b = m.prefill(toks[n - 40:], n - 40, all_logits=True)
            got[ap], splits[ap] = [np.array(a), np.array(b)], _count("tl_debug_split_launches") - before
        assert splits["0"] - splits["1"] == 2 * cfg["n_layers"], (terms, splits)
        for a, b in zip(got["0"], got["1"]):
            assert a.shape == b.shape and np.array_equal(a, b), (terms, np.abs(a - b).max())
    m.free()


def test_expanded_planes_of_models(E, pkg, oracle, monkeypatch):
    """A model whose matrices all have the f16 form keeps no expanded planes, whatever TL_PREFILL_PLANES says: no chunk of it reads
    them. One with a matrix that has none does (unless 0), and its chunks go through them: the logits of the oracle, and bit for bit
    those of the kernel that unpacks the quantized planes."""
    cfg, tensors = pkg.synth.build_model("tiny-gqa", "q8_0", seed=4)
    monkeypatch.setenv("TL_PREFILL_PLANES", "1")
    m = E.Model(cfg).load(tensors)
    assert m.prefill_planes_bytes() == 0
    m.free()
    cfg, tensors = pkg.synth.build_model(ODD_Q8, "q8_0", seed=4)
    toks = np.random.default_rng(3).integers(0, cfg["vocab"], 100).astype(np.int32)
    monkeypatch.setenv("TL_GEMM_PX_SLICES", "0")  # the unpacking kernel's K slices
    got = []
    for planes in ("1", "0"):
        monkeypatch.setenv("TL_PREFILL_PLANES", planes)
        m = E.Model(cfg).load(tensors)
        assert (m.prefill_planes_bytes() > 0) == (planes == "1")
        before = _count("tl_debug_gemm_px_launches")
        got.append(np.array(m.prefill(toks, 0, all_logits=True)[1]))
        assert (_count("tl_debug_gemm_px_launches") > before) == (planes == "1")
        m.free()
    assert np.array_equal(got[0], got[1])
    om = OracleModel(oracle, cfg, tensors)
    _, want = om.forward_batch(np.stack([om.lookup_embedding(t) for t in toks]), 0)
    assert close(got[0], want, TOL[6]).all()


@pytest.mark.parametrize("name,rows,cols,T", [
    ("q4_k", 1, 256, 8), ("q4_k", 65, 512, 16), ("q4_k", 129, 4096, 17), ("q4_k", 300, 14336, 32), ("q6_k", 63, 256, 9),
    ("q6_k", 130, 2304, 16), ("q6_k", 97, 768, 31), ("q8_0", 31, 64, 8), ("q8_0", 70, 320, 13), ("q8_0", 129, 448, 27),
    ("q8_0", 64, 1088, 32), ("q8_k", 127, 512, 11), ("q8_k", 33, 1280, 30)])
def test_half_plane_gemm_edges(E, pkg, name, rows, cols, T):
    """tl_hgemm.hip through tl_matmul_q (16- and 32-token tiles): rows and tokens off the tiles, one and several super-blocks,
    K slices, Q8_0 rows that end inside a super-block; magnitudes 2^-20 .. 2^20 apart from super-block to super-block and
    rows of zeros. Against float64 over the dequantized weights: an activation is held to 2^-22 of its super-block's largest
    value at worst, a running sum of 256 products is rounded 16 to 48 times (2^-24 each), their sum once per super-block: with
    |w| . |x| as the scale of a row's dot, 2^-22 + 48 * 2^-24 + (cols / 256) * 2^-24 bounds the error; measured a tenth."""
    t, S = TYPES[name], pkg.synth
    rng = np.random.default_rng(rows + 7 * cols + T)
    w = E.QWeight(t, S.random_blocks(t, rows * cols // S.BLOCK_ELEMS[t], rng, w_std=1.0 / np.sqrt(cols)), rows, cols)
    x = rng.standard_normal((T, cols)).astype(np.float32)
    x *= np.exp2(rng.integers(-20, 21, (T, -(-cols // 256)))).astype(np.float32).repeat(256, axis=1)[:, :cols]
    x[T // 2] = 0.0
    W = w.dequantize().astype(np.float64)
    want = x.astype(np.float64) @ W.T
    # (Q4_K: the scale q and minimum m parts are summed apart, their sizes are what rounds)
    scale = np.abs(x).astype(np.float64) @ (np.abs(W) + 4.0 * np.abs(W).max(axis=1, keepdims=True)).T
    y = _matmul(E, w, x)
    assert (np.abs(y - want) <= (2.0 ** -22 + 48 * 2.0 ** -24 + cols / 256 * 2.0 ** -24) * scale).all(), (np.abs(y - want) / np.maximum(scale, 1e-30)).max()
    assert not y[T // 2].any()
    w.free()


@pytest.mark.parametrize("shape", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("name,rows,cols,T,slices", [
    ("q4_k", 1, 256, 65, 1), ("q4_k", 129, 768, 127, 2), ("q4_k", 257, 2304, 300, 5), ("q4_k", 300, 1280, 63, 5), ("q6_k", 1, 512, 129, 2),
    ("q6_k", 257, 1792, 65, 4), ("q6_k", 129, 256, 300, 1), ("q8_0", 129, 64, 65, 1), ("q8_0", 257, 320, 127, 2), ("q8_0", 1, 1088, 300, 5),
    ("q8_0", 255, 1984, 64, 3), ("q8_0", 70, 192, 129, 1), ("q8_k", 257, 1280, 127, 3), ("q8_k", 130, 256, 65, 1)])
def test_half_plane_gemm_shapes(E, pkg, shape, name, rows, cols, T, slices):
    """Every workgroup shape of tl_hgemm.hip by itself, those of long chunks (2, 3, 4: the ring of three 64-column steps, two row
    tiles a wave, eight waves) at sizes off their tiles: one row, one more than a tile, tokens around 64 and 128, one super-block,
    K slices with a short last one, Q8_0 rows that end inside a super-block. The bound of test_half_plane_gemm_edges."""
    from tinyllama_cpp_amd.capi import check, lib
    t, S = TYPES[name], pkg.synth
    rng = np.random.default_rng(rows + 7 * cols + T)
    w = E.QWeight(t, S.random_blocks(t, rows * cols // S.BLOCK_ELEMS[t], rng, w_std=1.0 / np.sqrt(cols)), rows, cols)
    x = rng.standard_normal((T, cols)).astype(np.float32)
    x *= np.exp2(rng.integers(-20, 21, (T, -(-cols // 256)))).astype(np.float32).repeat(256, axis=1)[:, :cols]
    x[T // 2] = 0.0
    xb, yb = E.DeviceBuffer.from_numpy(x), E.DeviceBuffer(4 * T * rows)
    check(lib().tl_memset(yb.ptr, 0xff, yb.nbytes, None))
    rc = lib().tl_debug_half_gemm(w.h, xb.ptr, yb.ptr, T, shape, slices, None)
    if shape == 3 and name in ("q6_k", "q8_0"):
        assert rc != 0  # (not instantiated)
        w.free()
        return
    check(rc)
    y = yb.to_numpy(np.float32, (T, rows))
    W = w.dequantize().astype(np.float64)
    want = x.astype(np.float64) @ W.T
    scale = np.abs(x).astype(np.float64) @ (np.abs(W) + 4.0 * np.abs(W).max(axis=1, keepdims=True)).T
    assert (np.abs(y - want) <= (2.0 ** -22 + 48 * 2.0 ** -24 + cols / 256 * 2.0 ** -24) * scale).all(), (np.abs(y - want) / np.maximum(scale, 1e-30)).max()
    assert not y[T // 2].any()
    assert lib().tl_debug_half_gemm(w.h, xb.ptr, yb.ptr, T, shape, 8 if cols <= 1792 else 7, None) != 0  # an empty slice: refused
    w.free()


@pytest.mark.parametrize("heads,kv_heads,hd", [(8, 1, 64), (6, 2, 128), (4, 4, 64)])
def test_short_prompts_attend_token_by_token(E, pkg, monkeypatch, heads, kv_heads, hd):
    """Chunks of few tokens over few keys take the batched FP32 attention. Tokens and starts on both sides of its line (with a CU's 400 keys)
    and around a workgroup a CU, against the FP32 prompt kernel (TL_HATTN=0): two layers, within 2^-22 a product and layer. Which attention
    ran is counted; where it is the batched one, the f16 kernel's logits (TL_ATTN_SHORT=0) are others, elsewhere the same."""
    E.init(0)
    cfg = dict(pkg.synth.SHAPES["tiny-gqa"], hidden=heads * hd, n_heads=heads, n_kv_heads=kv_heads, n_layers=2, max_pos=640)
    cfg, tensors = pkg.synth.build_model(cfg, "q4_k_m", seed=6)
    m = E.Model(cfg).load(tensors)
    toks = np.random.default_rng(hd).integers(0, cfg["vocab"], 620).astype(np.int32)
    cus, got = 256, {}  # (compute units of an MI355X)
    cases = [(0, 9), (0, 31), (0, 65), (0, 129), (0, 257), (65, 17), (300, 40), (380, 20), (380, 21), (390, 64), (560, 10)]
    few = {(start, n) for start, n in cases if max(n * kv_heads * (2 if heads == 8 * kv_heads else 1), cus) * (start + n) <= 400 * cus}
    assert few and len(few) < len(cases)
    for route, hattn, short in (("fp32", "0", "1"), ("f16", "1", "0"), ("rule", "1", "1")):
        for start, n in cases:
            m.reset_kv()
            monkeypatch.setenv("TL_HATTN", "0")  # (the same rows before the chunk)
            if start:
                m.prefill(toks[:start])
            monkeypatch.setenv("TL_HATTN", hattn)
            monkeypatch.setenv("TL_ATTN_SHORT", short)
            before = _count("tl_debug_half_attention_launches")
            got[route, start, n] = m.prefill(toks[start:start + n], start, all_logits=True)[1]
            half = _count("tl_debug_half_attention_launches") - before
            assert half == (0 if route == "fp32" or (route == "rule" and (start, n) in few) else 2), (route, start, n, half)
    m.free()
    for at in cases:
        want = got["fp32", at[0], at[1]]
        for route in ("f16", "rule"):
            assert np.linalg.norm(got[route, at[0], at[1]] - want) <= 4e-6 * np.linalg.norm(want), (route, at)
        assert np.array_equal(got["rule", at[0], at[1]], got["f16", at[0], at[1]]) == (at not in few), at


@pytest.mark.parametrize("shape", [5, 6, 7, 8])
@pytest.mark.parametrize("name,rows,cols,T,slices", [
    ("q4_k", 1, 256, 1, 1), ("q4_k", 63, 768, 7, 3), ("q4_k", 129, 2304, 9, 5), ("q4_k", 64, 512, 33, 1), ("q6_k", 65, 512, 8, 2),
    ("q6_k", 127, 768, 17, 1), ("q6_k", 128, 1792, 31, 4), ("q8_0", 129, 64, 3, 1), ("q8_0", 65, 320, 16, 2), ("q8_0", 1, 1088, 8, 5),
    ("q8_0", 255, 1984, 32, 3), ("q8_k", 130, 1280, 8, 3), ("q8_k", 63, 256, 15, 1)])
def test_half_plane_gemm_shapes_of_few_tokens(E, pkg, shape, name, rows, cols, T, slices):
    """Both parts of eight tokens in one instruction (5, 6), eight waves of 16 rows (6, 7), two fragments of 16 tokens (8): one token, one
    more than a tile, rows around 64 and 128, slices. The bound of test_half_plane_gemm_edges."""
    test_half_plane_gemm_shapes(E, pkg, shape, name, rows, cols, T, slices)


@pytest.mark.parametrize("name,rows,cols,T,slices", [
    ("q4_k", 255, 256, 63, 1), ("q4_k", 600, 2304, 129, 3), ("q6_k", 257, 768, 64, 1), ("q6_k", 255, 768, 65, 3), ("q6_k", 1, 256, 300, 1),
    ("q8_0", 511, 1280, 130, 2), ("q8_0", 70, 256, 65, 1), ("q8_k", 257, 768, 65, 2), ("q8_k", 33, 2304, 64, 1)])
def test_half_plane_gemm_lds_shape_has_the_sums_of_shape_4(E, pkg, name, rows, cols, T, slices):
    """256 rows in eight waves with weights through LDS against 128 rows in four with weights through registers: the same bits. Rows and
    tokens off the tiles, odd numbers of super-blocks (two rows' d in one dword, the last row's at the end of its plane), slices of
    one super-block and a short last one."""
    from tinyllama_cpp_amd.capi import check, lib
    t, S = TYPES[name], pkg.synth
    rng = np.random.default_rng(rows + 7 * cols + T)
    w = E.QWeight(t, S.random_blocks(t, rows * cols // S.BLOCK_ELEMS[t], rng, w_std=1.0 / np.sqrt(cols)), rows, cols)
    xb, yb = E.DeviceBuffer.from_numpy(rng.standard_normal((T, cols)).astype(np.float32)), E.DeviceBuffer(4 * T * rows)
    got = []
    for shape in (2, 4):
        check(lib().tl_memset(yb.ptr, 0xff, yb.nbytes, None))
        check(lib().tl_debug_half_gemm(w.h, xb.ptr, yb.ptr, T, shape, slices, None))
        got.append(yb.to_numpy(np.uint32, (T, rows)))
    assert np.array_equal(got[0], got[1])
    w.free()


@pytest.mark.parametrize("rows,cols,T,slices", [(511, 256, 64, 1), (513, 1280, 65, 2), (1030, 512, 63, 1)])
def test_half_plane_gemm_waves_of_64_rows(E, pkg, rows, cols, T, slices):
    """512 rows a workgroup around its tile. The bound of test_half_plane_gemm_edges."""
    from tinyllama_cpp_amd.capi import check, lib
    S = pkg.synth
    rng = np.random.default_rng(rows)
    w = E.QWeight(Q4_K, S.random_blocks(Q4_K, rows * cols // 256, rng, w_std=1.0 / np.sqrt(cols)), rows, cols)
    x = rng.standard_normal((T, cols)).astype(np.float32)
    xb, yb = E.DeviceBuffer.from_numpy(x), E.DeviceBuffer(4 * T * rows)
    check(lib().tl_debug_half_gemm(w.h, xb.ptr, yb.ptr, T, 3, slices, None))
    W = w.dequantize().astype(np.float64)
    scale = np.abs(x).astype(np.float64) @ (np.abs(W) + 4.0 * np.abs(W).max(axis=1, keepdims=True)).T
    y = yb.to_numpy(np.float32, (T, rows))
    assert (np.abs(y - x.astype(np.float64) @ W.T) <= (2.0 ** -22 + 48 * 2.0 ** -24 + cols / 256 * 2.0 ** -24) * scale).all()
    w.free()


@pytest.mark.parametrize("shape", [2, 3, 4])
@pytest.mark.parametrize("T", [512, 513, 1024, 1050, 1500])
def test_half_plane_gemm_panels_of_token_tiles(E, pkg, shape, T):
    """Workgroups walk panels of 64-token tiles: one panel (8 and 9 tiles), equal ones (16), a last one that is narrower, several row
    tiles and K slices. Every
    token's row equals, to the bit, that of a launch of 64 tokens."""
    from tinyllama_cpp_amd.capi import check, lib
    S, rows, cols = pkg.synth, 520, 512
    rng = np.random.default_rng(T)
    w = E.QWeight(Q4_K, S.random_blocks(Q4_K, rows * cols // 256, rng, w_std=1.0 / np.sqrt(cols)), rows, cols)
    x = rng.standard_normal((T, cols)).astype(np.float32)

    def run(a, slices):
        xb, yb = E.DeviceBuffer.from_numpy(np.ascontiguousarray(a)), E.DeviceBuffer(4 * a.shape[0] * rows)
        check(lib().tl_memset(yb.ptr, 0xff, yb.nbytes, None))
        check(lib().tl_debug_half_gemm(w.h, xb.ptr, yb.ptr, a.shape[0], shape, slices, None))
        return yb.to_numpy(np.float32, (a.shape[0], rows))

    for slices in (1, 2):
        want = np.concatenate([run(x[i:i + 64], slices) for i in range(0, T, 64)])
        assert np.array_equal(run(x, slices).view(np.uint32), want.view(np.uint32))
    w.free()


@pytest.mark.parametrize("name", ["q4_k", "q6_k", "q8_0", "q8_k"])
@pytest.mark.parametrize("power", [125, 121, -112, -120])
def test_half_plane_gemm_largest_and_smallest_activations(E, pkg, name, power):
    """Activations at the ends of FP32's range (a row's largest just below 2^128, or far below 2^-100), another row at 1: the power
    of two that brings a super-block into f16's range exists for all of them, and so do Q4_K's block sums. Finite products keep
    their relative error (test_half_plane_gemm_edges' bound; below 2^-126 an output rounds to 2^-149)."""
    t, S = TYPES[name], pkg.synth
    rows, cols, T = 70, 512, 9
    rng = np.random.default_rng(power + 200)
    w = E.QWeight(t, S.random_blocks(t, rows * cols // S.BLOCK_ELEMS[t], rng, w_std=1.0 / np.sqrt(cols)), rows, cols)
    x = rng.uniform(-4.0, 4.0, (T, cols)).astype(np.float32)
    x[3:] = np.ldexp(x[3:], power)
    W = w.dequantize().astype(np.float64)
    want = x.astype(np.float64) @ W.T
    scale = np.abs(x).astype(np.float64) @ (np.abs(W) + 4.0 * np.abs(W).max(axis=1, keepdims=True)).T
    fits = np.abs(want) < 2.0 ** 127
    assert fits.mean() > 0.5
    y = _matmul(E, w, x)
    assert (np.abs(y - want) <= (2.0 ** -22 + 50 * 2.0 ** -24) * scale + 2.0 ** -147)[fits].all()
    w.free()


@pytest.mark.parametrize("heads,kv,hd,start,T", [
    (4, 2, 64, 0, 8), (8, 1, 64, 33, 95), (16, 16, 64, 31, 33), (4, 1, 64, 900, 129), (6, 2, 128, 0, 129), (2, 2, 128, 63, 64),
    (6, 2, 128, 1000, 300), (8, 8, 128, 7, 150), (16, 2, 128, 2000, 9)])
def test_half_attention_edges(E, pkg, monkeypatch, heads, kv, hd, start, T):
    """tl_hattn.hip against the FP32 matrix kernel (TL_HATTN=0): groups of 1 to 8 heads, rows and keys on and off the tiles of
    128 and 32, one and several pieces of the keys, tiles whose values are 2^-9 .. 2^9 apart (the common exponent of the running
    sum) and an all-zero tile. A score's error is at most 2^-21 |q| |k| scale from the parts and hd 2^-24 of it from the sums;
    with |q| |k| scale below 16 here, and as much again from the values, the outputs agree to 2 * 16 * (2^-21 + hd 2^-24) < 3e-4
    at worst; errors are independent, so the L2 distance of the logits is held to 1e-5. (TL_ATTN_SHORT=0: the shorter ones would take
    the batched attention.)"""
    monkeypatch.setenv("TL_ATTN_SHORT", "0")
    cfg = dict(hidden=heads * hd, inter=256, n_heads=heads, n_kv_heads=kv, n_layers=1, vocab=64, max_pos=start + T, eps=1e-5,
               rope_theta=10000.0)
    _, tensors = pkg.synth.build_model(cfg, "q8_0", seed=heads + T)
    m = E.Model(cfg).load(tensors)
    m.set_prefill(terms=6, min_batch=8)
    rng = np.random.default_rng(start + T)
    K = rng.standard_normal((start, kv * hd)).astype(np.float32)
    V = rng.standard_normal((start, kv * hd)).astype(np.float32)
    V *= np.exp2(rng.integers(-9, 10, -(-start // 32))).astype(np.float32).repeat(32)[:start, None]
    K[32:64] = V[32:64] = 0.0
    toks = rng.integers(0, cfg["vocab"], T).astype(np.int32)
    got = []
    for route in ("0", "1"):
        monkeypatch.setenv("TL_HATTN", route)
        m.reset_kv()
        if start:
            m.set_kv_cache(0, K, V)
        before = _count("tl_debug_half_attention_launches")
        got.append(np.array(m.prefill(toks, start, all_logits=True)[1], np.float64))
        assert _count("tl_debug_half_attention_launches") - before == int(route)
    m.free()
    assert np.isfinite(got[1]).all() and not np.array_equal(got[0], got[1])
    assert np.linalg.norm(got[1] - got[0]) <= 1e-5 * np.linalg.norm(got[0]), np.linalg.norm(got[1] - got[0]) / np.linalg.norm(got[0])


@pytest.mark.parametrize("mix", ["q4_k_m", "q6_k"])
def test_split_products_of_long_chunks_stay_in_the_models_buffers(E, pkg, mix):
    """ffn_down of 3072 x 8192 in Q6_K and 1400 tokens takes four K slices: 17.2 million partial sums. They have a place in the
    model's own workspaces (summed by the next kernel), so once a first prompt has made those, prompts of other lengths allocate
    nothing, in the model or process-wide (tl_shutdown drops what other tests left there)."""
    import ctypes as C
    from tinyllama_cpp_amd.capi import check, lib
    hip = C.CDLL("libamdhip64.so")

    def free_bytes():
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    cfg = dict(hidden=3072, inter=8192, n_heads=24, n_kv_heads=8, n_layers=1, vocab=64, max_pos=2048, eps=1e-5, rope_theta=10000.0)
    _, tensors = pkg.synth.build_model(cfg, mix, seed=1)
    m = E.Model(cfg).load(tensors)
    check(lib().tl_shutdown(), "tl_shutdown")
    toks = np.random.default_rng(1).integers(0, cfg["vocab"], 2048).astype(np.int32)
    m.prefill(toks, 0)
    before = free_bytes()
    for T in (1100, 1380, 1400, 1660, 600, 300, 100, 20):
        m.reset_kv()
        m.prefill(toks[:T], 0)
        assert free_bytes() == before, T
    m.free()


@pytest.mark.parametrize("max_pos", [2048, 80])
def test_short_first_prompts_make_the_workspaces_of_long_ones(E, pkg, max_pos):
    """A first prompt of 20 tokens, whose attention needs no workspace, makes that of the f16 attention all the same (some 145 MB; with 80
    positions no chunk ever takes it): longer prompts and a prompt behind another allocate no more than their token ids."""
    import ctypes as C
    hip = C.CDLL("libamdhip64.so")

    def free_bytes():
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    E.init(0)
    cfg = dict(hidden=512, inter=512, n_heads=4, n_kv_heads=2, n_layers=1, vocab=64, max_pos=max_pos, eps=1e-5, rope_theta=10000.0)
    _, tensors = pkg.synth.build_model(cfg, "q6_k", seed=2)
    m = E.Model(cfg).load(tensors)
    toks = np.random.default_rng(1).integers(0, cfg["vocab"], max_pos).astype(np.int32)
    m.prefill(toks[:20], 0)
    before = free_bytes()
    for start, T in ((0, max_pos), (0, max_pos // 2), (max_pos // 2, max_pos // 2)):
        m.prefill(toks[start:start + T], start)
        assert before - free_bytes() <= (2 << 20), (start, T, before - free_bytes())
    m.free()


@pytest.mark.parametrize("T", [2048, 2049, 2600])
def test_prefill_chunks_of_2048(E, pkg, T):
    """Prompts around the largest chunk: the last logits of the whole prompt against the last row of an all-logits prefill, which
    walks the prompt in chunks of 512. The same products in the same grade; only which K slices and key pieces are summed apart
    differs: 32-bit rounding, some 2^-22 a layer. And the packed form of the same prompt."""
    cfg = dict(hidden=256, inter=512, n_heads=4, n_kv_heads=2, n_layers=2, vocab=64, max_pos=2700, eps=1e-5, rope_theta=10000.0)
    _, tensors = pkg.synth.build_model(cfg, "q4_k_m", seed=T)
    m = E.Model(cfg).load(tensors)
    m.batch_init(3)
    toks = np.random.default_rng(T).integers(0, cfg["vocab"], T).astype(np.int32)
    last = np.array(m.prefill(toks, 0), np.float64)
    m.reset_kv()
    rows = np.array(m.prefill(toks, 0, all_logits=True)[1], np.float64)
    packed = np.array(m.batch_prefill_packed([toks], slots=[2])[0][0], np.float64)
    for got in (last, packed):
        assert np.linalg.norm(got - rows[-1]) <= 4e-6 * np.linalg.norm(rows[-1])
    m.free()


@pytest.mark.parametrize("heads,kv,hd", [(3, 1, 64), (8, 8, 32), (2, 2, 128), (9, 3, 64)])
def test_prompt_rotation_and_cache_rows(E, pkg, heads, kv, hd):
    """A prompt in two portions (q, k and v below, at and above a block of the rotation kernel, positions from the second portion's
    start on), then decoding over its cache rows, against the same tokens decoded one by one: 32-bit rounding on both sides, the
    decode tests' tolerance."""
    cfg = dict(hidden=heads * hd if heads * hd % 64 == 0 else 64, inter=512, n_heads=heads, n_kv_heads=kv, n_layers=2, vocab=96, max_pos=64,
               eps=1e-5, rope_theta=10000.0)
    cfg, tensors = pkg.synth.build_model(cfg, "q8_0", seed=heads)
    m = E.Model(cfg).load(tensors)
    toks = np.random.default_rng(heads).integers(0, 96, 40).astype(np.int32)
    want = [np.array(m.decode(int(t), i)[0], np.float64) for i, t in enumerate(toks)]
    m.reset_kv()
    got = {16: np.array(m.prefill(toks[:17], 0)), 36: np.array(m.prefill(toks[17:37], 17))}
    got.update({i: np.array(m.decode(int(toks[i]), i)[0]) for i in (37, 38, 39)})
    for i, g in got.items():
        assert (np.abs(g - want[i]) <= 1e-4 * np.maximum(1.0, np.abs(want[i]))).all(), (i, np.abs(g - want[i]).max())
    m.free()
