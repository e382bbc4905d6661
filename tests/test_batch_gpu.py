"""Multi-sequence decode (generate_batch api.cpp:836, forward_cpu_batch_generation model.cpp:1158) on MI355X:
B sequences with prompts of different lengths share every step's weight stream (skinny GEMMs on the matrix cores) over a
sequence-major KV cache. The bar is the reference's sequential fallback: every sequence must decode exactly as it does
alone -- logits within the decode tolerance of the single-sequence CPU oracle, identical greedy ids -- whatever else is
in the batch, in whatever slot order, and while other sequences join or leave."""
import numpy as np
import pytest

from oracle.oracle import OracleModel

pytestmark = pytest.mark.gpu
LOGIT_TOL = 1e-4


def close(a, b, tol):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return np.abs(a - b) <= tol * np.maximum(1.0, np.abs(b))


def oracle_run(om, prompt, n_steps):
    """greedy ids + the logits that produced each of them, single sequence, no penalty"""
    om.reset_kv()
    logits = None
    for pos, t in enumerate(prompt):
        _, logits = om.forward(om.lookup_embedding(int(t)), pos)
    ids, rows = [], []
    for i in range(n_steps):
        rows.append(logits)
        tok = int(np.argmax(logits))
        ids.append(tok)
        if i + 1 < n_steps:
            _, logits = om.forward(om.lookup_embedding(tok), len(prompt) + i)
    return np.array(ids, np.int32), np.stack(rows)


@pytest.mark.parametrize("gemv_max", ["8", "0", "3"])
@pytest.mark.parametrize("shape,mix", [("tiny-gqa", "q4_k_m"), ("tiny", "q6_k"), ("tiny-tp", "q8_0")])
def test_batch_matches_single_sequence_oracle(pkg, oracle, monkeypatch, shape, mix, gemv_max):
    """gemv_max: steps with at most that many sequences use multi-vector GEMVs, larger ones matrix-core GEMMs
    (12 = default: every step of this test on GEMVs; 0: all on GEMMs; 3: the test crosses between the two)."""
    from tinyllama_cpp_amd import engine as E
    monkeypatch.setenv("TL_BATCH_GEMV_MAX", gemv_max)
    E.init(0)
    cfg, tensors = pkg.synth.build_model(shape, mix, seed=21)
    m = E.Model(cfg).load(tensors)
    om = OracleModel(oracle, cfg, tensors)
    rng = np.random.default_rng(4)
    lens = [5, 1, 17, 9, 3]
    prompts = [rng.integers(0, cfg["vocab"], n).astype(np.int32) for n in lens]
    slots = [3, 0, 6, 2, 5]  # sequence i lives in cache slot slots[i] (not the batch order)
    n_steps = 7
    want = [oracle_run(om, p, n_steps) for p in prompts]
    m.batch_init(8)
    # prompts: batched prefill per sequence into its slot; its last logits pick the first generated id
    first = []
    for p, s, (ids, rows) in zip(prompts, slots, want):
        last = m.batch_prefill(s, p)
        assert close(last, rows[0], LOGIT_TOL).all(), np.abs(last - rows[0]).max()
        first.append(int(np.argmax(last)))
        assert first[-1] == ids[0]
    # step by step with logits: all five active, then sequences 1 and 3 leave (as finished ones do in the reference)
    toks, pos = list(first), list(lens)
    active = list(range(5))
    for step in range(1, n_steps):
        if step == 3:
            active = [0, 2, 4]
        logits, nxt = m.batch_decode([toks[i] for i in active], [pos[i] for i in active], [slots[i] for i in active])
        for j, i in enumerate(active):
            assert close(logits[j], want[i][1][step], LOGIT_TOL).all(), (step, i, np.abs(logits[j] - want[i][1][step]).max())
            assert nxt[j] == want[i][0][step]
            toks[i], pos[i] = int(nxt[j]), pos[i] + 1
    # the device-resident loop from the same prompts (fresh prefill: the cache rows are simply overwritten)
    for p, s in zip(prompts, slots):
        m.batch_prefill(s, p)
    ids = m.batch_generate_greedy(first, lens, slots, n_steps - 1)
    for i in range(5):
        assert np.array_equal(ids[:, i], want[i][0][1:]), i
    # the single-sequence engine state is untouched by batch mode
    single = m.generate(prompts[2], n_steps)
    assert np.array_equal(single, want[2][0])
    m.free()
    om.close()


@pytest.mark.parametrize("shape,mix,lens", [("tiny-gqa", "q4_k_m", [5, 1, 17, 9, 3]), ("tiny", "q6_k", [40, 2, 33]),
                                            ("tiny-tp", "q4_k_m", [12] * 12 + [7] * 13)])
def test_packed_prefill_of_all_prompts(pkg, oracle, shape, mix, lens):
    """batch_prefill_parallel (api.cpp:1144): every prompt's tokens in ONE packed batch with sequence-aware attention; the
    last-token logits equal the single-sequence oracle's, and decode continues from the caches it left. (The layers of
    a 35..250-token batch take the GEMM route; the head runs on the n_last rows only: multi-vector GEMVs for <= 12 rows,
    a GEMM for the 25 of the third case.)"""
    from tinyllama_cpp_amd import engine as E
    E.init(0)
    cfg, tensors = pkg.synth.build_model(shape, mix, seed=31)
    m = E.Model(cfg).load(tensors)
    om = OracleModel(oracle, cfg, tensors)
    rng = np.random.default_rng(sum(lens))
    prompts = [rng.integers(0, cfg["vocab"], n).astype(np.int32) for n in lens]
    B = len(prompts)
    slots = list(rng.permutation(B + 2)[:B])
    m.batch_init(B + 2)
    logits, ids = m.batch_prefill_packed(prompts, slots)
    n_steps = 4
    want = [oracle_run(om, p, n_steps) for p in prompts]
    for i in range(B):
        assert close(logits[i], want[i][1][0], LOGIT_TOL).all(), (i, np.abs(logits[i] - want[i][1][0]).max())
        assert ids[i] == want[i][0][0]
    out = m.batch_generate_greedy(ids, lens, slots, n_steps - 1)
    for i in range(B):
        assert np.array_equal(out[:, i], want[i][0][1:]), i
    m.free()
    om.close()


def test_batch_long_contexts_and_eight_head_groups(pkg, oracle):
    """TinyLlama-1.1B's attention geometry (head_dim 64, 8 query heads per kv head: two workgroups per (kv head, token))
    at 2 layers, with contexts of 70..150 rows (several 64-row passes of the batched decode attention) next to a short one."""
    from tinyllama_cpp_amd import engine as E
    E.init(0)
    cfg = dict(pkg.synth.SHAPES["tinyllama-1.1b"], n_layers=2, vocab=2048, max_pos=256)
    cfg, tensors = pkg.synth.build_model(cfg, "q4_k_m", seed=23)
    m = E.Model(cfg).load(tensors)
    om = OracleModel(oracle, cfg, tensors)
    rng = np.random.default_rng(6)
    lens = [150, 70, 4]
    prompts = [rng.integers(0, cfg["vocab"], n).astype(np.int32) for n in lens]
    n_steps = 5
    want = [oracle_run(om, p, n_steps) for p in prompts]
    m.batch_init(4)
    logits, ids = m.batch_prefill_packed(prompts, slots=[2, 0, 3])
    for i in range(3):
        assert close(logits[i], want[i][1][0], LOGIT_TOL).all(), (i, np.abs(logits[i] - want[i][1][0]).max())
    toks, pos = [int(x) for x in ids], list(lens)
    for step in range(1, n_steps):
        lg, nxt = m.batch_decode(toks, pos, [2, 0, 3])
        for i in range(3):
            assert close(lg[i], want[i][1][step], LOGIT_TOL).all(), (step, i, np.abs(lg[i] - want[i][1][step]).max())
            assert nxt[i] == want[i][0][step]
        toks, pos = [int(x) for x in nxt], [p + 1 for p in pos]
    m.free()
    om.close()


@pytest.mark.parametrize("heads,kv_heads,hd,B", [(6, 2, 128, 130), (12, 4, 64, 65), (4, 2, 64, 129), (8, 1, 64, 129), (4, 4, 128, 65)])
def test_batched_attention_in_four_and_eight_waves(pkg, heads, kv_heads, hd, B):
    """One step of B sequences (more workgroups than CUs: four waves each) against the same sequences seven at a time (eight waves beyond a
    step of four), at contexts around one and several steps of either. Both are within 2^-22 of the exact sums a layer and product, as in the packed tests."""
    from tinyllama_cpp_amd import engine as E
    E.init(0)
    cfg = dict(pkg.synth.SHAPES["tiny-gqa"], hidden=heads * hd, n_heads=heads, n_kv_heads=kv_heads, n_layers=2, max_pos=320)
    cfg, tensors = pkg.synth.build_model(cfg, "q4_k_m", seed=5)
    m = E.Model(cfg).load(tensors)
    m.batch_init(B)
    rng = np.random.default_rng(heads + B)
    lens = [(1, 31, 63, 64, 127, 128, 255, 256, 300, 16)[i] if i < 10 else int(rng.integers(1, 40)) for i in range(B)]
    _, ids = m.batch_prefill_packed([rng.integers(0, cfg["vocab"], n).astype(np.int32) for n in lens], slots=list(range(B)))
    toks = [int(x) for x in ids]
    whole, _ = m.batch_decode(toks, lens, list(range(B)))
    for i in range(0, min(B, 28), 7):
        part, _ = m.batch_decode(toks[i:i + 7], lens[i:i + 7], list(range(i, i + 7)))
        assert np.isfinite(part).all() and np.linalg.norm(part - whole[i:i + 7]) <= 4e-6 * np.linalg.norm(part), i
    m.free()


@pytest.mark.parametrize("heads,kv_heads,hd", [(8, 1, 64), (8, 2, 128), (8, 4, 64), (4, 2, 128)])
def test_batched_attention_writes_the_products_input(pkg, monkeypatch, heads, kv_heads, hd):
    """A step of 7 and of 130 sequences and a prompt of 9 tokens, whose attention writes the two f16 parts itself where a workgroup's heads
    are whole super-blocks (64 x 2: they are not), bit for bit with the split in a launch of its own (TL_ATTN_HALF_PLANES=0): one launch
    a layer and call less, which are counted."""
    import ctypes as C
    from tinyllama_cpp_amd import engine as E
    from tinyllama_cpp_amd.capi import check, lib
    E.init(0)

    def splits():
        n = C.c_longlong()
        check(lib().tl_debug_split_launches(C.byref(n)))
        return n.value

    cfg = dict(pkg.synth.SHAPES["tiny-gqa"], hidden=heads * hd, n_heads=heads, n_kv_heads=kv_heads, n_layers=2, max_pos=320)
    cfg, tensors = pkg.synth.build_model(cfg, "q4_k_m", seed=8)
    rng = np.random.default_rng(heads)
    prompts = [rng.integers(0, cfg["vocab"], n).astype(np.int32) for n in rng.integers(1, 12, 130)]
    want, launches = None, []
    for switch in ("0", "1"):
        monkeypatch.setenv("TL_ATTN_HALF_PLANES", switch)
        m = E.Model(cfg).load(tensors)
        m.batch_init(130)
        first, ids = m.batch_prefill_packed(prompts, slots=list(range(130)))
        toks, lens = [int(x) for x in ids], [len(p) for p in prompts]
        got, counts = [], [splits()]
        for call in (lambda: m.batch_decode(toks, lens, list(range(130)))[0], lambda: m.batch_decode(toks[:7], lens[:7], list(range(7)))[0],
                     lambda: m.prefill(np.arange(9, dtype=np.int32))):
            got.append(call())
            counts.append(splits())
        launches.append(np.diff(counts))
        m.free()
        if want is None:
            want = got
        else:
            assert all(np.isfinite(a).all() and np.array_equal(a, b) for a, b in zip(got, want))
    group = min(heads // kv_heads, 4)
    assert (launches[0] - launches[1] == (2 if group * hd % 256 == 0 else 0)).all(), launches


@pytest.mark.parametrize("heads,kv_heads,hd", [(3, 3, 64), (2, 1, 128), (4, 2, 64), (3, 1, 128), (6, 2, 64), (4, 1, 64), (8, 1, 128)])
@pytest.mark.parametrize("T", [3, 300])
def test_batched_attention_of_keys_out_of_range(pkg, heads, kv_heads, hd, T):
    """Keys so large that their scores are -inf, at every 16th and 32nd position (all that a group of lanes of four or eight waves sees) and
    in the first positions: weight 0, as if they were not there; a token that sees no others gets 0. Bound of
    test_packed_attention_kernel. Three tokens take eight waves, 300 four."""
    from tinyllama_cpp_amd import engine as E
    from tinyllama_cpp_amd.capi import check, lib
    E.init(0)
    rng = np.random.default_rng(heads * hd + T)
    S, group, start = 340, heads // kv_heads, 30
    q = np.abs(rng.standard_normal((T, heads, hd))).astype(np.float32) + 0.5
    k, v = (rng.standard_normal((S, kv_heads, hd)).astype(np.float32) for _ in range(2))
    gone = np.zeros(S, bool)
    gone[:2] = gone[5::32] = gone[7::16] = gone[16::16] = True
    k[gone] = -3e38
    scale = float(np.float32(1.0 / np.sqrt(hd)))
    dev, out = [E.DeviceBuffer.from_numpy(a) for a in (q, k, v)], E.DeviceBuffer(4 * q.size)

    def run(at):
        check(lib().tl_memset(out.ptr, 0xff, out.nbytes, None))
        check(lib().tl_debug_batch_attention(*(d.ptr for d in dev), out.ptr, 0, None, None, at, T, heads, kv_heads, hd, S, 1, scale, None))
        return out.to_numpy(np.float32, q.shape)

    got = run(start)
    assert np.isfinite(got).all()
    for i in range(T):
        at = np.flatnonzero(~gone[:start + i + 1])
        K, V = (np.repeat(a[at].astype(np.float64), group, 1) for a in (k, v))
        sc = np.einsum("hd,jhd->hj", q[i].astype(np.float64), K) * scale
        w = np.exp(sc - sc.max(1, keepdims=True))
        w /= w.sum(1, keepdims=True)
        want = np.einsum("hj,jhd->hd", w, V)
        bound = 2.0 ** -24 * np.einsum("hj,jhd->hd", w * (12 + 8 * np.abs(sc).max()), np.abs(V))
        assert (np.abs(got[i] - want) <= bound).all(), (i, float((np.abs(got[i] - want) / bound).max()))
    assert not run(0)[:2].any()


@pytest.mark.parametrize("heads,kv_heads,hd", [(3, 3, 64), (2, 1, 128), (3, 1, 128), (4, 1, 64), (8, 1, 128)])
def test_batched_attention_of_one_step_takes_four_waves(pkg, heads, kv_heads, hd):
    """Positions that four waves take in one step (64 of 128 columns, 128 of 64) are theirs however few tokens there are: the bits of the same
    tokens in a launch of 300, which has four waves throughout. One position more, and eight waves sum in another order."""
    from tinyllama_cpp_amd import engine as E
    from tinyllama_cpp_amd.capi import check, lib
    E.init(0)
    rng = np.random.default_rng(heads * hd)
    S, T, step = 340, 300, 4096 * 2 // hd
    q = rng.standard_normal((T, heads, hd)).astype(np.float32)
    pos = np.resize(np.array([0, 1, 15, 16, 31, 33, step - 2, step - 1, step, step + 40], np.int32), T)
    dev = [E.DeviceBuffer.from_numpy(a) for a in (q, *(rng.standard_normal((S, kv_heads, hd)).astype(np.float32) for _ in range(2)))]
    posd, seqd, out = E.DeviceBuffer.from_numpy(pos), E.DeviceBuffer.from_numpy(np.zeros(T, np.int32)), E.DeviceBuffer(4 * q.size)

    def run(n):
        check(lib().tl_debug_batch_attention(*(d.ptr for d in dev), out.ptr, 0, posd.ptr, seqd.ptr, 0, n, heads, kv_heads, hd, S, 1, 0.125, None))
        return out.to_numpy(np.float32, q.shape)[:n]

    many, few = run(T)[:10], run(10)
    assert np.isfinite(many).all() and np.array_equal(many[:8], few[:8]) and not np.array_equal(many[8:], few[8:])
    assert np.linalg.norm(many[8:] - few[8:]) <= 2e-6 * np.linalg.norm(many[8:])


def test_packed_prefill_rejects_bad_batches(pkg):
    from tinyllama_cpp_amd import engine as E
    from tinyllama_cpp_amd.capi import TlError, check, lib
    E.init(0)
    cfg, tensors = pkg.synth.build_model("tiny", "q4_k_m", seed=1)
    m = E.Model(cfg).load(tensors)
    m.batch_init(2)

    def call(toks, pos, seq, last):
        a = [np.ascontiguousarray(x, np.int32) for x in (toks, pos, seq, last)]
        ids = np.zeros(max(len(last), 1), np.int32)
        check(lib().tl_model_batch_prefill_packed(m.h, a[0].size, a[0].ctypes.data, a[1].ctypes.data, a[2].ctypes.data,
                                                  a[3].size, a[3].ctypes.data, None, ids.ctypes.data), "packed")
        return ids
    call([1, 2, 3], [0, 1, 0], [0, 0, 1], [1, 2])  # fine
    with pytest.raises(TlError):
        call([1, 2], [1, 0], [0, 0], [1])  # positions of a sequence out of order
    with pytest.raises(TlError):
        call([1, 2], [0, 0], [0, 2], [1])  # sequence index out of range
    with pytest.raises(TlError):
        call([1, 2], [0, 1], [0, 0], [2])  # output row outside the batch
    with pytest.raises(TlError):
        call([1, 2, 3], [0, 0, 1], [0, 1, 1], [0, 1, 2])  # more output rows than max_batch
    with pytest.raises(TlError):
        call([1, cfg["vocab"]], [0, 1], [0, 0], [1])  # token id
    m.free()


def test_batch_argument_errors(pkg):
    from tinyllama_cpp_amd import engine as E
    from tinyllama_cpp_amd.capi import TlError
    E.init(0)
    cfg, tensors = pkg.synth.build_model("tiny", "q4_k_m", seed=1)
    m = E.Model(cfg).load(tensors)
    with pytest.raises(TlError):
        m.batch_decode([1], [0], [0])  # before batch_init
    with pytest.raises(TlError):
        m.batch_init(0)
    with pytest.raises(TlError):
        m.batch_init(100000)
    m.batch_init(4)
    with pytest.raises(TlError):
        m.batch_prefill(4, [1, 2, 3])  # slot out of range
    with pytest.raises(TlError):
        m.batch_decode([1, 2], [0, 0], [1, 1])  # repeated sequence index
    with pytest.raises(TlError):
        m.batch_decode([1], [cfg["max_pos"]], [0])  # position out of range
    with pytest.raises(TlError):
        m.batch_decode([cfg["vocab"]], [0], [0])  # token id out of range
    with pytest.raises(TlError):
        m.batch_decode([1, 2, 3, 4, 5], [0] * 5, [0, 1, 2, 3, 4])  # more than max_batch (and slot 4)
    with pytest.raises(TlError):
        m.batch_generate_greedy([1], [cfg["max_pos"] - 2], [0], 5)  # would run past max_pos
    m.free()
    with pytest.raises(TlError):
        E.Model(dict(pkg.synth.SHAPES["tiny-gqa"]), tp_rank=0, tp_size=2).batch_init(2)  # not finalized / sharded


def test_deferred_ksplit_reductions_are_bit_identical(pkg, monkeypatch):
    """Skinny GEMMs split K; their partial tiles are summed by the NEXT kernel (RMSNorm split, SwiGLU split, RoPE + cache
    write) instead of a reduction launch of their own. Same sums in the same order: logits of a batched step, a packed
    prefill and an all-logits prefill are bit-for-bit those of TL_GEMM_DEFER=0 (one ksplit_reduce launch per GEMM), with
    and without q | k | v and gate | up merged into one launch each. The last model's products are in bf16 parts (Q8_0 rows that
    are not whole pairs of blocks): its batched attention writes the attn_output GEMM's planes itself (TL_ATTN_PLANES)."""
    import ctypes as C
    from tinyllama_cpp_amd import engine as E
    from tinyllama_cpp_amd.capi import lib
    monkeypatch.setenv("TL_BATCH_GEMV_MAX", "0")
    E.init(0)
    rng = np.random.default_rng(8)
    odd = dict(hidden=512, inter=1056, n_heads=8, n_kv_heads=2, n_layers=2, vocab=128, max_pos=128, eps=1e-5, rope_theta=10000.0)
    for shape, mix in (("tiny-tp", "q4_k_m"), ("tiny-gqa", "q6_k"), (odd, "q8_0")):
        cfg, tensors = pkg.synth.build_model(shape, mix, seed=5)
        prompts = [rng.integers(0, cfg["vocab"], n).astype(np.int32) for n in [9, 3, 14, 6, 11, 2, 8, 5, 7, 10, 4, 12]]
        long_prompt = rng.integers(0, cfg["vocab"], 100).astype(np.int32)
        got, splits = {}, {}
        for defer, merge in (("0", "1"), ("1", "0"), ("1", "1")):
            monkeypatch.setenv("TL_GEMM_DEFER", defer)  # read when the model's prefill workspaces are made
            monkeypatch.setenv("TL_GEMM_MERGE", merge)  # q | k | v and gate | up in one launch each (needs DEFER)
            monkeypatch.setenv("TL_ATTN_PLANES", defer)
            m = E.Model(cfg).load(tensors)
            m.batch_init(12)
            n0, n1 = C.c_longlong(), C.c_longlong()
            assert lib().tl_debug_split_launches(C.byref(n0)) == 0
            logits, ids = m.batch_prefill_packed(prompts)
            assert lib().tl_debug_split_launches(C.byref(n1)) == 0
            splits[defer] = n1.value - n0.value
            step, nxt = m.batch_decode(list(ids), [len(p) for p in prompts], list(range(12)))
            more = m.batch_generate_greedy(list(nxt), [len(p) + 1 for p in prompts], list(range(12)), 3)
            _, all_logits = m.prefill(long_prompt, all_logits=True)       # 64-token tiles of the f16 form, 128-token ones of the other
            _, all_logits40 = m.prefill(long_prompt[:40], all_logits=True)  # 32- and 64-token tiles
            got[defer + merge] = [np.array(x) for x in (logits, ids, step, nxt, more, all_logits, all_logits40)]
            m.free()
        assert splits["0"] - splits["1"] == (cfg["n_layers"] if mix == "q8_0" else 0), (shape, splits)
        for other in ("10", "11"):
            for a, b in zip(got["01"], got[other]):
                assert a.shape == b.shape and np.array_equal(a, b), (shape, other, np.abs(a.astype(np.float64) - b).max())


@pytest.mark.parametrize("mix,n", [("q4_k_m", 330), ("q6_k", 200), ("q8_0", 150)])
def test_merged_and_separate_launches_round_alike(pkg, monkeypatch, mix, n):
    """gate | up of 2 x 5632 rows and 330 tokens fill the chip in another workgroup shape than one of them does, and the shapes do
    not round alike: launched one after another (TL_GEMM_MERGE=0) the matrices of a group keep the group's shape and slices, so
    every logit is the same bit for bit."""
    from tinyllama_cpp_amd import engine as E
    E.init(0)
    cfg, tensors = pkg.synth.build_model(dict(hidden=2048, inter=5632, n_heads=32, n_kv_heads=4, n_layers=1, vocab=64, max_pos=512, eps=1e-5,
                                              rope_theta=10000.0), mix, seed=6)
    m = E.Model(cfg).load(tensors)
    toks = np.random.default_rng(6).integers(0, cfg["vocab"], n).astype(np.int32)
    got = []
    for merge in ("0", "1"):
        monkeypatch.setenv("TL_GEMM_MERGE", merge)
        m.reset_kv()
        got.append(np.array(m.prefill(toks, 0, all_logits=True)[1]))
    m.free()
    assert np.array_equal(got[0], got[1]), np.abs(got[0].astype(np.float64) - got[1]).max()


@pytest.mark.parametrize("heads,kv", [(8, 4), (4, 4)])
def test_two_formats_in_one_launch(pkg, monkeypatch, heads, kv):
    """q | k in Q4_K and v in Q6_K share a launch, tokens around 8, 16, 32 and 64 and many more, in the workgroup shapes of narrow matrices (the
    next test has those of wide ones), with rows that end inside a tile and K slices: the same bits as a launch of each with the shared launch's shapes and slices
    (TL_GEMM_MERGE=0), whose products are held against float64 elsewhere."""
    from tinyllama_cpp_amd import engine as E
    E.init(0)
    cfg, tensors = pkg.synth.build_model(dict(hidden=heads * 128, inter=512, n_heads=heads, n_kv_heads=kv, n_layers=1, vocab=64, max_pos=2048, eps=1e-5,
                                              rope_theta=10000.0), "q4_k_m", seed=16)
    assert [tensors["blk.0.attn_%s.weight" % n][0] for n in "qkv"] == [pkg.synth.Q4_K, pkg.synth.Q4_K, pkg.synth.Q6_K]
    m = E.Model(cfg).load(tensors)
    rng = np.random.default_rng(heads)
    for n in (1, 8, 9, 16, 17, 31, 33, 64, 65, 130, 520, 1999):
        toks = rng.integers(0, cfg["vocab"], n).astype(np.int32)
        got = []
        for merge in ("0", "1"):
            monkeypatch.setenv("TL_GEMM_MERGE", merge)
            m.reset_kv()
            got.append(np.array(m.prefill(toks, 0, all_logits=True)[1]))
        assert np.array_equal(got[0], got[1]), (n, np.abs(got[0].astype(np.float64) - got[1]).max())
    m.free()


@pytest.mark.parametrize("heads,tokens", [(32, {8: 5, 20: 1, 40: 1, 63: 1, 844: 3, 900: 3, 1200: 3, 1350: 3}), (40, {8: 6, 9: 7, 16: 7, 130: 3, 650: 3}),
                                          (64, {8: 6, 9: 7, 16: 7, 17: 1, 32: 1, 33: 2, 200: 3, 450: 3})])
def test_two_formats_in_one_launch_of_wide_matrices(pkg, monkeypatch, heads, tokens):
    """As above in the shapes that wide matrices take: 128 rows x 32 tokens (1), waves of 64 rows in Q4_K with twice the rows of a Q6_K tile
    beside them (3), 128 rows x 8 and x 16 tokens (6 and 7), one and several K slices of either format; the shape that ran is counted."""
    import ctypes as C
    from tinyllama_cpp_amd import engine as E
    from tinyllama_cpp_amd.capi import check, lib
    E.init(0)
    cfg, tensors = pkg.synth.build_model(dict(hidden=heads * 128, inter=512, n_heads=heads, n_kv_heads=8, n_layers=1, vocab=64, max_pos=1408, eps=1e-5,
                                              rope_theta=10000.0), "q4_k_m", seed=16)
    m = E.Model(cfg).load(tensors)
    rng = np.random.default_rng(heads)
    counts = (C.c_longlong * 9)()

    def launches():
        check(lib().tl_debug_half_pair_launches(counts))
        return np.array(counts)

    for n, shape in tokens.items():
        toks = rng.integers(0, cfg["vocab"], n).astype(np.int32)
        got = []
        for merge in ("0", "1"):
            monkeypatch.setenv("TL_GEMM_MERGE", merge)
            m.reset_kv()
            before = launches()
            every = n <= 512  # (chunks whose logits are all asked for end there)
            logits = m.prefill(toks, 0, all_logits=True)[1] if every else m.prefill(toks, 0)
            got.append(np.concatenate([np.ravel(logits)] + [np.ravel(x) for i in range(0, n, 5) for x in m.kv_cache(0, i)]))  # (in every column of a tile)
            assert np.array_equal(np.flatnonzero(launches() - before), [shape] if merge == "1" else []), (n, merge)
        assert np.array_equal(got[0], got[1]), (n, np.abs(got[0].astype(np.float64) - got[1]).max())
    m.free()


def test_packed_output_rows_in_any_order(pkg):
    """Output rows of a packed batch that come in no order, from two chunks in turn, twice, and more of them than one gather takes: each is the
    logits row of its own sequence's prefill, up to the order of 32-bit sums (2^-22 a layer and product)."""
    from tinyllama_cpp_amd import engine as E
    from tinyllama_cpp_amd.capi import check, lib
    E.init(0)
    cfg, tensors = pkg.synth.build_model(dict(pkg.synth.SHAPES["tiny-gqa"], max_pos=96), "q4_k_m", seed=18)
    m = E.Model(cfg).load(tensors)
    n_seq = 96
    m.batch_init(n_seq)
    rng = np.random.default_rng(18)
    prompts = [rng.integers(0, cfg["vocab"], n).astype(np.int32) for n in rng.integers(9, 48, n_seq)]
    toks, pos = np.concatenate(prompts), np.concatenate([np.arange(p.size, dtype=np.int32) for p in prompts])
    seq = np.concatenate([np.full(p.size, i, np.int32) for i, p in enumerate(prompts)])
    assert toks.size > 2048 + 64
    want = []
    for p in prompts:
        m.reset_kv()
        want.append(m.prefill(p, 0, all_logits=True)[1])
    want = np.concatenate(want)
    for rows in (rng.integers(0, toks.size, n_seq), np.arange(toks.size - n_seq, toks.size), np.array([2047, 2048, 0, 2048, toks.size - 1]), np.arange(64)):
        rows = np.ascontiguousarray(rows, np.int32)
        logits, ids = np.empty((rows.size, cfg["vocab"]), np.float32), np.empty(rows.size, np.int32)
        check(lib().tl_model_batch_prefill_packed(m.h, toks.size, toks.ctypes.data, pos.ctypes.data, seq.ctypes.data, rows.size, rows.ctypes.data,
                                                  logits.ctypes.data, ids.ctypes.data), "tl_model_batch_prefill_packed")
        # (the bound of the next test, which is one of all rows together; another row's logits are as far off as their size)
        assert np.linalg.norm(logits - want[rows]) <= 4e-6 * np.linalg.norm(want[rows])
        assert all(np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(b) for a, b in zip(logits, want[rows]))
        assert np.array_equal(ids, logits.argmax(1))
    m.free()


def test_packed_prompts_longer_than_a_sequence(pkg):
    """A packed batch of more tokens than a sequence has positions goes through as one chunk: every prompt's last logits are those
    of its own prefill, up to the order of 32-bit sums (2^-22 a layer and product)."""
    from tinyllama_cpp_amd import engine as E
    E.init(0)
    cfg, tensors = pkg.synth.build_model(dict(pkg.synth.SHAPES["tiny-gqa"], max_pos=96), "q4_k_m", seed=8)
    m = E.Model(cfg).load(tensors)
    m.batch_init(9)
    rng = np.random.default_rng(8)
    prompts = [rng.integers(0, cfg["vocab"], n).astype(np.int32) for n in (96, 95, 61, 96, 33, 96, 90, 17, 96)]  # 680 tokens
    alone = np.stack([m.batch_prefill(i, p) for i, p in enumerate(prompts)])
    packed, ids = m.batch_prefill_packed(prompts)
    assert np.linalg.norm(packed - alone) <= 4e-6 * np.linalg.norm(alone)
    assert np.array_equal(ids, packed.argmax(1))
    m.free()


@pytest.mark.parametrize("heads,kv_heads,hd", [(8, 1, 64), (6, 2, 128), (4, 4, 64)])
def test_packed_attention_by_row_tiles(pkg, monkeypatch, heads, kv_heads, hd):
    """A packed batch large enough for the matrix-core attention: runs of 1, 31, 32, 33, 127, 129 tokens, slots out of order, a
    second batch that goes on behind the first one's rows and two runs of one sequence in a batch. Against the per-token FP32
    kernel: both are within 2^-22 of the exact sums a layer and product (two layers, a handful of products each)."""
    from tinyllama_cpp_amd import engine as E
    E.init(0)
    cfg = dict(pkg.synth.SHAPES["tiny-gqa"], hidden=heads * hd, n_heads=heads, n_kv_heads=kv_heads, n_layers=2, max_pos=640)
    cfg, tensors = pkg.synth.build_model(cfg, "q4_k_m", seed=4)
    m = E.Model(cfg).load(tensors)
    m.batch_init(9)
    rng = np.random.default_rng(9)
    lens, slots = (33, 1, 129, 320, 31, 127, 32, 300), [8, 3, 0, 5, 2, 7, 1, 4]
    runs = [(s, 0, rng.integers(0, cfg["vocab"], n)) for s, n in zip(slots, lens)]
    more = [(s, n, rng.integers(0, cfg["vocab"], k)) for s, n, k in zip(slots, lens, (40, 300, 1, 200, 65, 5, 96, 7))]
    more.append((more[3][0], more[3][1] + 200, rng.integers(0, cfg["vocab"], 90)))  # goes on behind other sequences' tokens
    want = {}
    for switch in ("0", "1"):
        monkeypatch.setenv("TL_HATTN", switch)
        m.reset_kv()
        for k, part in enumerate((runs, more)):
            toks = np.concatenate([t for _, _, t in part]).astype(np.int32)
            pos = np.concatenate([np.arange(p, p + len(t)) for _, p, t in part]).astype(np.int32)
            seq = np.concatenate([np.full(len(t), s) for s, _, t in part]).astype(np.int32)
            last = np.cumsum([len(t) for _, _, t in part]).astype(np.int32) - 1
            logits, ids = np.zeros((len(last), cfg["vocab"]), np.float32), np.zeros(len(last), np.int32)
            from tinyllama_cpp_amd.capi import check, lib
            check(lib().tl_model_batch_prefill_packed(m.h, toks.size, toks.ctypes.data, pos.ctypes.data, seq.ctypes.data, last.size,
                                                      last.ctypes.data, logits.ctypes.data, ids.ctypes.data), "packed")
            if switch == "0":
                want[k] = logits
            else:
                assert not np.array_equal(logits, want[k])  # (the other kernel ran)
                assert np.linalg.norm(logits - want[k]) <= 4e-6 * np.linalg.norm(want[k])
    m.free()


def test_many_logits_reach_the_caller(pkg):
    """Logits of 4 MB and more come through four threads' stripes: every row where it belongs, whole pages and not, one buffer after
    another. Against steps of a few sequences (the runtime's own copy): the same products in another order of sums."""
    from tinyllama_cpp_amd import engine as E
    E.init(0)
    cfg, tensors = pkg.synth.build_model(dict(pkg.synth.SHAPES["tiny-gqa"], vocab=50003, n_layers=1), "q4_k_m", seed=6)
    m = E.Model(cfg).load(tensors)
    m.batch_init(101)
    toks = np.random.default_rng(1).integers(0, cfg["vocab"], 101).astype(np.int32)
    at = lambda lo, hi: m.batch_decode(toks[lo:hi], np.zeros(hi - lo, np.int32), np.arange(lo, hi))
    want = np.concatenate([at(lo, min(lo + 15, 101))[0] for lo in range(0, 101, 15)])
    for n in (20, 21, 22, 50, 101):
        logits, ids = at(0, n)
        assert np.linalg.norm(logits - want[:n]) <= 4e-6 * np.linalg.norm(want[:n]) and np.array_equal(ids, logits.argmax(1)), n
        assert np.abs(logits - want[:n]).max() <= 1e-4 * np.abs(want).max(), n
    m.free()

@pytest.mark.parametrize("heads,kv_heads,hd,lens", [(4, 4, 64, (320, 40)), (6, 2, 128, (500, 300))])
@pytest.mark.parametrize("bad", ["nan", "huge"])
def test_packed_attention_before_a_row_out_of_range(pkg, monkeypatch, heads, kv_heads, hd, lens, bad):
    """A token whose key and value rows are NaN, or 2^30 times and more as large as its neighbours', in the middle of a key tile: the tokens in
    front of it give what the per-token FP32 kernel gives, to the tolerance of finite batches; those behind it are NaN in both."""
    from tinyllama_cpp_amd import engine as E
    from tinyllama_cpp_amd.capi import check, lib
    E.init(0)
    cfg = dict(pkg.synth.SHAPES["tiny-gqa"], hidden=heads * hd, n_heads=heads, n_kv_heads=kv_heads, n_layers=1, max_pos=640)
    cfg, tensors = pkg.synth.build_model(cfg, "q4_k_m", seed=8)
    typ, emb, rows, cols = tensors["token_embd.weight"]
    blocks = emb.copy().reshape(rows, cols // 256, 144)
    half = blocks[7, :, :4].copy().view(np.float16)  # a block's scale and minimum
    half[:] = np.nan if bad == "nan" else 6e4
    blocks[7, :, :4] = half.view(np.uint8)
    if bad == "huge":  # norms that keep a row's size (eps over its mean square), and everybody else small
        others = np.arange(rows) != 7
        small = blocks[others, :, :4].copy().view(np.float16) * np.float16(2.0 ** -10)
        blocks[others, :, :4] = small.view(np.uint8)
        cfg["eps"] = 1e24
        for name in ("blk.0.attn_norm.weight", "blk.0.ffn_norm.weight", "output_norm.weight"):
            t, w, r, c = tensors[name]
            tensors[name] = (t, (w * np.float32(0.0 if "ffn" in name else 1e12)).astype(w.dtype), r, c)
    tensors["token_embd.weight"] = (typ, blocks.reshape(emb.shape), rows, cols)
    m = E.Model(cfg).load(tensors)
    m.batch_init(8)
    rng = np.random.default_rng(2)
    toks = rng.integers(8, cfg["vocab"], sum(lens)).astype(np.int32)
    at = 290
    toks[at] = 7
    pos = np.concatenate([np.arange(n) for n in lens]).astype(np.int32)
    seq = np.concatenate([np.full(n, s) for s, n in zip((3, 1), lens)]).astype(np.int32)
    last = np.array([5, 200, 287, 288, at - 1, at, lens[0] - 1, sum(lens) - 1], np.int32)
    got = []
    for switch in ("0", "1"):
        monkeypatch.setenv("TL_HATTN", switch)
        m.reset_kv()
        logits, ids = np.zeros((last.size, cfg["vocab"]), np.float32), np.zeros(last.size, np.int32)
        check(lib().tl_model_batch_prefill_packed(m.h, toks.size, toks.ctypes.data, pos.ctypes.data, seq.ctypes.data, last.size,
                                                  last.ctypes.data, logits.ctypes.data, ids.ctypes.data), "packed")
        got.append(logits)
    assert not np.array_equal(got[0], got[1])  # (the other kernel ran)
    for j, r in enumerate(last):
        if bad == "nan" and at <= r < lens[0]:
            assert np.isnan(got[0][j]).all() and np.isnan(got[1][j]).all(), r
        else:
            assert np.isfinite(got[0][j]).all() and np.linalg.norm(got[1][j] - got[0][j]) <= 4e-6 * np.linalg.norm(got[0][j]), r
    m.free()


def test_packed_prompts_need_no_memory_of_their_own(pkg):
    """What the attention of packed prompts converts its rows into is laid out with the sequences' caches: neither a small batch (the
    per-token kernel) nor a large one takes device memory when the first one comes."""
    import ctypes as C
    from tinyllama_cpp_amd import engine as E
    E.init(0)
    hip = C.CDLL("libamdhip64.so")

    def free_bytes():
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    cfg = dict(pkg.synth.SHAPES["tiny-gqa"], hidden=256, n_heads=4, n_kv_heads=4, n_layers=1, max_pos=640)
    cfg, tensors = pkg.synth.build_model(cfg, "q4_k_m", seed=8)
    rng = np.random.default_rng(3)
    prompts = [rng.integers(0, cfg["vocab"], n).astype(np.int32) for n in (320, 40, 9)]
    for warm in (True, False):  # (the first model's calls make what the process keeps: loaded kernels, scratch)
        m = E.Model(cfg).load(tensors)
        m.batch_init(4)
        m.batch_decode(np.array([1]), np.array([0]), np.array([3]))
        before = free_bytes()
        m.batch_prefill_packed(prompts[2:])
        m.batch_prefill_packed(prompts)
        if not warm:
            assert free_bytes() == before
        m.free()


@pytest.mark.parametrize("heads,kv_heads,hd", [(8, 1, 64), (6, 2, 64), (3, 3, 64), (4, 2, 128), (8, 1, 128), (3, 1, 128)])
def test_packed_attention_kernel(pkg, heads, kv_heads, hd):
    """Row tiles of one to 32 rows and tiles of one to 32 keys, at the edges of both, one key and many; NaN behind every sequence's last
    position. Against float64: half a dozen roundings on the way to a score (a sum of eight, met in a tree; sizes up to 8 in here), as many on
    the way of the values."""
    from tinyllama_cpp_amd import engine as E
    from tinyllama_cpp_amd.capi import check, lib
    E.init(0)
    rng = np.random.default_rng(heads * hd + kv_heads)
    runs = [(3, 0, 1), (0, 0, 33), (4, 31, 1), (1, 30, 5), (2, 0, 64), (6, 97, 31), (5, 200, 40), (7, 0, 2)]
    S, group = 256, heads // kv_heads
    pos = np.concatenate([np.arange(p, p + n) for _, p, n in runs]).astype(np.int32)
    seq = np.concatenate([np.full(n, s) for s, _, n in runs]).astype(np.int32)
    q = rng.standard_normal((pos.size, heads, hd)).astype(np.float32)
    k, v = (rng.standard_normal((8, S, kv_heads, hd)).astype(np.float32) for _ in range(2))
    for s, p, n in runs:
        k[s, p + n:], v[s, p + n:] = np.nan, np.nan
    scale = float(np.float32(2.0 / np.sqrt(hd)))

    def run(v):
        dev = [E.DeviceBuffer.from_numpy(a) for a in (q, k, v)]
        out = E.DeviceBuffer(4 * q.size)
        check(lib().tl_memset(out.ptr, 0xff, out.nbytes, None))
        check(lib().tl_debug_packed_attention(*(d.ptr for d in dev), out.ptr, S * kv_heads * hd, pos.ctypes.data, seq.ctypes.data, pos.size, heads,
                                              kv_heads, hd, scale, None), "tl_debug_packed_attention")
        return out.to_numpy(np.float32, q.shape)

    got = run(v)
    for i, (p, s) in enumerate(zip(pos, seq)):
        K, V = (np.repeat(a[s, :p + 1].astype(np.float64), group, 1) for a in (k, v))
        sc = np.einsum("hd,jhd->hj", q[i].astype(np.float64), K) * scale
        w = np.exp(sc - sc.max(1, keepdims=True))
        w /= w.sum(1, keepdims=True)
        want = np.einsum("hj,jhd->hd", w, V)
        bound = 2.0 ** -24 * np.einsum("hj,jhd->hd", w * (12 + 8 * np.abs(sc).max()), np.abs(V))
        assert (np.abs(got[i] - want) <= bound).all(), (i, p, s, float((np.abs(got[i] - want) / bound).max()))
    # an infinity and a NaN in two columns of one position: seen from there on, and nowhere else
    s, p, n = runs[1]
    v[s, 20, 0, 3], v[s, 20, kv_heads - 1, hd - 2] = np.inf, np.nan
    odd = run(v)
    sees = (seq == s) & (pos >= 20)
    assert (odd[sees][:, :group, 3] == np.inf).all() and np.isnan(odd[sees][:, heads - group:, hd - 2]).all()
    odd[np.ix_(sees, np.arange(group), [3])] = got[np.ix_(sees, np.arange(group), [3])]
    odd[np.ix_(sees, np.arange(heads - group, heads), [hd - 2])] = got[np.ix_(sees, np.arange(heads - group, heads), [hd - 2])]
    assert np.array_equal(odd, got)


def test_many_logits_into_memory_that_the_runtime_knows(pkg):
    """Logits of 4 MB and more into pinned memory, a device's memory and ordinary memory: what the runtime knows it copies to itself (no
    thread of the host could write a device's), and every destination holds the same."""
    import ctypes as C
    from tinyllama_cpp_amd import engine as E
    from tinyllama_cpp_amd.capi import check, lib
    E.init(0)
    cfg, tensors = pkg.synth.build_model(dict(pkg.synth.SHAPES["tiny-gqa"], vocab=50003, n_layers=1), "q4_k_m", seed=6)
    m = E.Model(cfg).load(tensors)
    m.batch_init(24)
    n = 24
    toks = np.random.default_rng(1).integers(0, cfg["vocab"], n).astype(np.int32)
    pos, seq, nxt = np.zeros(n, np.int32), np.arange(n, dtype=np.int32), np.zeros(n, np.int32)
    want, ids = m.batch_decode(toks, pos, seq)
    hip = C.CDLL("libamdhip64.so")
    pinned = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(pinned), C.c_size_t(want.nbytes), 0) == 0
    on_device = E.DeviceBuffer(want.nbytes)

    def step(dst):
        nxt[:] = -1
        check(lib().tl_model_batch_decode(m.h, n, toks.ctypes.data, pos.ctypes.data, seq.ctypes.data, dst, nxt.ctypes.data), "tl_model_batch_decode")
        assert np.array_equal(nxt, ids)

    C.memset(pinned.value, 0xff, want.nbytes)
    step(pinned.value)
    assert np.array_equal(np.ctypeslib.as_array(C.cast(pinned, C.POINTER(C.c_float)), want.shape), want)
    step(on_device.ptr)
    assert np.array_equal(on_device.to_numpy(np.float32, want.shape), want)
    assert hip.hipHostFree(pinned) == 0
    m.free()


@pytest.mark.parametrize("heads,kv,hd", [(4, 4, 64), (4, 2, 128), (6, 2, 128), (8, 2, 64), (16, 2, 64), (16, 2, 128), (12, 4, 64)])
def test_step_attention_takes_new_keys(pkg, monkeypatch, heads, kv, hd):
    """A step whose attention rotates, sums and stores the new queries, keys and values itself against the same step with a launch of its own
    for that (TL_ATTN_STEP=0): every group size and head size, sequences at their first position, at the edges of a wave's and a
    workgroup's rows and beyond, slots out of order, four and eight waves; three steps, so that what was stored is read. Both sum the same
    numbers in another order (the new position last): 2^-22 a layer and product, as packed prompts."""
    from tinyllama_cpp_amd import engine as E
    E.init(0)
    cfg, tensors = pkg.synth.build_model(dict(hidden=heads * hd, inter=512, n_heads=heads, n_kv_heads=kv, n_layers=2, vocab=64, max_pos=320, eps=1e-5,
                                              rope_theta=10000.0), "q4_k_m", seed=26)
    lengths = [0, 1, 3, 4, 15, 16, 31, 32, 33, 63, 64, 65, 127, 128, 129, 200, 255, 256, 257, 300]
    m = E.Model(cfg).load(tensors)
    m.batch_init(140)
    rng = np.random.default_rng(heads)
    for n in (len(lengths), 140):  # (140 sequences: four waves a workgroup)
        lens = (lengths * 7)[:n]
        slots = rng.permutation(140)[:n].astype(np.int32)
        prompts = [rng.integers(0, cfg["vocab"], k).astype(np.int32) for k in lens]
        first = rng.integers(0, cfg["vocab"], n).astype(np.int32)
        got = []
        for step in ("0", "1"):
            monkeypatch.setenv("TL_ATTN_STEP", step)
            for s, p in zip(slots, prompts):
                if p.size:
                    m.batch_prefill(int(s), p)
            out = [m.batch_decode(first, np.array(lens, np.int32) + i, slots)[0] for i in range(3)]
            got.append(np.concatenate(out).astype(np.float64))
        assert np.isfinite(got[1]).all() and np.linalg.norm(got[1] - got[0]) <= 4e-6 * np.linalg.norm(got[0])
    m.free()
