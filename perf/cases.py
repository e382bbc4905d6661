"""The work that users of this framework have it do, as cases that can be timed and checked.

Quantized Llama models (the three shapes of tinyllama.cpp_amd/synth.py up to 8 billion weights, in the three GGUF mixes) in the
four ways a program drives them: tokens one by one (`decode`, greedy or sampled), a prompt (`prompt`), many prompts at once
(`packed`) and many sequences side by side (`batch`). Layer-list models (bf16 checkpoints): a prompt through latent attention,
sink attention and a delta rule (`layers_prompt`), and decoding of a model with routed experts (`layers_decode`).
Weights are random in the formats' own blocks; a model has every layer of its shape.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)
from _pkg import load_package  # noqa: E402

S = load_package().synth

LLAMA = ("tinyllama-1.1b", "llama-3.2-3b", "llama-3-8b")
MIXES = ("q4_k_m", "q6_k", "q8_0")
LAYERED = {  # the sizes of bench.py --family
    "s": dict(width=1024, layers=8, heads=16, kv_heads=4, dim=64, window=512, experts=8, top=2, ff=512, shared_ff=1024, vocab=32000),
    "m": dict(width=2048, layers=12, heads=32, kv_heads=8, dim=64, window=1024, experts=16, top=4, ff=768, shared_ff=1024, vocab=32000),
}


def listed():
    return [
        # the first words of an answer from the smallest model: launches and latency count, hardly any context
        dict(name="decode_1b_q4km", op="decode", model="tinyllama-1.1b", mix="q4_k_m", context=5, steps=16),
        # the headline: one user's greedy answer from the 8-billion-weight model
        dict(name="decode_8b_q4km", op="decode", model="llama-3-8b", mix="q4_k_m", context=64, steps=16),
        # an answer about a long document: the key/value cache is read beside the weights
        dict(name="decode_3b_q6k_long", op="decode", model="llama-3.2-3b", mix="q6_k", context=7901, steps=8),
        # chat with sampling as the session's callers ask for it (repetition penalty, top-k, top-p)
        dict(name="sampled_1b_q8", op="sampled", model="tinyllama-1.1b", mix="q8_0", context=187, steps=16),
        # a one-line question: time to the first token
        dict(name="prompt_1b_q8_short", op="prompt", model="tinyllama-1.1b", mix="q8_0", tokens=23),
        # an ordinary prompt with instructions and context
        dict(name="prompt_8b_q4km", op="prompt", model="llama-3-8b", mix="q4_k_m", tokens=512),
        # a document as the prompt, of a length that no tile divides
        dict(name="prompt_3b_q6k_long", op="prompt", model="llama-3.2-3b", mix="q6_k", tokens=3989),
        # prompts of many lengths that arrive together
        dict(name="packed_1b_q4km", op="packed", model="tinyllama-1.1b", mix="q4_k_m", sequences=21, tokens=150),
        # a handful of users served side by side
        dict(name="batch_3b_q4km_8", op="batch", model="llama-3.2-3b", mix="q4_k_m", sequences=8, context=90, steps=8),
        # a server at full load
        dict(name="batch_8b_q4km_128", op="batch", model="llama-3-8b", mix="q4_k_m", sequences=128, context=30, steps=6),
        # a document through a layer-list model at serving precision (bf16 activations)
        dict(name="layers_prompt_m", op="layers_prompt", size="m", tokens=1999),
        # an answer from a layer-list model with routed experts
        dict(name="layers_decode_m", op="layers_decode", size="m", context=700, steps=16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(("decode", "decode", "sampled", "prompt", "prompt", "packed", "batch", "batch", "layers_prompt", "layers_decode"))
    if op == "layers_prompt":
        return dict(op=op, size=rng.choice(sorted(LAYERED)), tokens=_log_int(rng, 24, 1990))
    if op == "layers_decode":
        return dict(op=op, size=rng.choice(sorted(LAYERED)), context=_log_int(rng, 4, 1500), steps=rng.randint(8, 16))
    model, mix = rng.choice(LLAMA), rng.choice(MIXES)
    c = dict(op=op, model=model, mix=mix)
    longest = {"tinyllama-1.1b": 1990, "llama-3.2-3b": 3900, "llama-3-8b": 1400}[model]
    if op in ("decode", "sampled"):
        c.update(context=_log_int(rng, 4, longest), steps=rng.randint(5, 8))
    elif op == "prompt":
        c.update(tokens=_log_int(rng, 9, longest))
    elif op == "packed":
        c.update(sequences=rng.randint(2, 24), tokens=_log_int(rng, 6, 150))
    else:
        c.update(sequences=_log_int(rng, 2, 125), context=_log_int(rng, 4, 200), steps=rng.randint(3, 5))
    return c


# ---- what a pass cannot do without ------------------------------------------------------------------------------------------
def work(case):
    op = case["op"]
    if op.startswith("layers"):
        z = LAYERED[case["size"]]
        W, V, H, G, d, n = z["width"], z["vocab"], z["heads"], z["kv_heads"], z["dim"], z["layers"]
        if op == "layers_decode":
            per = (2 * H * d + 2 * G * d) * W + W * z["experts"] + 3 * W * (z["top"] * z["ff"] + z["shared_ff"])
            seen = min(z["window"], case["context"]) * 2 * G * d
            steps = case["steps"]
            return {"bytes": steps * (2.0 * (n * per + V * W) + 4.0 * n * seen), "flops": steps * (2.0 * (n * per + V * W) + 4.0 * n * seen * (H // G))}
        T, params, attn = case["tokens"], 0.0, 0.0
        for i, (kind, own) in enumerate(_sogalix_kinds(n)):
            params += 2.0 * W * _sogalix_ff(z)
            if kind == "latent_attention":
                rq, rk, rd = W // 2, 4 * d, d // 2
                params += W * (rq + (rk + rd if own else 0) + H) + rq * H * (d + rd) + 2.0 * rk * H * d + H * d * W
                attn += T * T / 2.0 * H * 2 * (2 * d + rd)
            elif kind == "attention":
                params += (2 * H * d + 2 * G * d) * W
                attn += T * T / 2.0 * H * 4 * d
            else:
                params += (6 * H * d + d) * W + H * d * d
                attn += T * 8.0 * H * d * d
        return {"bytes": 2.0 * (params + V * W) + 4.0 * T * W, "flops": 2.0 * T * params + attn + 2.0 * V * W}
    c = S.SHAPES[case["model"]]
    hd, plan = c["hidden"] // c["n_heads"], S.tensor_plan(c, case["mix"])
    kvd, L, A = c["n_kv_heads"] * hd, c["n_layers"], c["hidden"]
    layer_w = float(sum(r * k for n, t, r, k in plan if n.startswith("blk.") and t != S.F32))
    head_w = float(c["vocab"]) * A
    weights = float(S.weight_bytes_per_token(c, case["mix"]))
    if op in ("decode", "sampled"):
        n, p = case["steps"], case["context"] + case["steps"] / 2.0
        return {"bytes": n * (weights + 8.0 * p * kvd * L), "flops": n * (2.0 * (layer_w + head_w) + 4.0 * p * A * L)}
    if op == "prompt":
        T = case["tokens"]
        return {"bytes": weights + 8.0 * T * kvd * L, "flops": 2.0 * T * layer_w + 2.0 * head_w + 2.0 * T * T * A * L}
    if op == "packed":
        lens = _packed_lengths(case)
        T, n = sum(lens), len(lens)
        return {"bytes": weights + 8.0 * T * kvd * L + 4.0 * n * c["vocab"],
                "flops": 2.0 * T * layer_w + 2.0 * n * head_w + 2.0 * sum(t * t for t in lens) * A * L}
    n, B, p = case["steps"], case["sequences"], case["context"] + case["steps"] / 2.0
    return {"bytes": n * (weights + 8.0 * B * p * kvd * L) + 4.0 * B * c["vocab"],
            "flops": n * B * (2.0 * (layer_w + head_w) + 4.0 * p * A * L)}


# ---- inputs -----------------------------------------------------------------------------------------------------------------
# odd lengths: where a large vocabulary goes round the pool, its rows stay distinct (equal rows of the head would tie)
POOL_BLOCKS = {S.Q4_K: 400_009, S.Q6_K: 300_007, S.Q8_0: 2_000_003}


class _Tensors:
    """The quantized tensors of one model, cut out of one random pool of blocks per format (distinct cuts per tensor), with
    scales that give weights of standard deviation 1 / sqrt(columns)."""

    def __init__(self, case, seed):
        self.cfg = dict(S.SHAPES[case["model"]])
        self.plan = S.tensor_plan(self.cfg, case["mix"])
        self.seed, self.pools = seed, {}

    def pool(self, typ, std):
        if (typ, std) not in self.pools:
            if (typ, 1.0) not in self.pools:
                rng = np.random.default_rng([self.seed, typ])
                self.pools[typ, 1.0] = S.random_blocks(typ, POOL_BLOCKS[typ], rng, w_std=1.0)
            b = self.pools[typ, 1.0].copy()
            for off in {S.Q4_K: (0, 2), S.Q6_K: (208,), S.Q8_0: (0,)}[typ]:
                d = b[:, off:off + 2].copy().view(np.float16).astype(np.float32) * std
                b[:, off:off + 2] = d.astype(np.float16).view(np.uint8)
            self.pools[typ, std] = b
        return self.pools[typ, std]

    def __iter__(self):
        rng = np.random.default_rng([self.seed, 7])
        for name, typ, rows, cols in self.plan:
            if typ == S.F32:
                yield name, typ, (1.0 + 0.1 * rng.standard_normal(cols)).astype(np.float32), rows, cols
                continue
            pool = self.pool(typ, 1.0 if name == "token_embd.weight" else float(cols) ** -0.5)
            n, at = rows * cols // S.BLOCK_ELEMS[typ], int(rng.integers(0, len(pool)))
            if n > len(pool) // 2:  # embedding and head of the large vocabularies
                yield name, typ, np.resize(np.roll(pool, at, axis=0), (n, pool.shape[1])), rows, cols
            else:
                at = at % (len(pool) - n)
                yield name, typ, pool[at:at + n], rows, cols


def _max_pos(case):
    need = case.get("context", 0) + case.get("steps", 0) + case.get("tokens", 0) + 8
    return 512 if need <= 512 else 2048 if need <= 2048 else 8192


def _prompts(case, cfg, seed):
    rng = np.random.default_rng([seed, 11])
    n = case.get("sequences", 1)
    if case["op"] == "packed":
        lens = _packed_lengths(case)
    elif case["op"] == "batch":  # sequences of a running server stand at different lengths
        lens = [max(1, case["context"] - (3 * i) % max(1, case["context"] // 2)) for i in range(n)]
    else:
        lens = [case.get("tokens") or case["context"]] * n
    return [rng.integers(0, cfg["vocab"], k).astype(np.int32) for k in lens]


def _packed_lengths(case):
    """From a few words up to `tokens`, in no order."""
    n, top = case["sequences"], case["tokens"]
    return [max(3, top * ((7 * i) % n + 1) // n) for i in range(n)]


def prepare(case, seed):
    from tinyllama_cpp_amd import engine
    if case["op"].startswith("layers"):
        return _prepare_layers(engine, case, seed)
    t = _Tensors(case, seed)
    t.cfg["max_pos"] = _max_pos(case)
    m = engine.Model(t.cfg)
    for name, typ, arr, rows, cols in t:
        m.set_tensor(name, typ, arr, rows, cols)
    m.finalize()
    st = dict(case=case, model=m, seed=seed, prompts=_prompts(case, t.cfg, seed))
    if case["op"] in ("decode", "sampled"):
        st["first"] = int(np.argmax(m.prefill(st["prompts"][0])))
    elif case["op"] in ("packed", "batch"):
        m.batch_init(case["sequences"])
        if case["op"] == "batch":
            st["first"] = m.batch_prefill_packed(st["prompts"], want_logits=False)[1]
    return st


def run(state):
    c, m, p = state["case"], state["model"], state["prompts"]
    op, n = c["op"], c.get("steps", 0)
    if op == "prompt":
        m.reset_kv()
        return {"logits": m.prefill(p[0])}
    if op == "layers_prompt":
        m.reset_kv()
        return {"logits": m.prefill_rows(p[0], 0, np.array([p[0].size - 1], np.int32))}
    if op == "packed":
        logits, ids = m.batch_prefill_packed(p)
        return {"logits": logits, "ids": ids}
    if op == "batch":
        pos = np.array([x.size for x in p], np.int32)
        slots = np.arange(len(p), dtype=np.int32)
        ids = m.batch_generate_greedy(state["first"], pos, slots, n - 1)
        logits, last = m.batch_decode(ids[-1], pos + n - 1, slots)
        return {"ids": np.concatenate([ids, last[None]]), "logits": logits}
    pos = p[0].size
    if op == "sampled":
        ids = m.generate_sampled(state["first"], pos, n - 1, penalty=1.1, history=p[0][-64:], temperature=0.8, top_k=40, top_p=0.9,
                                 seed=state["seed"])
    else:
        ids = m.generate_greedy(state["first"], pos, n - 1)
    logits, last = m.decode(ids[-1], pos + n - 1)
    return {"ids": np.append(ids, np.int32(last)), "logits": logits}


def tolerance(case):
    # measured against exact(): 1e-6 (one token) to 3.5e-6 (a prompt through 32 layers, 12 layers with routed experts); an
    # arg-max over two logits closer than that may fall either way, and every later token with it: none does in these inputs
    if case["op"] == "layers_prompt":
        return {"rel": 2e-2, "max": 0.1}  # activations in bf16: 5e-3 measured
    return {"rel": 1.4e-5, "max": 1e-4, "differ": 0.0}


# ---- the same answers in 64 bits, from torch alone --------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _f16(b, off):
    return b[:, off:off + 2].contiguous().view(torch.float16).double()


def _dequantize(typ, blocks, rows, cols):
    """float64 weights of GGUF blocks (uint8 array [n, block bytes])."""
    dev = _device()
    if typ == S.F32:
        return torch.from_numpy(blocks).to(dev).double()
    b = torch.from_numpy(np.ascontiguousarray(blocks)).to(dev)
    n = b.shape[0]
    if typ == S.Q8_0:
        w = b[:, 2:34].contiguous().view(torch.int8).double() * _f16(b, 0).abs()
    elif typ == S.Q4_K:
        s = b[:, 4:16].int()
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double() * _f16(b, 0)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double() * _f16(b, 2)
        q = b[:, 16:144].reshape(n, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(n, 8, 32)
        w = sc[:, :, None] * q.double() - mn[:, :, None]
    else:  # Q6_K: two halves of 128 weights
        ql, qh = b[:, 0:128].reshape(n, 2, 2, 32).int(), b[:, 128:192].reshape(n, 2, 1, 32).int()
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * _f16(b, 208)
        lo = torch.cat([ql & 15, ql >> 4], 2)  # [n, half, 4, 32]
        hi = torch.cat([(qh >> k) & 3 for k in (0, 2, 4, 6)], 2)
        q = (lo | (hi << 4)) - 32
        w = q.reshape(n, 16, 16).double() * sc[:, :, None]
    return w.reshape(rows, cols)


class _Llama64:
    """Weights are kept as float32 (their values are exact there or within 2^-24) and widened for each product."""

    def __init__(self, case, seed, sequences, max_pos):
        t = _Tensors(case, seed)
        self.c, self.w = t.cfg, {}
        for name, typ, arr, rows, cols in t:
            w = _dequantize(typ, arr, rows, cols)
            self.w[name] = w.float() if typ != S.F32 else w
        c = self.c
        self.hd, self.G = c["hidden"] // c["n_heads"], c["n_kv_heads"]
        shape = (c["n_layers"], sequences, self.G, max_pos, self.hd)
        self.k, self.v = (torch.zeros(shape, dtype=torch.float64, device=_device()) for _ in range(2))
        f = np.float64(c["rope_theta"]) ** -(np.arange(0, self.hd, 2, dtype=np.float32) / np.float32(self.hd)).astype(np.float64)
        ang = np.arange(max_pos, dtype=np.float32)[:, None] * f.astype(np.float32)[None, :]  # the table's angles are 32-bit
        self.cos, self.sin = (torch.from_numpy(fn(ang.astype(np.float64))).to(_device()) for fn in (np.cos, np.sin))

    def mul(self, x, name):
        return x @ self.w[name].double().T

    def norm(self, x, name):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + max(self.c["eps"], 1e-5)) * self.w[name]

    def rope(self, x, pos):  # [n, heads, hd], neighbouring pairs
        c, s = self.cos[pos][:, None], self.sin[pos][:, None]
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)

    def attend(self, q, k, v, pos):
        """q [S, G, rep, hd] with k, v [S, G, P, hd]: row r of a group sees positions up to pos[S, rep]."""
        s = (q @ k.transpose(-1, -2).contiguous()) * self.hd ** -0.5
        hide = torch.arange(k.shape[2], device=q.device)[None, None, None] > pos[:, None, :, None]
        return torch.softmax(s.masked_fill(hide, -math.inf), -1) @ v

    def forward(self, tokens, pos, seq, rows):
        """Tokens in sequence order at their positions; logits of the listed rows. One token a sequence, or whole sequences."""
        c, dev = self.c, _device()
        H, G, hd, n = c["n_heads"], self.G, self.hd, len(tokens)
        rep, dpos, dseq = H // G, torch.as_tensor(pos, device=dev), torch.as_tensor(seq, device=dev)
        one = len(set(seq)) == n
        x = self.w["token_embd.weight"][torch.as_tensor(tokens, device=dev).long()].double()
        for i in range(c["n_layers"]):
            p = "blk.%d." % i
            h = self.norm(x, p + "attn_norm.weight")
            q = self.rope(self.mul(h, p + "attn_q.weight").view(n, H, hd), dpos)
            self.k[i].transpose(1, 2)[dseq, dpos] = self.rope(self.mul(h, p + "attn_k.weight").view(n, G, hd), dpos)
            self.v[i].transpose(1, 2)[dseq, dpos] = self.mul(h, p + "attn_v.weight").view(n, G, hd)
            if one:
                P = int(max(pos)) + 1
                o = self.attend(q.view(n, G, rep, hd), self.k[i][dseq, :, :P], self.v[i][dseq, :, :P], dpos[:, None].expand(n, rep)).reshape(n, H * hd)
            else:
                o = torch.empty(n, H * hd, dtype=torch.float64, device=dev)
                for a in sorted(set(seq)):
                    at = (dseq == a).nonzero()[:, 0]
                    for part in at.split(256):
                        P, r = int(dpos[part[-1]]) + 1, len(part)
                        y = self.attend(q[part].view(r, G, rep, hd).permute(1, 2, 0, 3).reshape(1, G, rep * r, hd), self.k[i][a:a + 1, :, :P],
                                        self.v[i][a:a + 1, :, :P], dpos[part].repeat(rep)[None])
                        o[part] = y.view(G, rep, r, hd).permute(2, 0, 1, 3).reshape(r, H * hd)
            x = x + self.mul(o, p + "attn_output.weight")
            h = self.norm(x, p + "ffn_norm.weight")
            g = self.mul(h, p + "ffn_gate.weight")
            x = x + self.mul(g * torch.sigmoid(g) * self.mul(h, p + "ffn_up.weight"), p + "ffn_down.weight")
        return self.mul(self.norm(x[torch.as_tensor(rows, device=dev)], "output_norm.weight"), "output.weight")


def exact(case, seed):
    op = case["op"]
    if op == "sampled":
        return None  # the tokens come from the sampler's own random numbers
    with torch.no_grad():
        if op.startswith("layers"):
            return _exact_layers(case, seed)
        cfg = S.SHAPES[case["model"]]
        prompts = _prompts(case, cfg, seed)
        m = _Llama64(case, seed, len(prompts), max(len(p) for p in prompts) + case.get("steps", 0) + 1)
        flat = np.concatenate(prompts)
        pos = np.concatenate([np.arange(len(p)) for p in prompts])
        seq = np.concatenate([np.full(len(p), i) for i, p in enumerate(prompts)])
        z = m.forward(flat, pos, seq.tolist() if len(prompts) > 1 else [0] * len(flat), np.cumsum([len(p) for p in prompts]) - 1)
        if op == "prompt":
            return {"logits": z[0].cpu().numpy()}
        if op == "packed":
            return {"logits": z.cpu().numpy(), "ids": z.argmax(-1).int().cpu().numpy()}
        ids, at = [], np.array([len(p) for p in prompts])
        for k in range(case["steps"]):
            z = m.forward(z.argmax(-1).cpu().numpy(), at + k, list(range(len(prompts))), list(range(len(prompts))))
            ids.append(z.argmax(-1).int().cpu().numpy())
        if op == "batch":
            return {"ids": np.stack(ids), "logits": z.cpu().numpy()}
        return {"ids": np.concatenate(ids), "logits": z[0].cpu().numpy()}


# ---- layer-list models ------------------------------------------------------------------------------------------------------
def _sogalix_kinds(n):
    """Latent attention (every second one over the cache of the one before it), delta rule, sink attention, delta rule in turn."""
    return [("latent_attention", i % 8 != 4) if i % 4 == 0 else ("attention", True) if i % 4 == 2 else ("general_delta", True) for i in range(n)]


def _sogalix_ff(z):
    return z["top"] * z["ff"] + z["shared_ff"]


def _layers_tensors(case, seed):
    """(configuration, iterator over (name, bf16 bits)) of a layer-list model."""
    z = LAYERED[case["size"]]
    W, V, H, G, d, n = z["width"], z["vocab"], z["heads"], z["kv_heads"], z["dim"], z["layers"]
    rng = np.random.default_rng([seed, 5])
    pool = rng.standard_normal((1 << 23) + 9).astype(np.float32)  # (odd: rows that go round it stay distinct)
    scaled = {}

    def mat(name, r, c, std=None):
        std = std or c ** -0.5
        if std not in scaled:
            scaled[std] = S.to_bf16(pool * np.float32(std))
        k, at = r * c, int(rng.integers(0, pool.size))
        if k > pool.size // 2:
            return name, np.resize(np.roll(scaled[std], at), (r, c))
        at %= pool.size - k
        return name, scaled[std][at:at + k].reshape(r, c)

    def vec(name, k, centre, spread=0.05):
        return name, S.to_bf16((centre + spread * rng.standard_normal(k)).astype(np.float32))

    if case["op"] == "layers_decode":
        layer = S.stack_layer(H, G, d, d, z["window"], v_mix=True, experts=z["experts"], top=z["top"], ff=z["ff"], shared_ff=z["shared_ff"])

        def routed():
            yield from (mat("embed", V, W, 1.0), mat("head", V, W), vec("embed.norm", W, 0.0), vec("final.norm", W, 0.0))
            for i in range(n):
                p = "l%d." % i
                yield from (mat(p + "mix.q", H * d, W), mat(p + "mix.k", G * d, W), mat(p + "mix.v", G * d, W), mat(p + "mix.o", W, H * d))
                yield from (vec(p + "mix.q.norm", H * d, 1.0), vec(p + "mix.k.norm", G * d, 1.0), vec(p + "norm1", W, 0.0), vec(p + "norm2", W, 0.0))
                yield p + "mix.vmix", S.to_bf16(np.array(0.5, np.float32))
                yield from (mat(p + "mlp.router", z["experts"], W), vec(p + "mlp.router.b", z["experts"], 0.0))
                for q, ff in [(p + "mlp.e%d." % e, z["ff"]) for e in range(z["experts"])] + [(p + "mlp.shared.", z["shared_ff"])]:
                    yield from (mat(q + "gate", ff, W), mat(q + "up", ff, W), mat(q + "down", W, ff))

        return S.stack_config(W, V, [layer] * n), routed()
    rq, rk, rd, F, layers = W // 2, 4 * d, d // 2, _sogalix_ff(z), []
    for i, (kind, own) in enumerate(_sogalix_kinds(n)):
        mx = (S.sogalix_latent(H, d, rd, d, rq, rk, base=250000.0, kv_from=None if own else i - 4) if kind == "latent_attention" else
              S.sogalix_attention(H, G, d, d, q_temp=(0.1, 512)) if kind == "attention" else S.sogalix_delta(H, d))
        layers.append(S.sogalix_layer(kind, mx, F))

    def dense():
        yield from (mat("embed", V, W, 1.0), mat("head", V, W))
        for nm in ["embed.norm", "final.norm"] + ["l%d.norm%d" % (i, k) for i in range(n) for k in (1, 2)]:
            yield from (vec(nm, W, 1.0), vec(nm + ".b", W, 0.0))
        for i, (kind, own) in enumerate(_sogalix_kinds(n)):
            p = "l%d.mix." % i
            yield mat(p + "o", W, H * d)
            if kind == "latent_attention":
                yield from (mat(p + "dq", rq, W), vec(p + "dq.norm", rq, 1.0), mat(p + "uq", H * (d + rd), rq))
                if own:
                    yield from (mat(p + "dkv", rk + rd, W), vec(p + "dkv.norm", rk, 1.0))
                yield from (mat(p + "uk", H * d, rk), mat(p + "uv", H * d, rk), mat(p + "g", H, W))
            elif kind == "attention":
                yield from (mat(p + "q", H * d, W), mat(p + "k", G * d, W), mat(p + "v", G * d, W))
            else:
                yield from (mat(p + x, H * d, W) for x in "rkvga")
                yield from (mat(p + "w1", d, W), mat(p + "w2", H * d, d), vec(p + "a.b", H * d, 0.0, 0.3), vec(p + "w0", H * d, -1.0, 0.5), vec(p + "norm", H * d, 1.0))
            yield from (mat("l%d.mlp.up" % i, F, W), mat("l%d.mlp.down" % i, W, F))
            yield "l%d.mlp.act" % i, S.to_bf16(np.array([0.3, -0.2], np.float32))

    return S.sogalix_config(W, V, layers), dense()


def _prepare_layers(engine, case, seed):
    cfg, tensors = _layers_tensors(case, seed)
    d = LAYERED[case["size"]]["dim"]
    m = engine.StackModel(cfg, _max_pos(case), {"l%d.mix.w1" % i: np.empty((d, 0)) for i in range(len(cfg["layers"]))})
    for name, arr in tensors:
        m.set_tensor(name, arr)
    m.finalize()
    st = dict(case=case, model=m, seed=seed, prompts=_prompts(case, {"vocab": cfg["vocab"]}, seed))
    if case["op"] == "layers_decode":
        m.set_prefill(3, 1)  # the context that an answer starts from, at 32-bit precision
        last = np.array([case["context"] - 1], np.int32)
        st["first"] = int(np.argmax(m.prefill_rows(st["prompts"][0], 0, last)[0]))
    else:
        m.set_prefill(1, 1)  # serving precision: activations in bf16
    return st


def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _window_softmax(q, k, v, scale, first, window=None, sink=False):
    """q [T, H, d] at positions first.., k [P, G, d], v [P, G, vd] -> [T, H * vd]; sink: a score 0 joins the denominator."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    s = (q.view(T, G, H // G, -1).permute(1, 2, 0, 3).reshape(G, H // G * T, -1) @ k.permute(1, 2, 0).contiguous()) * scale
    gap = (first + torch.arange(T, device=q.device))[:, None] - torch.arange(k.shape[0], device=q.device)[None]
    hide = gap < 0 if window is None else (gap < 0) | (gap >= window)
    s = s.view(G, H // G, T, -1).masked_fill(hide, -math.inf)
    top = s.amax(-1, keepdim=True).clamp(min=0.0) if sink else s.amax(-1, keepdim=True)
    e = torch.exp(s - top)
    e = e / (e.sum(-1, keepdim=True) + (torch.exp(-top) if sink else 0.0))
    return (e.view(G, H // G * T, -1) @ v.permute(1, 0, 2).contiguous()).view(G, H // G, T, -1).permute(2, 0, 1, 3).reshape(T, -1)


def _exact_layers(case, seed):
    cfg, tensors = _layers_tensors(case, seed)
    w = {k: torch.from_numpy(S.from_bf16(v).copy()).to(_device()).double() for k, v in tensors}
    tokens = _prompts(case, {"vocab": cfg["vocab"]}, seed)[0]
    if case["op"] == "layers_prompt":
        return {"logits": _sogalix64(cfg, w, tokens).cpu().numpy()}
    state, ids = {}, []
    z = _ralasun64(cfg, w, tokens, state)
    for _ in range(case["steps"]):
        z = _ralasun64(cfg, w, [int(z.argmax())], state)
        ids.append(int(z.argmax()))
    return {"ids": np.array(ids, np.int32), "logits": z.cpu().numpy()}


def _ralasun64(cfg, w, tokens, state):
    """The next tokens of a sequence (state: its caches): logits of the last one."""
    eps, first, T = cfg["norm"]["eps"], state.get("n", 0), len(tokens)
    x = _rms(w["embed"][torch.as_tensor(np.asarray(tokens), device=_device()).long()], eps) * (1 + w["embed.norm"])
    v1 = None

    def unit(h, q, limit):
        g, u = (h @ w[q + "gate"].T).clamp(max=limit), (h @ w[q + "up"].T).clamp(-limit, limit)
        return (g * torch.sigmoid(1.702 * g) * (u + 1)) @ w[q + "down"].T

    for i, L in enumerate(cfg["layers"]):
        mx, ml, p = L["mixer"], L["mlp"], "l%d." % i
        H, G, d = mx["heads"], mx["kv_heads"], mx["dim"]
        q = (_rms(x @ w[p + "mix.q"].T, eps) * w[p + "mix.q.norm"]).view(T, H, d)
        k = (_rms(x @ w[p + "mix.k"].T, eps) * w[p + "mix.k.norm"]).view(T, G, d)
        v = (x @ w[p + "mix.v"].T).view(T, G, d)
        if v1 is None:
            v1 = v
        else:
            v = v + w[p + "mix.vmix"] * (v1 - v)
        for nm, a in (("k", k), ("v", v)):
            state[nm, i] = torch.cat([state[nm, i], a]) if first else a
        o = _window_softmax(q, state["k", i], state["v", i], mx["scale"], first, mx["mask"]["size"])
        x = x + _rms(o @ w[p + "mix.o"].T, eps) * (1 + w[p + "norm1"])
        z, ids = (x @ w[p + "mlp.router"].T + w[p + "mlp.router.b"]).topk(ml["router"]["top"], -1)
        part, y = torch.softmax(z, -1), unit(x, p + "mlp.shared.", ml["shared"]["limit"])
        for e in range(ml["router"]["experts"]):
            t, j = (ids == e).nonzero(as_tuple=True)
            if len(t):
                y[t] += part[t, j][:, None] * unit(x[t], p + "mlp.e%d." % e, ml["expert"]["limit"])
        x = x + _rms(y, eps) * (1 + w[p + "norm2"])
    state["n"] = first + T
    return (_rms(x[-1], eps) * (1 + w["final.norm"])) @ w["head"].T


def _sogalix64(cfg, w, tokens):
    """Logits [1, vocab] of the last token of a sequence."""
    eps, T, dev, keep = cfg["norm"]["eps"], len(tokens), _device(), {}

    def norm(x, nm):
        x = x - x.mean(-1, keepdim=True)
        return _rms(x, eps) * w[nm] + w[nm + ".b"]

    def turn(x, dims, base):  # [T, heads, n]: neighbouring pairs of the first `dims`
        f = base ** (-torch.arange(0, dims, 2, dtype=torch.float64, device=dev) / dims)
        ang = torch.arange(T, dtype=torch.float64, device=dev)[:, None, None] * f
        a, b = x[..., 0:dims:2], x[..., 1:dims:2]
        return torch.cat([torch.stack([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], -1).flatten(-2), x[..., dims:]], -1)

    x = norm(w["embed"][torch.as_tensor(tokens, device=dev).long()], "embed.norm")
    for i, L in enumerate(cfg["layers"]):
        mx, p = L["mixer"], "l%d.mix." % i
        H, d = mx["heads"], mx["dim"]
        h = norm(x, "l%d.norm1" % i)
        if L["type"] == "attention":
            q, k, v = ((h @ w[p + nm].T).view(T, -1, d) for nm in "qkv")
            pos = torch.arange(T, dtype=torch.float64, device=dev)
            q = q * (1 + mx["q_temp"]["coef"] * torch.log(torch.floor((pos + 1) / mx["q_temp"]["every"]) + 1))[:, None, None]
            y = _window_softmax(q, k, v, mx["scale"], 0, sink=True)
        elif L["type"] == "latent_attention":
            rk, rot = mx["kv_rank"], mx["rot"]
            q = ((_rms(h @ w[p + "dq"].T, eps) * w[p + "dq.norm"]) @ w[p + "uq"].T).view(T, H, -1)
            q = torch.cat([q[..., :d], turn(q[..., d:], rot["dims"], rot["base"])], -1)
            if mx.get("kv_from") is None:
                c = h @ w[p + "dkv"].T
                keep[i] = _rms(c[:, :rk], eps) * w[p + "dkv.norm"], turn(c[:, None, rk:], rot["dims"], rot["base"])
            c, kr = keep[i if mx.get("kv_from") is None else mx["kv_from"]]
            k = torch.cat([(c @ w[p + "uk"].T).view(T, H, d), kr.expand(T, H, -1)], -1)
            y = _window_softmax(q, k, (c @ w[p + "uv"].T).view(T, H, -1), mx["scale"], 0)
            y = (y.view(T, H, -1) * torch.sigmoid(h @ w[p + "g"].T)[:, :, None]).reshape(T, -1)
        else:
            r, k, v = ((h @ w[p + nm].T).view(T, H, d) for nm in "rkv")
            dec = torch.exp(-math.exp(-0.5) * torch.sigmoid(torch.tanh(h @ w[p + "w1"].T) @ w[p + "w2"].T + w[p + "w0"])).view(T, H, d, 1)
            u = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
            au = torch.sigmoid(h @ w[p + "a"].T + w[p + "a.b"]).view(T, H, d) * u
            s, y = torch.zeros(H, d, d, dtype=torch.float64, device=dev), torch.empty(T, H, d, dtype=torch.float64, device=dev)
            for t in range(T):
                s = dec[t] * s - au[t, :, :, None] * (u[t, :, None] @ s) + k[t, :, :, None] * v[t, :, None]
                y[t] = (r[t, :, None] @ s)[:, 0]
            y = _rms(y, eps).reshape(T, -1) * w[p + "norm"] * torch.sigmoid(h @ w[p + "g"].T)
        x = x + y @ w[p + "o"].T
        z = norm(x, "l%d.norm2" % i) @ w["l%d.mlp.up" % i].T
        sp = torch.nn.functional.softplus(w["l%d.mlp.act" % i])
        neg = z.clamp(max=0.0)
        z = torch.where(z > 0, sp[0] * z * z + 0.5 * z, (0.5 + sp[1]) * (torch.expm1(neg) - neg) + 0.5 * z)
        x = x + z @ w["l%d.mlp.down" % i].T
    return norm(x[-1:], "final.norm") @ w["head"].T
