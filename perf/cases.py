"""The calls a serving program makes of this sampler, as measurable cases.

Each case is one pass through a public entry point on inputs that are already
on the GPU: the batched sampler (`BatchSampler.launch` on a prepared
descriptor, which is one `oxs_sample_batch`), the decode loop (`DecodeLoop`,
captured once and replayed, tokens polled on the host), the greedy argmax
(`oxs_argmax`), the Q8_0 LM head (`quantize_q8_1`, `LmHeadQ8_0.project`) and the
grammar masks (`DfaSchemaGrammar.token_masks`). Sizes are those of the seeded
workloads (`oxide_sampler/workloads.py`), of the tests, and generic ones.

Results are whole: tokens, statuses, kept candidates and their probabilities,
histories, generator and Mirostat states, logits, masks. They are the
reference's to the last bit (the tests assert it against the CPU oracle: no
float of a kept probability, a mu or a logit may differ), so the tolerance is
"exact" everywhere.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "oxide-tech-llm-engine_amd"))

from oxide_sampler import (  # noqa: E402
    BatchSampler, DecodeLoop, DfaSchemaGrammar, LmHeadQ8_0, MirostatMode, SamplerState, SamplingConfig, TokenBytes,
    _abi, configs_to_array, load_library, quantize_q8_1,
)
from oxide_sampler.workloads import disabled_config  # noqa: E402

POOL = 256        # the reference's smallest candidate pool: max(top_k, 256)
HISTORY_ROOM = 32  # free history slots per row beyond the prompt
NEWLINE = 10


def listed():
    return [
        # one lightly loaded request on a 32k vocabulary (the seeded config 1): launches and latency
        {"name": "sample_b1_v32000", "kind": "sample", "batch": 1, "vocab": 32000, "dtype": "f32", "logits": "normal",
         "chain": "repeat", "top_k": 40, "history": 64, "mask": 0.0, "biases": 0},
        # the headline decode batch (config 2): every penalty, then top-k, top-p and min-p
        {"name": "sample_b64_v128256", "kind": "sample", "batch": 64, "vocab": 128256, "dtype": "f32",
         "logits": "zipf", "chain": "penalties", "top_k": 50, "history": 512, "mask": 0.0, "biases": 0},
        # structured output (config 3): a grammar mask with about 3% of the tokens allowed, top-p
        {"name": "sample_mask_b128_v128256", "kind": "sample", "batch": 128, "vocab": 128256, "dtype": "f32",
         "logits": "zipf", "chain": "top_p", "top_k": 0, "history": 0, "mask": 0.03, "biases": 0},
        # a large batch of bf16 logits with long windows, tail-free and typical (config 4)
        {"name": "sample_bf16_b256_v151936", "kind": "sample", "batch": 256, "vocab": 151936, "dtype": "bf16",
         "logits": "heavy", "chain": "typical", "top_k": 0, "history": 1024, "mask": 0.0, "biases": 0},
        # the largest batch and vocabulary, Mirostat v2 (config 5)
        {"name": "sample_mirostat_b512_v262144", "kind": "sample", "batch": 512, "vocab": 262144, "dtype": "f32",
         "logits": "normal", "chain": "mirostat", "top_k": 0, "history": 256, "mask": 0.0, "biases": 0},
        # a vocabulary nobody padded (odd size, rows on 4-byte boundaries), the default chain with
        # biased and banned tokens: a handful of chat requests
        {"name": "sample_ragged_b24_v50257", "kind": "sample", "batch": 24, "vocab": 50257, "dtype": "f32",
         "logits": "zipf", "chain": "default", "top_k": 40, "history": 300, "mask": 0.0, "biases": 16},
        # a wide candidate pool (creative settings, draft sampling): top_k above the default pool of 256
        {"name": "sample_topk1000_b16_v128256", "kind": "sample", "batch": 16, "vocab": 128256, "dtype": "f32",
         "logits": "zipf", "chain": "penalties", "top_k": 1000, "history": 512, "mask": 0.0, "biases": 0},
        # the scheduler's decode stage, 64 slots of mixed requests: greedy, default, DRY and Mirostat rows
        {"name": "decode_mixed_b64_v128256", "kind": "decode", "batch": 64, "vocab": 128256, "history": 512},
        # the greedy path
        {"name": "argmax_b32_v151936", "kind": "argmax", "batch": 32, "vocab": 151936},
        # the LM head for the last prompt token, and for a decode batch
        {"name": "lm_head_b1_m128256_k4096", "kind": "lm_head", "batch": 1, "m": 128256, "k": 4096},
        {"name": "lm_head_b64_m128256_k4096", "kind": "lm_head", "batch": 64, "m": 128256, "k": 4096},
        # grammar masks for a structured decode batch (the 8-state JSON validator)
        {"name": "dfa_mask_b128_v128256", "kind": "dfa", "batch": 128, "vocab": 128256, "prefix": 0},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _vocab(rng, most=262144):
    v = _log_int(rng, 32000, most)
    return v if rng.random() < 0.5 else max(32000, v // 128 * 128)  # half padded, half any size


def draw(rng):
    kind = rng.choice(["sample", "sample", "sample", "sample", "sample", "decode", "argmax", "lm_head", "lm_head",
                       "dfa"])
    if kind == "lm_head":
        k = 128 * rng.randint(7, 32)
        return {"kind": kind, "batch": _log_int(rng, 1, 128), "m": _vocab(rng, 128256), "k": k}
    if kind == "dfa":
        return {"kind": kind, "batch": _log_int(rng, 1, 128), "vocab": _vocab(rng, 160000),
                "prefix": rng.choice([0, 0, rng.randint(1, 70)])}
    if kind == "argmax":
        return {"kind": kind, "batch": _log_int(rng, 1, 64), "vocab": _vocab(rng)}
    if kind == "decode":
        return {"kind": kind, "batch": _log_int(rng, 1, 128), "vocab": _vocab(rng), "history": _log_int(rng, 16, 1024)}
    chain = rng.choice(["repeat", "penalties", "top_p", "typical", "mirostat", "default"])
    return {"kind": kind, "batch": _log_int(rng, 1, 256), "vocab": _vocab(rng), "dtype": rng.choice(["f32", "bf16"]),
            "logits": rng.choice(["normal", "zipf", "heavy"]), "chain": chain,
            "top_k": 0 if chain in ("top_p", "typical", "mirostat") else _log_int(rng, 10, 1000),
            "history": _log_int(rng, 16, 1024), "mask": rng.choice([0.0, 0.0, 0.0, 0.03, 0.3]),
            "biases": rng.choice([0, 0, 16])}


# ------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _logits(g, batch, vocab, shape):
    """normal: N(0, 2). zipf: N(0, 3) plus -1.1 ln(rank) over a permutation per row.
    heavy: N(0, 2.5), 1% of the entries U[6, 10]."""
    x = torch.randn(batch, vocab, generator=g, device="cuda")
    if shape == "normal":
        return x * 2.0
    if shape == "zipf":
        rank = torch.rand(batch, vocab, generator=g, device="cuda").argsort(dim=1)
        return x * 3.0 - 1.1 * torch.log(rank.float() + 1.0)
    x *= 2.5
    heavy = torch.rand(batch, vocab, generator=g, device="cuda")
    return torch.where(heavy < 0.01, 6.0 + 4.0 * (heavy * 100.0), x)


def _history(g, batch, vocab, n):
    """Prompt ids skewed to a common part of the vocabulary, so that some repeat."""
    u = torch.rand(batch, n + HISTORY_ROOM, generator=g, device="cuda")
    return (u.pow(3) * vocab).to(torch.int32).clamp_(0, vocab - 1)


def _config(case, g):
    chain, k = case["chain"], case["top_k"]
    if chain == "repeat":
        c = disabled_config(repeat_penalty=1.1, repeat_last_n=64, temperature=0.8, top_k=k, top_p=0.95)
    elif chain == "penalties":
        c = disabled_config(frequency_penalty=0.3, presence_penalty=0.2, repeat_penalty=1.05, repeat_last_n=512,
                            temperature=0.7, top_k=k, top_p=0.9, min_p=0.05)
    elif chain == "top_p":
        c = disabled_config(temperature=1.0, top_p=0.95)
    elif chain == "typical":
        c = disabled_config(repeat_penalty=1.1, repeat_last_n=1024, temperature=0.9, typical_p=0.95, tfs_z=0.95)
    elif chain == "mirostat":
        c = disabled_config(presence_penalty=0.5, mirostat_mode=MirostatMode.V2, mirostat_tau=5.0, mirostat_eta=0.1)
    else:
        c = SamplingConfig(top_k=k)
    if case["biases"]:
        ids = torch.randint(0, case["vocab"], (2 * case["biases"],), generator=g, device="cuda").tolist()
        vals = (torch.rand(case["biases"], generator=g, device="cuda") * 4 - 2).tolist()
        c.logit_biases = dict(zip(ids[: case["biases"]], vals))
        c.banned_tokens = set(ids[case["biases"]:])
    return c


def _sample_inputs(case, seed):
    g = _gen(seed)
    B, V, H = case["batch"], case["vocab"], case["history"]
    x = _logits(g, B, V, case["logits"])
    if case["dtype"] == "bf16":
        x = x.to(torch.bfloat16)
    mask = None
    if case["mask"] > 0:
        words = (V + 31) // 32
        bits = torch.rand(B, words * 32, generator=g, device="cuda") < case["mask"]
        bits[:, V:] = False
        bits.scatter_(1, torch.randint(0, V, (B, 1), generator=g, device="cuda"), True)  # never an empty row
        weight = torch.ones(32, dtype=torch.int64, device="cuda") << torch.arange(32, device="cuda")
        mask = (bits.view(B, words, 32).long() * weight).sum(2)
        mask = (mask - (mask >> 31 << 32)).to(torch.int32)  # the low 32 bits, two's complement
    hist = _history(g, B, V, H)
    mu = torch.full((B,), 10.0, device="cuda")
    rng = torch.randint(1, 1 << 62, (B,), generator=g, device="cuda")
    return {"logits": x, "mask": mask, "history": hist, "mu": mu, "rng": rng, "config": _config(case, g)}


def _prepare_sample(case, seed):
    s = _sample_inputs(case, seed)
    B, V, H, dev = case["batch"], case["vocab"], case["history"], "cuda"
    raw, bias_ids, bias_vals, ban_ids = configs_to_array([s["config"]], NEWLINE)
    s["configs"] = torch.from_numpy(raw).to(dev)
    s["bias_ids"] = torch.from_numpy(bias_ids.view(np.int32)).to(dev)
    s["bias_values"] = torch.from_numpy(bias_vals).to(dev)
    s["ban_ids"] = torch.from_numpy(ban_ids.view(np.int32)).to(dev)
    s["history_len"] = torch.full((B,), H, dtype=torch.int32, device=dev)
    kept = max(POOL, case["top_k"])
    out = {"tokens": torch.zeros(B, dtype=torch.int32, device=dev),
           "status": torch.zeros(B, dtype=torch.int32, device=dev),
           "kept_count": torch.zeros(B, dtype=torch.int32, device=dev),
           "kept_ids": torch.zeros(B, kept, dtype=torch.int32, device=dev),
           "kept_probs": torch.zeros(B, kept, device=dev)}
    b = _abi.OxsBatch()
    b.batch, b.vocab = B, V
    b.logits_dtype = _abi.OXS_DTYPE_F32 if case["dtype"] == "f32" else _abi.OXS_DTYPE_BF16
    b.flags = _abi.OXS_FLAG_RECORD_HISTORY | _abi.OXS_FLAG_SHARED_CONFIG
    b.logits_ld, b.logits = V, s["logits"].data_ptr()
    b.configs = s["configs"].data_ptr()
    if case["biases"]:
        b.bias_ids, b.bias_values = s["bias_ids"].data_ptr(), s["bias_values"].data_ptr()
        b.ban_ids = s["ban_ids"].data_ptr()
    if s["mask"] is not None:
        b.allowed_mask, b.mask_ld = s["mask"].data_ptr(), s["mask"].shape[1]
    b.history, b.history_ld = s["history"].data_ptr(), H + HISTORY_ROOM
    b.history_len, b.history_cap = s["history_len"].data_ptr(), H + HISTORY_ROOM
    b.rng_state, b.mirostat_mu = s["rng"].data_ptr(), s["mu"].data_ptr()
    b.out_tokens, b.out_status = out["tokens"].data_ptr(), out["status"].data_ptr()
    b.out_kept_count, b.out_kept_ids = out["kept_count"].data_ptr(), out["kept_ids"].data_ptr()
    b.out_kept_probs, b.kept_ld = out["kept_probs"].data_ptr(), kept
    s["batch"], s["out"] = b, out
    s["sampler"] = BatchSampler(B, V, kept)
    return s


def _run_sample(s):
    s["sampler"].launch(s["batch"])
    return dict(s["out"], history=s["history"], history_len=s["history_len"], rng=s["rng"], mu=s["mu"])


# decode: slot i's request by i % 8
def _slot_config(i):
    k = i % 8
    if k == 0:
        return SamplingConfig(temperature=0.0)  # greedy: the raw argmax
    if k == 5:
        return SamplingConfig(dry_multiplier=0.8)
    if k == 6:
        return SamplingConfig(mirostat_mode=MirostatMode.V2)
    if k == 7:
        return SamplingConfig(temperature=1.0, top_k=0, min_p=0.02, frequency_penalty=0.2)
    return SamplingConfig()


def _decode_inputs(case, seed):
    g = _gen(seed)
    x = _logits(g, case["batch"], case["vocab"], "zipf")
    hist = _history(g, case["batch"], case["vocab"], case["history"])[:, : case["history"]].contiguous()
    n = case["history"]
    if n >= 16:  # the prompt ends in a repeated phrase, which DRY acts on
        hist[:, n - 8: n - 4] = hist[:, n - 4:]
        hist[:, n - 16: n - 12] = hist[:, n - 4:]
    return x, hist


def _prepare_decode(case, seed):
    B, V, H = case["batch"], case["vocab"], case["history"]
    x, hist = _decode_inputs(case, seed)
    loop = DecodeLoop(B, V, history_cap=H + HISTORY_ROOM)
    rows = hist.cpu().numpy().view(np.uint32)
    for i in range(B):
        c = _slot_config(i)
        st = SamplerState(2.0 * c.mirostat_tau, rows[i].tolist(), int(seed) * 1000003 + 977 * i + 1)
        loop.add_sequence(i, temperature=c.temperature, top_p=c.top_p, current_token=int(rows[i, -1]),
                          current_position=H, max_tokens=1 << 30, config=c, state=st)
    loop.capture(x)
    return {"loop": loop, "logits": x}


def _run_decode(s):
    loop = s["loop"]
    loop.replay()
    tokens = loop.wait()
    return {"tokens": tokens.view(np.int32), "status": loop.out["status"], "history": loop.history,
            "history_len": loop.history_len, "mu": loop.mirostat_mu, "rng": loop.rng_state,
            "current_token": loop.current_token, "position": loop.current_position, "count": loop.generated_count}


def _prepare_argmax(case, seed):
    B, V = case["batch"], case["vocab"]
    return {"lib": load_library(), "B": B, "V": V, "logits": _logits(_gen(seed), B, V, "normal"),
            "token": torch.zeros(B, dtype=torch.int32, device="cuda"), "value": torch.zeros(B, device="cuda")}


def _run_argmax(s):
    _abi.check(s["lib"].oxs_argmax(s["logits"].data_ptr(), s["V"], s["V"], s["B"], s["token"].data_ptr(),
                                   s["value"].data_ptr(), torch.cuda.current_stream().cuda_stream), "oxs_argmax")
    return {"token": s["token"], "value": s["value"]}


def _lm_head_inputs(case, seed):
    """GGUF Q8_0 rows ({f16 d, int8 qs[32]} per 32 weights) and hidden states."""
    g = _gen(seed)
    m, nb = case["m"], case["k"] // 32
    w = torch.empty(m, nb, 34, dtype=torch.uint8, device="cuda")
    for r in range(0, m, 16384):
        n = min(16384, m - r)
        q = torch.randn(n, nb, 32, generator=g, device="cuda").mul_(42.0).round_().clamp_(-127, 127)
        w[r:r + n, :, 2:] = q.to(torch.int8).view(torch.uint8)
        d = torch.rand(n, nb, 1, generator=g, device="cuda").mul_(4e-4).add_(2e-4).half()
        w[r:r + n, :, :2] = d.view(torch.uint8)
    x = torch.randn(case["batch"], case["k"], generator=g, device="cuda") * 1.5
    return w, x


def _prepare_lm_head(case, seed):
    w, x = _lm_head_inputs(case, seed)
    head = LmHeadQ8_0(w.view(-1), case["m"], case["k"])
    return {"head": head, "x": x,
            "xq": torch.zeros(case["batch"], case["k"] // 32 * 36, dtype=torch.uint8, device="cuda"),
            "y": torch.zeros(case["batch"], case["m"], device="cuda")}


def _run_lm_head(s):
    quantize_q8_1(s["x"], out=s["xq"])
    s["head"].project(s["xq"], out=s["y"])
    return {"xq": s["xq"], "logits": s["y"]}


def _prepare_dfa(case, seed):
    rng = np.random.default_rng(int(seed))
    V = case["vocab"]
    if case["prefix"]:
        grammar = DfaSchemaGrammar.new_json_with_fixed_prefix(
            "".join(chr(int(c)) for c in rng.integers(0x61, 0x7B, case["prefix"])))
    else:
        grammar = DfaSchemaGrammar.new_simple_json_validator()
    # token texts of 1 to 16 bytes, mostly letters, digits and JSON punctuation
    lens = np.clip(rng.geometric(0.2, V), 1, 16)
    alphabet = np.frombuffer(b"abcdefghijklmnopqrstuvwxyz ABCDEFGHIJ0123456789\"\"{}::,,_-.\xc3\xa9", np.uint8)
    flat = alphabet[rng.integers(0, len(alphabet), int(lens.sum()))].tobytes()
    ends = np.cumsum(lens).tolist()
    tokens = TokenBytes([flat[e - n: e] for e, n in zip(ends, lens.tolist())])
    states = torch.from_numpy(rng.integers(0, grammar.num_states, case["batch"]).astype(np.int32)).to("cuda")
    grammar.token_masks(tokens, states[:1])  # the grammar's table goes to the device on its first use
    return {"grammar": grammar, "tokens": tokens, "states": states}


def _run_dfa(s):
    return s["grammar"].token_masks(s["tokens"], s["states"])


_PREPARE = {"sample": _prepare_sample, "decode": _prepare_decode, "argmax": _prepare_argmax,
            "lm_head": _prepare_lm_head, "dfa": _prepare_dfa}
_RUN = {"sample": _run_sample, "decode": _run_decode, "argmax": _run_argmax, "lm_head": _run_lm_head,
        "dfa": _run_dfa}


def prepare(case, seed):
    s = _PREPARE[case["kind"]](case, seed)
    s["kind"] = case["kind"]
    return s


def run(state):
    return _RUN[state["kind"]](state)


# ------------------------------------------------------------------ what a pass cannot do without

def work(case):
    B = case["batch"]
    if case["kind"] == "lm_head":
        m, k = case["m"], case["k"]
        return {"bytes": m * k // 32 * 34 + B * k * 4 + 2 * B * k // 32 * 36 + B * m * 4, "flops": 2 * m * k * B}
    V = case["vocab"]
    if case["kind"] == "dfa":
        states = 8 if not case["prefix"] else case["prefix"] + 4
        return {"bytes": V * 4 + V * 5 + states * 1024 + B * 4 + B * ((V + 31) // 32) * 4, "flops": 0}
    if case["kind"] == "argmax":
        return {"bytes": B * V * 4 + B * 8, "flops": 0}
    if case["kind"] == "decode":
        return {"bytes": B * V * 4 + B * (case["history"] * 4 + 104 + 40), "flops": 0}
    kept = min(max(POOL, case["top_k"]), case["top_k"] or POOL)
    logits = B * V * (4 if case["dtype"] == "f32" else 2)
    mask = B * ((V + 31) // 32) * 4 if case["mask"] else 0
    return {"bytes": logits + mask + B * (case["history"] * 4 + kept * 8 + 40), "flops": 0}


def tolerance(case):
    # every float is the reference's to the last bit: its order of sums is part of the contract
    return "exact"


# ------------------------------------------------------------------ 64-bit results

def _penalised(x, cfg, hist, hlen, bias=True):
    """The stages before the pool, in float64, on x [B, V] (in place)."""
    B, V = x.shape
    for t in cfg.banned_tokens:
        x[:, t] = -math.inf
    for t, v in cfg.logit_biases.items():
        x[:, t] += v
    rep = abs(cfg.repeat_penalty - 1.0) > 1e-5 and cfg.repeat_penalty > 0
    fp = abs(cfg.frequency_penalty) > 1e-5 or abs(cfg.presence_penalty) > 1e-5
    if hlen and (rep or fp):
        n = min(hlen, cfg.repeat_last_n) if cfg.repeat_last_n > 0 else hlen
        win = hist[:, hlen - n: hlen].long()
        cnt = torch.zeros(B, V, dtype=torch.float64, device=x.device)
        cnt.scatter_add_(1, win, torch.ones_like(win, dtype=torch.float64))
        seen = cnt > 0
        if rep:
            x.copy_(torch.where(seen, torch.where(x > 0, x / cfg.repeat_penalty, x * cfg.repeat_penalty), x))
        if fp:
            x.copy_(torch.where(seen, x - (cnt * cfg.frequency_penalty + cfg.presence_penalty), x))
    if cfg.temperature > 0 and cfg.mirostat_mode == MirostatMode.Disabled:
        x *= 1.0 / cfg.temperature
    return x


def _cut(p, stop):
    """Length of the prefix that ends with the first running sum >= stop."""
    over = np.nonzero(np.cumsum(p) >= stop)[0]
    return int(over[0]) + 1 if over.size else len(p)


def _kept(p, cfg):
    """The candidates' probabilities after the chain, from the softmax of the sorted pool."""
    if cfg.min_p > 0:
        p = p[p >= p[0] * cfg.min_p]
    if cfg.top_k > 0:
        p = p[: cfg.top_k]
    if cfg.tfs_z < 1.0 and len(p) > 2:
        d2 = np.abs(np.diff(p, n=2))
        if d2.sum() > 0:
            over = np.nonzero(np.cumsum(d2 / d2.sum()) >= cfg.tfs_z)[0]
            p = p[: max(1, int(over[0]) + 1 if over.size else len(p))]
    if cfg.typical_p < 1.0 and len(p) > 1:
        s = -np.log(p)
        p = p[np.argsort(np.abs(s - (p * s).sum()), kind="stable")]
        p = p[: _cut(p, cfg.typical_p)]
    if cfg.top_p < 1.0:
        p = p[: _cut(p, cfg.top_p)]
    return p / p.sum()


def _mirostat_v2(p, cfg, mu):
    over = np.nonzero(-np.log2(np.maximum(p, 1e-8))[1:] > mu)[0]
    n = int(over[0]) + 1 if over.size else len(p)
    surprise = -math.log2(max(p[0] / max(p[:n].sum(), 1e-6), 1e-8))
    return mu - cfg.mirostat_eta * (surprise - cfg.mirostat_tau)


def _pool(x, m):
    """Softmax of each row's m largest finite values: a list of arrays, largest first."""
    top = torch.topk(x, min(m, x.shape[1]), dim=1).values.cpu().numpy()
    rows = []
    for v in top:
        v = v[np.isfinite(v)]
        e = np.exp(v - v[0])
        rows.append(e / e.sum())
    return rows


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        s = _sample_inputs(case, seed)
        cfg, H = s["config"], case["history"]
        B, V = case["batch"], case["vocab"]
        kept = np.zeros((B, max(POOL, case["top_k"])))
        mu = np.full(B, 10.0)
        for r in range(0, B, 64):  # 64 rows at a time keep the 64-bit copies small
            x = s["logits"][r:r + 64].double()
            if s["mask"] is not None:
                bits = (s["mask"][r:r + 64].unsqueeze(2) >> torch.arange(32, device="cuda", dtype=torch.int32)) & 1
                x.masked_fill_(bits.reshape(x.shape[0], -1)[:, :V] == 0, -math.inf)
            x = _penalised(x, cfg, s["history"][r:r + 64], H)
            for i, p in enumerate(_pool(x, max(POOL, case["top_k"]))):
                if cfg.mirostat_mode != MirostatMode.Disabled:
                    mu[r + i] = _mirostat_v2(p, cfg, 10.0)
                else:
                    p = _kept(p, cfg)
                kept[r + i, : len(p)] = p
        return {"tokens": None, "status": None, "kept_count": None, "kept_ids": None,
                "kept_probs": torch.from_numpy(kept), "history": None, "history_len": None, "rng": None,
                "mu": torch.from_numpy(mu)}
    if kind == "decode":
        x, hist = _decode_inputs(case, seed)
        mu = np.zeros(case["batch"])
        for i in range(case["batch"]):
            c = _slot_config(i)
            mu[i] = 2.0 * c.mirostat_tau
            if c.mirostat_mode != MirostatMode.Disabled:
                row = _penalised(x[i:i + 1].double(), c, hist[i:i + 1], case["history"])
                mu[i] = _mirostat_v2(_pool(row, POOL)[0], c, mu[i])
        return {"tokens": None, "status": None, "history": None, "history_len": None, "mu": torch.from_numpy(mu),
                "rng": None, "current_token": None, "position": None, "count": None}
    if kind == "argmax":
        x = _logits(_gen(seed), case["batch"], case["vocab"], "normal")
        return {"token": None, "value": x.double().max(dim=1).values}
    if kind == "lm_head":
        w, x = _lm_head_inputs(case, seed)
        m, nb, B = case["m"], case["k"] // 32, case["batch"]
        xb = x.double().view(B, nb, 32)
        d = xb.abs().amax(dim=2, keepdim=True) / 127.0
        q = torch.where(d > 0, torch.round(xb / d), torch.zeros_like(xb))
        xd = (q * d.half().double()).view(B, nb * 32)  # what q8_1 stores: whole quants, a half scale
        y = torch.empty(B, m, dtype=torch.float64, device="cuda")
        for r in range(0, m, 16384):
            blk = w[r:r + 16384]
            wd = blk[:, :, :2].contiguous().view(torch.float16).double() * blk[:, :, 2:].contiguous().view(
                torch.int8).double()
            y[:, r:r + 16384] = xd @ wd.view(wd.shape[0], -1).t()
        return {"xq": None, "logits": y}
    return None  # masks are whole numbers
