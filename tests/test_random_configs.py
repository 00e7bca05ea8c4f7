"""Randomised parity sweep: every SamplingConfig stage switched on at random, per row.

Each case draws a batch shape, a logits dtype (f32 or bf16), a logit
distribution (Gaussian, heavy spikes, long runs of equal values, -inf rows), a
grammar mask (none, per row or shared), a softcap, histories of random
length, and for every row a SamplingConfig whose fields are each enabled with
probability 1/2 at random values (sampler.rs:16-73), top_k up to 50000 (the
wide kernel past 1024), DRY ranges up to 4096
over histories up to 4400 ids. The HIP path must match
the oracle exactly: tokens, status, kept ids and probabilities, history, mu.
`test_random_configs_large_vocab` draws vocabularies above 131072 (more than 16
stream chunks per row, the 4096-key candidate union) with batches divisible by 8
(rows grouped by XCD).
"""
import numpy as np
import pytest

from harness import compare, run_gpu, run_oracle
from oxide_sampler import MirostatMode, configs_to_array
from oxide_sampler import workloads as wl

RTOL_F32 = 1e-5
RTOL_BF16 = 1e-3


def banner(msg):
    print(f"\n[case] {msg}", flush=True)


def random_config(rng, V):
    kw = {}
    coin = lambda: rng.random() < 0.5  # noqa: E731
    kw["temperature"] = float(rng.choice([0.0, 1e-7, 0.3, 0.7, 1.0, 1.6])) if coin() else 1.0
    if coin():
        kw["top_k"] = int(rng.choice([1, 2, 40, 50, 255, 256, 300, 1024, 2000, 50000]))
    if coin():
        kw["top_p"] = float(rng.choice([0.5, 0.9, 0.95, 0.999]))
    if coin():
        kw["min_p"] = float(rng.choice([0.01, 0.05, 0.2]))
    if coin():
        kw["tfs_z"] = float(rng.choice([0.5, 0.9, 0.99]))
    if coin():
        kw["typical_p"] = float(rng.choice([0.2, 0.8, 0.95]))
    if coin():
        kw["xtc_threshold"] = float(rng.choice([0.01, 0.1, 0.3]))
        kw["xtc_probability"] = float(rng.choice([0.3, 1.0]))
    if rng.random() < 0.2:
        kw["mirostat_mode"] = MirostatMode.V1 if coin() else MirostatMode.V2
        kw["mirostat_tau"] = float(rng.choice([2.0, 5.0]))
        kw["mirostat_eta"] = float(rng.choice([0.1, 0.3]))
    if rng.random() < 0.25:
        kw["dry_multiplier"] = float(rng.choice([0.5, 1.5]))
        kw["dry_base"] = float(rng.choice([1.1, 1.75, -1.2]))  # (< 0: alternating-sign penalties)
        kw["dry_allowed_length"] = int(rng.choice([0, 2, 3]))
        kw["dry_range"] = int(rng.choice([16, 128, 1024, 4096]))
    if coin():
        kw["repeat_penalty"] = float(rng.choice([0.9, 1.1, 1.3]))
        kw["repeat_last_n"] = int(rng.choice([0, 8, 64, 512]))
    if coin():
        kw["frequency_penalty"] = float(rng.choice([-0.3, 0.2, 0.6]))
    if coin():
        kw["presence_penalty"] = float(rng.choice([-0.2, 0.3]))
    if coin():
        kw["penalize_nl"] = True
        kw["newline_penalty"] = float(rng.choice([0.5, 2.0]))
    if coin():
        ids = rng.integers(0, V + 3, size=int(rng.integers(1, 6)))
        kw["logit_biases"] = {int(i): float(rng.choice([-5.0, -0.5, 0.75, 4.0])) for i in ids}
    if coin():
        kw["banned_tokens"] = {int(i) for i in rng.integers(0, V + 3, size=int(rng.integers(1, 6)))}
    return wl.disabled_config(**kw)


def random_workload(seed, large_vocab=False):
    rng = np.random.default_rng(seed)
    if large_vocab:
        B = int(rng.choice([8, 16, 24, 40]))
        V = int(rng.choice([151936, 262144]))
    else:
        B = int(rng.choice([1, 3, 8, 17, 33]))
        V = int(rng.choice([5, 100, 1000, 4097, 20000, 65537]))
    kind = rng.integers(0, 3)
    x = rng.standard_normal((B, V)).astype(np.float32) * np.float32(rng.choice([0.5, 2.0, 4.0]))
    if kind == 1:  # a heavy tail of spikes
        x[rng.random((B, V)) < 0.01] += np.float32(8.0)
    elif kind == 2 and V > 20:  # long runs of equal values: ties broken by the lower id
        x[:, V // 4: V // 2] = np.float32(1.5)
    if B > 2 and rng.random() < 0.5:
        x[1, :] = -np.inf
    bf16 = rng.random() < 0.3
    logits = wl.f32_to_bf16_bits(x) if bf16 else x
    cap = 4500
    history = rng.integers(0, V, size=(B, cap), dtype=np.uint32)
    history[:, ::9] = np.uint32(min(10, V - 1))
    hlen = rng.integers(0, 1090, size=B).astype(np.uint32)
    long_rows = rng.random(B) < 0.3  # DRY slices past the 1024 ids an LDS copy holds
    hlen[long_rows] = rng.integers(1100, 4400, size=int(long_rows.sum())).astype(np.uint32)
    for b in range(B):
        n = int(hlen[b])
        if n >= 30 and rng.random() < 0.5:  # repeated motifs: DRY n-gram matches
            history[b, n - 30:n] = np.tile(rng.integers(0, V, size=3, dtype=np.uint32), 10)
    mask = None
    mchoice = rng.integers(0, 3)
    if mchoice:
        words = (V + 31) // 32
        bits = rng.random((1 if mchoice == 2 else B, words * 32)) < rng.choice([0.03, 0.5])
        bits[:, int(rng.integers(0, V))] = True
        mask = np.packbits(bits.astype(np.uint8), axis=1, bitorder="little").view(np.uint32)[:, :words].copy()
    configs = [random_config(rng, V) for _ in range(B)]
    w = wl.Workload(name=f"random seed={seed} B={B} V={V}", logits=logits, dtype="bf16" if bf16 else "f32",
                    configs=configs, history=history, history_len=hlen, uniforms=wl.xorshift_uniforms(B, seed),
                    mask=mask, mu=np.full(B, 10.0, np.float32))
    if rng.random() < 0.3:
        w.extra["softcap"] = float(rng.choice([5.0, 30.0]))
    return w, mchoice == 2


@pytest.mark.gpu
@pytest.mark.parametrize("seed", range(24))
def test_random_configs(torch_gpu, seed):
    w, shared = random_workload(1000 + seed)
    banner(f"{w.name} {w.dtype} mask={'shared' if shared else w.mask is not None} "
           f"softcap={w.extra.get('softcap', 0)}")
    g = run_gpu(w, torch_gpu, kept_ld=1024, logits_out=True, max_top_k=50000, shared_mask=shared)
    r = run_oracle(w, kept_ld=1024, logits_out=True, shared_mask=shared)
    compare(g, r, RTOL_BF16 if w.dtype == "bf16" else RTOL_F32, w.name)


@pytest.mark.gpu
@pytest.mark.parametrize("seed", range(8))
def test_random_configs_large_vocab(torch_gpu, seed):
    w, shared = random_workload(2000 + seed, large_vocab=True)
    banner(f"{w.name} {w.dtype} mask={'shared' if shared else w.mask is not None} "
           f"softcap={w.extra.get('softcap', 0)}")
    g = run_gpu(w, torch_gpu, kept_ld=1024, logits_out=True, max_top_k=50000, shared_mask=shared)
    r = run_oracle(w, kept_ld=1024, logits_out=True, shared_mask=shared, n_threads=8)
    compare(g, r, RTOL_BF16 if w.dtype == "bf16" else RTOL_F32, w.name)


@pytest.mark.gpu
def test_logits_out_when_penalty_ids_overflow_the_chunk_hash(torch_gpu):
    # V = 1024 is one stream chunk; a whole-history window of all of its ids overflows its hash (1023
    # ids), so the row goes to the exact path, which must write every id of logits_out with its
    # penalties (sampler.rs:207-245)
    rng = np.random.default_rng(77)
    B, V = 4, 1024
    logits = (rng.standard_normal((B, V)) * 2.0).astype(np.float32)
    history = np.stack([rng.permutation(V)[:1024].astype(np.uint32) for _ in range(B)])
    configs = [wl.disabled_config(frequency_penalty=0.6, presence_penalty=0.2, repeat_last_n=0),
               wl.disabled_config(repeat_penalty=1.3, repeat_last_n=0, temperature=0.7),
               wl.disabled_config(presence_penalty=-0.2, top_k=40, top_p=0.9),
               wl.disabled_config(frequency_penalty=0.3, repeat_penalty=1.1, repeat_last_n=1024, min_p=0.05)]
    w = wl.Workload(name="hash overflow", logits=logits, dtype="f32", configs=configs, history=history,
                    history_len=np.full(B, 1024, np.uint32), uniforms=wl.xorshift_uniforms(B, 77))
    banner("logits_out with 1024 distinct penalty ids in one chunk")
    g = run_gpu(w, torch_gpu, logits_out=True, record=False)
    r = run_oracle(w, logits_out=True, record=False)
    compare(g, r, RTOL_F32, w.name)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [255, 256, 257, 320, 321, 960, 961, 1024])
def test_penalty_ids_at_the_sizes_of_the_chunk_hash(torch_gpu, n):
    # n distinct window ids in one stream chunk: its hash takes 256 slots (built again in 1024 where they
    # do not suffice), 512 or 1024 by the row's ids, full at 256, 512 and 1023
    rng = np.random.default_rng(n)
    B, V = 3, 1024
    logits = (rng.standard_normal((B, V)) * 2.0).astype(np.float32)
    history = np.stack([rng.permutation(V)[:n].astype(np.uint32) for _ in range(B)])
    configs = [wl.disabled_config(frequency_penalty=0.6, presence_penalty=0.2, repeat_last_n=0),
               wl.disabled_config(repeat_penalty=1.3, repeat_last_n=0, temperature=0.7),
               wl.disabled_config(presence_penalty=-0.2, top_k=300, top_p=0.9, repeat_last_n=0)]
    w = wl.Workload(name=f"{n} penalty ids in a chunk", logits=logits, dtype="f32", configs=configs,
                    history=history, history_len=np.full(B, n, np.uint32), uniforms=wl.xorshift_uniforms(B, n))
    banner(w.name)
    for out in (True, False):
        g = run_gpu(w, torch_gpu, logits_out=out, record=False, max_top_k=300)
        r = run_oracle(w, logits_out=out, record=False)
        compare(g, r, RTOL_F32, w.name)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [256, 257, 384, 385, 512, 513, 768, 769, 1000, 1023, 1024, 3000])
def test_skewed_windows_keep_the_candidate_path(torch_gpu, n):
    # n distinct window ids in the first of 16 stream chunks, with bans, biases and repeats among them:
    # up to 1023 the chunk's marks fit its hash (built again from 257 on where a smaller one was tried)
    # and the row keeps the candidate path; more overflow it and the row is re-scanned, which also
    # repairs logits_out
    rng = np.random.default_rng(n)
    B, V = 4, 128256
    logits = (rng.standard_normal((B, V)) * 2.0).astype(np.float32)
    ids = np.stack([rng.permutation(8192)[:n].astype(np.uint32) for _ in range(B)])
    history = np.concatenate([ids, ids[:, : n // 8]], axis=1) if n in (257, 769) else ids
    configs = []
    for i in range(B):
        c = wl.disabled_config(frequency_penalty=0.3, presence_penalty=0.2, repeat_penalty=1.2, repeat_last_n=0,
                               temperature=0.7, top_k=50, top_p=0.9)
        if i % 2 and n < 1023:  # of the window's own ids, so that the chunk's distinct ids stay n
            c.banned_tokens = {int(t) for t in ids[i, :3]}
            c.logit_biases = {int(t): 1.5 for t in ids[i, 2:5]}
        configs.append(c)
    w = wl.Workload(name=f"{n} ids in one chunk", logits=logits, dtype="f32", configs=configs, history=history,
                    history_len=np.full(B, history.shape[1], np.uint32), uniforms=wl.xorshift_uniforms(B, n))
    banner(w.name)
    from harness import gpu_sampler
    for out in (True, False):
        s = gpu_sampler(B, V, exact_limits=True)
        s.count_paths(True)
        try:
            g = run_gpu(w, torch_gpu, logits_out=out, record=False, exact_limits=True)
            counts = s.path_counts()
        finally:
            s.count_paths(False)
        compare(g, run_oracle(w, logits_out=out, record=False), RTOL_F32, w.name)
        assert counts["exact"] == (0 if n <= 1023 else B), counts


@pytest.mark.gpu
def test_ids_past_the_chunk_hash_cost_no_full_probes(torch_gpu):
    # more distinct window ids in a chunk than its hash takes: the answers are the oracle's, and the row's
    # cost grows with the window it reads, not with the slots its failing insertions look at. (A row of
    # 30000 ids takes 3.1 times as long as one of 1100; 13 times when each insertion probed a full table.)
    rng = np.random.default_rng(5)
    cfg = wl.disabled_config(repeat_penalty=1.1, repeat_last_n=0, temperature=0.8, top_k=40, top_p=0.95)
    w = wl.Workload(name="3000 ids in a chunk", logits=(rng.standard_normal((2, 5000)) * 2.0).astype(np.float32),
                    dtype="f32", configs=[cfg] * 2,
                    history=np.stack([rng.permutation(5000)[:3000].astype(np.uint32) for _ in range(2)]),
                    history_len=np.full(2, 3000, np.uint32), uniforms=wl.xorshift_uniforms(2, 5))
    banner("windows past the chunk hash")
    compare(run_gpu(w, torch_gpu, record=False), run_oracle(w, record=False), RTOL_F32, w.name)

    from harness import gpu_sampler
    torch, B, V = torch_gpu, 64, 128256
    g = torch.Generator(device="cuda").manual_seed(5)
    logits = torch.randn(B, V, generator=g, device="cuda") * 2.0
    raw, _, _, _ = configs_to_array([cfg] * B, 10)
    configs = torch.from_numpy(raw).cuda()
    u = torch.full((B,), 0.5, device="cuda")
    s = gpu_sampler(B, V, exact_limits=True)

    def milliseconds(n, span):
        hist = torch.stack([torch.randperm(span, generator=g, device="cuda")[:n] for _ in range(B)])
        hist = hist.to(torch.int32).contiguous()
        hlen = torch.full((B,), n, dtype=torch.int32, device="cuda")
        best = float("inf")
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            s.sample(logits, configs, history=hist, history_len=hlen, history_cap=n, record=False, uniforms=u)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    few, many = milliseconds(1100, 2048), milliseconds(30000, 32000)
    print(f"1100 ids {few:.3f} ms, 30000 ids {many:.3f} ms", flush=True)
    assert many < 6.0 * few, (few, many)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,vocab,dtype,kind", [
    (3, 16384, "f32", "topk"), (3, 50257, "f32", "topk"), (3, 128256, "bf16", "topk"), (64, 151936, "bf16", "topk"),
    (3, 50257, "f32", "ties"), (3, 128256, "bf16", "ties"), (3, 128256, "f32", "nan"), (2, 300001, "f32", "topk")])
def test_top_m_from_the_wavefront_records(torch_gpu, batch, vocab, dtype, kind):
    # rows whose candidate lists do not prove their top M, so that the wavefronts' thresholds bound it and
    # part of the row is read again: pools of 257 to 1024 keys; runs of equal values that overflow some
    # lists; NaN and infinities. Masks, biases, bans and window ids among the values read again.
    rng = np.random.default_rng(batch * 1000003 + vocab)
    x = (rng.standard_normal((batch, vocab)) * 3.0).astype(np.float32)
    if kind == "ties":
        x[:, 2048:2048 + 400] = 7.0
        x[:, vocab - 300:] = 7.0
    if kind == "nan":
        x[:, 100:6000] = np.nan
        x[0, 7000], x[1, 9000:9500] = np.inf, -np.inf
    if dtype == "bf16":
        x = (x.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)
    hist = (rng.random((batch, 700)) ** 3 * vocab).astype(np.uint32)
    hist[:, :40] = np.argsort(-np.nan_to_num(x, nan=-9.0), axis=1)[:, :40]  # penalised ids among the largest
    configs = []
    for i in range(batch):
        c = wl.disabled_config(repeat_penalty=1.2, frequency_penalty=-0.3, repeat_last_n=0, temperature=0.8,
                               top_k=[257, 1000, 1024][i % 3] if kind == "topk" else 256, top_p=0.99)
        c.logit_biases = {int(j): float(v) for j, v in zip(rng.integers(0, vocab, 40), rng.uniform(-4, 12, 40))}
        c.banned_tokens = {int(j) for j in hist[i, :5]}
        configs.append(c)
    mask = rng.integers(0, 2**32, size=(batch, (vocab + 31) // 32), dtype=np.uint32) if vocab != 50257 else None
    logits = (x.view(np.uint32) >> 16).astype(np.uint16) if dtype == "bf16" else x
    w = wl.Workload(name=f"{kind} {batch} x {vocab} {dtype}", logits=logits, dtype=dtype, configs=configs,
                    history=hist, history_len=np.full(batch, 700, np.uint32), mask=mask,
                    uniforms=wl.xorshift_uniforms(batch, vocab))
    banner(w.name)
    g = run_gpu(w, torch_gpu, kept_ld=1024, record=False, max_top_k=1024)
    r = run_oracle(w, kept_ld=1024, record=False, n_threads=8)
    compare(g, r, RTOL_BF16 if dtype == "bf16" else RTOL_F32, w.name)


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["records", "wide rows beside it", "ids", "write-back", "dry", "few wavefronts",
                                  "candidates"])
def test_which_rows_the_records_settle(torch_gpu, case):
    # pools of 1000 keys over 64 wavefronts of 128256 logits are settled by the wavefront records; a row
    # falls through to the radix select with more than 1536 penalised ids, a write-back, DRY that can raise
    # a value, wavefronts too few to bound 1000 keys (12 of 32 keys), or more than 2048 keys above the bound
    # (every wavefront holds a run of equal values, larger than its list)
    rng = np.random.default_rng(31)
    B, V = 4, 3000 if case == "few wavefronts" else 128256
    x = (rng.standard_normal((B, V)) * 3.0).astype(np.float32)
    if case == "candidates":
        x = np.minimum(x, 5.0)
        x.reshape(B, -1, 16)[:, :, 0] = 5.0  # 8016 equal largest values
    n = 1600 if case == "ids" else 500
    hist = (rng.random((B, n)) * V).astype(np.uint32)
    c = dict(repeat_penalty=1.2, repeat_last_n=0, temperature=1.0, top_k=1000, top_p=0.99)
    if case == "dry":
        hist[:, -8:-4] = hist[:, -4:]
        c.update(dry_multiplier=0.8, dry_base=-1.2, dry_allowed_length=2)
    configs = [wl.disabled_config(**c) for _ in range(B)]
    if case == "wide rows beside it":
        configs[1] = wl.disabled_config(**dict(c, top_k=1500))
    w = wl.Workload(name=f"records: {case}", logits=x, dtype="f32", configs=configs, history=hist,
                    history_len=np.full(B, n, np.uint32), uniforms=wl.xorshift_uniforms(B, 31))
    banner(w.name)
    from harness import gpu_sampler
    most = 1500 if case == "wide rows beside it" else 1000
    s = gpu_sampler(B, V, most, exact_limits=True)
    s.count_paths(True)
    try:
        out = case == "write-back"
        g = run_gpu(w, torch_gpu, kept_ld=most, record=False, max_top_k=most, exact_limits=True, logits_out=out)
        counts, settled = s.path_counts(), s.record_rows()
    finally:
        s.count_paths(False)
    print(counts, settled, flush=True)
    compare(g, run_oracle(w, kept_ld=most, record=False, logits_out=out, n_threads=4), RTOL_F32, w.name)
    assert counts["exact"] == B, counts
    assert settled == {"records": B, "wide rows beside it": B - 1}.get(case, 0), settled


@pytest.mark.gpu
@pytest.mark.parametrize("seed", range(5000, 5008))
def test_random_decode_steps(torch_gpu, seed):
    # oxs_decode_step over three steps with random configs (raw-argmax rows included) and
    # the device rng: tokens, kept sets, history, mu, rng state and the per-row advance
    import ctypes
    import test_decode_loop as td
    from oxide_sampler import BatchSampler, _abi, configs_to_array
    from oxide_sampler._abi import OxsDecodeIo
    t = torch_gpu
    rng = np.random.default_rng(seed)
    B, V, cap = int(rng.choice([3, 17, 40])), int(rng.choice([1000, 50001])), 1200
    cfgs = []
    for _ in range(B):
        c = random_config(rng, V)
        c.logit_biases, c.banned_tokens = {}, set()  # the decode loop's configs carry no lists
        if rng.random() < 0.25:
            c.temperature = float(rng.choice([0.0, 1e-6, -1.0]))
        cfgs.append(c)
    cfg_bytes = configs_to_array(cfgs, 10)[0]
    history = rng.integers(0, V, size=(B, cap), dtype=np.uint32)
    hlen = rng.integers(0, 1100, size=B).astype(np.uint32)
    mu = np.full(B, 10.0, np.float32)
    rng_state = np.array([(0x853C49E6748FEA9B + 977 * b * seed) & (2**64 - 1) or 1 for b in range(B)], np.uint64)
    dec = {"current_token": rng.integers(0, V, size=B).astype(np.uint32),
           "current_position": rng.integers(0, 5000, size=B).astype(np.int32),
           "generated_count": rng.integers(0, 50, size=B).astype(np.uint32)}
    d_cfg = td._to_dev(t, cfg_bytes)
    d_hist, d_hlen, d_mu, d_rng = (td._to_dev(t, a) for a in (history, hlen, mu, rng_state))
    d_dec = {k: td._to_dev(t, v) for k, v in dec.items()}
    lib = _abi.load_library()
    host = ctypes.c_void_p()
    _abi.check(lib.oxs_host_alloc(8 * B, ctypes.byref(host)), "oxs_host_alloc")
    s = BatchSampler(B, V, 50000)  # rows with top_k > 1024 take the wide kernel's decode form
    try:
        io = OxsDecodeIo(d_dec["current_token"].data_ptr(), d_dec["current_position"].data_ptr(),
                         d_dec["generated_count"].data_ptr(), host.value)
        out = {"tokens": t.zeros(B, dtype=t.int32, device="cuda"), "status": t.zeros(B, dtype=t.int32, device="cuda"),
               "kept_count": t.zeros(B, dtype=t.int32, device="cuda"),
               "kept_ids": t.zeros(B, 256, dtype=t.int32, device="cuda"),
               "kept_probs": t.zeros(B, 256, dtype=t.float32, device="cuda")}
        sent = int(np.uint32(td.SENT).view(np.int32))
        for step in range(3):
            banner(f"random decode seed={seed} B={B} V={V} step {step}")
            x = (rng.standard_normal((B, V)) * 2.0).astype(np.float32)
            x[rng.random((B, V)) < 0.003] += np.float32(6.0)
            for k in ("kept_count", "kept_ids"):
                out[k].fill_(sent)
            out["kept_probs"].view(t.int32).fill_(sent)
            s.sample(td._to_dev(t, x), d_cfg, history=d_hist, history_len=d_hlen, history_cap=cap, record=True,
                     rng_state=d_rng, mirostat_mu=d_mu, kept_ld=256, decode=io, out=out)
            t.cuda.synchronize()
            ref = td.oracle_decode(cfg_bytes, x, history, hlen, mu, rng_state, dec, cap)
            np.testing.assert_array_equal(td._u32(out["tokens"]), ref["tokens"])
            np.testing.assert_array_equal(out["status"].cpu().numpy(), ref["status"])
            np.testing.assert_array_equal(td._u32(out["kept_count"]), ref["kept_count"])
            kid, kpr = td._u32(out["kept_ids"]), out["kept_probs"].cpu().numpy().view(np.uint32)
            for b in range(B):
                n = 256 if ref["kept_count"][b] == td.SENT else min(int(ref["kept_count"][b]), 256)
                np.testing.assert_array_equal(kid[b, :n], ref["kept_ids"][b, :n])
                np.testing.assert_array_equal(kpr[b, :n], ref["kept_probs"][b, :n].view(np.uint32))
            np.testing.assert_array_equal(td._u32(d_hlen), hlen)
            np.testing.assert_array_equal(td._u32(d_hist), history)
            np.testing.assert_array_equal(d_mu.cpu().numpy().view(np.uint32), mu.view(np.uint32))
            np.testing.assert_array_equal(d_rng.cpu().numpy().view(np.uint64), rng_state)
            for k in dec:
                np.testing.assert_array_equal(d_dec[k].cpu().numpy().view(dec[k].dtype), dec[k])
    finally:
        t.cuda.synchronize()
        s.close()
        lib.oxs_host_free(host)
