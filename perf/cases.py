"""The calls whose speed matters: one decode step's sampling over the range of
batches, vocabularies and request settings that a server meets, and the
adjacent calls of a step (LM head, draft verification, MoE router, sparse
attention's block select, history and RNG upkeep).

A case is a dict of plain values.  `prepare` makes what a program holds
before the call (device inputs, the sampler's workspace, parameters), `run`
makes one call through the public entry points, `exact` gives the computed
numbers in 64 bits.  Sampled tokens are integers that the sampler defines
exactly, so they have no 64-bit form and no tolerance.
"""
import ctypes
import math

import numpy as np
import torch

from hi_amd import _lib
from hi_amd import sampler as S
from hi_amd.index_select import launch_dsv4_indexer_select

_streams = {}


def _stream():
    """The decode stream: the reference-compatible launchers take no null stream."""
    dev = torch.cuda.current_device()
    if dev not in _streams:
        _streams[dev] = torch.cuda.Stream()
    return _streams[dev]


def listed():
    return [
        # One interactive user: a single row, the usual top-k / top-p settings
        # with a repetition penalty over a short history, and the top
        # logprobs returned.  Latency of one launch.
        {"name": "one_request", "kind": "sample", "batch": 1, "vocab": 151936, "dtype": "f32", "logits": "normal",
         "rows": "topk", "top_k": 40, "history": 64, "mask": False, "logprobs": 40},
        # A small server that returns no logprobs: bf16 logits straight from
        # the model, half the requests greedy and half nucleus sampling.
        {"name": "greedy_and_nucleus", "kind": "sample", "batch": 64, "vocab": 151936, "dtype": "bf16",
         "logits": "zipf", "rows": "greedy_nucleus", "top_k": 0, "history": 0, "mask": False, "logprobs": 0},
        # A large server: every filter in use and 2048-token histories.
        {"name": "full_pipeline", "kind": "sample", "batch": 256, "vocab": 129280, "dtype": "f32", "logits": "spiked",
         "rows": "full", "top_k": 0, "history": 2048, "mask": False, "logprobs": 0},
        # Flat logits, a wide top-k and the top logprobs (distillation data,
        # evaluation runs): the long ranked draw.
        {"name": "wide_topk_logprobs", "kind": "sample", "batch": 128, "vocab": 256000, "dtype": "f32",
         "logits": "flat", "rows": "topk", "top_k": 1024, "history": 0, "mask": False, "logprobs": 20},
        # Constrained decoding: a grammar's allowed-token mask, nucleus rows.
        {"name": "grammar_mask", "kind": "sample", "batch": 32, "vocab": 151936, "dtype": "f32", "logits": "zipf",
         "rows": "nucleus", "top_k": 0, "history": 0, "mask": True, "logprobs": 0},
        # A large server whose requests each bring their own settings
        # (greedy, temperature only, nucleus, top-k), through the per-row
        # launcher that the reference's decode loop calls.
        {"name": "mixed_requests", "kind": "per_row", "batch": 256, "vocab": 129280, "logits": "zipf"},
        # A whole decode step of a small server around the sampler: uniforms,
        # sampling with penalties (requests with and without a top-k beside
        # their top-p), history append and pack, next inputs; a vocabulary
        # that is no multiple of anything.
        {"name": "decode_step", "kind": "step", "batch": 24, "vocab": 50257, "prompt": 384, "capacity": 512},
        # Single-stream decoding's output projection: one hidden row against
        # the whole head, logits written for the caller's own sampler.
        {"name": "lm_head_one_row", "kind": "lm_logits", "batch": 1, "hidden": 4096, "vocab": 151936, "softcap": 0.0},
        # The projection fused with sampling at the largest batch it takes,
        # greedy and top-k requests.
        {"name": "lm_head_sample", "kind": "lm_sample", "batch": 64, "hidden": 4096, "vocab": 151936,
         "softcap": 30.0},
        # Speculative decoding: a draft of 4 tokens verified for 8 requests.
        {"name": "draft_verify", "kind": "verify", "batch": 8, "draft": 4, "vocab": 151936},
        # The MoE router over a prefill chunk of tokens.
        {"name": "router_prefill", "kind": "router", "rows": 4096, "experts": 256, "top_k": 8, "sigmoid": True},
        # The sparse-attention indexer's block select at a long context.
        {"name": "block_select", "kind": "select", "blocks": 65536, "top_k": 2048},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _vocab(rng, lo, hi):
    """A vocabulary size: half of them padded to 64, as most models' are."""
    v = _log_int(rng, lo, hi)
    return min(hi, (v + 63) // 64 * 64) if rng.random() < 0.5 else v


def draw(rng):
    kind = rng.choice(["sample"] * 5 + ["per_row"] * 2 + ["step", "lm_logits", "lm_sample", "verify", "router", "select"])
    if kind in ("sample", "per_row"):
        vocab = _vocab(rng, 32000, 256000)
        batch = _log_int(rng, 1, min(256, 256 * 129280 // vocab))
        logits = rng.choice(["normal", "spiked", "zipf"])
        if kind == "per_row":
            return {"kind": kind, "batch": batch, "vocab": vocab, "logits": logits}
        rows = rng.choice(["topk", "topk", "greedy_nucleus", "nucleus", "full"])
        return {"kind": kind, "batch": batch, "vocab": vocab, "dtype": rng.choice(["f32", "bf16"]), "logits": logits,
                "rows": rows, "top_k": _log_int(rng, 5, 1024) if rows == "topk" else 0,
                "history": rng.choice([0, _log_int(rng, 16, 2048)]) if rows != "full" else _log_int(rng, 16, 2048),
                "mask": rng.random() < 0.2, "logprobs": _log_int(rng, 1, 40) if rng.random() < 0.3 else 0}
    if kind == "step":
        prompt = _log_int(rng, 32, 1024)
        return {"kind": kind, "batch": _log_int(rng, 1, 128), "vocab": _vocab(rng, 32000, 151936), "prompt": prompt,
                "capacity": prompt + 128}
    if kind in ("lm_logits", "lm_sample"):
        return {"kind": kind, "batch": _log_int(rng, 1, 64), "hidden": 32 * rng.randrange(32, 129),
                "vocab": _vocab(rng, 32000, 151936), "softcap": rng.choice([0.0, 30.0])}
    if kind == "verify":
        return {"kind": kind, "batch": _log_int(rng, 1, 33), "draft": rng.randrange(1, 8),
                "vocab": _vocab(rng, 32000, 151936)}
    if kind == "router":
        return {"kind": kind, "rows": _log_int(rng, 1, 8192), "experts": rng.choice([8, 64, 128, 160, 256, 300, 512]),
                "top_k": rng.choice([2, 4, 6, 8]), "sigmoid": rng.random() < 0.5}
    return {"kind": "select", "blocks": _log_int(rng, 513, 1 << 20), "top_k": rng.choice([512, 1024, 2048])}


# ---- inputs ----------------------------------------------------------------

def _logits(g, shape, B, V):
    """f32 logits on the device: N(0, 3) with 8 raised ids a row, N(0, 2.5)
    with 16, flat N(0, 0.5), or the log of a Zipf law over a permuted
    vocabulary with noise."""
    dev = "cuda"
    if shape == "zipf":
        logp = -1.1 * torch.log(torch.arange(1, V + 1, device=dev, dtype=torch.float64))
        logp = (logp - torch.logsumexp(logp, 0)).float()
        x = torch.empty(B, V, device=dev)
        for b in range(B):
            x[b, torch.randperm(V, generator=g, device=dev)] = logp
        return x.add_(torch.randn(B, V, generator=g, device=dev), alpha=0.5)
    sd, spikes, up = {"normal": (3.0, 8, 10.0), "spiked": (2.5, 16, 8.0), "flat": (0.5, 0, 0.0)}[shape]
    x = torch.randn(B, V, generator=g, device=dev).mul_(sd)
    if spikes:
        at = torch.randint(0, V, (B, spikes), generator=g, device=dev)
        x.scatter_(1, at, x.gather(1, at) + up)
    return x


def _zipf_ids(g, B, n, V):
    """n token ids a row under a Zipf law over one permutation of the vocabulary."""
    cdf = torch.cumsum(torch.arange(1, V + 1, device="cuda", dtype=torch.float64) ** -1.1, 0)
    r = torch.searchsorted(cdf / cdf[-1], torch.rand(B, n, generator=g, device="cuda", dtype=torch.float64))
    return torch.randperm(V, generator=g, device="cuda")[r.clamp_(max=V - 1)]


def _history(g, B, n, V):
    """Per-row (id, count) lists in CSR form: offsets, ids, counts."""
    key = _zipf_ids(g, B, n, V) + V * torch.arange(B, device="cuda")[:, None]
    key, count = torch.unique(key, return_counts=True)
    off = torch.zeros(B + 1, dtype=torch.int64, device="cuda")
    off[1:] = torch.cumsum(torch.bincount(key // V, minlength=B), 0)
    return off.int(), (key % V).int(), count.int()


def _mask(g, B, V):
    """Allowed-token words: 0.5%, 5% or 50% of the vocabulary a row."""
    W = (V + 31) // 32
    density = torch.tensor([0.005, 0.05, 0.5], device="cuda")[torch.randint(0, 3, (B,), generator=g, device="cuda")]
    words = torch.empty(B, W, dtype=torch.int32, device="cuda")
    bit = (1 << torch.arange(32, device="cuda")).view(1, 32)
    for b in range(B):
        on = torch.rand(W * 32, generator=g, device="cuda") < density[b]
        on[V:] = False
        words[b] = (on.view(W, 32) * bit).sum(1).int()  # keeps the low 32 bits
    return words


def _row_params(rows, top_k, B, history, seed):
    r = np.random.default_rng(seed)
    p = S.row_params(B, eos_id=2)
    if rows == "topk":
        p["temperature"], p["top_k"], p["top_p"] = (1.0, top_k, 0.99) if top_k > 256 else (0.7, top_k, 0.9)
        if history:
            p["repetition_penalty"] = 1.1
    elif rows == "greedy_nucleus":
        p["temperature"][B // 2:] = 1.0
        p["top_p"][B // 2:] = 0.95
    elif rows == "nucleus":
        p["temperature"], p["top_p"] = 0.8, 0.9
        if history:
            p["presence_penalty"] = 0.3
    else:  # full: every filter
        p["temperature"] = r.uniform(0.3, 1.2, B)
        p["top_k"] = r.choice([20, 50, 100], B)
        p["top_p"] = r.uniform(0.8, 0.99, B)
        p["min_p"], p["frequency_penalty"], p["presence_penalty"] = 0.05, 0.2, 0.3
    return p


def _ptr(t):
    return 0 if t is None else t.data_ptr()


def _sample_inputs(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    B, V = c["batch"], c["vocab"]
    x = _logits(g, c["logits"], B, V)
    s = {"logits": x.bfloat16() if c["dtype"] == "bf16" else x, "uniforms": torch.rand(B, generator=g, device="cuda"),
         "hist": _history(g, B, c["history"], V) if c["history"] else (None, None, None),
         "mask": _mask(g, B, V) if c["mask"] else None,
         "host_params": _row_params(c["rows"], c["top_k"], B, c["history"], seed)}
    s["params"] = S.params_to_device(s["host_params"])
    return s


def _prepare_sample(c, seed):
    s = _sample_inputs(c, seed)
    B, n = c["batch"], c["logprobs"]
    s["sampler"] = S.Sampler(B, c["vocab"], n)
    s["out"] = {"tokens": torch.zeros(B, dtype=torch.int32, device="cuda")}
    if n:
        s["out"].update(logprobs=torch.zeros(B, n, device="cuda"),
                        logprob_ids=torch.zeros(B, n, dtype=torch.int32, device="cuda"),
                        token_logprobs=torch.zeros(B, device="cuda"))
    s["n"] = n
    return s


def _prepare_per_row(c, seed):
    """Greedy, temperature only, nucleus and top-k requests by turns."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    B, V = c["batch"], c["vocab"]
    r = np.random.default_rng(seed)
    cls = r.permutation(B) % 4
    T = np.where(cls == 0, 0.0, r.uniform(0.6, 1.0, B)).astype(np.float32)
    top_p = np.where(cls == 2, 0.9, np.where(cls == 3, 0.95, 1.0)).astype(np.float32)
    top_k = np.where(cls == 3, r.choice([20, 40, 50, 100], B), 0).astype(np.int32)
    x = _logits(g, c["logits"], B, V)
    s = {"logits": x, "uniforms": torch.rand(B, generator=g, device="cuda"), "B": B, "V": V,
         "T": torch.from_numpy(T).cuda(), "top_p": torch.from_numpy(top_p).cuda(),
         "top_k": torch.from_numpy(top_k).cuda(), "tokens": torch.zeros(B, dtype=torch.int32, device="cuda")}
    # the launcher's workspace, reserved once on the decode stream
    _lib.check(_lib.load().hi_rocm_sampler_reserve(B, V, 0, _stream().cuda_stream))
    return s


def _prepare_step(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    lib = _lib.load()
    B, V, cap = c["batch"], c["vocab"], c["capacity"]
    i32 = lambda *n: torch.zeros(*n, dtype=torch.int32, device="cuda")  # noqa: E731
    p = S.row_params(B, temperature=0.7, top_p=0.9, top_k=40 * (np.arange(B) % 2 == 0), repetition_penalty=1.1,
                     presence_penalty=0.2, flags=_lib.FLAG_REP_ONCE)
    keys = np.zeros((B, 8), np.uint32)
    for b in range(B):
        _lib.check(lib.hi_rocm_rng_key_from_seed(seed * 1000 + b, keys[b].ctypes.data))
    s = {"B": B, "cap": cap, "logits": _logits(g, "spiked", B, V), "params": S.params_to_device(p),
         "keys": torch.from_numpy(keys.view(np.int32)).cuda(),
         "used": torch.zeros(B, dtype=torch.int64, device="cuda"), "uniforms": torch.zeros(B, device="cuda"),
         "slot_ids": i32(B, cap), "slot_counts": i32(B, cap), "lens": i32(B), "overflow": i32(1), "offs": i32(B + 1),
         "ids": i32(B * cap), "counts": i32(B * cap), "next": i32(B), "pos": i32(B) + c["prompt"],
         "sampler": S.Sampler(B, V), "out": {"tokens": i32(B)}}
    # the prompts' histories: distinct ids with their counts
    off, ids, cnt = (t.cpu() for t in _history(g, B, c["prompt"], V))
    for b in range(B):
        n = int(off[b + 1] - off[b])
        s["slot_ids"][b, :n] = ids[off[b]:off[b + 1]].cuda()
        s["slot_counts"][b, :n] = cnt[off[b]:off[b + 1]].cuda()
        s["lens"][b] = n
    s["offs"], s["ids"][:len(ids)], s["counts"][:len(cnt)] = off.cuda(), ids.cuda(), cnt.cuda()
    return s


def _lm_inputs(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    H = c["hidden"]
    h = torch.randn(c["batch"], H, generator=g, device="cuda").bfloat16()
    w = torch.empty(c["vocab"], H, dtype=torch.bfloat16, device="cuda")
    for a in range(0, c["vocab"], 16384):  # a block at a time: the f32 form is twice the size
        w[a:a + 16384] = torch.randn(min(16384, c["vocab"] - a), H, generator=g, device="cuda").mul_(2.5 / H ** 0.5)
    return h, w


def _prepare_lm(c, seed):
    h, w = _lm_inputs(c, seed)
    B, V = c["batch"], c["vocab"]
    s = {"h": h, "w": w, "B": B, "V": V, "H": c["hidden"], "cap": c["softcap"]}
    if c["kind"] == "lm_logits":
        s["logits"] = torch.zeros(B, V, device="cuda")
        return s
    r = np.random.default_rng(seed)
    p = S.row_params(B, temperature=0.8, top_p=0.95, top_k=40)
    p["temperature"][r.permutation(B)[:B // 4]] = 0.0  # a quarter greedy
    n = ctypes.c_size_t()
    _lib.check(_lib.load().hi_rocm_lm_head_workspace_bytes(B, V, ctypes.byref(n)))
    s.update(params=S.params_to_device(p), uniforms=torch.from_numpy(r.random(B).astype(np.float32)).cuda(),
             ws=torch.zeros(n.value, dtype=torch.uint8, device="cuda"),
             tokens=torch.zeros(B, dtype=torch.int32, device="cuda"))
    return s


def _prepare_verify(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    B, K, V = c["batch"], c["draft"], c["vocab"]
    x = torch.randn(B, K + 1, V, generator=g, device="cuda").mul_(2.0)
    draft = x[:, :K].argmax(2).int()  # the target's own choice, wrong from a random place on
    wrong = torch.arange(K, device="cuda")[None] >= torch.randint(0, K + 1, (B, 1), generator=g, device="cuda")
    draft = torch.where(wrong, (draft + 1) % V, draft).int().contiguous()
    out = [torch.full((B, K + 1), -1, dtype=torch.int32, device="cuda") for _ in range(2)]
    return {"x": x, "draft": draft, "greedy": out[0], "tokens": out[1],
            "count": torch.zeros(B, dtype=torch.int32, device="cuda"), "B": B, "K": K, "V": V}


def _router_inputs(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(c["rows"], c["experts"], generator=g, device="cuda").mul_(2.5)
    return x, torch.randn(c["experts"], generator=g, device="cuda").mul_(0.1) if c["sigmoid"] else None


def _prepare_router(c, seed):
    x, bias = _router_inputs(c, seed)
    n, k = c["rows"], c["top_k"]
    return {"x": x, "bias": bias, "ids": torch.zeros(n, k, dtype=torch.int32, device="cuda"),
            "w": torch.zeros(n, k, device="cuda"), "n": n, "E": c["experts"], "k": k, "sigmoid": int(c["sigmoid"])}


def _prepare_select(c, seed):
    n = c["blocks"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    return {"x": torch.randn(n, generator=g, device="cuda"), "k": c["top_k"], "n": n,
            "marks": torch.zeros(n, dtype=torch.uint8, device="cuda"),
            "sel": torch.zeros(min(n, c["top_k"]), dtype=torch.int32, device="cuda")}


_PREPARE = {"sample": _prepare_sample, "per_row": _prepare_per_row, "step": _prepare_step, "lm_logits": _prepare_lm,
            "lm_sample": _prepare_lm, "verify": _prepare_verify, "router": _prepare_router,
            "select": _prepare_select}


def prepare(case, seed):
    with torch.cuda.stream(_stream()):  # everything of a state belongs to the decode stream
        s = _PREPARE[case["kind"]](case, seed)
    s["kind"] = case["kind"]
    return s


# ---- one call --------------------------------------------------------------

def _run_sample(s, lib, st):
    n = s["n"]
    return s["sampler"].sample(s["logits"], s["params"], s["uniforms"], *s["hist"], s["mask"], n_logprobs=n,
                               token_logprobs=n > 0, out=s["out"], stream=_stream())


def _run_per_row(s, lib, st):
    _lib.check(lib.hi_rocm_launch_select_batched_last_token_per_row(
        s["logits"].data_ptr(), s["tokens"].data_ptr(), s["uniforms"].data_ptr(), s["T"].data_ptr(),
        s["top_p"].data_ptr(), s["top_k"].data_ptr(), s["B"], 1, s["V"], 1, st))
    return {"tokens": s["tokens"]}


def _run_step(s, lib, st):
    B, cap, tok = s["B"], s["cap"], s["out"]["tokens"]
    _lib.check(lib.hi_rocm_rng_uniforms(s["keys"].data_ptr(), s["used"].data_ptr(), 0, s["uniforms"].data_ptr(), B, st))
    s["sampler"].sample(s["logits"], s["params"], s["uniforms"], s["offs"], s["ids"], s["counts"], out=s["out"],
                        stream=_stream())
    slots = (s["slot_ids"].data_ptr(), s["slot_counts"].data_ptr(), s["lens"].data_ptr(), B, cap)
    _lib.check(lib.hi_rocm_history_append(*slots, 0, tok.data_ptr(), B, s["overflow"].data_ptr(), st))
    _lib.check(lib.hi_rocm_history_pack(*slots, s["offs"].data_ptr(), s["ids"].data_ptr(), s["counts"].data_ptr(), st))
    _lib.check(lib.hi_rocm_decode_step_advance(tok.data_ptr(), s["next"].data_ptr(), s["pos"].data_ptr(), B, B, st))
    return {k: s[k] for k in ("uniforms", "used", "slot_ids", "slot_counts", "lens", "overflow", "offs", "ids",
                              "counts", "next", "pos")}


def _run_lm_logits(s, lib, st):
    _lib.check(lib.hi_rocm_lm_head_logits(s["h"].data_ptr(), s["w"].data_ptr(), 0, s["cap"], s["B"], s["H"], s["V"],
                                          s["logits"].data_ptr(), st))
    return {"logits": s["logits"]}


def _run_lm_sample(s, lib, st):
    _lib.check(lib.hi_rocm_sample_lm_head(s["h"].data_ptr(), s["w"].data_ptr(), 0, s["cap"], s["B"], s["H"], s["V"],
                                          s["params"].data_ptr(), s["uniforms"].data_ptr(), s["tokens"].data_ptr(),
                                          s["ws"].data_ptr(), s["ws"].numel(), st))
    return {"tokens": s["tokens"]}


def _run_verify(s, lib, st):
    _lib.check(lib.hi_rocm_spec_verify_greedy(s["x"].data_ptr(), s["B"], s["K"], s["V"], s["draft"].data_ptr(), 0,
                                              s["greedy"].data_ptr(), s["tokens"].data_ptr(), s["count"].data_ptr(),
                                              st))
    return {"greedy": s["greedy"], "tokens": s["tokens"], "count": s["count"]}


def _run_router(s, lib, st):
    _lib.check(lib.hi_rocm_launch_moe_topk_router(s["x"].data_ptr(), s["ids"].data_ptr(), s["w"].data_ptr(),
                                                  _ptr(s["bias"]), s["n"], s["E"], s["k"], 1, s["sigmoid"], 2.5, st))
    return {"ids": s["ids"], "weights": s["w"]}


def _run_select(s, lib, st):
    launch_dsv4_indexer_select(s["x"], s["n"], s["k"], s["marks"], s["sel"], stream=_stream())
    return {"sel": s["sel"], "marks": s["marks"]}


_RUN = {"sample": _run_sample, "per_row": _run_per_row, "step": _run_step, "lm_logits": _run_lm_logits,
        "lm_sample": _run_lm_sample, "verify": _run_verify, "router": _run_router, "select": _run_select}


def run(state):
    return _RUN[state["kind"]](state, _lib.load(), _stream().cuda_stream)


# ---- what a pass cannot do without, and how far results may be off ---------

def work(case):
    """Inputs read once and outputs written once; a history or mask entry
    counts as stored (8 bytes a distinct id at most, one bit a token)."""
    c, k = case, case["kind"]
    if k in ("sample", "per_row", "step"):
        B, V = c["batch"], c["vocab"]
        n = B * V * (2 if c.get("dtype") == "bf16" else 4) + B * 48
        if k == "sample":
            n += B * c["history"] * 8 + (B * ((V + 31) // 32) * 4 if c["mask"] else 0) + B * c["logprobs"] * 8
        elif k == "step":  # the packed history read, and read and written again by the upkeep
            n += 3 * B * c["prompt"] * 8
        return {"bytes": n, "flops": 0}
    if k in ("lm_logits", "lm_sample"):
        B, H, V = c["batch"], c["hidden"], c["vocab"]
        return {"bytes": 2 * V * H + 2 * B * H + (4 * B * V if k == "lm_logits" else 44 * B), "flops": 2 * B * H * V}
    if k == "verify":
        rows = c["batch"] * (c["draft"] + 1)
        return {"bytes": 4 * rows * c["vocab"] + 12 * rows, "flops": 0}
    if k == "router":
        return {"bytes": 4 * c["rows"] * c["experts"] + 4 * c["experts"] + 8 * c["rows"] * c["top_k"], "flops": 0}
    return {"bytes": 5 * c["blocks"] + 4 * min(c["blocks"], c["top_k"]), "flops": 0}


def tolerance(case):
    if case["kind"] == "sample" and case["logprobs"]:
        return {"rel": 1e-6, "max": 1e-5}  # f32 masses of the chunks beside double sums
    if case["kind"] == "lm_logits":
        return {"rel": 2e-6, "max": 2e-5}  # f32 sums over the hidden size in another order
    if case["kind"] == "router":
        return {"rel": 5e-7, "max": 5e-6}
    return "exact"


def _exact_sample(c, seed):
    if not c["logprobs"]:
        return None
    s = _sample_inputs(c, seed)
    B, V, p = c["batch"], c["vocab"], s["host_params"]
    col = lambda name: torch.from_numpy(p[name].astype(np.float64)).cuda()  # noqa: E731
    x = s["logits"].double()
    if s["hist"][0] is not None:
        off, ids, cnt = (t.long() for t in s["hist"])
        row = torch.repeat_interleave(torch.arange(B, device="cuda"), off[1:] - off[:-1])
        l, n, rep = x[row, ids], cnt.double(), col("repetition_penalty")[row]
        l = torch.where(l < 0, l * rep ** n, l / rep ** n)
        x[row, ids] = l - col("frequency_penalty")[row] * n - col("presence_penalty")[row]
    if s["mask"] is not None:
        bits = (s["mask"][:, :, None] >> torch.arange(32, device="cuda", dtype=torch.int32)) & 1
        x.masked_fill_(bits.view(B, -1)[:, :V] == 0, -math.inf)
    T = col("temperature")
    lp = torch.log_softmax(x / torch.where(T > 0, T, torch.ones_like(T))[:, None], 1)
    return {"tokens": None, "logprobs": lp.topk(c["logprobs"], 1).values, "logprob_ids": None, "token_logprobs": None}


def _exact_lm(c, seed):
    h, w = _lm_inputs(c, seed)
    h = h.double()
    x = torch.cat([h @ w[a:a + 16384].double().t().contiguous() for a in range(0, c["vocab"], 16384)], 1)
    return {"logits": c["softcap"] * torch.tanh(x / c["softcap"]) if c["softcap"] > 0 else x}


def _exact_router(c, seed):
    x, bias = _router_inputs(c, seed)
    p = torch.sigmoid(x.double()) if c["sigmoid"] else torch.softmax(x.double(), 1)
    at = (p + bias.double() if bias is not None else p).topk(c["top_k"], 1).indices
    w = p.gather(1, at)
    return {"ids": None, "weights": 2.5 * w / w.sum(1, keepdim=True)}


_EXACT = {"sample": _exact_sample, "lm_logits": _exact_lm, "router": _exact_router}


def exact(case, seed):
    with torch.cuda.stream(_stream()):
        r = _EXACT[case["kind"]](case, seed) if case["kind"] in _EXACT else None
        torch.cuda.synchronize()
    return r
