"""GPU parity of the draws over a row's whole distribution (top-p without
top-k, min-p alone, temperature only, top-k above 1024) against the oracle:
tokens equal, at the edges of the tiles (1024 logits), of the pieces sorted at
a time (4096 weights) and of a row's 256 tiles (262,144 logits: beyond, one
workgroup's tiles are longer and the wide pass chains them 256 at a time),
over one launch or two, 16-byte aligned rows and others, and over weights that
all differ, come in long runs, or are all equal."""
import numpy as np
import pytest

from hi_amd._lib import ROW_PARAMS_DTYPE
from hi_amd.workloads import f32_to_bf16_bits

pytestmark = pytest.mark.gpu

F32 = np.float32


def _rows(kind, B, V, seed):
    rng = np.random.default_rng(seed)
    if kind == "spiked":
        x = rng.normal(0, 2.5, (B, V))
        x[:, rng.choice(V, max(1, min(16, V // 4)), replace=False)] += 8.0
    elif kind == "flat":
        x = rng.normal(0, 0.5, (B, V))
    elif kind == "runs":
        x = rng.integers(-3, 4, (B, V)).astype(float)
    else:  # equal
        x = np.full((B, V), 0.75)
    return x.astype(F32)


def _params(B):
    p = np.zeros(B, ROW_PARAMS_DTYPE)
    p["repetition_penalty"] = 1.0
    p["top_p"] = 1.0
    p["temperature"] = 0.9
    p["top_p"][0::5] = 0.9       # nucleus
    p["top_p"][1::5] = 0.999
    p["min_p"][2::5] = 0.02      # min-p alone; rows 3::5 are temperature only
    p["top_k"][4::5] = 1500
    p["top_p"][4::5] = 0.95
    return p


@pytest.mark.parametrize("V", [1, 4, 255, 257, 1023, 1024, 1025, 4097, 16388, 50257, 262149])
@pytest.mark.parametrize("kind", ["spiked", "flat", "runs", "equal"])
def test_draw_parity(hip, oracle, V, kind):
    import torch
    from hi_amd import sampler as S
    B = 5 if V > 100000 else 15
    x = _rows(kind, B, V, V)
    p = _params(B)
    u = np.random.default_rng(V + 1).random(B).astype(F32)
    u[-1] = 0.99999994
    for bf16 in (False, True):
        logits = f32_to_bf16_bits(x) if bf16 else x
        t = torch.from_numpy(logits.view(np.int16) if bf16 else logits).cuda()
        smp = S.Sampler(B, V)
        print(f"draw V={V} {kind} bf16={bf16}", flush=True)
        out = smp.sample(t.view(torch.bfloat16) if bf16 else t, S.params_to_device(p), torch.from_numpy(u).cuda())
        torch.cuda.synchronize()
        want = oracle.sample_rows(logits, p, u)["tokens"]
        got = out["tokens"].cpu().numpy().view(np.uint32)
        bad = np.flatnonzero(got != want)
        assert bad.size == 0, (bad, got[bad], want[bad])


@pytest.mark.parametrize("with_mask,V", [(False, 65537), (True, 65540), (True, 65537)])
def test_row_kernel_other_classes(hip, oracle, with_mask, V):
    """256 rows in one workgroup each (masked rows of an odd vocabulary: the
    general scan): every class but
    the streamed top-k, with histories (repeated ids, ids past the
    vocabulary, one longer than the kernel's table), penalties, masks (one
    row fully masked), rows without a finite logit, infinities and NaN."""
    import torch
    from hi_amd import sampler as S
    B = 256
    rng = np.random.default_rng(9 + with_mask)
    x = _rows("spiked", B, V, 5)
    p = _params(B)
    p["temperature"][0::7] = 0.0
    p["eos_id"] = 3
    p["repetition_penalty"][1::3] = 1.2
    p["frequency_penalty"][1::2] = 0.1
    x[3, :] = -np.inf
    x[8, 17] = np.inf
    x[13, 5] = np.nan
    x[14, :] = np.round(x[14, :])
    off, ids, cnt = [0], [], []
    for b in range(B):
        n = 3500 if b == 20 else (0 if b % 4 == 0 else int(rng.integers(1, 300)))
        i = rng.integers(0, V + 50, n)
        if n:
            i[:8] = np.argsort(np.nan_to_num(x[b], nan=-1e30, posinf=-1e30))[-8:][:n]  # likely tokens penalised
        ids.append(np.concatenate([i, i[:5]]).astype(np.uint32))
        cnt.append(rng.integers(1, 4, len(ids[-1])).astype(np.uint32))
        off.append(off[-1] + len(ids[-1]))
    off, ids, cnt = np.array(off, np.uint32), np.concatenate(ids), np.concatenate(cnt)
    mask = None
    if with_mask:
        mask = rng.integers(0, 2 ** 32, (B, (V + 31) // 32), dtype=np.uint64).astype(np.uint32)
        mask[30] = 0
    u = rng.random(B).astype(F32)
    i32 = lambda a: torch.from_numpy(a.view(np.int32)).cuda()  # noqa: E731
    print(f"row kernel classes mask={with_mask}", flush=True)
    out = S.Sampler(B, V).sample(torch.from_numpy(x).cuda(), S.params_to_device(p), torch.from_numpy(u).cuda(),
                                 i32(off), i32(ids), i32(cnt), None if mask is None else i32(mask))
    torch.cuda.synchronize()
    want = oracle.sample_rows(x, p, u, off, ids, cnt, mask)["tokens"]
    got = out["tokens"].cpu().numpy().view(np.uint32)
    bad = np.flatnonzero(got != want)
    assert bad.size == 0, (bad, got[bad], want[bad])


@pytest.mark.parametrize("B,V", [(256, 4096), (257, 100), (129, 4097), (37, 33001), (512, 257), (12, 151936), (2, 1048575)])
def test_one_launch_grids(hip, oracle, B, V):
    """Grids of 256 to 512 workgroups (4096 logits each), whose workgroups
    are dealt to the rows by CU: every row class, tokens equal the oracle's."""
    import torch
    from hi_amd import sampler as S
    x = _rows("spiked", B, V, B + V)
    p = _params(B)
    p["temperature"][0::7] = 0.0
    p["top_k"][1::6] = 40
    u = np.random.default_rng(B).random(B).astype(F32)
    smp = S.Sampler(B, V)
    print(f"one launch B={B} V={V}", flush=True)
    for _ in range(2):
        out = smp.sample(torch.from_numpy(x).cuda(), S.params_to_device(p), torch.from_numpy(u).cuda())
        torch.cuda.synchronize()
        got = out["tokens"].cpu().numpy().view(np.uint32)
        want = oracle.sample_rows(x, p, u)["tokens"]
        bad = np.flatnonzero(got != want)
        assert bad.size == 0, (bad, got[bad], want[bad])


GRID = [(9, 262143), (9, 262144), (9, 262145), (12, 262208), (2, 1048577), (40, 70001), (64, 50257), (128, 50257)]


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("B,V", GRID)
def test_finish_grid(hip, oracle, B, V, bf16):
    """Two launches (more than 512 workgroups of 4096 logits): nucleus and
    min-p rows through the wide pass, which the path codes show, and
    temperature-only rows split over workgroups (up to 64 rows) or not, on
    both sides of 256 tiles and 256 chunks, rows of any alignment, with and
    without logprobs."""
    import torch
    from hi_amd import sampler as S
    n = B * ((V + 4095) // 4096)
    assert n > 512 and B * ((V + 16383) // 16384) < 1024
    x = _rows("spiked", B, V, V + B)
    p = _params(B)
    p["top_k"][4::5] = 40
    u = np.random.default_rng(V).random(B).astype(F32)
    logits = f32_to_bf16_bits(x) if bf16 else x
    t = torch.from_numpy(logits.view(np.int16) if bf16 else logits).cuda()
    t = t.view(torch.bfloat16) if bf16 else t
    # (rows of top-p 0.999 list more than a quarter of the row, or more bf16
    # values than the merge's table holds: finish_row then)
    whole = np.flatnonzero((p["top_k"] == 0) & ((p["top_p"] < 0.99) | (p["min_p"] > 0)))
    for n_lp in (0, 3):
        smp = S.Sampler(B, V, n_lp)
        print(f"finish grid B={B} V={V} bf16={bf16} logprobs={n_lp}", flush=True)
        out = smp.sample(t, S.params_to_device(p), torch.from_numpy(u).cuda(), n_logprobs=n_lp)
        torch.cuda.synchronize()
        want = oracle.sample_rows(logits, p, u, n_logprobs=n_lp)
        got = out["tokens"].cpu().numpy().view(np.uint32)
        bad = np.flatnonzero(got != want["tokens"])
        assert bad.size == 0, (bad, got[bad], want["tokens"][bad])
        names = [S.WIDE_PATHS[int(c)] for c in S.debug_wide_paths(smp, B, V)[whole]]
        assert names == ["wide"] * len(whole), names
        if n_lp:
            np.testing.assert_allclose(out["logprobs"].cpu().numpy(), want["logprobs"], rtol=1e-5, atol=0)
            assert np.array_equal(out["logprob_ids"].cpu().numpy().view(np.uint32), want["logprob_ids"])


@pytest.mark.parametrize("kind", ["levels", "equal", "bf16 values", "both", "own levels", "short", "flat"])
@pytest.mark.parametrize("B,V", [(16, 151936), (56, 70003)])
def test_f32_rows_of_few_values(hip, oracle, B, V, kind):
    """f32 rows whose long lists share values: counted by value; rows with a unit of other values, which stays
    listed beside counted ones; units with levels of their own, too many together for the merge's table
    (their ranks come from the lists after all); rows that share none."""
    import torch
    from hi_amd import sampler as S
    assert B * ((V + 4095) // 4096) > 512
    rng = np.random.default_rng(V)
    x = rng.normal(0, 2.5 if kind in ("bf16 values", "own levels", "short") else 1.5, (B, V))
    if kind == "levels":
        x = np.round(x)
    elif kind == "equal":
        x = np.full((B, V), 0.25)
    elif kind == "both":
        x[:, :-1000] = np.round(x[:, :-1000] * 4) / 4
    elif kind == "own levels":
        x = np.round(x * 16) / 16 + np.arange(V) // 4096 * 2.0 ** -12
    x = x.astype(F32)
    if kind == "bf16 values":
        x = (f32_to_bf16_bits(x).astype(np.uint32) << 16).view(F32)
    p = _params(B)
    p["top_k"][4::5] = 0
    u = rng.random(B).astype(F32)
    smp = S.Sampler(B, V)
    print(f"few values B={B} V={V} {kind}", flush=True)
    out = smp.sample(torch.from_numpy(x).cuda(), S.params_to_device(p), torch.from_numpy(u).cuda())
    torch.cuda.synchronize()
    want = oracle.sample_rows(x, p, u)["tokens"]
    got = out["tokens"].cpu().numpy().view(np.uint32)
    bad = np.flatnonzero(got != want)
    assert bad.size == 0, (bad, got[bad], want[bad])
    nucleus = np.flatnonzero(p["top_p"] < 0.99)
    names = [S.WIDE_PATHS[int(c)] for c in S.debug_wide_paths(smp, B, V)[nucleus]]
    want = {"flat": {"long-list"}, "own levels": {"wide", "merge-full"}}.get(kind, {"wide"})
    assert set(names) <= want and ("wide" in names or kind == "flat"), sorted(set(names))


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("B,V,n_hist", [(3, 50257, 3500), (45, 50257, 3500), (5, 50304, 700), (4, 16387, 16000)])
def test_dense_histories(hip, oracle, B, V, n_hist, bf16):
    """Greedy and top-k rows whose histories mark more than 64 tokens of a
    chunk (the select pass leaves them out of its maxima), the likeliest
    tokens among them, with penalties that keep, lower or raise them, one
    launch and two, with logprobs."""
    import torch
    from hi_amd import sampler as S
    rng = np.random.default_rng(V + B)
    x = _rows("spiked", B, V, V + B)
    logits = f32_to_bf16_bits(x) if bf16 else x
    p = np.zeros(B, ROW_PARAMS_DTYPE)
    p["temperature"] = np.where(np.arange(B) % 3 == 0, 0.0, 0.9)
    p["top_k"], p["top_p"] = 40, 0.95
    p["repetition_penalty"] = np.array([1.3, 1.0, 0.8], F32)[np.arange(B) % 3]
    p["frequency_penalty"] = np.array([0.0, 0.2, -0.1], F32)[np.arange(B) % 3]
    ids = np.stack([np.concatenate([np.argsort(x[b])[-30:], rng.permutation(V)[:n_hist]]) for b in range(B)])
    off = (np.arange(B + 1) * ids.shape[1]).astype(np.uint32)
    ids = ids.astype(np.uint32).ravel()
    cnt = rng.integers(1, 4, ids.size).astype(np.uint32)
    u = rng.random(B).astype(F32)
    t = torch.from_numpy(logits.view(np.int16) if bf16 else logits).cuda()
    i32 = lambda a: torch.from_numpy(a.view(np.int32)).cuda()  # noqa: E731
    print(f"dense histories B={B} V={V} bf16={bf16}", flush=True)
    out = S.Sampler(B, V, 5).sample(t.view(torch.bfloat16) if bf16 else t, S.params_to_device(p),
                                    torch.from_numpy(u).cuda(), i32(off), i32(ids), i32(cnt), n_logprobs=5)
    torch.cuda.synchronize()
    want = oracle.sample_rows(logits, p, u, off, ids, cnt, n_logprobs=5)
    got = out["tokens"].cpu().numpy().view(np.uint32)
    bad = np.flatnonzero(got != want["tokens"])
    assert bad.size == 0, (bad, got[bad], want["tokens"][bad])
    np.testing.assert_allclose(out["logprobs"].cpu().numpy(), want["logprobs"], rtol=1e-5, atol=1e-6)
    assert np.array_equal(out["logprob_ids"].cpu().numpy().view(np.uint32), want["logprob_ids"])


@pytest.mark.parametrize("V", [65540, 70001])
def test_row_kernel_finite_lane_argmax(hip, oracle, new_stream, V):
    """256 greedy rows by the launchers' finite-lane rule (ties by the
    bit-reversed lane) in one workgroup each, and the same rows by temperature
    alone: ties across lanes and tiles, signed zeros, infinities, NaN, rows
    without a finite logit."""
    import torch
    from test_gpu_parity import _finite_lane_rows
    B = 256
    x = _finite_lane_rows(V, B, np.random.default_rng(V))
    u = np.random.default_rng(1).random(B).astype(F32)
    logits, samples = torch.from_numpy(x).cuda(), torch.from_numpy(u).cuda()
    out = torch.zeros(B, dtype=torch.int32, device="cuda")
    st = new_stream()
    torch.cuda.synchronize()
    print(f"finite-lane rows V={V}", flush=True)
    for t in (0.0, 0.8):
        hip.check(hip.load().hi_rocm_launch_sample_batched_last_token(
            logits.data_ptr(), out.data_ptr(), samples.data_ptr(), B, 1, V, t, float("inf"), 0, 1, st.cuda_stream))
        st.synchronize()
        got = out.cpu().numpy().view(np.uint32).tolist()
        want = [oracle.argmax_finite_lane(x[b])[0] if t <= 0 else oracle.temp_only_sample(x[b], t, float(u[b]))
                for b in range(B)]
        assert got == want, [(b, g, w) for b, (g, w) in enumerate(zip(got, want)) if g != w][:8]


@pytest.mark.parametrize("with_mask", [False, True])
def test_row_kernel_path_of_other_classes(hip, with_mask):
    """Which rows of a 256-row batch all waves finish: every class but top-k,
    unless the history is too long for their table or no logit is finite."""
    import torch
    from hi_amd import sampler as S
    B, V = 256, 65540
    rng = np.random.default_rng(3)
    x = _rows("spiked", B, V, 5)
    x[3, :] = -np.inf
    p = _params(B)
    p["top_k"][4::5] = 40
    p["temperature"][10::20] = 0.0
    n = np.where(np.arange(B) == 21, 3500, 50)
    off = np.concatenate([[0], np.cumsum(n)]).astype(np.uint32)
    ids = rng.integers(0, V, off[-1]).astype(np.uint32)
    mask = np.full((B, (V + 31) // 32), 0xffffffff, np.uint32) if with_mask else None
    i32 = lambda a: torch.from_numpy(a.view(np.int32)).cuda()  # noqa: E731
    smp = S.Sampler(B, V)
    print(f"row kernel paths mask={with_mask}", flush=True)
    smp.sample(torch.from_numpy(x).cuda(), S.params_to_device(p), torch.full((B,), 0.5, device="cuda"), i32(off),
               i32(ids), i32(np.ones_like(ids)), None if mask is None else i32(mask))
    torch.cuda.synchronize()
    names = np.array([S.WIDE_PATHS.get(int(c) & 0xff) for c in S.debug_wide_paths(smp, B, V)])
    topk = (p["top_k"] > 0) & (p["temperature"] > 0)
    left = np.isin(np.arange(B), [21] if with_mask else [3, 21])  # (masked rows without a finite logit give eos)
    assert set(names[~topk & ~left]) == {"row-all"}, names
    assert set(names[left]) == {"row-general"}, names[left]
    assert "row-all" not in names[topk]
