"""GPU parity of the draws over a row's whole distribution (top-p without
top-k, min-p alone, temperature only, top-k above 1024) against the oracle:
tokens equal, at the edges of the tiles (1024 logits), of the pieces sorted at
a time (4096 weights) and of the tile limit (262,144 logits), over one launch
or two, 16-byte aligned rows and others, and over weights that all differ,
come in long runs, or are all equal."""
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
