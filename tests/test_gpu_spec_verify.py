"""GPU parity of hi_rocm_spec_verify_greedy against the oracle's literal
restatement of gpu.rs:10725-10762 (host argmax gpu.rs:6406-6435): per-row
argmax, accepted counts and emitted tokens bit for bit, over drafts that
are fully accepted, rejected at each position, per-request draft lengths,
K = 0, ties, NaN and infinities, and a 151,936-token vocabulary."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

F32 = np.float32


@pytest.mark.parametrize("B,K,V", [(8, 4, 151936), (33, 1, 5000), (5, 0, 777), (16, 7, 32000)])
def test_spec_verify_parity(hip, oracle, B, K, V):
    import torch
    lib = hip.load()
    rng = np.random.default_rng(B * 100 + K)
    x = (rng.standard_normal((B, K + 1, V)) * 2).astype(F32)
    x[0, :, :] = np.round(x[0, :, :])  # ties
    x[1 % B, 0, 0] = np.nan
    x[2 % B, -1, 5] = np.inf
    x[3 % B, 0, 7] = np.nan
    g_ref = np.argmax(np.nan_to_num(x, nan=-np.inf), axis=2)
    # drafts: copy the target's argmax for a prefix of random length, then differ
    d = np.zeros((B, max(K, 1)), np.uint32)
    for b in range(B):
        cut = rng.integers(0, K + 1)
        for i in range(K):
            d[b, i] = g_ref[b, i] if i < cut else (g_ref[b, i] + 1) % V
    d = d[:, :K]
    dl = rng.integers(0, K + 1, B).astype(np.int32)
    for use_len in (False, True):
        dx = torch.from_numpy(x).cuda()
        dd = torch.from_numpy(d.view(np.int32).copy() if K else np.zeros(1, np.int32)).cuda()
        ddl = torch.from_numpy(dl).cuda()
        g = torch.full((B, K + 1), -1, dtype=torch.int32, device="cuda")
        t = torch.full((B, K + 1), -1, dtype=torch.int32, device="cuda")
        c = torch.full((B,), -1, dtype=torch.int32, device="cuda")
        s = torch.cuda.Stream()
        torch.cuda.synchronize()
        print(f"spec verify B={B} K={K} V={V} lens={use_len}", flush=True)
        hip.check(lib.hi_rocm_spec_verify_greedy(dx.data_ptr(), B, K, V, dd.data_ptr(),
                                                 ddl.data_ptr() if use_len else 0, g.data_ptr(), t.data_ptr(),
                                                 c.data_ptr(), s.cuda_stream))
        s.synchronize()
        wg, wt, wc = oracle.spec_verify_greedy(x, d, dl if use_len else None)
        gg, tt, cc = g.cpu().numpy().view(np.uint32), t.cpu().numpy().view(np.uint32), c.cpu().numpy()
        assert np.array_equal(gg, wg)
        assert np.array_equal(cc, wc)
        for b in range(B):
            assert np.array_equal(tt[b, :cc[b]], wt[b, :wc[b]]), b
            assert (tt[b, cc[b]:] == 0xffffffff).all(), "write past the emitted tokens"


class _Call:
    """One verification's device arrays and what the oracle says of them."""

    def __init__(self, torch, oracle, x, d):
        self.want = oracle.spec_verify_greedy(x, d, None)
        self.B, self.K, self.V = x.shape[0], x.shape[1] - 1, x.shape[2]
        self.x, self.d = torch.from_numpy(x).cuda(), torch.from_numpy(d.view(np.int32)).cuda()
        self.g, self.t = (torch.full((self.B, self.K + 1), -1, dtype=torch.int32, device="cuda") for _ in range(2))
        self.c = torch.full((self.B,), -1, dtype=torch.int32, device="cuda")

    def launch(self, hip, handle):
        hip.check(hip.load().hi_rocm_spec_verify_greedy(
            self.x.data_ptr(), self.B, self.K, self.V, self.d.data_ptr(), 0, self.g.data_ptr(), self.t.data_ptr(),
            self.c.data_ptr(), handle))

    def clear(self, greedy=-1):
        for o in (self.g, self.t, self.c):
            o.fill_(-1)
        self.g.fill_(greedy)

    def same(self):
        wg, wt, wc = self.want
        assert np.array_equal(self.g.cpu().numpy().view(np.uint32), wg)
        assert np.array_equal(self.c.cpu().numpy(), wc)
        t = self.t.cpu().numpy().view(np.uint32)
        assert all(np.array_equal(t[b, :wc[b]], wt[b, :wc[b]]) for b in range(self.B))
        assert all((t[b, wc[b]:] == 0xffffffff).all() for b in range(self.B)), "write past the emitted tokens"


@pytest.mark.parametrize("V", [1, 8191, 8193, 50257, 70001])
def test_spec_verify_parts(hip, oracle, new_stream, V):
    """Rows split over workgroups (8192 logits each), eagerly and in a capture
    on a stream of no earlier call: maxima on both sides of every part's edge,
    equal maxima in two parts, -inf and NaN rows, and whatever the greedy
    array holds before: no index, one past the row, a NaN's, an equal maximum
    that is not the first."""
    import torch
    B, K = 6, 2
    rng = np.random.default_rng(V)
    x = (rng.standard_normal((B, K + 1, V)) * 2).astype(F32)
    edges = [i for i in (0, 8191, 8192, V - 1) if i < V]
    for n, e in enumerate(edges):
        x[n % B, n % (K + 1), e] = 50.0
    x[4, 0, edges] = 60.0
    x[4, 1, :] = 0.0
    x[4, 1, ::2] = -0.0
    x[5, 0, :] = -np.inf
    x[5, 1, :] = np.nan
    x[5, 2, V // 2:] = np.nan
    d = rng.integers(0, V, (B, K)).astype(np.uint32)
    d[:, 0] = oracle.spec_verify_greedy(x, d, None)[0][:, 0]
    call = _Call(torch, oracle, x, d)
    s = new_stream()
    torch.cuda.synchronize()
    print(f"spec verify parts V={V}", flush=True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        call.launch(hip, s.cuda_stream)
    for before in (-1, 0, V, V - 1, V // 2):
        call.clear(before)
        graph.replay()
        torch.cuda.synchronize()
        call.same()
        call.clear(before)
        torch.cuda.synchronize()
        call.launch(hip, s.cuda_stream)
        s.synchronize()
        call.same()
    del graph


def test_spec_verify_calls_share_nothing(hip, oracle, new_stream):
    """Calls with different outputs at once: two graphs captured on one stream
    and replayed on two others, beside eager calls on the capture stream, each
    checked after every round; releasing the stream's library buffers leaves
    the graphs whole, and no call allocates."""
    import torch
    B, K, V = 8, 4, 151936
    calls = []
    for seed in range(3):
        rng = np.random.default_rng(seed)
        x = rng.standard_normal((B, K + 1, V), dtype=F32)
        d = x[:, :K].argmax(2).astype(np.uint32)
        d[::3, seed] += 1
        calls.append(_Call(torch, oracle, x, d))
    s = new_stream()
    others = [new_stream(), new_stream()]
    for c in calls:  # the kernels' first launches
        c.launch(hip, others[0].cuda_stream)
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    calls[2].launch(hip, s.cuda_stream)  # the stream's first call
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] == free0, "a verification allocated"
    graphs = []
    for c in calls[:2]:
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1], stream=s):
            c.launch(hip, s.cuda_stream)
    hip.check(hip.load().hi_rocm_sampler_release(s.cuda_stream))
    print("spec verify: concurrent calls", flush=True)
    for _ in range(20):
        for c in calls:
            c.clear()
        torch.cuda.synchronize()
        for _ in range(3):
            for graph, o in zip(graphs, others):
                with torch.cuda.stream(o):
                    graph.replay()
            calls[2].launch(hip, s.cuda_stream)
        torch.cuda.synchronize()
        for c in calls:
            c.same()
    del graphs


def test_spec_verify_beyond_32_bit_bytes(hip, new_stream):
    """A row of more than 2^32 bytes: the maximum is found wherever it lies,
    and of two equal ones the first."""
    import torch
    lib = hip.load()
    V = 2 ** 30 + 5
    x = torch.full((V,), -1.0, device="cuda")
    d, g, t, c = (torch.zeros(2, dtype=torch.int32, device="cuda") for _ in range(4))
    st = new_stream()
    for at in ([3], [2 ** 29 - 1, 2 ** 29 + 3], [2 ** 29 + 3], [2 ** 30 - 1, 2 ** 30 + 2], [2 ** 30 + 2], [V - 1]):
        x[at] = 2.0
        torch.cuda.synchronize()
        print(f"spec verify V={V} {at}", flush=True)
        hip.check(lib.hi_rocm_spec_verify_greedy(x.data_ptr(), 1, 0, V, 0, 0, g.data_ptr(), t.data_ptr(), c.data_ptr(),
                                                 st.cuda_stream))
        torch.cuda.synchronize()
        assert (int(g[0]), int(t[0]), int(c[0])) == (at[0], at[0], 1)
        x[at] = -1.0
