"""The weight-streaming decode GEMM (csrc/kernels/gemm_stream.hip) against fp64, and its rule."""
import pytest
import torch

from drtc_amd import ops
from drtc_amd.ops import gemm as G


def test_rule_takes_only_what_the_kernel_takes():
    """Every shape that the rule accepts has a slice count whose K steps the kernel is built for, whole
    tiles of rows and a workspace that holds the parts; others keep their routes."""
    seen = set()
    for M in range(0, 70):
        for N in (8, 16, 48, 2048, 2560, 6144, 16384, 32000, 256000):
            for K in (256, 512, 2048, 3584, 4096, 5632, 7168, 8192, 14336, 16384, 28672):
                for epi in G.STREAM_ACT:
                    s = G.stream_slices(M, N, K, epi)
                    if G.stream_ok(M, N, K, epi):
                        assert s
                    if not s:
                        continue
                    mt = 1 if M <= 16 else 2 if M <= 32 else 4
                    assert 1 <= M <= 64 and N % 16 == 0 and K % (256 * s) == 0 and K // (256 * s) in G.STREAM_KS[mt]
                    parts = N // 16 * mt * (1 + G.STREAM_ACT[epi][0])
                    assert s == 1 or s * parts * 1024 <= G.WS_SLAB_BYTES and parts < G.WS_COUNTERS - 1
                    assert s == 1 or s <= 4 and M <= 32 and not G.STREAM_ACT[epi][0]
                    seen.add((mt, K // (256 * s), s > 1))
    assert {(m, k) for m, k, _ in seen} == {(m, k) for m in G.STREAM_KS for k in G.STREAM_KS[m]}


def _want(x, w, epi, N, limit):
    r = x.double() @ w.double().t()
    if epi == "relu2":
        return torch.relu(r).square()
    if epi == "store":
        return r
    g, u = r[:, :N], r[:, N:]
    if epi == "clamped":
        g = g.clamp(max=limit)
        return g * torch.sigmoid(1.702 * g) * (u.clamp(-limit, limit) + 1)
    f = torch.nn.functional
    return (f.silu(g) if epi == "silu" else f.gelu(g, approximate="tanh")) * u


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 3, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K,epi", [(16, 2048, "store"), (4112, 4096, "store"), (8208, 2048, "silu"),
                                     (48, 7168, "relu2"), (4096, 14336, "store"), (80, 16384, "store"),
                                     (2064, 4096, "gelu_tanh"), (112, 4096, "clamped")])
def test_stream_gemm(hipk, M, N, K, epi):
    """One tile and many, more tiles than workgroups, one slice and several, rows in strides; the same
    bits twice, tickets left at zero, and in replays of a graph on new inputs between other work."""
    if not G.stream_slices(M, N, K, epi):
        pytest.skip("not an instance")
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    buf = torch.randn(M, K + 24, device="cuda", generator=g).to(torch.bfloat16)
    x = buf[:, 8:K + 8]
    w = (torch.randn(N * (1 + G.STREAM_ACT[epi][0]), K, device="cuda", generator=g) * 0.03).to(torch.bfloat16)
    out = torch.full((M + 1, N + 8), 7.0, device="cuda", dtype=torch.bfloat16)

    def check(y):
        # fp32 sums of K products: far below the rounding of the result to bf16 (2^-9 of each value)
        r = _want(x, w, epi, N, 0.8)
        assert (y.double() - r).norm() <= 2 ** -9 * 1.1 * r.norm() + 1e-5 * K ** 0.5

    G.stream_gemm(x, w, epi, out=out[:M, :N], limit=0.8)
    check(out[:M, :N])
    assert (out[M] == 7).all() and (out[:, N:] == 7).all()
    assert torch.equal(G.stream_gemm(x, w, epi, limit=0.8), out[:M, :N])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = G.stream_gemm(x, w, epi, limit=0.8)
    for _ in range(3):
        buf.normal_(generator=g)
        graph.replay()
        check(y)
        assert torch.equal(G.stream_gemm(x, w, epi, limit=0.8), y)
    assert int(G.gemm_workspace(x.device)[1].abs().sum()) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("M", [3, 16, 32])
def test_routes_to_the_stream(hipk, M):
    """linear, norm_glu, gated and squared_relu at a shape of the rule: the same numbers as the kernel
    itself, unaligned rows through another route."""
    K, N = 4096, 16384
    g = torch.Generator(device="cuda").manual_seed(M)
    buf = torch.randn(M * K + 8, device="cuda", generator=g).to(torch.bfloat16)
    x, nw = buf[:M * K].view(M, K), torch.ones(K, device="cuda", dtype=torch.bfloat16)
    w = (torch.randn(N, K, device="cuda", generator=g) * 0.03).to(torch.bfloat16)
    G.reset()
    assert G.route(M, N, K, K) == ("skinny", G.STREAM)
    assert torch.equal(ops.linear(x, w), G.stream_gemm(x, w))
    odd = buf[1:M * K + 1].view(M, K)
    assert (ops.linear(odd, w).double() - odd.double() @ w.double().t()).norm() < 0.01 * (K ** 0.5) * (M * N) ** 0.5
    assert ops.gemm.fused_glu_ok(x, w, "silu")
    xn = ops.rmsnorm(x, nw, 1e-5)
    assert torch.equal(ops.norm_glu(ops.PendingNorm(x, None, nw, 1e-5, False), w, "silu"), G.stream_gemm(xn, w, "silu"))
    assert torch.equal(ops.gated(x, w, "clamped", 0.9), G.stream_gemm(x, w, "clamped", limit=0.9))
    out = torch.zeros(M, N + 8, device="cuda", dtype=torch.bfloat16)
    ops.squared_relu(x, w, out[:, 8:])
    assert torch.equal(out[:, 8:], G.stream_gemm(x, w, "relu2")) and (out[:, :8] == 0).all()


@pytest.mark.gpu
def test_measured_shapes_keep_their_kernels(hipk):
    """Entries of the tuning table that say the streaming kernel is slower: the table's kernel, for the batches
    that pad to the entry's bucket too; the bucket above takes the rule again."""
    G.reset()
    tab = {tuple(int(v) for v in k.split(",")) for k, e in G.load_table()[str(hipk.lt_version())].items()
           if e.get("stream") == 0}
    assert tab
    for M, N, K, ldx in tab:
        assert G.stream_ok(M, N, K) and G.route(M, N, K, ldx) != ("skinny", G.STREAM)
    assert (4, 1280, 8192, 8192) in tab
    assert G.route(3, 1280, 8192, 8192) != ("skinny", G.STREAM) and G.route(8, 1280, 8192, 8192) == ("skinny", G.STREAM)
    x = torch.randn(3, 8192, device="cuda").to(torch.bfloat16)
    w = (torch.randn(1280, 8192, device="cuda") / 8192 ** 0.5).to(torch.bfloat16)
    want = x.double() @ w.double().t()
    assert ((ops.linear(x, w).double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-3).all()


# tiles of 16 rows in an entry, 0: not taken; 2048 x 4096 and 4096 x 3584 leave registers for 32 rows (gated: 16)
STREAMED_TILES = {(2048, "silu", 0): {1: 1, 5: 1, 16: 1, 37: 1, 80: 2, 150: 4},
                  (4096, "relu2", 0): {1: 1, 5: 1, 16: 1, 37: 1, 80: 2, 150: 0},
                  (2048, "gelu_tanh", 0): {1: 1, 5: 1, 16: 1, 37: 1, 80: 0, 150: 0},
                  (1792, "clamped", 0): {1: 1, 5: 1, 16: 1, 37: 1, 80: 2, 150: 4},
                  (2048, "silu", 4): {1: 1, 5: 1, 16: 1, 37: 2, 80: 4, 150: 0}}


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 5, 16, 37, 80, 150])
@pytest.mark.parametrize("H,I,E,k,act,e_off", [(2048, 1792, 16, 4, "silu", 0), (4096, 3584, 20, 4, "relu2", 0),
                                              (2048, 4096, 8, 2, "gelu_tanh", 0), (1792, 2048, 24, 6, "clamped", 0),
                                              (2048, 2048, 12, 3, "silu", 4)])
def test_streamed_experts(hipk, T, H, I, E, k, act, e_off):
    """Experts with no row, one, a tile and more than an entry holds (every third token goes to the first
    expert first), a part of the experts on this rank; against the fp32 oracle, and the same bits in
    replays of a graph."""
    e_local = E // 2 if e_off else E
    g = torch.Generator(device="cuda").manual_seed(T + E)
    x = torch.randn(T, H, device="cuda", generator=g).to(torch.bfloat16)
    lg = torch.randn(T, E, device="cuda", generator=g)
    lg[::3, e_off] = 9.0
    n_in = I if act == "relu2" else 2 * I
    w_in = (torch.randn(e_local, n_in, H, device="cuda", generator=g) * 0.02).to(torch.bfloat16)
    w_out = (torch.randn(e_local, H, I, device="cuda", generator=g) * 0.02).to(torch.bfloat16)
    ws = ops.moe.make_workspace(T, H, I, e_local, k, "cuda")
    G.gemm_workspace(x.device)

    def run(v=5):
        return ops.fused_moe(x, lg, w_in, w_out, k, act, E, e_off, ws, variant=v, limit=0.9)

    mt = hipk.stream_moe_tiles(T * k // e_local, H, I, act != "relu2")
    assert mt == STREAMED_TILES[(H, act, e_off)][T]
    if mt:
        y = run()
    else:  # more rows to an expert than the registers hold
        with pytest.raises(RuntimeError):
            run()
        y = run(-1)
    want = ops.fused_moe_ref(x, lg, w_in, w_out, k, act, e_off, limit=0.9).double()
    # both round the hidden rows and the experts' outputs to bf16: a few of them differ by one unit
    assert (y.double() - want).norm() <= 2e-3 * want.norm() + 1e-6
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        z = run(-1)
    for _ in range(3):
        x.normal_(generator=g)
        lg.normal_(generator=g)
        graph.replay()
        assert torch.equal(z, run(-1))


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 255, 256, 257, 1000, 1024, 1025])
@pytest.mark.parametrize("E,k,groups,keep", [(16, 4, 1, 1), (250, 16, 1, 1), (24, 5, 4, 2)])
def test_routing_plan(hipk, T, E, k, groups, keep):
    """Logits on a coarse grid, so that most choices are ties, with both zeros and infinities among them,
    in one workgroup (T <= 1024) and in three passes: identical experts must come out of a model whose
    experts return their number (the weighted sum tells which were chosen)."""
    g = torch.Generator(device="cuda").manual_seed(T + E)
    lg = (torch.randn(T, E, device="cuda", generator=g) * 2).round() / 2
    lg[::5] *= -0.0
    lg[1::7, 3] = float("-inf")
    x = torch.ones(T, 128, device="cuda")
    w_in = torch.ones(E, 8, 128, device="cuda") / 128  # hidden 1 for all
    w_out = (torch.arange(E, device="cuda").float() + 1).view(E, 1, 1).expand(E, 128, 8).contiguous() / 8
    for logits in (lg, lg.t().contiguous().t(), lg.to(torch.bfloat16)):
        y = ops.fused_moe(x, logits, w_in, w_out, k, "relu2", E, groups=groups, keep=keep)
        ids, w = ops.moe.route_ref(logits, k, groups, keep)
        want = (w * (ids + 1)).sum(-1)
        # a wrong expert moves the sum by a weight times a whole number; the fp32 sums by 1e-5 of it
        assert (y[:, 0] - want).abs().max() <= 1e-4 * E


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,e_off", [(64, 256, 0), (256, 256, 0), (200, 255, 0), (300, 256, 0), (256, 256, 128)])
def test_routing_plan_group_offsets(hipk, T, E, e_off):
    """As many experts as threads: the end of the last expert's rows, which the grouped GEMM reads, over a
    workspace of other bytes; hidden rows and outputs rounded to bf16 as in test_streamed_experts."""
    H, I, k = 256, 128, 4
    g = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn(T, H, device="cuda", generator=g).to(torch.bfloat16)
    lg = torch.randn(T, E, device="cuda", generator=g)
    lg[::3, E - 1] = 9.0
    lg[::7, e_off] = 8.0
    w_in = (torch.randn(E - e_off, 2 * I, H, device="cuda", generator=g) * 0.05).to(torch.bfloat16)
    w_out = (torch.randn(E - e_off, H, I, device="cuda", generator=g) * 0.05).to(torch.bfloat16)
    ws = ops.moe.make_workspace(T, H, I, E - e_off, k, "cuda")
    want = ops.fused_moe_ref(x, lg, w_in, w_out, k, "silu", e_off).double()
    for fill in (0xff, 0x00, 0x01):
        ws.fill_(fill)
        y = ops.fused_moe(x, lg, w_in, w_out, k, "silu", E, e_off, ws, variant=4).double()
        assert (y - want).norm() <= 4e-3 * want.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("M,I,K,act", [(17, 8192, 2048, "silu"), (33, 14336, 1024, "gelu_tanh"), (127, 10240, 4096, "silu"),
                                       (129, 3584, 4096, "silu"), (257, 7168, 1024, "clamped"), (511, 5632, 512, "silu"),
                                       (700, 1792, 2048, "silu"), (130, 28672, 512, "gelu_tanh")])
def test_gated_default_form(hipk, M, I, K, act):
    """Shapes that no table measured, through the rule that sends them to gemm_xd: rows of x apart, M
    around its tiles, against 64 bits (bf16 rounding of the result, 2^-9 of it, and of nothing else)."""
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K + 16, generator=g).bfloat16().to("cuda")[:, :K]
    w = (torch.randn(2 * I, K, generator=g) / K ** 0.5).bfloat16().to("cuda")
    form = ops.gemm.glu_form(M, 2 * I, K, x.stride(0), act)
    assert form == ops.gemm._glu_default(M, I, K) != 0 and ops.gemm.fused_glu_ok(x, w, act)
    got = ops.gemm.gated(x, w, act, limit=1.0).double()
    a, b = (x.double() @ w.double().t()).chunk(2, -1)
    if act == "clamped":
        a, b = a.clamp(max=1.0), b.clamp(-1.0, 1.0)
        want = a * torch.sigmoid(1.702 * a) * (b + 1)
    else:
        want = (torch.nn.functional.silu(a) if act == "silu" else torch.nn.functional.gelu(a, approximate="tanh")) * b
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all()


def test_gated_default_leaves_what_the_library_does_faster():
    """Tiles of 128 columns a half: not above 128 rows with long K, nor from 257 rows to gemm_w4's first; the
    neighbours on the other side of each line keep theirs."""
    none = [(160, 28672, 8192), (256, 20480, 8192), (320, 14336, 4096), (513, 7168, 4096), (600, 7168, 2048),
            (639, 5632, 2048)]
    assert not any(G._glu_default(*s) for s in none)
    some = [(128, 28672, 8192), (160, 16384, 4096), (256, 32768, 4096), (512, 7168, 4096), (640, 7168, 4096),
            (600, 3584, 2048)]
    assert all(G._glu_default(*s) for s in some), [G._glu_default(*s) for s in some]


@pytest.mark.parametrize("xd", [True, False])
def test_streaming_yields_to_forms_that_run(monkeypatch, xd):
    """Where a gated product of 33 to 64 rows leaves the streaming kernel for gemm_xd, gemm_xd has a form for its
    activation; the clamped one gets a form of its own tiles; without gemm_xd the stream takes all it can."""
    monkeypatch.setattr(G, "_xd_enabled", xd)
    seen = set()
    for act in G.GATED:
        for M in (33, 48, 64):
            for I in (1024, 3584, 5632, 7168, 8192, 14336, 16384):
                for K in (2048, 4096):
                    form = G.glu_form(M, 2 * I, K, K, act)
                    assert not form or xd and G.xd_supported(M, I, K, form, True)
                    assert act != "clamped" or not form or G.xd_form(form)[1] in G.XD_CLAMP_NF
                    if G.stream_slices(M, I, K, act) == 1 and 2 * I >= 14336:
                        assert G.stream_ok(M, I, K, act) != bool(form)
                        seen.add((act, bool(form)))
    assert seen >= {(a, xd) for a in G.GATED}
    if xd:
        assert G.glu_form(48, 14336, 2048, 2048, "clamped") == 1141 and G.glu_form(48, 14336, 2048, 2048, "silu") == 121


@pytest.mark.gpu
@pytest.mark.parametrize("M", [17, 64, 128])
def test_clamped_default_form(hipk, M):
    """A shape whose default tiles the clamped activation lacks, against 64 bits (bf16 rounding of the result)."""
    I, K = 7168, 1024
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).bfloat16().to("cuda")
    w = (torch.randn(2 * I, K, generator=g) / K ** 0.5).bfloat16().to("cuda")
    assert G.glu_form(M, 2 * I, K, K, "clamped") == 1141
    got = G.gated(x, w, "clamped", limit=1.0).double()
    a, b = (x.double() @ w.double().t()).chunk(2, -1)
    a, b = a.clamp(max=1.0), b.clamp(-1.0, 1.0)
    want = a * torch.sigmoid(1.702 * a) * (b + 1)
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,kind", [(6145, 4096, 10304, "w4"), (7681, 4352, 11264, "w4"), (11520, 4096, 17472, "w4"),
                                        (8960, 4096, 17472, "torch"), (9216, 4096, 11264, "torch"),
                                        (4096, 4096, 10304, "torch"), (8192, 4096, 10304, "torch"),
                                        (6400, 4096, 8256, "torch"), (6400, 2048, 11264, "torch")])
def test_long_k_prefill_route(hipk, M, N, K, kind):
    """K above the limit of the measured shapes, without a tuned solution: gemm_w4 between the quarter rounds of its
    tiles (9216 rows: 2.25; 4096 and 8192: whole), from K 10240 and 4096 columns on.  Rows against 64 bits: bf16
    rounding of the result and fp32 sums of K products."""
    G.reset()
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda", generator=g) / K ** 0.5).to(torch.bfloat16)
    assert G.route(M, N, K, K)[0] == kind
    rows = torch.tensor([0, 255, 256, M // 2, M - 1], device="cuda")
    want = x[rows].double() @ w.double().t()
    assert ((ops.linear(x, w)[rows].double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-3).all()


@pytest.mark.gpu
@pytest.mark.parametrize("H,I,E,k,act,e_off,T", [
    (128, 64, 4, 2, "silu", 0, 1),       # one K tile of the down projection, fewer columns than workgroups
    (256, 192, 8, 2, "gelu_tanh", 0, 9),
    (384, 320, 8, 4, "clamped", 4, 70),  # some of the experts on this rank
    (2048, 1792, 16, 4, "silu", 0, 128), (2048, 1792, 20, 4, "relu2", 0, 129),  # tiles of 3 fragments and of 4
    (1024, 640, 5, 3, "relu2", 0, 170),  # entries of all 128 rows, and of a few
    (128, 128, 256, 4, "relu2", 0, 500),  # more entries than workgroups: runs over several of them
    (192 * 2, 64, 130, 8, "silu", 0, 300),  # one workgroup to an entry, several tiles each
])
def test_ring_experts(hipk, H, I, E, k, act, e_off, T):
    """The experts' ring at the edges of its tiles, entries and runs, against the fp32 oracle; the same bits
    in replays of a graph, and with no row for any expert of this rank."""
    e_local = E - e_off
    g = torch.Generator(device="cuda").manual_seed(T + E)
    x = torch.randn(T, H, device="cuda", generator=g).to(torch.bfloat16)
    lg = torch.randn(T, E, device="cuda", generator=g)
    lg[::3, e_off] = 9.0
    n_in = I if act == "relu2" else 2 * I
    w_in = (torch.randn(e_local, n_in, H, device="cuda", generator=g) * 0.02).to(torch.bfloat16)
    w_out = (torch.randn(e_local, H, I, device="cuda", generator=g) * 0.02).to(torch.bfloat16)
    ws = ops.moe.make_workspace(T, H, I, e_local, k, "cuda")
    G.gemm_workspace(x.device)

    def run():
        return ops.fused_moe(x, lg, w_in, w_out, k, act, E, e_off, ws, variant=6, limit=0.9)

    y = run()
    want = ops.fused_moe_ref(x, lg, w_in, w_out, k, act, e_off, limit=0.9).double()
    # both round the hidden rows and the experts' outputs to bf16: a few of them differ by one unit
    assert (y.double() - want).norm() <= 2e-3 * want.norm() + 1e-6
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        z = run()
    for _ in range(3):
        x.normal_(generator=g)
        lg.normal_(generator=g)
        graph.replay()
        assert torch.equal(z, run())
    if e_off >= k:  # every token to the other rank
        lg[:, :e_off] += 100.0
        assert not run().any()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,form", [(23, 32768, 2048, 0), (24, 32768, 2048, 1141), (128, 27648, 2112, 1141),
                                       (129, 27648, 2112, 1241), (256, 65536, 2048, 1281), (64, 32768, 1984, 0),
                                       (64, 50176, 2048, 0), (129, 64128, 2048, 0), (65, 64128, 2048, 1141)])
def test_wide_products(hipk, M, N, K, form):
    """Both sides of the rule for wide plain products, and what linear then gives: every workgroup starts its walk
    of K (33 tiles of 64 in two cases) elsewhere.  bf16 rounding of the result and fp32 sums of K products."""
    G.reset()
    assert G.wide_form(M, N, K) == form
    kind = G.route(M, N, K, K)
    assert not form or kind[0] == "xd"
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda", generator=g) / K ** 0.5).to(torch.bfloat16)
    got, want = ops.linear(x, w).double(), x.double() @ w.double().t()
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all()
    if form:
        glu = ops.gemm.xd_gemm(x, w[:N // 512 * 512], "silu", form=form)
        a, b = (x.double() @ w[:N // 512 * 512].double().t()).chunk(2, -1)
        want = a * torch.sigmoid(a) * b
        assert ((glu.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all()


def test_parts_forms():
    """The cut of every shape that the rule takes fits the kernel; what lies outside of it stays with linear."""
    seen = set()
    for K in (2048, 2112, 3584, 4096, 5120, 5632, 8192, 14336, 28672):
        for N in (1024, 1088, 2048, 4096, 5120, 8192):
            for M in (1, 2, 3, 16, 17, 33, 64, 65, 128, 129, 160, 161, 256, 257):
                form = G.parts_form(M, N, K)
                if form:
                    nf, s = form
                    assert nf in (2, 4) and N % (32 * nf) == 0 and 2 <= s <= G.MAX_PARTS and K // 64 // s >= 4
                    assert N // (32 * nf) * s <= 256 and 3 <= M <= 256
                    seen.add(form)
    assert len(seen) > 6
    assert not any(G.parts_form(*s) for s in [(2, 4096, 14336), (257, 4096, 14336), (161, 4096, 4096), (16, 2048, 2048),
                                              (65, 4096, 2048), (64, 4096, 1984), (64, 8256, 4096), (64, 4096, 4104)])


@pytest.mark.parametrize("limits", [(4, G.MAX_PARTS), (G.MAX_PARTS, 4)])
def test_parts_forms_of_up_to_four_slices(monkeypatch, limits):
    """A reader of up to four slices gets no more, whichever limit was asked first; 3 rows on from K = 4096, 17 from 2048."""
    monkeypatch.setattr(G, "_parts_forms", {})
    seen = {most: set() for most in limits}
    for M in (2, 3, 16, 17, 33, 64):
        for N, K in ((6144, 4096), (3072, 2048), (2304, 2048), (4096, 5120), (5120, 4096)):
            for most in limits:
                form = G.parts_form(M, N, K, most)
                assert (form is not None) == (M >= (3 if K >= 4096 else 17)), (M, N, K, most)
                if form:
                    assert 2 <= form[1] <= most and N % (32 * form[0]) == 0 and K // 64 // form[1] >= 4
                    seen[most].add(form)
    assert max(s for _, s in seen[4]) == 4 and max(s for _, s in seen[G.MAX_PARTS]) > 4


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,form", [(1, 1024, 256, (2, 1)), (17, 1088, 320, (2, 5)), (33, 2048, 4096, (2, 8)),
                                       (64, 4096, 704, (4, 8)), (96, 1024, 2112, (4, 3)), (150, 4096, 5632, (2, 4)),
                                       (160, 2048, 1024, (4, 2)), (200, 1152, 7168, (4, 7)), (256, 1024, 448, (4, 1))])
def test_product_parts(hipk, M, N, K, form):
    """K slices at the edges of the tiles and rings (fewer K tiles than stages, slices of unequal length, rows
    that are no multiple of 32) and the three ops that add them up, each against 64 bits."""
    g = torch.Generator(device="cuda").manual_seed(M + K)
    buf = torch.randn(M, K + 8, device="cuda", generator=g).to(torch.bfloat16)
    x = buf[:, :K]
    w = (torch.randn(N, K, device="cuda", generator=g) / K ** 0.5).to(torch.bfloat16)
    nf, s = form
    slab = torch.full((s, M, N), float("nan"), device="cuda")
    assert hipk.midm_gemm(0, x.data_ptr(), w.data_ptr(), 0, M, N, K, x.stride(0), N, 0, 4, s, nf, slab.data_ptr(),
                          slab.numel() * 4, torch.cuda.current_stream().cuda_stream) == 0
    want = x.double() @ w.double().t()
    # fp32 sums of K products in whatever order
    assert (slab.double().sum(0) - want).abs().max() <= 2.0 ** -24 * K ** 0.5 * 16
    parts = G.Parts(slab, torch.bfloat16)
    near = 2.0 ** -8  # of a rounding to bf16
    # residual add and RMS norm
    res = torch.randn(M, N, device="cuda", generator=g).to(torch.bfloat16)
    nw = (1 + 0.1 * torch.randn(N, device="cuda", generator=g)).to(torch.bfloat16)
    h = want + res.double()
    for gemma in (False, True):
        r = res.clone()
        p = ops.PendingNorm(parts, r, nw, 1e-5, gemma)
        assert p.stream().data_ptr() == r.data_ptr()
        assert ((r.double() - h).abs() <= near * h.abs() + 1e-5).all()
        n = h * torch.rsqrt((h * h).mean(-1, keepdim=True) + 1e-5) * (nw.double() + gemma)
        assert ((p.materialize().double() - n).abs() <= 2 * near * n.abs() + 1e-4).all()
    # Dynamic Tanh on the 32-bit stream
    st, b = res.float(), torch.randn(N, device="cuda", generator=g)
    out = ops.dyt(st, nw.float(), b, 0.7, y=parts)
    assert (st.double() - h).abs().max() <= 1e-5
    t = torch.tanh(0.7 * h) * nw.double() + b.double()
    assert ((out.double() - t).abs() <= near * t.abs() + 1e-5).all()
    # the experts' combine: experts that return zeros leave the sum alone
    if N % 128 == 0:
        st = res.float()
        zero = torch.zeros(2, 128, N, device="cuda", dtype=torch.bfloat16)
        out = ops.fused_moe(res, torch.randn(M, 2, device="cuda", generator=g), zero, zero.transpose(1, 2).contiguous(), 1,
                            "relu2", stream=st, y=parts)
        assert (st.double() - h).abs().max() <= 1e-5 and torch.equal(out, st.to(torch.bfloat16))
    # a K slice's sums do not depend on what else is in the batch
    if M > 32:
        few = torch.empty(s, 32, N, device="cuda")
        assert hipk.midm_gemm(0, x.data_ptr(), w.data_ptr(), 0, 32, N, K, x.stride(0), N, 0, 4, s, nf, few.data_ptr(),
                              few.numel() * 4, torch.cuda.current_stream().cuda_stream) == 0
        assert torch.equal(few, slab[:, :32])


@pytest.mark.gpu
@pytest.mark.parametrize("family", ["llama", "ralesun"])
def test_slices_sums_live_until_their_norm(hipk, monkeypatch, family):
    """A layer stack holds the sums of one product's K slices at a time."""
    import weakref

    from drtc_amd.engine import LLMEngine, Request
    from drtc_amd.models import build_model
    from drtc_amd.models.config import HybridConfig, LatentAttention, Layer, ModelConfig

    if family == "llama":
        cfg = ModelConfig("three layers", 512, 2048, 7168, 3, 16, 4, 128)
    else:
        att = LatentAttention(16, 128, 64, 128, 512, 192 ** -0.5, 1024, 500000.0, 64)
        cfg = HybridConfig("three layers", 512, 2048, (Layer(att, 7168),) * 3, norm_eps=1e-5)
    real, live, seen = G.linear_parts, [], []

    def watch(x, w):
        assert not [r for r in live if r() is not None]
        y = real(x, w)
        if isinstance(y, ops.Parts):
            live.append(weakref.ref(y.slab))
            seen.append(y.shape)
        return y

    eng = LLMEngine(build_model(cfg, "cuda", seed=1), max_batch=4, max_model_len=128, num_blocks=16)
    monkeypatch.setattr(ops, "linear_parts", watch)
    monkeypatch.setattr(G, "linear_parts", watch)
    eng.feed([(Request([]), list(range(3, 51)), [47])])
    torch.cuda.synchronize()
    assert len(seen) >= 4


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(17, 1024, 64), (64, 4096, 256), (128, 1088, 256), (170, 2048, 192), (256, 2048, 128)])
def test_short_k_products(hipk, M, N, K):
    """Products of one to four K tiles, fewer than the ring has stages, as linear routes them; rows of a wider
    buffer.  bf16 rounding of the result; unaligned rows through another route."""
    G.reset()
    assert G.brief_ok(M, N, K) and not G.brief_ok(M, N, K + 256) and not G.brief_ok(16, N, K) and not G.brief_ok(M, 512, K)
    g = torch.Generator(device="cuda").manual_seed(M)
    wide = torch.randn(M, K + 72, device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda", generator=g) / K ** 0.5).to(torch.bfloat16)
    for x in (wide[:, 8:K + 8], wide[:, 3:K + 3], wide[:, :K].contiguous()):
        got, want = ops.linear(x, w).double(), x.double() @ w.double().t()
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 17, 63, 64, 65, 200, 256])
@pytest.mark.parametrize("form", [11, 21, 41, 1011, 1021, 1041])
@pytest.mark.parametrize("N,K", [(256, 512), (384, 2048)])
def test_row_tiles_of_64(hipk, M, form, N, K):
    """gemm_xd on tiles of 64 rows: one row tile (each workgroup starts K at another tile) and several, rows of a
    wider buffer, residual and squared epilogues.  bf16 rounding of the result (twice with the residual)."""
    g = torch.Generator(device="cuda").manual_seed(M + form)
    x = torch.randn(M, K + 8, device="cuda", generator=g).to(torch.bfloat16)[:, :K]
    w = (torch.randn(N, K, device="cuda", generator=g) / K ** 0.5).to(torch.bfloat16)
    res = torch.randn(M, N, device="cuda", generator=g).to(torch.bfloat16)
    want = x.double() @ w.double().t()
    near = lambda got, ref, add=0.0: bool(((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + add + 1e-5).all())
    assert near(G.xd_gemm(x, w, form=form), want)
    assert near(G.xd_gemm(x, w, "relu2", form=form), want.clamp(min=0) ** 2, 1e-5 * want.abs().max())
    assert near(G.xd_gemm(x, w, "residual", residual=res.clone(), form=form), want + res.double(), 2.0 ** -8 * want.abs())
    assert not G.xd_supported(M, N, K, form + 1) and not G.xd_supported(M, N, K, form, glu=True)


@pytest.mark.gpu
def test_variants_by_pairs(hipk):
    """A few pairs of large experts are gemm_xd's, from eight on or more than one an expert the ring's, as are small
    experts; few rows an expert of gemm_stream's widths its form; nothing off 16 bytes the ring's."""
    v = lambda T, k, E, H, I, glu=True, whole=True: hipk.moe_variant(T, T * k, E, H, I, glu, whole)
    assert [v(T, 2, 4, 2048, 5632) for T in (1, 2, 3)] == [3, 3, 6]
    assert [v(T, 2, 12, 1536, 4096) for T in (1, 2, 3, 4)] == [3, 3, 3, 6]
    assert [v(T, 2, 64, 2560, 2816) for T in (2, 3, 4, 16)] == [3, 3, 6, 6]
    assert [v(T, 2, 8, 4096, 14336) for T in (1, 3, 4, 16, 500, 2000)] == [3, 3, 6, 6, 3, 4]
    assert v(1, 2, 16, 1024, 1024) == 6 and v(1, 2, 16, 1024, 1024, whole=False) == 1
    assert [v(T, 4, 16, 2048, 1792) for T in (1, 4, 224)] == [5, 6, 6] and v(224, 4, 16, 2048, 1792, whole=False) == 1
    assert v(13, 4, 16, 4096, 3584) == 5 and v(16, 4, 20, 4096, 3584, glu=False) == 6


@pytest.mark.gpu
@pytest.mark.parametrize("T,act", [(4, "silu"), (24, "silu"), (128, "silu"), (64, "relu2")])
def test_experts_at_any_address(hipk, T, act):
    """Rows or weights that start off 16 bytes, at sizes that the ring of LDS pieces takes otherwise: the form that
    streams into registers takes them, within the tolerance of the tests above."""
    E, k, H, I = 16, 4, 2048, 1792
    g = torch.Generator(device="cuda").manual_seed(T)

    def at(off, scale, *shape):
        n = torch.Size(shape).numel()
        flat = torch.randn(n + 8, device="cuda", generator=g).mul_(scale).to(torch.bfloat16)
        return flat[off:off + n].view(shape)

    lg = torch.randn(T, E, device="cuda", generator=g).to(torch.bfloat16)
    n_in = I if act == "relu2" else 2 * I
    for ox, oi, oo in ((3, 0, 0), (0, 5, 0), (0, 0, 1), (0, 0, 0)):
        x, w_in, w_out = at(ox, 1.0, T, H), at(oi, 0.02, E, n_in, H), at(oo, 0.02, E, H, I)
        got, want = ops.fused_moe(x, lg, w_in, w_out, k, act).double(), ops.fused_moe_ref(x, lg, w_in, w_out, k, act).double()
        assert (got - want).norm() <= 1e-2 * want.norm()


def test_medium_m_cuts_fill_the_chip_once():
    """The K slices that the medium-M kernel takes by itself: one workgroup to a CU, all of whose LDS its ring takes."""
    for M in (17, 64, 128, 129, 256):
        for N, K in ((4096, 4096), (4096, 14336), (6144, 4096), (8192, 28672), (2048, 16384), (65536, 4096)):
            s = G.midm_splits(M, N, K)
            assert K % (256 * s) == 0 and (s == 1 or N // 128 * s <= 256)
    assert G.midm_splits(64, 4096, 4096) == 8 and G.midm_splits(64, 8192, 28672) == 4


def test_medium_m_entries_decide():
    """The tuning table's medium-M cuts: shapes that no rule ahead of the table takes, at most a workgroup to a CU,
    whole K tiles to a slice, faster than what the table has otherwise."""
    seen = 0
    for entries in G.load_table().values():
        for key, e in entries.items():
            cut = e.get("midm")
            if not cut:
                continue
            M, N, K, ldx = (int(v) for v in key.split(","))
            nf, s = cut // 100 or 4, cut % 100
            assert G.midm_supported(M, N, K) and N % (32 * nf) == 0 and nf in (2, 4) and 1 <= s <= K // 64
            assert N // (32 * nf) * s <= 256, key
            assert not (G.wide_form(M, N, K) or G.small_form(M, N, K) or G.brief_ok(M, N, K) or e.get("xd")), key
            assert e["midm_us"] < e["midm_base_us"]
            seen += 1
    assert seen


def test_prompts_ask_once(monkeypatch):
    """What a prompt's products ask for on the host: no K slices above the rows that they take, and a shape's tile once."""
    asked = []
    real = G._gpu_bf16
    monkeypatch.setattr(G, "_gpu_bf16", lambda x, w: asked.append(x.shape[0]) or real(x, w))
    w = torch.randn(64, 128)
    for rows in (G.MIDM_MAX_M + 1, 1000):
        x = torch.randn(rows, 128)
        assert torch.equal(ops.linear_parts(x, w), ops.linear(x, w))
    assert len(asked) == 4
    supported = G.xd_supported
    monkeypatch.setattr(G, "xd_supported", lambda *a: asked.append(a) or supported(*a))
    first, n = G.xd_default_form(397, 2048, 2048, True), len(asked)
    assert n > 4 and G.xd_default_form(397, 2048, 2048, True) == first and len(asked) == n


def test_short_k_rule():
    """Short K stays with the library's pick where many rows lose: above 64, wide products 128, but for shapes
    whose tuned solution is slower."""
    for M, N, K in ((17, 1024, 64), (64, 1024, 256), (64, 8192, 64), (112, 6144, 128), (128, 3072, 192), (128, 8192, 256)):
        assert G.brief_ok(M, N, K) and G.brief_pays(M, N, K, False) and G._resolve(M, N, K, K) == ("midm", 201)
    for M, N, K in ((65, 1024, 128), (128, 1024, 256), (112, 2048, 192), (160, 4096, 192), (200, 8192, 128), (256, 1536, 128)):
        assert G.brief_ok(M, N, K) and not G.brief_pays(M, N, K, False) and G.brief_pays(M, N, K, True)
        assert G._resolve(M, N, K, K) == ("torch", 0)  # (no such shape in the table)


def test_small_products_rule():
    """Which products the 64-row tiles take: at most a workgroup a CU of their tiles, long K on more than half of
    them."""
    forms = {(M, N, K): G.small_form(M, N, K) for M in (16, 17, 32, 64, 100, 128, 224, 256, 257)
             for N in (1024, 2048, 3584, 6144, 8448, 32000) for K in (1984, 2048, 4096, 4160)}
    assert not any(f for (M, N, K), f in forms.items() if M in (16, 257) or N in (1024, 32000) or K in (1984, 4160))
    assert forms[64, 3584, 2048] == 11 and forms[224, 3584, 2048] == 21 and forms[224, 2048, 2048] == 11
    assert forms[64, 6144, 4096] == 1011 and forms[100, 6144, 4096] == 21 and forms[128, 6144, 4096] == 0
    assert forms[32, 8448, 2048] == 0 and forms[64, 8448, 2048] == 1021 and forms[224, 8448, 2048] == 0
    assert forms[64, 2048, 4096] == 0 and forms[128, 8448, 2048] == 0


def test_dot2_rule():
    """One and two rows from 2^25 weights on, K in whole waves and N in whole rows of them; rows 16 bytes apart."""
    assert G.dot2_ok(1, 8192, 4096, 4096) and G.dot2_ok(2, 65536, 512, 520)
    for M, N, K, ldx in ((3, 8192, 4096, 4096), (2, 8188, 4096, 4096), (2, 65538, 512, 512), (1, 32768, 1088, 1088),
                         (2, 8192, 4096, 4100)):
        assert not G.dot2_ok(M, N, K, ldx)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2])
@pytest.mark.parametrize("N,K", [(8192, 4096), (65540, 512), (16388, 2048), (2624, 12800)])
def test_dot2_rule_products(hipk, M, N, K):
    """The rule's products, and one row's with its norm, against fp32: twice the 2^-9 of a bf16 result, and fp32 sums;
    with the norm its bf16 rows too (2^-9 of every product, signs at random: of the products' norm, 12 deviations)."""
    g = torch.Generator(device="cuda").manual_seed(N + M)
    x, w = (torch.randn(*s, device="cuda", generator=g).bfloat16() for s in ((M, K), (N, K)))
    assert G.route(M, N, K, K) == ("skinny", 1)
    want = x.float() @ w.float().T
    assert ((ops.linear(x, w).float() - want).abs() <= 2 ** -8 * want.abs() + 1e-6 * K).all()
    if K > 8192:  # no norm of such rows
        return
    nw = torch.rand(K, device="cuda", generator=g).bfloat16()
    y = ops.norm_linear(ops.PendingNorm(x, None, nw, 1e-5, False), w).float()
    xf = x.float()
    n = xf * (xf.pow(2).mean(-1, keepdim=True) + 1e-5).rsqrt() * nw.float()
    want = n @ w.float().T
    assert ((y - want).abs() <= 2 ** -8 * want.abs() + 6 * 2 ** -8 * (n.pow(2) @ w.float().pow(2).T).sqrt()).all()
