"""CPU checks of the decode-GEMM router's gemm_xd forms and of the in-tree tuning table
(ops/gemm.py; no GPU work: forms are parsed and shape-checked on the host)."""
import json
import types

import pytest
import torch

from drtc_amd.ops import gemm as G


def test_xd_form_parsing():
    assert G.xd_form(244) == (2, 4, 4) and not G.xd_nt(244)
    assert G.xd_form(1244) == (2, 4, 4) and G.xd_nt(1244)
    assert G.xd_form(1281) == (2, 8, 1)


def test_nontemporal_forms_only_for_built_tiles():
    assert G.xd_supported(256, 8192, 28672, 1244)
    assert G.xd_supported(256, 28672, 8192, 1281, glu=True)
    assert not G.xd_supported(256, 1536, 2048, 1121)  # 128 x 64: no non-temporal build
    assert not G.xd_supported(256, 1536, 2048, 2244)  # not a form


@pytest.mark.parametrize("M,N,K,glu,want", [
    (129, 14336, 4096, True, 1341), (160, 14336, 4096, True, 1341), (161, 14336, 4096, True, 1441), (193, 14336, 4096, True, 1541),
    (224, 32000, 2048, False, 1541), (160, 7168, 2048, True, 1321), (161, 7168, 2048, True, 0), (128, 32000, 4096, False, 0),
    (225, 32000, 4096, False, 0), (160, 28672, 4096, True, 0), (160, 32000, 1024, False, 0), (160, 8448, 2048, False, 0),
    (160, 32016, 4096, False, 0),
    (148, 6656, 5120, True, 0), (148, 6656, 4096, True, 1321), (148, 13312, 3072, False, 0), (148, 13312, 11008, False, 1321),
    (148, 25600, 5120, False, 1341),  # tiles of 128 columns at any K
])
def test_tall_tiles_rule(monkeypatch, M, N, K, glu, want):
    monkeypatch.setattr(G, "_xd_nt", True)
    monkeypatch.setattr(G, "_xd_enabled", True)
    assert G.tall_form(M, N, K, glu) == want
    if want:
        assert not G.xd_supported(G.XD_ROWS[want // 100 % 10] + 1, N, K, want, glu)  # one row tile
        assert not G.xd_supported(M, N, K, want - 1000, glu) and not G.xd_supported(M, N, K, want + 1, glu)


@pytest.mark.parametrize("N,K", [(2048, 7168), (2048, 14336), (1024, 5632), (4096, 8192), (3072, 5696), (2080, 7168)])
def test_deep_products_rule(monkeypatch, N, K):
    monkeypatch.setattr(G, "_xd_enabled", True)
    for M in (257, 300, 512, 640, 641, 768, 769, 1024):
        form = G.deep_form(M, N, K)
        if 640 < M <= 768 and N >= 4096 or N == 2080 and not form:  # the library; no whole tiles
            assert form == 0
            continue
        mt, nf, sk = G.xd_form(form)
        assert sk > 1 and G.xd_supported(M, N, K, form)
        assert 100 <= -(-M // G.XD_ROWS[mt]) * (N // (32 * nf)) * sk <= 256  # a workgroup a CU
    assert not G.deep_form(256, N, K) and not G.deep_form(1025, N, K) and not G.deep_form(512, N, 5568)


@pytest.mark.parametrize("M,N,K,want", [
    (256, 6656, 2048, 121), (448, 6656, 2048, 141), (1024, 6656, 2048, 241), (2048, 3072, 2048, 161), (300, 12800, 4096, 241),
    (256, 25600, 4096, 1241),                   # one row tile: weights past the caches
    (129, 4096, 512, 121), (1024, 4096, 512, 141), (192, 8192, 512, 121),
    (640, 6656, 2048, 0), (128, 12800, 4096, 0), (3073, 3072, 2048, 0), (300, 6640, 2048, 0), (256, 4096, 256, 0),
    (261, 12800, 12800, 0), (383, 12800, 7232, 0), (384, 12800, 7232, 241), (261, 12800, 7168, 241),  # rows of the tiles used
    (160, 6656, 12288, 121), (161, 14336, 8192, 0), (192, 14336, 8192, 141),
    (614, 13824, 4096, 0), (615, 13824, 4096, 261), (520, 13824, 1536, 261),
    (2049, 768, 8192, 0), (2049, 768, 3072, 121), (1100, 1536, 8192, 121),  # tiles of 64 columns
])
def test_full_round_rule(monkeypatch, M, N, K, want):
    monkeypatch.setattr(G, "_xd_nt", True)
    monkeypatch.setattr(G, "_xd_enabled", True)
    assert G.full_form(M, N, K) == want
    if want:
        assert G.xd_supported(M, N, K, want) and G.xd_form(want)[2] == 1


@pytest.mark.parametrize("M,I,K,want", [
    (513, 7168, 2048, 281), (639, 7168, 2048, 281), (512, 7168, 2048, 241), (600, 5632, 2048, 0), (600, 7168, 2112, 0),
    (600, 14336, 2048, 0), (769, 7168, 4096, 281), (1024, 7168, 4096, 281), (640, 8192, 4096, 281), (1024, 8320, 4096, 0),
    (1024, 5632, 4096, 281), (910, 8192, 1024, 0), (910, 8192, 1728, 0), (910, 8192, 1792, 281), (560, 8192, 1024, 281),
])
@pytest.mark.parametrize("act", ["silu", "clamped"])
def test_gated_tiles_of_one_round(monkeypatch, M, I, K, want, act):
    monkeypatch.setattr(G, "_xd_enabled", True)
    monkeypatch.setattr(G, "_activate", lambda: {})
    assert G.glu_form(M, 2 * I, K, K, act) == want


@pytest.mark.parametrize("M,form,want", [
    (256, 244, 1244),   # one 256-row tile: every weight byte read once
    (128, 141, 1141),
    (160, 141, 141),    # two 128-row tiles share the weight panel through L2
    (1024, 281, 281),
    (256, 121, 121),    # 128 x 64 tile: no non-temporal build
    (256, 1243, 1243),  # tuned non-temporal form: as tuned
    (512, 0, 0),
])
def test_router_policy_picks_nontemporal_twin(monkeypatch, M, form, want):
    monkeypatch.setattr(G, "_xd_nt", True)
    monkeypatch.setattr(G, "_xd_enabled", True)
    assert G._xd_policy(M, form) == want
    monkeypatch.setattr(G, "_xd_nt", False)
    assert G._xd_policy(M, form) == form % 1000  # DRTC_XD_NT=0: every form plain
    monkeypatch.setattr(G, "_xd_enabled", False)
    assert G._xd_policy(M, form) == 0


def test_router_keeps_nt_tuned_plain_winner(monkeypatch):
    """An entry the nt-aware re-tune measured (profiles/r4ab: Llama-3-8B gate_up at M = 160-256
    picked plain 241 over 1241) runs exactly its pick; its nt picks stay nt unless
    DRTC_XD_NT=0; the committed table marks those entries."""
    monkeypatch.setattr(G, "_xd_enabled", True)
    monkeypatch.setattr(G, "_xd_nt", True)
    assert G._xd_policy(160, 241, nt_tuned=True) == 241
    assert G._xd_policy(160, 241, nt_tuned=False) == 1241
    assert G._xd_policy(256, 1244, nt_tuned=True) == 1244
    monkeypatch.setattr(G, "_xd_nt", False)
    assert G._xd_policy(256, 1244, nt_tuned=True) == 244
    with open(G.table_path()) as f:
        data = json.load(f)
    e = next(iter(data.values()))["160,28672,4096,4096"]
    assert e["xd"] == 241 and e["nt_tuned"]


def test_every_tuned_xd_form_fits_its_shape():
    """Each xd / xd_glu entry of the committed table names a built form that takes its own
    shape (what the router would run, including the non-temporal twin)."""
    with open(G.table_path()) as f:
        data = json.load(f)
    n = 0
    for entries in data.values():
        for key, e in entries.items():
            M, N, K, _ = (int(v) for v in key.split(","))
            if e.get("xd"):
                n += 1
                assert G.xd_supported(M, N, K, e["xd"]), (key, e["xd"])
                assert G.xd_supported(M, N, K, G._xd_policy(M, e["xd"]) or e["xd"]), key
            if e.get("xd_glu"):
                n += 1
                assert N % 2 == 0
                assert G.xd_supported(M, N // 2, K, e["xd_glu"], glu=True), (key, e["xd_glu"])
    assert n > 100


def test_gemma_2048_decode_shapes_carry_a_gemm_xd_form():
    """Gemma-2B's 2,048-row decode batch (above the 1,024 decode buckets): the tuned table
    gives its qkv / o / down shapes a gemm_xd form next to their prefill library entries
    (profiles/r6ak), and every such form fits its shape."""
    tab = json.load(open(G.table_path()))
    for ver, ents in tab.items():
        for k, want in (("2048,2560,2048,2048", 241), ("2048,2048,2048,2048", 141),
                        ("2048,2048,16384,16384", 242)):
            e = ents.get(k)
            if e is None:
                continue
            assert e.get("prefill") and e["xd"] == want
            M, N, K, _ = (int(v) for v in k.split(","))
            assert G.xd_supported(M, N, K, want)


@pytest.mark.parametrize("M,N,want", [
    (8159, 1024, ("w4", 0)), (7680, 1024, ("w4", 0)), (7424, 1024, ("xd", 241)), (7936, 1024, ("xd", 241)), (7168, 1024, ("xd", 241)),
    (16384, 512, ("w4", 0)), (16384, 256, ("xd", 141)), (10000, 768, ("w4", 0)), (10400, 768, ("xd", 241)), (4096, 2048, ("xd", 241)),
    (6100, 1280, ("xd", 241)), (9000, 2048, ("w4", 0)),
])
def test_half_a_round_of_large_tiles(monkeypatch, M, N, want):
    monkeypatch.setattr(G, "_xd_enabled", True)
    assert G._resolve(M, N, 4096, 4096) == want


@pytest.mark.parametrize("op,M,N,K", [("squared_relu", 256, 25600, 4096), ("gated", 513, 14336, 2048), ("gated", 160, 25600, 2048)])
@pytest.mark.parametrize("stride", [1 << 22, 4104])
def test_rows_far_apart_stay_with_the_library(monkeypatch, op, M, N, K, stride):
    """gemm_xd's tiles of 256 rows have 32-bit offsets; the products with something behind them keep ``linear``'s bound."""
    monkeypatch.setattr(G, "on_gpu", lambda t: True)
    monkeypatch.setattr(G, "_activate", lambda: {})
    monkeypatch.setattr(G, "_prefill_algo", lambda *a: -1)
    monkeypatch.setattr(G, "_routes", {})
    monkeypatch.setattr(G, "hipk", lambda: types.SimpleNamespace(relu2=lambda *a: 0))
    monkeypatch.setattr(G, "stream_ptr", lambda t: 0)
    monkeypatch.setattr("drtc_amd.ops.activation.act_glu", lambda y, act, limit=0.0: y)
    taken = []
    monkeypatch.setattr(G, "xd_gemm", lambda *a, **k: taken.append("xd"))
    monkeypatch.setattr(G.F, "linear", lambda x, w: taken.append("library") or torch.empty(1, dtype=x.dtype))
    x = torch.empty((M - 1) * stride + K, dtype=torch.bfloat16).as_strided((M, K), (stride, 1))
    w = torch.empty(N, K, dtype=torch.bfloat16)
    G.squared_relu(x, w, torch.empty(M, N, dtype=torch.bfloat16)) if op == "squared_relu" else G.gated(x, w)
    assert taken == ["library" if stride == 1 << 22 else "xd"]


@pytest.mark.parametrize("M,N,K", [(1, 2048, 4096), (16, 2048, 4096), (300, 2048, 5632), (256, 6656, 2048), (129, 25600, 2048)])
@pytest.mark.parametrize("less", [64, -64])
def test_widths_that_differ_are_refused(monkeypatch, M, N, K, less):
    """Ahead of every kernel, which would take the rows of W for K apart and K long."""
    monkeypatch.setattr(G, "on_gpu", lambda t: True)
    monkeypatch.setattr(G, "_activate", lambda: {})
    monkeypatch.setattr(G, "_prefill_algo", lambda *a: -1)
    monkeypatch.setattr(G, "_routes", {})
    monkeypatch.setattr(G, "hipk", lambda: pytest.fail("a kernel took it"))
    monkeypatch.setattr(G, "stream_ptr", lambda t: 0)
    x, w, wrong = (torch.empty(n, k, dtype=torch.bfloat16) for n, k in ((M, K), (N, K), (N, K - less)))
    out = torch.empty(M, N, dtype=torch.bfloat16)
    for call in (lambda: G.linear(x, wrong), lambda: G.squared_relu(x, wrong, out), lambda: G.linear_parts(x, wrong),
                 lambda: G.linear_beside(x, wrong, x, wrong)):
        with pytest.raises(RuntimeError, match="shapes cannot be multiplied"):
            call()
    if M <= 16:
        monkeypatch.setattr(G, "hipk", lambda: types.SimpleNamespace(skinny_gemm=lambda *a: 0 if a[15] == 0 else pytest.fail("both")))
        with pytest.raises(RuntimeError, match="shapes cannot be multiplied"):
            G.linear_beside(x, w, x, wrong)


@pytest.mark.parametrize("K", [128, 192])
def test_rows_by_a_list_want_four_k_tiles(K):
    """Fewer, and a tile's row indexes would be read ahead of the first wait that covers them.  (Refused on the host.)"""
    from drtc_amd.ops._ext import hipk

    N, rows, p = 512, 600, 1 << 20
    args = (p, p, p, p, 2, rows, N, K, K, K, N, 2 * N * K, G.EPI["silu"], N, 4, 1, 0, 0.0, 0, p, rows)
    assert hipk().gemm_grouped(*args) == -1


@pytest.mark.parametrize("T,k,E,H,I,glu,want", [
    (3664, 2, 16, 1024, 3584, False, 4), (7490, 2, 32, 512, 3584, False, 4), (7141, 1, 16, 1024, 3584, True, 4),  # 208 / 151, ... us in 128 rows
    (2367, 3, 16, 1024, 1792, False, 4), (3200, 4, 32, 2048, 7168, True, 4),
    (1408, 4, 20, 2048, 1792, False, 3), (1152, 4, 16, 4096, 3584, True, 3), (2048, 4, 16, 4096, 3584, True, 4), (4096, 4, 16, 4096, 3584, True, 4),
])
def test_rows_to_an_experts_tile(T, k, E, H, I, glu, want):
    """128 rows (variant 3) where both estimates of a layer's time say so, 256 (4) elsewhere."""
    from drtc_amd.ops._ext import hipk

    assert hipk().moe_variant(T, T * k, E, H, I, glu, True) == want


def test_few_rows_ways_up_add_up_their_splits():
    """Two vectors of the rows to a thread, 64 KB of splits."""
    from drtc_amd.ops._ext import hipk

    take = lambda *a: hipk().latent_up_merges(*a)
    assert take(1, 512, 2) and take(1, 512, 32) and take(4, 512, 8) and take(8, 256, 8) and take(16, 128, 8)
    assert not (take(5, 512, 2) or take(16, 512, 2) or take(9, 256, 4) or take(16, 256, 4) or take(1, 512, 33) or take(17, 64, 2))
