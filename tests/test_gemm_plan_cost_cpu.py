"""Estimated tile plans (gemm.hip cake_gemm_plan): what they pick can run, at every size."""
import random

import pytest
import torch

from cake_amd.build import GEMM_LIB

pytestmark = pytest.mark.skipif(not GEMM_LIB.exists(), reason="native libraries not built")


def test_estimated_plans_can_run():
    from cake_amd.ops import gemm as G
    rng = random.Random(4)
    epis = list(G.EPI)
    for _ in range(3000):
        M = int(2 ** rng.uniform(0, 17))
        Nv = 32 * int(2 ** rng.uniform(0, 12))
        K = 8 * int(2 ** rng.uniform(0, 13))
        epi, big = rng.choice(epis), rng.random() < 0.2
        cfg, splits = G.resolve(M, Nv, K, epi, big)
        assert cfg in G.CFG_TILES and 1 <= splits <= 16
        if cfg in G.K64_ONLY:
            assert K % 64 == 0 and not big
        if epi in ("swiglu", "geglu"):
            assert cfg not in G.NO_GATED
        if splits > 1:
            assert -(-K // 64) // splits >= 4


def test_measured_entry_of_the_size_stands_unless_well_behind(monkeypatch):
    from cake_amd.ops import gemm as G

    def at(cfg, splits):
        monkeypatch.setattr(G, "_TUNED", [{"M": 2048, "Nv": 4096, "K": 4096, "epi": "store",
                                           "cfg": cfg, "splits": splits}])
        monkeypatch.setattr(G, "_resolved", {})
        return G.resolve(2048, 4096, 4096, "store", False)
    assert at(27, 1) == (27, 1)     # close to the best estimate
    assert at(13, 1) != (13, 1)     # 64 x 64 tiles of a large product
    assert at(20, 1) == (20, 1)     # a tile the estimate does not cover


@pytest.mark.parametrize("size,times", [
    # us of the tiles (unsplit) on an MI355X: the estimate's choice is within a tenth of the best
    ((12288, 320, 320, "add16"), {14: 11.6, 4: 11.8, 1: 13.0, 13: 13.2, 8: 13.4, 27: 18.4}),
    ((7040, 640, 640, "add16"), {14: 16.3, 6: 18.7, 8: 19.0, 4: 20.6, 27: 21.5}),
    ((7040, 640, 2560, "add16"), {14: 37.4, 6: 41.8, 27: 43.8, 8: 45.2}),
    ((18432, 2560, 320, "geglu"), {5: 53.9, 22: 57.5, 8: 60.8, 26: 63.5, 27: 64.3}),
    ((3200, 2560, 320, "geglu"), {27: 12.6, 8: 12.7, 12: 16.4, 4: 17.1, 26: 17.2}),
    ((800, 5120, 640, "geglu"), {6: 15.1, 8: 15.2, 27: 15.6, 4: 17.5, 26: 20.0}),
    ((18432, 960, 320, "store"), {8: 29.1, 14: 29.1, 26: 30.6, 6: 32.7, 27: 32.8, 12: 34.7}),
    ((113, 57344, 8192, "swiglu"), {27: 193.0, 8: 204.7, 7: 209.5, 22: 221.2})], ids=str)
def test_estimate_picks_a_measured_best(monkeypatch, size, times):
    """Short products, residual and GEGLU epilogues, and tiles that all wait for the weights."""
    from cake_amd.ops import gemm as G
    monkeypatch.setattr(G, "_TUNED", [])
    monkeypatch.setattr(G, "_resolved", {})
    cfg, splits = G.resolve(*size)
    assert splits == 1 and times[cfg] <= 1.1 * min(times.values())


@pytest.mark.parametrize("size,times", [
    # us of (tile, splits) on an MI355X, the fastest and some that an estimate has taken for them
    ((6000, 57344, 8192, "swiglu"), {(22, 1): 3969, (25, 1): 4188, (33, 1): 4252}),
    ((1800, 57344, 8192, "swiglu"), {(22, 1): 1275, (25, 1): 1306, (31, 2): 1354, (32, 1): 1393}),
    ((3000, 10240, 8192, "store"), {(22, 1): 353, (31, 1): 374, (33, 1): 380}),
    ((6000, 10240, 8192, "store"), {(22, 1): 746, (31, 1): 762, (33, 1): 775}),
    ((1600, 8192, 8192, "resid32"), {(35, 1): 172.5, (22, 1): 178.8, (31, 4): 193.6}),
    ((100, 57344, 8192, "swiglu"), {(27, 1): 169.5, (31, 1): 170.6, (28, 1): 179.2, (7, 1): 181.8}),
    ((260, 4096, 14336, "resid32"), {(6, 4): 58.6, (28, 2): 59.7, (30, 4): 65.4}),
    ((350, 2048, 11776, "resid32"), {(6, 8): 34.9, (7, 4): 38.0, (28, 4): 42.2}),
    ((560, 1024, 4096, "resid32"), {(18, 4): 17.0, (7, 4): 18.8, (13, 1): 21.7}),
    ((113, 16384, 2048, "swiglu"), {(12, 1): 21.9, (13, 1): 22.8, (28, 1): 24.2}),
    ((512, 5120, 1280, "gelu"), {(18, 1): 17.9, (28, 1): 19.2, (7, 1): 20.5}),
    ((1200, 5120, 1280, "gelu"), {(6, 1): 27.2, (32, 1): 27.6, (27, 1): 28.9})], ids=str)
def test_estimate_picks_a_measured_best_of_all_splits(monkeypatch, size, times):
    """Prompts of wide models, tiles that wait for the weights, short k: within 4 % of the best."""
    from cake_amd.ops import gemm as G
    monkeypatch.setattr(G, "_TUNED", [])
    monkeypatch.setattr(G, "_resolved", {})
    assert times[G.resolve(*size)] <= 1.04 * min(times.values())


@pytest.mark.parametrize("M,Nv", [(3072, 57344), (2500, 57344), (1024, 28672), (1024, 14336)])
def test_measured_eight_wave_tiles_behind_the_four_wave_ones(monkeypatch, M, Nv):
    """3072 x 57344 x 8192 SwiGLU on 256 x 256: eight waves 2326 us, four 2056; 2500 rows 1902, 1688."""
    from cake_amd.ops import gemm as G
    monkeypatch.setattr(G, "_TUNED", [{"M": M, "Nv": Nv, "K": 8192, "epi": "swiglu", "cfg": 5, "splits": 1}])
    monkeypatch.setattr(G, "_resolved", {})
    assert G.resolve(M, Nv, 8192, "swiglu")[0] == 22


def test_library_plan_falls_back_to_the_plan_without_it(monkeypatch):
    """A call that the library form does not carry (a bias) runs what a table without the library's
    entries plans, as the native engines do, not the nearest measured size."""
    from cake_amd.ops import gemm as G
    near = {"M": 1000, "Nv": 4096, "K": 4096, "epi": "store", "cfg": 13, "splits": 4}
    lib = {**near, "M": 1100, "cfg": G.LIB, "splits": 1}
    monkeypatch.setattr(G, "_TUNED", [near])
    monkeypatch.setattr(G, "_resolved", {})
    want = G.resolve(1100, 4096, 4096, "store")
    assert want[0] != 13
    monkeypatch.setattr(G, "_TUNED", [near, lib])
    monkeypatch.setattr(G, "_resolved", {})
    assert G.resolve(1100, 4096, 4096, "store") == (G.LIB, 1)
    assert G.resolve(1100, 4096, 4096, "store", mfma_only=True) == want
    monkeypatch.setattr(G, "_plans", {(1100, 4096, 4096, "store"): (G.LIB, 1)})
    assert G.resolve(1100, 4096, 4096, "store", mfma_only=True) == want


def test_workspace_covers_the_pieces():
    """Tiles in pieces need a slab each; whole tiles need none."""
    from cake_amd.ops import gemm as G
    L = G._lib()
    assert L.cake_gemm_ws_floats(22, 4, 777, 4096, 14336, 0) == 64 * 4 * 256 * 256
    assert L.cake_gemm_ws_floats(25, 8, 4500, 4096, 14336, 0) == 32 * 8 * 256 * 256   # 288 tiles
    assert L.cake_gemm_ws_floats(27, 2, 1100, 4096, 14336, 0) == 0                     # 144 tiles
    assert L.cake_gemm_ws_floats(22, 2, 2048, 8192, 8192, 0) == 0                      # one wave


@pytest.mark.skipif(torch.cuda.is_available(), reason="makes launches without operands")
@pytest.mark.parametrize("cfg,splits,M", [(22, 4, 777), (27, 2, 129)])
def test_pieces_take_the_callers_counters(cfg, splits, M):
    """Tiles in pieces need the workspace and the counters of the caller's stream: refused without
    either; with both, and whole tiles without, the call ends at its launch (no device)."""
    from cake_amd.ops import gemm as G
    L, invalid = G._lib(), 1

    def call(splits, ws, tick):
        return L.cake_gemm_scaled(0, 0, cfg, splits, 64, 4096, 64, 4096, 64, 4096, None, None, 0, ws,
                                  tick, 64, M, 4096, 4096, 1.0, None)
    assert call(splits, 64, 64) not in (0, invalid) and call(1, None, None) not in (0, invalid)
    assert call(splits, None, 64) == invalid and call(splits, 64, None) == invalid
    assert 0 < L.cake_gemm_ticks() <= L.cake_gemm_rows_ticks()


def test_workspaces_are_of_a_stream_or_of_a_graph(monkeypatch):
    """An eager launch takes its stream's slabs, of the newest 16 streams; a captured one slabs of
    its own, which nothing but the graph keeps (graphs share PyTorch's capture stream, and may be
    replayed side by side)."""
    from types import SimpleNamespace

    from cake_amd.ops import gemm as G
    state = SimpleNamespace(stream=1, capturing=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: SimpleNamespace(cuda_stream=state.stream))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state.capturing)
    monkeypatch.setattr(G, "_ws", {})
    dev = torch.device("cpu")
    first = G._workspace(dev, 100)
    assert G._workspace(dev, 50) is first
    state.capturing = True
    a, b = G._workspace(dev, 100), G._workspace(dev, 100)
    assert a.numel() >= 100 and len({t.data_ptr() for t in (first, a, b)}) == 3
    state.capturing = False
    assert G._workspace(dev, 100) is first and len(G._ws) == 1
    grown = G._workspace(dev, first.numel() + 1)
    assert grown is not first and list(G._ws.values()) == [grown]
    for state.stream in range(2, 40):
        assert G._workspace(dev, 100) is not grown
    assert len(G._ws) == 16
