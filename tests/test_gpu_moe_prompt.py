"""The whole-prompt expert launches (esp_grouped_prompt over esp_group_tiles' list): windows' tokens bit for bit those of the
32-row window launches, at K splits of 4, 6 and 8 steps, tiles of 32 and 64 members, one to four row groups."""
import pytest
import torch

from vllm_espalier import experts as G
from vllm_espalier import workloads as WL

pytestmark = pytest.mark.gpu

# (D, I, routed experts, shared, k): K splits of 8 / 4 steps, of 12 / 6, of 4 / 6; a layer of few experts, many members
SHAPES = {
    "wide": (1024, 512, 24, True, 4),
    "odd": (768, 768, 9, False, 2),
    "narrow": (512, 384, 6, True, 3),
}
GRIDS = {1: "e2m1", 2: "e2m1", 3: "int5", 4: "mcg", 5: "int6", 8: "mcg"}


def _layer(shape, dev, seed=2):
    D, I, E, shared, k = SHAPES[shape]
    gen = torch.Generator().manual_seed(seed)
    bits = [1, 2, 3, 4, 5, 8]
    mats = [tuple(WL.matrix(K, N, b, GRIDS[b], gen, dev) for K, N in ((D, I), (D, I), (I, D)))
            for b in (bits[e % 6] for e in range(E))]
    sh = tuple(WL.matrix(K, N, 4, "int5", gen, dev) for K, N in ((D, I), (D, I), (I, D))) if shared else None
    gw = (torch.randn((D,), generator=gen) * 0.05).to(torch.bfloat16).to(dev) if shared else None
    router = (torch.randn((E, D), generator=gen) * 0.05).to(torch.bfloat16).to(dev)
    L = G.prepare(mats, sh, gw)
    return L, router, k, G.Scratch(L.E, L.D, L.I, 32, k + shared, dev)


def _x(T, D, dev, seed):
    return torch.randn((T, D), generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16).to(dev)


def _by_window(x, pick, wts, L, s, k, gate):
    outs = [G.windows(x[r:r + 32], None if pick is None else pick[r:r + 32], None if wts is None else wts[r:r + 32], L, s,
                      k=k, gate=gate) for r in range(0, x.shape[0], 32)]
    return tuple(None if o[0] is None else torch.cat(o) for o in zip(*outs))


def _same(a, b):
    for u, v in zip(a, b):
        assert (u is None) == (v is None)
        assert u is None or torch.equal(u, v)


@pytest.mark.parametrize("rows", [32, 64])
@pytest.mark.parametrize("T", [33, 100, 300])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_windows_whole_prompt_equals_windows(dev, monkeypatch, shape, T, rows):
    monkeypatch.setattr(G, "tile_rows", lambda *a: rows)
    L, router, k, s = _layer(shape, dev)
    x = _x(T, L.D, dev, T)
    want = _by_window(x, None, None, L, s, k, router)
    assert s.prompt is None
    _same(G.windows(x, None, None, L, s, k=k, gate=router), want)
    assert s.prompt is not None
    G.check_status()


@pytest.mark.parametrize("plan", ["8,4", "16,4", "4,4;8,4", "8,4;4,4"])
def test_windows_keep_decode_bits_under_a_forced_plan(dev, monkeypatch, plan):
    """A forced plan of 8 or 16 waves sums several k slots a split: a prompt's tokens, a window's and those of one to four
    rows still have the same bits."""
    monkeypatch.setenv("ESPALIER_GROUPED_TILE_PLAN", plan)
    L, router, k, s = _layer("wide", dev)
    x = _x(70, L.D, dev, 11)
    want = _by_window(x, None, None, L, s, k, router)
    _same(G.windows(x, None, None, L, s, k=k, gate=router), want)
    for n in (1, 3, 4, 5):
        _same(G.windows(x[:n], None, None, L, s, k=k, gate=router), [t[:n] for t in want])


def test_windows_given_picks_and_chunks(dev, monkeypatch):
    """vLLM's picks handed in, and a prompt of several passes."""
    monkeypatch.setattr(G, "WINDOWS_PROMPT_ROWS", 64)
    L, _, k, s = _layer("wide", dev)
    T = 150
    gen = torch.Generator().manual_seed(1)
    x = _x(T, L.D, dev, 4)
    pick = torch.stack([torch.randperm(L.E - 1, generator=gen)[:k] for _ in range(T)]).to(torch.int32).to(dev)
    wts = torch.rand((T, k), generator=gen).to(dev)
    _same(G.windows(x, pick, wts, L, s, k=k), _by_window(x, pick, wts, L, s, k, None))


@pytest.mark.parametrize("rows", [32, 64])
def test_windows_of_no_finite_values(dev, monkeypatch, rows):
    """Tokens of infinities, NaN and overflow on the way among ordinary ones: NaN where the window launches give NaN, their
    bits elsewhere, the other tokens' and the signs of zeros included."""
    monkeypatch.setattr(G, "tile_rows", lambda *a: rows)
    L, router, k, s = _layer("wide", dev)
    x = _x(120, L.D, dev, 15)
    x[7, 3], x[40, L.D // 2], x[41, L.D - 1] = float("inf"), float("nan"), float("-inf")
    x[42] = torch.finfo(x.dtype).max
    x[100] = 0.0
    want = _by_window(x, None, None, L, s, k, router)
    for got, w in zip(G.windows(x, None, None, L, s, k=k, gate=router), want):
        nan = torch.isnan(w)
        assert bool(nan.any()) and not bool(nan[100].any()) and torch.equal(torch.isnan(got), nan)
        assert torch.equal(got.view(torch.int16)[~nan], w.view(torch.int16)[~nan])


def test_windows_rows_of_8_bytes_alignment(dev):
    """Rows that route_rows does not take (8-byte aligned) still run, as windows."""
    L, router, k, s = _layer("narrow", dev)
    x = _x(70, L.D + 4, dev, 6)[:, 4:]
    assert not G._whole_prompt(x, L, router)
    _same(G.windows(x, None, None, L, s, k=k, gate=router), _by_window(x, None, None, L, s, k, router))
    assert s.prompt is None


def test_windows_graph_outlives_a_longer_prompt(dev):
    """A captured prompt keeps its scratch when a longer prompt outgrows it."""
    L, router, k, s = _layer("wide", dev)
    x = _x(50, L.D, dev, 7)
    want = G.windows(x, None, None, L, s, k=k, gate=router)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        got = G.windows(x, None, None, L, s, k=k, gate=router)
    first = s.prompt
    G.windows(_x(400, L.D, dev, 8), None, None, L, s, k=k, gate=router)
    assert s.prompt is not first and s.kept == [first]
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
        _same(got, want)
        torch.randn((256, 256), device=dev).sum()             # eager work between replays


@pytest.mark.parametrize("mode", ["windows", "prefill"])
def test_outgrown_prompt_scratch_outlives_its_streams(dev, mode):
    """A prompt scratch allocated on stream a, used on b and outgrown there while b still has that prompt to run: a's next
    allocations of the same sizes get other memory, and b's results are right."""
    L, router, k, s = _layer("wide", dev)
    slots = k + 1

    def run(x):
        if mode == "windows":
            return G.windows(x, None, None, L, s, k=k, gate=router)
        return G.prefill(x, None, None, L, G.prefill_scratch(L, x.shape[0], slots, dev), k, gate=router)

    def held():
        return s.prompt if mode == "windows" else G._PREFILL[(L.E, L.D, L.I, slots, str(dev))]
    if mode == "prefill":
        G._PREFILL.pop((L.E, L.D, L.I, slots, str(dev)), None)
    x, longer = _x(50, L.D, dev, 7), _x(700, L.D, dev, 8)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        want = run(x)
    first = {t.data_ptr(): t.numel() * t.element_size() for t in held().tensors}
    a.synchronize()
    b.wait_stream(a)
    with torch.cuda.stream(b):
        torch.cuda._sleep(400_000_000)                     # ~0.17 s
        got = run(x)
        run(longer)                                           # drops the first scratch
    with torch.cuda.stream(a):
        other = [torch.empty(n, dtype=torch.uint8, device=dev) for n in first.values()]
        busy = not b.query()
        for t in other:
            t.fill_(255)
    torch.cuda.synchronize()
    assert busy, "b was done before a allocated: nothing tested"
    for t in other:
        assert all(t.data_ptr() + t.numel() <= p or p + n <= t.data_ptr() for p, n in first.items())
    _same(got, want)


@pytest.mark.parametrize("table", ["k2", "cb"])
def test_grouped_prompt_refuses_bad_table_entries(dev, ext, table):
    """A width outside the launch's range, or a codebook with no kernel: NaN sums and a status bit, no copy."""
    L, router, k, s = _layer("narrow", dev)
    ext.status(True)
    (L.k2[0] if table == "k2" else L.cb[0])[0] = 16 if table == "k2" else 9
    x = _x(40, L.D, dev, 9)
    out, _ = G.windows(x, None, None, L, s, k=k, gate=router)
    torch.cuda.synchronize()
    hit = (s.prompt.pick[:40 * s.slots].view(40, s.slots) == 0).any(dim=1)
    assert bool(hit.any()) and not bool(hit.all())
    assert bool(torch.isnan(out[hit].float()).all()) and bool(torch.isfinite(out[~hit].float()).all())
    assert int(ext.status(True)) != 0


@pytest.mark.parametrize("rows", [32, 64])
@pytest.mark.parametrize("T,slots,E", [(1, 1, 3), (33, 9, 257), (517, 9, 257), (2048, 9, 257), (2100, 4, 17), (300, 8, 4096)])
def test_group_tiles_equals_group_and_tile_list(dev, ext, T, slots, E, rows):
    """One launch's tables against group's, and its list against the member counts: random picks, ids out of range among
    them, an id twice a row, more picks than one batch of a workgroup (16384)."""
    gen = torch.Generator().manual_seed(T + rows)
    pick = torch.randint(-1, E + 1, (T, slots), generator=gen, dtype=torch.int32)
    pick[::3, -1] = E - 1
    pick = pick.reshape(-1).to(dev)
    maxu, P = min(T * slots, E), T * slots
    maxm = min(P, 2 * T)
    cap = min(maxu * -(-maxm // rows), -(-P // rows) + maxu)

    def tables():
        return [torch.full(shape, -7, dtype=torch.int32, device=dev) for shape in ((maxu,), (1,), (maxu, maxm))]
    (ids, count, members), (ids2, count2, members2) = tables(), tables()
    tiles = torch.full((1 + cap,), -7, dtype=torch.int32, device=dev)
    ext.group(pick, ids, count, members, T, slots, E)
    ext.group_tiles(pick, ids2, count2, members2, T, slots, E, rows, tiles)
    u = int(count.item())
    assert int(count2.item()) == u and torch.equal(ids2[:u], ids[:u])
    have = (members[:u] >= 0).sum(dim=1).tolist()
    want = [i << 16 | t for i, h in enumerate(have) for t in range(-(-h // rows))]
    assert tiles[:1 + len(want)].tolist() == [len(want)] + want
    for i, h in enumerate(have):
        full = min(-(-h // rows) * rows, maxm)
        assert torch.equal(members2[i, :full], members[i, :full]), i
    G.check_status()
