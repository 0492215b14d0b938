"""esp_dense_prompt (Dense.forward_prompt, and forward_tile past its rule): every weight decoded once, with the bits of the
launches whose sums it keeps. No tolerance: the windows (esp_dense) and the tile launch (esp_dense_tile), themselves held
to the oracle elsewhere, are the reference, bit for bit."""
import dataclasses

import pytest
import torch

from vllm_espalier import dense as D
from vllm_espalier import workloads as WL

pytestmark = pytest.mark.gpu

# K splits of 4 slots of 2 or 3 steps, of 2, of 1; one split; odd widths and codebooks; several launches
LAYERS = {
    "uneven_slots": [(2048, 4096, 4, "int6"), (2048, 512, 4, "int6"), (2048, 512, 4, "int6")],
    "two_steps": [(4096, 2048, 4, "int6")],
    "one_step": [(2048, 512, 4, "int5"), (2048, 512, 4, "int5")],
    "one_split": [(128, 384, 8, "mcg")],
    "nine_blocks": [(1152, 384, 5, "mcg"), (1152, 128, 5, "mcg")],
    "one_bit": [(640, 256, 1, "e2m1")],
    "two_codes": [(512, 256, 3, "int5"), (512, 128, 2, "e2m1")],
}


def _layer(name, dev, seed=1, n_out=None):
    gen = torch.Generator().manual_seed(seed)
    return D.Dense([WL.matrix(K, N, b, g, gen, dev) for K, N, b, g in LAYERS[name]], n_out)


def _rows(T, K, dtype, dev, seed):
    return torch.randn((T, K), generator=torch.Generator().manual_seed(seed)).to(dtype).to(dev)


def _windows(d, x):
    y = torch.empty((x.shape[0], d.n_out), dtype=x.dtype, device=x.device)
    for r in range(0, x.shape[0], D.MAX_ROWS):
        d.forward(x[r:r + D.MAX_ROWS], out=y[r:r + D.MAX_ROWS])
    return y


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T", [1, 17, 63, 64, 65, 200])
@pytest.mark.parametrize("name", list(LAYERS))
def test_prompt_equals_windows(dev, name, T, dtype):
    d = _layer(name, dev)
    assert d.prompts()
    x = _rows(T, d.K, dtype, dev, T)
    assert torch.equal(d.forward_prompt(x), _windows(d, x))


@pytest.mark.parametrize("w", [4, 8])
@pytest.mark.parametrize("sk", [1, 3, 5])
def test_prompt_equals_windows_at_fewer_slots(dev, w, sk):
    d = _layer("nine_blocks", dev)
    d.plans = [(sk, w, 2)]
    x = _rows(130, d.K, torch.bfloat16, dev, 3)
    assert torch.equal(d.forward_prompt(x), _windows(d, x))


def test_prompt_strided_padded_and_chunked(dev):
    """Rows a slice of a wider tensor, an output with padding columns, and more rows than one call takes."""
    d = _layer("two_codes", dev, n_out=512)
    T = D.PROMPT_ROWS + 33
    x = _rows(T, d.K + 64, torch.bfloat16, dev, 5)[:, 64:]
    y = d.forward_prompt(x)
    assert torch.equal(y, _windows(d, x))
    assert int(y[:, d.N:].abs().sum()) == 0


def test_prompt_signed_zeros(dev):
    """Zero rows and rows of -0: every sum's zero keeps the sign the windows give it."""
    d = _layer("uneven_slots", dev)
    x = torch.zeros((70, d.K), dtype=torch.bfloat16, device=dev)
    x[35:] = -0.0
    x[50, 7] = 1.0
    assert torch.equal(d.forward_prompt(x).view(torch.int16), _windows(d, x).view(torch.int16))


def _hows(d, T):
    return [how for *_, how in d._tiles(T)]


@pytest.mark.parametrize("name", ["uneven_slots", "two_steps", "one_step"])
def test_tile_mode_rows_alone_equal_prompt(dev, name):
    """forward_tile past its rule runs as esp_dense_prompt: its rows alone (esp_dense_tile) have the same bits."""
    d = _layer(name, dev)
    T = 2100
    assert _hows(d, T) == ["once"] and _hows(d, 1) == _hows(d, 128) == ["tile"]
    x = _rows(T, d.K, torch.bfloat16, dev, 8)
    y = d.forward_tile(x)
    for r in (0, 63, 64, 1000, 2099):
        assert torch.equal(d.forward_tile(x[r:r + 1]), y[r:r + 1]), r
    assert torch.equal(d.forward_tile(x[128:256]), y[128:256])


@pytest.mark.parametrize("name", ["one_split", "nine_blocks"])
def test_prompt_in_tile_order_equals_tile(dev, name):
    """esp_dense_prompt at esp_dense_tile's sums (its K splits, two k slots), on layers too small for the rule to take it."""
    d = _layer(name, dev)
    T = 300
    assert _hows(d, T) == ["tile"]
    x = _rows(T, d.K, torch.bfloat16, dev, 8)
    l, y = d.launches[0], torch.empty((T, d.n_out), dtype=x.dtype, device=dev)
    d._prompt(x, [m.trellis for m in d.mats], [m.suh for m in d.mats], [m.svh for m in d.mats], y, l, D.tile_plan(d.K, l.n),
              D.TILE_SLOTS)
    assert torch.equal(y, d.forward_tile(x))


def test_prompt_graph_replay(dev):
    d = _layer("two_steps", dev)
    x = _rows(150, d.K, torch.bfloat16, dev, 9)
    want = d.forward_prompt(x)
    y = torch.empty_like(want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        d.forward_prompt(x, out=y)
    for i in range(3):
        y.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), i
        torch.randn((64, 64), device=dev).sum()                # eager work between replays


def test_tile_mode_few_rows_of_a_wide_layer(dev):
    """A layer with one K split and two k slots (an LM head's plan): up to 32 rows of the tile mode are decode launches,
    with the bits of the same rows in a longer prompt."""
    gen = torch.Generator().manual_seed(3)
    d = D.Dense([WL.matrix(256, 128 * 260, 2, "mcg", gen, dev)])
    assert d._tile_is_window(32, d.launches[0]) and not d._tile_is_window(33, d.launches[0])
    x = _rows(100, d.K, torch.bfloat16, dev, 2)
    y = d.forward_tile(x)
    for T in (1, 7, 32):
        assert torch.equal(d.forward_tile(x[:T]), y[:T]), T


def test_reserve_prompt_only_for_tile_launches(dev, monkeypatch):
    """reserve_prompt grows the scratch for launches that run as esp_dense_tile at T rows, and for no others; forward_tile
    then allocates none."""
    for name in ("_PROMPT", "_PROMPT_COUNTERS"):
        monkeypatch.setattr(D, name, type(D._PROMPT)(getattr(D, name).fill, getattr(D, name).dtype))
    gen = torch.Generator().manual_seed(4)
    head = D.Dense([WL.matrix(256, 128 * 260, 2, "mcg", gen, dev)])
    head.reserve_prompt(1)                                     # a decode launch
    d = _layer("two_steps", dev)
    d.reserve_prompt(2048)                                     # every weight decoded once
    assert [how for *_, how in head._tiles(1) + d._tiles(2048)] == ["window", "once"]
    assert D._PROMPT.current == {} == D._PROMPT_COUNTERS.current
    d.reserve_prompt(100)
    assert [how for *_, how in d._tiles(100)] == ["tile"]
    held = [t.data_ptr() for t in D.prompt_scratch(dev, 0, 0, 0)]
    x = _rows(100, d.K, torch.bfloat16, dev, 2)
    want = d.forward_tile(x)
    assert [t.data_ptr() for t in D.prompt_scratch(dev, 0, 0, 0)] == held
    assert torch.equal(d.forward_tile(x[:17]), want[:17])


def _streamed(d):
    """d with its launch as esp_dense_stream for 1 to 6 rows, whatever the package's rule: any layer at one K split and 8
    waves (its shares may be one workgroup a CU)."""
    l = d.launches[0]
    assert (l.sk, l.w) == (1, 8)
    d.launches = [dataclasses.replace(l, stream=range(1, D.STREAM_MAX_ROWS + 1))]
    return d


@pytest.mark.parametrize("M", [1, 2, 5, 6])
@pytest.mark.parametrize("K,blocks,bits,grid", [(256, 600, 2, "mcg"), (1024, 260, 4, "int6"), (2048, 517, 6, "mcg"),
                                                (768, 1187, 3, "int5"), (512, 513, 5, "mcg"), (1280, 700, 8, "mcg")])
def test_stream_equals_one_workgroup_a_block(dev, ext, monkeypatch, K, blocks, bits, grid, M):
    """esp_dense_stream against esp_dense: shares that end inside blocks, blocks of one stage, as many blocks as workgroups;
    launches in a row, the hand-off buffer left all-ones and no wait timed out."""
    gen = torch.Generator(device=dev).manual_seed(K + blocks)
    d = _streamed(D.Dense([WL.matrix(K, 128 * blocks, bits, grid, gen, dev)]))
    for dtype in (torch.bfloat16, torch.float16):
        x = _rows(M, K, dtype, dev, M)
        monkeypatch.setattr(D, "STREAM", False)
        want = d.forward(x)
        monkeypatch.setattr(D, "STREAM", True)
        for _ in range(3):
            assert torch.equal(d.forward(x), want)
    assert bool((d._stream_part(dev).view(torch.int32) == -1).all())
    assert int(ext.status(True)) == 0


@pytest.mark.parametrize("wait", [-1, 200])
@pytest.mark.parametrize("M,K,blocks,bits,grid", [(5, 1280, 700, 8, "mcg"), (6, 1280, 257, 8, "mcg"), (6, 4096, 300, 4, "int6"),
                                                  (6, 8192, 260, 2, "mcg")])
def test_stream_one_workgroup_a_cu(dev, ext, monkeypatch, M, K, blocks, bits, grid, wait):
    """esp_dense_stream where its shared memory passes 80 KiB (the package runs esp_dense there): one workgroup a CU."""
    gen = torch.Generator(device=dev).manual_seed(K + blocks)
    m = WL.matrix(K, 128 * blocks, bits, grid, gen, dev)
    d = D.Dense([m])
    l = d.launches[0]
    assert not d._streams(M, l)
    l = D.Launch(l.members, l.k2, l.cb, l.n, 1, 8, 2)             # the plan whose sums the launch keeps
    d.launches = [l]
    x = _rows(M, K, torch.bfloat16, dev, M)
    monkeypatch.setattr(D, "STREAM", False)
    want = d.forward(x)
    part, y = d._new_parts(dev, 1)[0], torch.full_like(want, float("nan"))
    for _ in range(2):
        ext.dense_stream(x, None, None, None, 0.0, None, m.trellis, m.suh, m.svh, 0, y, part, wait, l.k2, l.cb)
        assert torch.equal(y, want)
    assert bool((part.view(torch.int32) == -1).all())


def _specials(x):
    """Rows of infinities, NaN, overflow on the way, the largest and the smallest values among ordinary ones."""
    T, K = x.shape
    fin = torch.finfo(x.dtype)
    x[0, 3], x[1, K // 2], x[2, K - 1] = float("inf"), float("nan"), float("-inf")
    if T > 5:
        x[3] = fin.max
        x[4, ::7], x[4, 1::7] = float("inf"), float("-inf")
        x[5] = fin.smallest_normal
    return x


def _same_values(got, want):
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan) and bool(nan.any())
    assert torch.equal(got[~nan], want[~nan])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("name", ["uneven_slots", "two_steps", "one_step", "nine_blocks", "two_codes"])
def test_prompt_equals_windows_of_no_finite_values(dev, name, dtype):
    d = _layer(name, dev)
    x = _specials(_rows(100, d.K, dtype, dev, 12))
    _same_values(d.forward_prompt(x), _windows(d, x))


@pytest.mark.parametrize("M", [3, 6])
def test_stream_equals_dense_of_no_finite_values(dev, ext, monkeypatch, M):
    gen = torch.Generator(device=dev).manual_seed(31)
    d = D.Dense([WL.matrix(1024, 128 * 700, 4, "int6", gen, dev)])
    assert d._streams(M, d.launches[0])
    x = _specials(_rows(M, d.K, torch.bfloat16, dev, 13))
    monkeypatch.setattr(D, "STREAM", False)
    want = d.forward(x)
    monkeypatch.setattr(D, "STREAM", True)
    _same_values(d.forward(x), want)
    assert bool((d._stream_part(dev).view(torch.int32) == -1).all()) and int(ext.status(True)) == 0


@pytest.mark.parametrize("wait", [-1, 0])
@pytest.mark.parametrize("M", [1, 6])
@pytest.mark.parametrize("K,blocks,bits,grid", [(256, 600, 2, "mcg"), (2048, 513, 4, "int6"), (1024, 1187, 3, "int5")])
def test_stream_without_its_predecessors_sums(dev, ext, monkeypatch, K, blocks, bits, grid, M, wait):
    """Workgroups that give up on their predecessor's sums (all of them; those that come too early) make them themselves: the
    same bits, and the hand-off buffer all-ones for the launches after, which wait as ever."""
    gen = torch.Generator(device=dev).manual_seed(K + blocks)
    d = _streamed(D.Dense([WL.matrix(K, 128 * blocks, bits, grid, gen, dev)]))
    monkeypatch.setattr(D, "STREAM", False)
    xs = [_rows(M, K, torch.bfloat16, dev, M + i) for i in range(4)]
    want = [d.forward(x) for x in xs]
    monkeypatch.setattr(D, "STREAM", True)
    for us in (wait, D.STREAM_WAIT_US, wait, wait):
        monkeypatch.setattr(D, "STREAM_WAIT_US", us)
        got = [d.forward(x) for x in xs]
        torch.cuda.synchronize()
        assert all(torch.equal(g, w) for g, w in zip(got, want)), us
        assert bool((d._stream_part(dev).view(torch.int32) == -1).all()), us
    assert int(ext.status(True)) == 0


@pytest.mark.parametrize("M", [1, 2])
def test_stream_rmsnorm_equals_dense_rmsnorm(dev, monkeypatch, M):
    gen = torch.Generator(device=dev).manual_seed(9)
    d = D.Dense([WL.matrix(2048, 128 * 530, 4, "mcg", gen, dev)])
    assert d.norm_fusable(M) and d._streams(M, d.launches[0])
    h, d1, d2 = (_rows(M, d.K, torch.bfloat16, dev, s) for s in (1, 2, 3))
    w = (1 + 0.1 * torch.randn((d.K,), generator=torch.Generator().manual_seed(4))).to(torch.bfloat16).to(dev)
    outs = []
    for stream in (False, True):
        monkeypatch.setattr(D, "STREAM", stream)
        h_out, y = torch.zeros_like(h), torch.empty((M, d.n_out), dtype=h.dtype, device=dev)
        d.forward_rmsnorm(h, d1, d2, w, 1e-6, h_out, y)
        d.forward_rmsnorm(h, None, None, w, 1e-6, torch.zeros_like(h), y.clone())
        outs.append((h_out, y))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


def test_stream_graph_replay(dev):
    gen = torch.Generator(device=dev).manual_seed(10)
    d = D.Dense([WL.matrix(1024, 128 * 700, 4, "mcg", gen, dev)])
    x = _rows(1, d.K, torch.bfloat16, dev, 1)
    want = d.forward(x)
    calls = D.STREAM_SPARES + 2                                # the last ones run as esp_dense
    y = torch.empty((calls, *want.shape), dtype=want.dtype, device=dev)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for i in range(calls):
            d.forward(x, out=y[i])
    for i in range(4):
        y.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(v, want) for v in y), i
        assert torch.equal(d.forward(x), want)                 # eager work between replays
    side = torch.cuda.Stream()                                 # another stream, another hand-off buffer
    own = d._stream_part(dev)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        assert d._stream_part(dev).data_ptr() != own.data_ptr()
        ys = [d.forward(x) for _ in range(3)]
    ym = [d.forward(x) for _ in range(3)]
    torch.cuda.synchronize()
    assert all(torch.equal(v, want) for v in ys + ym)
