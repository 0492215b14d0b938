"""esp_dense_prompt (Dense.forward_prompt, and forward_tile past its rule): every weight decoded once, with the bits of the
launches whose sums it keeps. No tolerance: the windows (esp_dense) and the tile launch (esp_dense_tile), themselves held
to the oracle elsewhere, are the reference, bit for bit."""
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


@pytest.mark.parametrize("name", ["uneven_slots", "two_steps", "one_step", "one_split"])
def test_tile_mode_rows_alone_equal_prompt(dev, name):
    """forward_tile past its rule runs as esp_dense_prompt: its rows alone (esp_dense_tile) have the same bits."""
    d = _layer(name, dev)
    T = 2100
    x = _rows(T, d.K, torch.bfloat16, dev, 8)
    y = d.forward_tile(x)
    for r in (0, 63, 64, 1000, 2099):
        assert torch.equal(d.forward_tile(x[r:r + 1]), y[r:r + 1]), r
    assert torch.equal(d.forward_tile(x[128:256]), y[128:256])


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
