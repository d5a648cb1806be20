"""The fp32 tiles that multiply on the bf16 matrix instruction (each float as three bf16
planes, six products): single products to the last bits, infinities, NaN, the largest and
the subnormal values as the fp32 instruction gives them, on every such tile, both B
layouts, both loads (16- and 4-byte) and split K, against float64."""
import pytest
import torch

import cmpext3

pytestmark = pytest.mark.gpu
TILES = ["f32tile128x128", "f32tile96x64", "f32tile64x64"]


def _run(monkeypatch, tile, a, b, nk, splits=1):
    monkeypatch.setenv("CMPEXT3_GEMM_CONFIG", f"kernel={tile},splits={splits}")
    out = cmpext3.fp32_matmul(a, b.t().contiguous().t() if nk else b)
    desc = cmpext3.last_plan()
    print(tuple(a.shape), b.shape[1], desc, flush=True)
    assert desc.startswith(f"kernel={tile} ") and ("splits=" in desc) == (splits > 1), desc
    return out


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("M,N,K", [(130, 132, 4), (97, 65, 1), (128, 64, 33), (100, 200, 31)])
def test_single_products(monkeypatch, tile, nk, M, N, K):
    """One nonzero k: the result is one product, off by the three left-out plane products
    (each below 2^-23 of it) and six roundings of 2^-24."""
    g = torch.Generator().manual_seed(M + K)
    a, b = torch.zeros(M, K), torch.zeros(K, N)
    scale = lambda n: 2.0 ** torch.randint(-40, 41, (n,), generator=g)  # noqa: E731
    a[:, K - 1] = (torch.rand(M, generator=g) + 1) * scale(M)
    b[K - 1] = -(torch.rand(N, generator=g) + 1) * scale(N)
    out = _run(monkeypatch, tile, a.cuda(), b.cuda(), nk).double().cpu()
    exact = a[:, K - 1].double()[:, None] * b[K - 1].double()[None]
    assert ((out - exact).abs() / exact.abs()).max().item() <= 3 * 2.0 ** -23 + 6 * 2.0 ** -24


def _special(kind, M, N, K):
    g = torch.Generator().manual_seed(7)
    a, b = torch.randn(M, K, generator=g), torch.randn(K, N, generator=g)
    big = torch.finfo(torch.float32).max
    if kind == "infinity":
        a[5, 7], b[9, 33] = float("inf"), float("-inf")
    elif kind == "infinity times zero":
        a[5, 7], a[5, 8], b[7, 11] = float("inf"), float("-inf"), 0.0
    elif kind == "nan":
        a[M - 1, K - 1] = float("nan")
    elif kind == "largest":  # one in each row: the sums stay finite
        a[:, 3], b[3] = -big, 2.0 ** -20
    elif kind == "tiny":
        a, b = a * 2.0 ** -122, b * 2.0 ** 60
    elif kind == "subnormal":
        a, b = a * 2.0 ** -135, b * 2.0 ** 100
    elif kind == "mixed rows":  # rows of very different size: each to its own precision
        a = a * (2.0 ** torch.linspace(-130, 20, M))[:, None]
        b = b * 2.0 ** 60
    return a, b


@pytest.mark.parametrize("tile,nk,splits", [(t, n, 1) for t in TILES for n in (False, True)] + [(t, False, 3) for t in TILES])
@pytest.mark.parametrize("kind", ["infinity", "infinity times zero", "nan", "largest", "tiny", "subnormal", "mixed rows"])
def test_special_values(monkeypatch, tile, nk, splits, kind):
    for M, N, K in [(200, 260, 768), (131, 67, 75)][: 1 if splits > 1 else 2]:  # 16- and 4-byte loads
        a, b = _special(kind, M, N, K)
        out = _run(monkeypatch, tile, a.cuda(), b.cuda(), nk, splits).double().cpu()
        ref = a.double() @ b.double()
        assert torch.equal(torch.isnan(out), torch.isnan(ref))
        inf = torch.isinf(ref)
        assert torch.equal(torch.isinf(out), inf) and torch.equal(out[inf], ref[inf])
        # fp32 sums of K products: K roundings of 2^-24 of the row's products at most
        fine = torch.isfinite(ref)
        size = (a.double().nan_to_num(0, 0, 0).abs() @ b.double().nan_to_num(0, 0, 0).abs())
        assert ((out - ref).abs()[fine] <= (K + 8) * 2.0 ** -24 * size[fine] + 2.0 ** -149).all()
