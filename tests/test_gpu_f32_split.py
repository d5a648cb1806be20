"""The fp32 tiles that multiply on the bf16 matrix instruction (each float as three bf16
planes, six products): single products to the last bits, sums no further from the exact
ones than a chain of fused multiply-adds, infinities, NaN, the largest and the subnormal
values as the fp32 instruction gives them, on every such tile, both B layouts, both loads
(16- and 4-byte) and split K, against float64."""
import numpy as np
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
    """One nonzero k: the result is one product.  The left-out plane products come to at
    most 2 * 2^-8 * 2^-16 of it, adding the two sums rounds by 2^-24, and the five small
    products, 2^-7 of it, are added with a unit (2^-23) of their sum each."""
    g = torch.Generator().manual_seed(M + K)
    a, b = torch.zeros(M, K), torch.zeros(K, N)
    scale = lambda n: 2.0 ** torch.randint(-40, 41, (n,), generator=g)  # noqa: E731
    x, y = torch.rand(M, generator=g) + 1, -(torch.rand(N, generator=g) + 1)
    for i, bits in enumerate([0x3F807FFF, 0x3F80FFFF, 0x3F808001, 0x3FFF7FFF, 0x3FFFFFFF, 0x3F800001]):
        x[i] = y[i] = torch.tensor(bits, dtype=torch.int32).view(torch.float32)  # long rests
    a[:, K - 1], b[K - 1] = x * scale(M), y * scale(N)
    out = _run(monkeypatch, tile, a.cuda(), b.cuda(), nk).double().cpu()
    exact = a[:, K - 1].double()[:, None] * b[K - 1].double()[None]
    assert ((out - exact).abs() / exact.abs()).max().item() <= 3 * 2.0 ** -24 + 5 * 2.0 ** -30


@pytest.mark.parametrize("tile,nk", [(t, n) for t in TILES for n in (False, True)])
def test_single_products_of_tiny_floats(monkeypatch, tile, nk):
    """Floats down to the smallest subnormal: no plane loses a bit (bounds as above; the
    results, 2^-69 and more, are ordinary numbers)."""
    M, N, K = 150, 68, 36
    g = torch.Generator().manual_seed(1)
    a, b = torch.zeros(M, K), torch.zeros(K, N)
    a[:, K - 1] = (torch.rand(M, generator=g) + 1) * 2.0 ** torch.arange(-149, 1)
    b[K - 1] = (torch.rand(N, generator=g) - 2) * 2.0 ** 80
    assert (a[:, K - 1] > 0).all()
    exact = a[:, K - 1].double()[:, None] * b[K - 1].double()[None]
    for x, y, ref in ((a, b, exact), (b.t().contiguous(), a.t().contiguous(), exact.t())):
        out = _run(monkeypatch, tile, x.cuda(), y.cuda(), nk).double().cpu()
        assert ((out - ref).abs() / ref.abs()).max().item() <= 3 * 2.0 ** -24 + 5 * 2.0 ** -30


@pytest.mark.parametrize("tile,nk", [(t, n) for t in TILES for n in (False, True)])
@pytest.mark.parametrize("tiny", [1.2345e-35, 3e-39, 1.4e-45])
def test_tiny_floats_stay_on_the_planes(monkeypatch, tile, nk, tiny):
    """A tiny element does not send its tile to the fp32 instruction: every row and column
    but its own has the bits that it has with a zero in its place."""
    M, N, K = 130, 132, 200
    g = torch.Generator().manual_seed(2)
    a, b = torch.randn(M, K, generator=g), torch.randn(K, N, generator=g)
    a[7, 100] = b[33, 70] = 0.0
    ref = _run(monkeypatch, tile, a.cuda(), b.cuda(), nk)
    a[7, 100] = b[33, 70] = tiny
    out = _run(monkeypatch, tile, a.cuda(), b.cuda(), nk)
    rows, cols = torch.arange(M) != 7, torch.arange(N) != 70
    assert torch.equal(out[rows][:, cols], ref[rows][:, cols])


def _chain(a, b):
    """Each element as one chain of fused multiply-adds over k in fp32 (a product of two
    floats is exact in float64, and rounding their sum twice moves a last bit in 2^29)."""
    a, b = a.numpy().astype(np.float64), b.numpy().astype(np.float64)
    c = np.zeros((a.shape[0], b.shape[1]), np.float32)
    for k in range(a.shape[1]):
        c = (c + a[:, k, None] * b[k]).astype(np.float32)
    return c


def _draw(kind, g, *shape):
    x = torch.randn(shape, generator=g) if kind != "positive" else torch.rand(shape, generator=g)
    return x.exp() if kind == "lognormal" else x


@pytest.mark.parametrize("tile,nk", [(t, n) for t in TILES for n in (False, True)])
@pytest.mark.parametrize("kind", ["normal", "positive", "lognormal"])
def test_sums_against_a_chain(monkeypatch, tile, nk, kind):
    for M, N, K in [(130, 68, 24), (96, 64, 100), (70, 65, 515), (130, 132, 2048), (64, 96, 8192)]:
        g = torch.Generator().manual_seed(K)
        a, b = _draw(kind, g, M, K), _draw(kind, g, K, N)
        out = _run(monkeypatch, tile, a.cuda(), b.cuda(), nk).cpu().numpy().astype(np.float64)
        exact = a.double().numpy() @ b.double().numpy()
        err, chain = (np.linalg.norm(x - exact) / np.linalg.norm(exact) for x in (out, _chain(a, b)))
        print(f"{tile} {kind} K={K}: {err:.2e}, a chain {chain:.2e}", flush=True)
        assert err <= chain


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("K", [1, 3, 16])
def test_short_sums_keep_the_fp32_instruction(monkeypatch, tile, nk, K):
    """K <= 16: one product is rounded once, on every tile."""
    g = torch.Generator().manual_seed(K)
    a, b = torch.zeros(130, K), torch.zeros(K, 132)
    a[:, K - 1], b[K - 1] = torch.randn(130, generator=g), torch.randn(132, generator=g)
    out = _run(monkeypatch, tile, a.cuda(), b.cuda(), nk).cpu()
    assert torch.equal(out, a[:, K - 1, None] * b[K - 1])


@pytest.mark.parametrize("M,N", [(1, 1), (63, 64), (64, 65), (129, 200), (1000, 1001), (4, 3000)])
@pytest.mark.parametrize("K", [0, 1, 2, 4, 15, 16, 17, 31, 32, 33])
@pytest.mark.parametrize("nk", [False, True])
def test_short_k(M, N, K, nk):
    """The kernel for one stage and the first sizes past it, with a bias: no element further
    off than K + 1 roundings of its terms."""
    g = torch.Generator().manual_seed(M + K)
    x, w, bias = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g), torch.randn(N, generator=g)
    if nk:
        out = cmpext3.linear(x.cuda(), w.cuda(), bias.cuda())
    else:
        out, bias = cmpext3.fp32_matmul(x.cuda(), w.t().contiguous().cuda()), torch.zeros(N)
    desc = cmpext3.last_plan()
    print(M, N, K, desc, flush=True)
    assert K > 16 or desc.startswith("kernel=f32tile64x64 ")
    x, w, bias = x.double(), w.double(), bias.double()
    err = (out.double().cpu() - (x @ w.t() + bias)).abs()
    assert (err <= (K + 1) * 2.0 ** -24 * (x.abs() @ w.abs().t() + bias.abs())).all()


def test_short_k_batches():
    g = torch.Generator().manual_seed(0)
    for B, M, N, K in [(3, 65, 70, 16), (2, 100, 33, 7), (5, 1, 64, 16)]:
        a, b = torch.randn(B, M, K, generator=g), torch.randn(B, K, N, generator=g)
        out = cmpext3.bmm(a.cuda(), b.cuda()).double().cpu()
        for i in range(B):
            size = a[i].double().abs() @ b[i].double().abs()
            assert ((out[i] - a[i].double() @ b[i].double()).abs() <= K * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("M,N,K,nk", [(198, 896, 5976, True), (512, 512, 4096, False), (329, 392, 8002, True),
                                      (23, 2236, 8230, True), (656, 140, 7368, False)])
def test_splits_past_the_end_of_k(M, N, K, nk):
    """Splits are whole numbers of 64 k, so the last may start past K: it adds zeros."""
    g = torch.Generator().manual_seed(K)
    x, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g)
    torch.full((1 << 24,), float("nan"), device="cuda")  # (what the workspace may have held)
    out = cmpext3.linear(x.cuda(), w.cuda()) if nk else cmpext3.fp32_matmul(x.cuda(), w.t().contiguous().cuda())
    desc = cmpext3.last_plan()
    print(M, N, K, desc, flush=True)
    assert "splits=" in desc
    ref = (x.double() @ w.double().t()).numpy()
    # K / 32 roundings of the partial sums, and one for each split
    assert np.linalg.norm(out.double().cpu().numpy() - ref) <= 1e-6 * np.linalg.norm(ref)


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
