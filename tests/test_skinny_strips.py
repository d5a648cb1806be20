"""skinny_nk's strips of W rows: the height rule (CPU), and every height the rule or the
override can choose, with whole and partial last strips, against the float64 oracle."""
import re

import pytest
import torch

from cmp_ext_amd import cabi
from oracle import gemm_oracle as O

CUS = 256


def _strip(M, N, K=4096, batch=1):
    _, desc = cabi.plan(cabi.BF16, cabi.B_NK, M, N, K, batch=batch, workspace_bytes=1 << 40)
    assert desc.startswith("kernel=skinny_nk"), desc
    return int(re.search(r"tile=\d+x(\d+) ", desc).group(1)), "splits=" in desc


def test_strip_heights():
    for M, N, expect in [(64, 4096, 16), (64, 4104, 32), (64, 8192, 32), (64, 8200, 48), (64, 11008, 48),
                         (64, 12288, 48), (64, 14336, 64), (33, 16384, 64), (33, 17000, 80), (64, 20480, 80),
                         (64, 24576, 96), (64, 28672, 112), (32, 20480, 80), (32, 24576, 48), (17, 32000, 64),
                         (16, 4096, 16), (16, 4104, 32), (16, 11008, 48),
                         (1, 12288, 48), (1, 12296, 32), (16, 28672, 32)]:
        assert _strip(M, N) == (expect, False), (M, N)


@pytest.mark.parametrize("M", [17, 40, 64])
def test_strips_never_stream_more_than_another_height(M):
    mb = -(-M // 16)
    rounds = lambda n, rows: -(-(-(-n // rows)) // CUS)  # noqa: E731
    for N in range(4104, 32700, 616):
        rows, split = _strip(M, N)
        if not split:
            best = min(rounds(N, r) * (r + 16 * mb) for r in range(16, 81 if mb == 2 else 129, 16))
            assert rounds(N, rows) * (rows + 16 * mb) == best, (M, N, rows)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("M,strips", [(16, (16, 32, 48, 64)), (17, (16, 48, 64, 80, 96, 112, 128)),
                                      (48, (32, 48, 80, 96, 112, 128)), (64, (48, 64, 80, 96, 112, 128))])
def test_every_strip_height(monkeypatch, dtype, M, strips):
    import cmpext3

    for strip in strips:
        for N, K in [(2 * strip, 512), (strip + 8, 264), (3 * strip - 8, 1032)]:
            monkeypatch.setenv("CMPEXT3_GEMM_CONFIG", f"kernel=skinny_nk,strip={strip}")
            x, w = O.make_inputs(dtype, M, N, K, "normal", K ** -0.5, strip + N, b_layout="NK")
            b = torch.linspace(-1, 1, N).to(x.dtype)
            out = cmpext3.linear(x.cuda(), w.cuda(), b.cuda())
            desc = cmpext3.last_plan()
            print(dtype, M, N, K, desc, flush=True)
            assert desc.startswith("kernel=skinny_nk") and f"x{strip} " in desc, desc
            assert O.reference_check(out.cpu(), x, w, dtype, b, "NK") <= O.TOLERANCE[dtype]


@pytest.mark.gpu
def test_strips_of_a_batch_and_of_whole_layers():
    import cmpext3

    for M, N, K, batch, strip in [(40, 3000, 256, 3, 48), (64, 20488, 264, 1, 96), (20, 9216, 128, 1, 48),
                                  (3, 11008, 512, 1, 48)]:
        g = torch.Generator().manual_seed(N)
        x = torch.randn((batch, M, K), generator=g).half()
        w = (torch.randn((batch, N, K), generator=g) * K ** -0.5).half()
        out = cmpext3.bmm(x.cuda(), w.cuda().transpose(1, 2))
        desc = cmpext3.last_plan()
        print(M, N, K, batch, desc, flush=True)
        assert desc.startswith("kernel=skinny_nk") and f"x{strip} " in desc, desc
        for i in range(batch):
            assert O.reference_check(out[i].cpu(), x[i], w[i], "fp16", None, "NK") <= O.TOLERANCE["fp16"]


@pytest.mark.gpu
def test_linear_without_rows_or_outputs():
    import cmpext3

    x, w = torch.randn(16, 14336).half().cuda(), torch.randn(8, 14336).half().cuda()
    assert cmpext3.linear(x, w[:0]).shape == (16, 0)
    assert cmpext3.linear(x[:0], w).shape == (0, 8)
    assert cmpext3.bmm(x[None][:0], w.t()[None][:0]).shape == (0, 16, 8)
