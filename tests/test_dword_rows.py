"""16-bit products whose B is [K, N] with rows aligned to 4 bytes only (an even N or pitch
that is no multiple of 8: images of 14x14 pixels) are read in place by the tile kernels and,
for at most 64 rows and N % 8 == 0, the skinny ones: which calls take that route (CPU), and
its results, with NaN after every row and after the operand, against the float64 oracle."""
import numpy as np
import pytest
import torch

from cmp_ext_amd import cabi
from oracle import gemm_oracle as O

A, B, C = 0x100000, 0x40000000, 0x80000000  # host addresses: plans only


def _plan(M, N, K, lda=None, ldb=None, batch=1, stride_b=None, off_a=0, off_b=0, layout=cabi.B_KN, ws=1 << 40):
    lda, ldb = lda or K, ldb or (N if layout == cabi.B_KN else K)
    st, call = cabi.prepare(cabi.F16, layout, A + 2 * off_a, lda, M * lda, B + 2 * off_b, ldb,
                            stride_b if stride_b is not None else K * ldb, C, N, M * N, None, M, N, K, batch, 0, ws)
    assert st == cabi.OK
    return cabi.describe(call)[1]


def test_route():
    rng = np.random.default_rng(7)
    taken = 0
    for _ in range(600):
        M, N, K = int(rng.integers(1, 3000)), int(rng.integers(1, 3000)), int(rng.integers(1, 1500))
        if rng.random() < 0.7:
            K = K // 8 * 8 or 8
        batch, off_b, off_a = int(rng.choice([1, 3])), int(rng.choice([0, 0, 2, 3])), int(rng.choice([0, 0, 0, 4]))
        ldb = N + int(rng.choice([0, 0, 1, 2, 8]))
        desc = _plan(M, N, K, ldb=ldb, batch=batch, off_b=off_b, off_a=off_a)
        aligned_a = K % 8 == 0 and off_a % 8 == 0
        aligned_b = off_b % 8 == 0 and ldb % 8 == 0 and N % 8 == 0
        even = off_b % 2 == 0 and ldb % 2 == 0 and (batch == 1 or K * ldb % 2 == 0)
        expect = aligned_a and even and not aligned_b and M * N * K * batch >= 1 << 24
        assert ("b_dword" in desc) == expect, (M, N, K, ldb, batch, off_a, off_b, desc)
        if expect:
            taken += 1
            # at least 256 tiles of 128 columns fill the GPU by themselves
            skinny = M <= 64 and N % 8 == 0 and -(-N // 128) * batch < 256
            assert ("kernel=skinny" if skinny else "kernel=tile") in desc and "padded" not in desc, desc
    assert taken > 60
    for M, N, K, kw in [(16, 4096, 4096, dict(off_b=2)), (16, 4096, 4096, dict(ldb=4098)), (1, 2048, 8192, dict(ldb=2050, off_b=2)),
                        (64, 1024, 1024, dict(ldb=1030, batch=3)), (33, 512, 2048, dict(ldb=516))]:
        desc = _plan(M, N, K, **kw)
        assert "kernel=skinny_wide " in desc and "b_dword" in desc and "padded" not in desc, desc
    assert "kernel=tile" in _plan(16, 4090, 4096)                  # N % 8: a piece would cross the row's end
    for ws in (0, 1 << 20):                                        # nothing is copied: no workspace needed
        assert "kernel=tile128x128 " in _plan(2048, 60, 2048, ws=ws) and "b_dword" in _plan(2048, 60, 2048, ws=ws)
        assert "b_dword" in _plan(4096, 4090, 4096, ws=ws)
    assert "generic" in _plan(2048, 61, 2048, ws=0)                # odd rows: copied, or element by element
    assert "padded" in _plan(1000, 1002, 1004)                     # K % 8: A is copied, and B
    assert "padded=B" in _plan(1000, 1001, 1000)                   # odd rows
    assert "b_dword" not in _plan(1000, 1002, 1000, layout=cabi.B_NK)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("M,N,K,gap,off,batch", [
    (200, 196, 1024, 0, 0, 3), (200, 1002, 512, 0, 0, 1), (257, 1030, 520, 6, 0, 1), (128, 2044, 264, 2, 2, 1),
    (300, 500, 72, 4, 6, 2), (70, 4098, 320, 0, 0, 1), (513, 130, 4104, 0, 2, 1), (4090, 4090, 128, 0, 0, 1),
    (64, 70002, 136, 0, 0, 1),
    # skinny_wide: one to four 16-row blocks, K split and not, streamed once (64 MiB), ragged K, a batch
    (16, 4096, 4096, 0, 2, 1), (1, 2048, 8192, 2, 0, 1), (33, 8192, 4096, 2, 2, 1), (64, 16392, 264, 4, 6, 1),
    (48, 1024, 520, 6, 0, 3), (20, 136, 8200, 2, 0, 1), (7, 32000, 128, 2, 2, 1), (16, 128, 8192, 4, 2, 2),
])
def test_results(dtype, M, N, K, gap, off, batch):
    import cmpext3

    dt = {"fp16": torch.float16, "bf16": torch.bfloat16}[dtype]
    g = torch.Generator().manual_seed(N)
    a = (torch.randn((batch, M, K), generator=g) * K ** -0.5).to(dt)
    b = torch.randn((batch, K, N), generator=g).to(dt)
    ldb = N + gap
    buf = torch.full((off + batch * K * ldb + 64,), float("nan"), dtype=dt, device="cuda")  # gaps and what follows
    view = buf[off : off + batch * K * ldb].view(batch, K, ldb)[:, :, :N]
    view.copy_(b)
    if batch == 1:
        fn = cmpext3.fp16_matmul if dtype == "fp16" else cmpext3.bf16_matmul
        out = fn(a[0].cuda(), view[0])[None]
    else:
        out = cmpext3.bmm(a.cuda(), view)
    desc = cmpext3.last_plan()
    print(dtype, M, N, K, gap, off, batch, desc, flush=True)
    assert "b_dword" in desc, desc
    for i in range(batch):
        assert O.reference_check(out[i].cpu(), a[i], b[i], dtype) <= O.TOLERANCE[dtype]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("M,N,K,gap,off,batch", [
    (512, 1001, 1024, 1, 0, 1), (200, 1003, 264, 3, 2, 1), (130, 999, 136, 5, 6, 2), (300, 129, 2048, 1, 0, 1),
    (4095, 4097, 64, 1, 0, 1), (200, 1001, 1024, 7, 0, 1), (512, 1002, 1024, 0, 0, 1), (130, 1004, 136, 2, 2, 2),
    (16, 1024, 4096, 2, 0, 1), (64, 4096, 1032, 6, 2, 1), (5, 2000, 2056, 0, 2, 3),
])
def test_last_column_of_the_last_row(dtype, M, N, K, gap, off, batch):
    """B's last element, at the very end of the operand (in the middle of a dword where N is
    odd and the pitch even), outweighs the rest of its column, with NaN after it: the last
    columns element by element."""
    import cmpext3

    dt = {"fp16": torch.float16, "bf16": torch.bfloat16}[dtype]
    g = torch.Generator().manual_seed(N + K)
    a = torch.rand((batch, M, K), generator=g).add_(0.5).to(dt)
    b = (torch.randn((batch, K, N), generator=g) / K).to(dt)
    b[:, K - 1] *= 64
    b[:, K - 1, N - 1] = 7
    ldb = N + gap
    buf = torch.full((off + batch * K * ldb,), float("nan"), dtype=dt, device="cuda")
    view = buf[off:].view(batch, K, ldb)[:, :, :N]
    view.copy_(b)
    matmul = cmpext3.fp16_matmul if dtype == "fp16" else cmpext3.bf16_matmul
    out = matmul(a[0].cuda(), view[0])[None] if batch == 1 else cmpext3.bmm(a.cuda(), view)
    desc = cmpext3.last_plan()
    print(dtype, M, N, K, gap, off, batch, desc, flush=True)
    assert "b_dword" in desc, desc
    a, b = a.double(), b[:, :, N - 9 :].double()
    ref, size = a @ b, a @ b.abs()
    # fp32 sums of K products and one rounding to 11 or 8 bits
    bound = K * 2.0 ** -24 * size + 2.0 ** (-11 if dtype == "fp16" else -8) * ref.abs() + 2.0 ** -24
    assert ((out[:, :, N - 9 :].double().cpu() - ref).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 16, 17, 64])
def test_narrow_strips_without_a_workspace(M):
    """The narrow skinny kernel on B at an offset of 4 bytes, with a bias per column."""
    N, K, ldb = 2056, 8200, 2058
    g = torch.Generator().manual_seed(M)
    a = (torch.randn((M, K), generator=g) * K ** -0.5).half()
    b, bias = torch.randn((K, N), generator=g).half(), torch.randn(N, generator=g).half()
    buf = torch.full((2 + K * ldb + 64,), float("nan"), dtype=torch.half, device="cuda")
    view = buf[2 : 2 + K * ldb].view(K, ldb)[:, :N]
    view.copy_(b)
    c = torch.full((M, N), 3.0, dtype=torch.half, device="cuda")
    ac, bias_c = a.cuda(), bias.cuda()
    st, call = cabi.prepare(cabi.F16, cabi.B_KN, ac, K, 0, view.data_ptr(), ldb, 0, c, N, 0, bias_c, M, N, K, 1, 0, 0)
    assert st == cabi.OK
    desc = cabi.describe(call)[1]
    print(M, desc, flush=True)
    assert "kernel=skinny " in desc and "b_dword" in desc and cabi.call_workspace_size(call) == 0
    assert cabi.run(call) == cabi.OK
    assert O.reference_check(c.cpu(), a, b, "fp16", bias) <= O.TOLERANCE["fp16"]
