"""16-bit products whose columns run just past whole rounds of tiles run as two launches
over their columns, on operands as they lie or on one padded copy that both read: every
element against an fp32 product on the GPU, the columns around the cut against the float64
oracle, nothing written between C's rows (of even and odd pitch), and replays of a
captured graph bit for bit."""
import pytest
import torch

from cmp_ext_amd import cabi
from oracle import gemm_oracle as O

pytestmark = pytest.mark.gpu
DT = {"fp16": torch.float16, "bf16": torch.bfloat16}
CODE = {"fp16": cabi.F16, "bf16": cabi.BF16}


@pytest.mark.parametrize("dtype,layout,M,N,K,batch,bias,gap", [
    ("bf16", "KN", 4095, 4097, 1032, 1, None, 0),   # padded B, one column left: strips of A
    ("fp16", "KN", 2047, 4099, 1027, 2, "col", 0),  # both operands padded, a batch
    ("fp16", "NK", 4095, 4101, 1031, 1, "col", 1),  # [N, K] rows padded, C's rows of even pitch
    ("bf16", "NK", 4096, 4104, 1024, 1, "col", 8),
    ("bf16", "KN", 4096, 4104, 1024, 1, "row", 0),
    ("bf16", "KN", 4096, 4100, 4096, 1, None, 4),   # 4-byte aligned rows of B in both launches
    ("fp16", "NK", 2048, 8200, 512, 1, None, 1),    # 1032 columns left: tiles, odd pitch of C
    ("fp16", "KN", 1024, 4104, 1024, 4, "row", 0),
])
def test_col_split(dtype, layout, M, N, K, batch, bias, gap):
    g = torch.Generator().manual_seed(N + K)
    kn = layout == "KN"
    a = (torch.randn((batch, M, K), generator=g) * K ** -0.5).to(DT[dtype]).cuda()
    b = torch.randn((batch, K, N) if kn else (batch, N, K), generator=g).to(DT[dtype]).cuda()
    vec = torch.randn({"col": N, "row": M, None: 1}[bias], generator=g).to(DT[dtype]).cuda() if bias else None
    ldc = N + gap
    c = torch.full((batch, M, ldc), 3.0, dtype=DT[dtype], device="cuda")
    st, call = cabi.prepare(CODE[dtype], cabi.B_KN if kn else cabi.B_NK, a, K, M * K, b, N if kn else K, N * K, c, ldc,
                            M * ldc, vec, M, N, K, batch, cabi.BIAS_PER_ROW if bias == "row" else 0, 1 << 62)
    assert st == cabi.OK
    desc = cabi.describe(call)[1]
    print(desc, flush=True)
    assert " cols=" in desc, desc
    cut = int(desc.split(" cols=")[1].split()[0])
    ws = torch.empty(max(1, cabi.call_workspace_size(call)), dtype=torch.uint8, device="cuda")
    assert cabi.run(call, ws) == cabi.OK
    torch.cuda.synchronize()
    assert (c[:, :, N:] == 3.0).all()
    add = 0 if bias is None else (vec.float()[None, :] if bias == "col" else vec.float()[:, None])
    for i in range(batch):
        wide = b[i].float() if kn else b[i].float().t().contiguous()
        ref = a[i].float() @ wide + add
        assert O.rel_frobenius(O.to_f64(c[i, :, :N]), O.to_f64(ref)) <= O.TOLERANCE[dtype]
        cols = slice(cut - 3, min(N, cut + 40))
        exact = O.matmul_f64(O.to_f64(a[i]), O.to_f64(wide[:, cols]))
        if bias:
            exact = exact + (O.to_f64(vec)[None, cols] if bias == "col" else O.to_f64(vec)[:, None])
        assert O.rel_frobenius(O.to_f64(c[i, :, cols]), exact) <= O.TOLERANCE[dtype]


def test_graph_replays():
    import cmpext3

    g = torch.Generator().manual_seed(3)
    a, b = torch.randn(4095, 1032, generator=g).half().cuda(), (torch.randn(1032, 4097, generator=g) / 32).half().cuda()
    eager = cmpext3.fp16_matmul(a, b)
    assert " cols=4096 | cols 4096..4096: " in cmpext3.last_plan()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        cmpext3.fp16_matmul(a, b)
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = cmpext3.fp16_matmul(a, b)
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager) and torch.equal(cmpext3.fp16_matmul(a, b), eager)
