"""Kernels whose waves read a ring of LDS stages that the whole workgroup (or the wave)
refills by LDS-DMA: the same product 60 times over, every result bit for bit the first one
and each element of it near the float64 product.  K ends in the middle of a stage and the
loads past it return at once, which is when a slot refilled before everyone had read it was
lost (rows of one wave's load, a share of their sum) in one launch of five or so."""
import pytest
import torch

import cmpext3
from cmp_ext_amd import cabi

pytestmark = pytest.mark.gpu
DT = {cabi.F16: torch.half, cabi.BF16: torch.bfloat16, cabi.F32: torch.float32}
UNIT = {cabi.F16: 2.0 ** -11, cabi.BF16: 2.0 ** -8, cabi.F32: 2.0 ** -24}


@pytest.mark.parametrize("kernel,dtype,layout,B,M,N,K,limit", [
    ("tall", cabi.F16, cabi.B_NK, 7, 2905, 2, 1728, 1 << 40),     # 32-row strips, one 16-row block of B
    ("tall", cabi.BF16, cabi.B_NK, 3, 4000, 24, 1336, 1 << 40),   # two
    ("tall", cabi.F16, cabi.B_NK, 2, 3000, 64, 2008, 1 << 40),    # four
    ("tall", cabi.F16, cabi.B_KN, 4, 2900, 40, 1544, 1 << 40),
    ("tall", cabi.F16, cabi.B_KN, 8, 2048, 64, 2048, 1 << 40),    # 64-row strips
    ("tall", cabi.F16, cabi.B_NK, 1, 1024, 16, 14344, 1 << 40),   # K split
    ("skinny_nk", cabi.F16, cabi.B_NK, 1, 16, 11000, 1544, 1 << 40),
    ("skinny_nk", cabi.BF16, cabi.B_NK, 1, 64, 8200, 1160, 1 << 40),
    ("skinny_nk", cabi.F16, cabi.B_NK, 6, 30, 5000, 584, 1 << 40),
    ("skinny_wide", cabi.F16, cabi.B_KN, 1, 16, 8192, 1096, 1 << 40),
    ("skinny_wide", cabi.BF16, cabi.B_KN, 1, 64, 30000, 328, 1 << 40),
    ("skinny", cabi.F16, cabi.B_KN, 1, 16, 8192, 1304, 0),
    ("skinny", cabi.F16, cabi.B_KN, 1, 50, 4096, 648, 0),
    ("f32tile64x64k4", cabi.F32, cabi.B_KN, 1, 1000, 1000, 1013, 1 << 40),
    ("f32tile64x64k4", cabi.F32, cabi.B_NK, 1, 512, 2048, 520, 1 << 40),
    ("f32tile16x64k4", cabi.F32, cabi.B_KN, 1, 16, 8192, 1100, 1 << 40),
])
def test_repeats(kernel, dtype, layout, B, M, N, K, limit):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    dt = DT[dtype]
    a = torch.rand((B, M, K), generator=g, device="cuda").to(dt)
    b = (torch.rand((B, K, N) if layout == cabi.B_KN else (B, N, K), generator=g, device="cuda") / K).to(dt)
    out = torch.empty((60, B, M, N), dtype=dt, device="cuda")
    ws = None
    for i in range(60):
        st, call = cabi.prepare(dtype, layout, a, K, M * K, b, N if layout == cabi.B_KN else K, N * K, out[i], N, M * N,
                                None, M, N, K, B, 0, limit)
        assert st == cabi.OK
        if ws is None:
            desc = cabi.describe(call)[1]
            print(desc, flush=True)
            assert desc.startswith(f"kernel={kernel} "), desc
            ws = torch.empty(max(1, cabi.call_workspace_size(call)), dtype=torch.uint8, device="cuda")
        assert cabi.run(call, ws) == cabi.OK
    torch.cuda.synchronize()
    differ = [i for i in range(60) if not torch.equal(out[i], out[0])]
    assert not differ, differ
    for i in range(B):
        w = (b[i] if layout == cabi.B_KN else b[i].t().contiguous()).double()
        ref = a[i].double() @ w
        # K roundings of 2^-24 of the sum and one to the type; all terms are positive
        assert ((out[0, i].double() - ref).abs() <= (K * 2.0 ** -24 + UNIT[dtype]) * ref).all()
