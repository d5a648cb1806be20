"""128x128 tiles alone on their CU run with a ring of four K steps: every number of steps
around the ring's length and the rule's K, ragged K, grids of one, 256 and 257
workgroups, K splits, both B layouts and both bias forms, against the float64 oracle."""
import pytest
import torch

import cmpext3
from oracle import gemm_oracle as O

pytestmark = pytest.mark.gpu


def _check(dtype, layout, M, N, K, bias):
    a, b = O.make_inputs(dtype, M, N, K, "normal", K ** -0.5, M + N + K, b_layout=layout)
    bias_t = torch.linspace(-1, 1, N).to(a.dtype) if bias else None
    if layout == "NK":
        out = cmpext3.linear(a.cuda(), b.cuda(), bias_t.cuda() if bias else None)
    else:
        out = (cmpext3.fp16_matmul if dtype == "fp16" else cmpext3.bf16_matmul)(a.cuda(), b.cuda())
    desc = cmpext3.last_plan()
    print(f"{dtype} {layout} {M}x{N}x{K}: {desc}", flush=True)
    assert desc.startswith("kernel=tile128x128"), desc
    # every element: fp32 sums and one rounding, K products each
    err = O.reference_check(out.cpu(), a, b, dtype, bias_t, layout)
    assert err <= O.TOLERANCE[dtype]
    return desc


@pytest.mark.parametrize("dtype,layout", [("fp16", "KN"), ("bf16", "NK")])
@pytest.mark.parametrize("K", [448, 512, 520, 576, 640, 704, 768, 1000, 1024])
def test_steps_around_the_ring(dtype, layout, K):
    _check(dtype, layout, 129, 136, K, layout == "NK")


@pytest.mark.parametrize("layout", ["KN", "NK"])
@pytest.mark.parametrize("M,N", [(70, 8), (2048, 2048), (1900, 2040), (128 * 257, 128)])
def test_grids_up_to_a_workgroup_per_cu(layout, M, N):
    _check("fp16", layout, M, N, 576, layout == "NK")


def test_split_k_and_rows_of_a_batch():
    desc = _check("bf16", "NK", 100, 512, 4104, True)  # splits of whole steps, the last one short
    assert "splits=" in desc and "splits=1 " not in desc
    w, x = O.make_inputs("fp16", 130, 3 * 200, 600, "normal", 600 ** -0.5, 5)
    x, b = x.view(600, 3, 200).transpose(0, 1).contiguous(), torch.linspace(-1, 1, 130).half()
    out = cmpext3.conv2d(x.view(3, 600, 10, 20).cuda(), w.view(130, 600, 1, 1).cuda(), b.cuda())
    assert cmpext3.last_plan().startswith("kernel=tile128x128"), cmpext3.last_plan()
    for i in range(3):  # the bias per row
        ref = O.matmul_f64(O.to_f64(w), O.to_f64(x[i])) + O.to_f64(b)[:, None]
        assert O.rel_frobenius(O.to_f64(out[i].cpu()).reshape(130, 200), ref) <= O.TOLERANCE["fp16"]
