"""GEMMs whose rows the integer tiled kernels cannot take (N % 4 != 0 or
K % 128 != 0): the small-M kernel up to 64 rows, the FP6 route above or for the
other layouts, each against the generic kernel. The sums are exact on all of
them, so outputs are equal bit for bit."""
import pytest
import torch

from quant_ops_amd import capi
from quant_ops_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w_view", [True, False])
@pytest.mark.parametrize("out_dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m", [1, 17, 64, 65, 300])
@pytest.mark.parametrize("n,k", [(5, 32), (37, 64), (100, 96), (1027, 1064), (1631, 1024), (1630, 1152 + 64), (1632, 8128)])
def test_ragged_gemm_equals_generic_kernel(gpu, m, n, k, out_dtype, w_view, routing):
    print(f"[gpu-ragged] {m}x{n}x{k} {out_dtype} W.t()={w_view}", flush=True)
    case = wl.gemm_case(m, n, k, seed=m + n, b_transposed_view=w_view, out_dtype=out_dtype)
    a, b = case.a.to(gpu), case.b.to(gpu)
    sa, sb = case.scale_a.to(gpu).float(), case.scale_b.to(gpu)
    bias = wl.uniform(n, -1.0, 1.0, 7, out_dtype).to(gpu) if n % 2 else None
    assert capi.gemm_workspace_size(m, n, k, out_dtype) > 0
    wide = torch.full((m, n + 5), 7.0, dtype=out_dtype, device=gpu)   # rows at a stride above their length
    out = wide[:, :n]
    capi.int4_gemm(a, b, sa, sb, out_dtype=out_dtype, out=out, bias=bias, workspace=True)
    routing.on("GEMM_GENERIC")
    ref = capi.int4_gemm(a, b, sa, sb, out_dtype=out_dtype, bias=bias)
    routing.off("GEMM_GENERIC")
    torch.cuda.synchronize()
    assert torch.equal(out, ref) and bool((wide[:, n:] == 7.0).all())
