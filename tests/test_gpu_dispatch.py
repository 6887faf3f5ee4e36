"""Sizes on both sides of the lines where the dispatch changes kernels
(quant_ops_amd/csrc/dispatch_rules.h), each against the generic kernel."""
import pytest
import torch

from quant_ops_amd import capi
from quant_ops_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _codes(q, pack):
    if not pack:
        return q.int()
    shifts = torch.arange(0, 32, 4, dtype=torch.int32, device=q.device)
    return (((q.unsqueeze(-1) >> shifts) & 15) - 8).reshape(q.shape[0], -1)


@pytest.mark.parametrize("pack", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,tokens", [
    (56, 64, 768), (56, 64, 769), (56, 64, 1024), (56, 64, 1025), (64, 80, 512), (64, 80, 513), (64, 80, 2000),
    (64, 112, 257), (64, 112, 513), (72, 96, 256), (72, 96, 257), (72, 96, 512), (80, 112, 257), (80, 112, 512),
])
def test_padded_shapes_at_their_lines(gpu, m, n, tokens, dtype, pack, routing):
    """Each kernel rounds where the fallback does; their float32 sums run in other orders, so a code may
    differ by one at a rounding boundary (0.1 % of the codes, as in the parity tests) and a scale by a unit
    per rounding (max |Y|, its product with clip, that by 1/7)."""
    print(f"[gpu-dispatch] {tokens} x {m}x{n} {dtype} pack={pack}", flush=True)
    case = wl.quant_case("line", tokens, m, n, dtype, 0.9, pack, seed=tokens + m, outlier_frac=0.005, outlier_scale=30.0)
    case.x[tokens // 2].zero_()
    x, left, right = case.x.to(gpu), case.left.to(gpu), case.right.to(gpu)
    q, s = capi.flatquant_quantize(x, left, right, 0.9, pack)
    routing.on("FQ_GENERIC")
    qg, sg = capi.flatquant_quantize(x, left, right, 0.9, pack)
    routing.off("FQ_GENERIC")
    torch.cuda.synchronize()
    unit = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7
    assert ((s - sg).abs() <= 3 * unit * sg).all()
    same = s == sg
    assert same.float().mean() >= 0.97
    d = (_codes(q, pack) - _codes(qg, pack)).abs()[same]
    assert int(d.max()) <= 1 and (d > 0).float().mean().item() <= 1e-3


@pytest.mark.parametrize("w_view", [True, False])
@pytest.mark.parametrize("out_dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m", [1, 16, 17, 64, 65, 128, 300])
@pytest.mark.parametrize("n,k", [(5, 64), (5, 160), (37, 192), (2051, 32), (2052, 64), (1023, 288), (64, 200), (64, 264), (1001, 72)])
def test_ragged_gemm_at_the_lines(gpu, m, n, k, out_dtype, w_view, routing):
    """Small ragged products (generic kernel) and the next larger ones (small-M kernel with 1 to 3 lane groups in
    the last stage, FP6 route): the sums are exact on all of them, so outputs are equal bit for bit."""
    print(f"[gpu-dispatch] {m}x{n}x{k} {out_dtype} W.t()={w_view}", flush=True)
    case = wl.gemm_case(m, n, k, seed=m + n + k, b_transposed_view=w_view, out_dtype=out_dtype)
    a, b, sa, sb = case.a.to(gpu), case.b.to(gpu), case.scale_a.to(gpu).float(), case.scale_b.to(gpu)
    wide = torch.full((m, n + 5), 7.0, dtype=out_dtype, device=gpu)   # rows at a stride above their length
    out = wide[:, :n]
    capi.int4_gemm(a, b, sa, sb, out_dtype=out_dtype, out=out, workspace=True)
    routing.on("GEMM_GENERIC")
    ref = capi.int4_gemm(a, b, sa, sb, out_dtype=out_dtype)
    routing.off("GEMM_GENERIC")
    torch.cuda.synchronize()
    assert torch.equal(out, ref) and bool((wide[:, n:] == 7.0).all())
