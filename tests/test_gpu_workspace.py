"""Device memory that the torch operators take beside their outputs."""
import pytest
import torch

import quant_ops_amd as qo
from quant_ops_amd import capi
from quant_ops_amd import workloads as wl

pytestmark = pytest.mark.gpu

ROOM = 1 << 20   # outputs, codes and scales of these calls are well below; an FP6 workspace well above


def _peak(f):
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out = f()
    torch.cuda.synchronize()
    return out, torch.cuda.max_memory_allocated() - before


@pytest.mark.parametrize("m", [1, 16])
def test_decode_over_an_odd_vocabulary_takes_no_workspace(gpu, m):
    """W.t() of an odd number of rows, up to 64 tokens: the small-M kernel, which uses no workspace."""
    n, k = 15163, 4096
    case = wl.gemm_case(m, n, k, seed=m, b_transposed_view=True)
    a, b, sa, sb = case.a.to(gpu), case.b.to(gpu), case.scale_a.to(gpu), case.scale_b.to(gpu)
    out, peak = _peak(lambda: qo.int4_matmul(a, b, sa, sb))
    print(f"[gpu-workspace] int4_matmul {m}x{n}x{k}: {peak} bytes", flush=True)
    assert peak < ROOM
    ref = capi.int4_gemm(a, b, sa, sb)
    assert torch.equal(out, ref)
    left, right = wl.orthogonal(64, 1, torch.bfloat16).to(gpu), wl.orthogonal(64, 2, torch.bfloat16).to(gpu)
    x = wl.activations(m, k, torch.bfloat16, 3).to(gpu)
    _, peak = _peak(lambda: torch.ops.quant_ops.w4a4_linear(x, left, right, b.t(), sb, 0.9, None))
    print(f"[gpu-workspace] w4a4_linear {m}x{n}x{k}: {peak} bytes", flush=True)
    assert peak < ROOM


@pytest.mark.parametrize("m,w_view", [(16, False), (200, True), (300, True)])
def test_gemm_without_room_for_its_workspace(gpu, m, w_view):
    """Where the caching allocator cannot give the FP6 route's workspace (here: its share of the memory is
    capped from the host), the call takes the kernels without one and gives the same output."""
    n, k = 40001, 4096
    case = wl.gemm_case(m, n, k, seed=m, b_transposed_view=w_view)
    a, b, sa, sb = case.a.to(gpu), case.b.to(gpu), case.scale_a.to(gpu), case.scale_b.to(gpu)
    full, peak = _peak(lambda: qo.int4_matmul(a, b, sa, sb))
    ws = capi.gemm_workspace_size(m, n, k)
    assert peak > ws > (100 << 20)   # the FP6 route
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(gpu).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + ws // 2) / total)
    try:
        out, peak = _peak(lambda: qo.int4_matmul(a, b, sa, sb))
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    print(f"[gpu-workspace] {m}x{n}x{k} capped: {peak} bytes", flush=True)
    assert peak < ws and torch.equal(out, full)
