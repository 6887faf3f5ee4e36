"""fq_f32_kernel (float32 inputs on the float32 matrix cores): its sums run over
k in order with one rounding per product, as the generic kernel's do, so codes
and scales are equal bit for bit; at rounding ties against the oracle."""
import pytest
import torch

from quant_ops_amd import capi
from quant_ops_amd import workloads as wl
from oracle import fq_reference as ofq

pytestmark = pytest.mark.gpu


SHAPES = [(2, 8), (8, 2), (4, 10), (17, 24), (8, 13), (33, 40), (96, 96), (64, 64), (86, 128), (128, 128), (32, 202),
          (64, 254), (16, 255)]


@pytest.mark.parametrize("tokens", [1, 37, 1500])
@pytest.mark.parametrize("m,n,pack", [(m, n, p) for m, n in SHAPES for p in (True, False) if not (p and n % 2)])
def test_f32_matches_generic_kernel(gpu, m, n, tokens, pack, routing):
    print(f"[gpu-f32] {tokens} x {m}x{n} pack={pack}", flush=True)
    f = m * n
    x = wl.activations(tokens, f, torch.float32, tokens + m, 0.005, 30.0)
    if tokens > 8:   # an all-zero token, infinities, a NaN, tiny and huge values
        x[tokens // 2].zero_()
        x[3, f // 3] = float("inf")
        x[4, f // 2] = float("nan")
        x[5] *= 1e-9
        x[6] *= 1e30
    wide = torch.full((tokens, f + 12), 7.0)   # rows at a stride above their length
    wide[:, :f] = x
    x = wide.to(gpu)[:, :f]
    left, right = wl.orthogonal(m, m + 1).to(gpu), wl.orthogonal(n, n + 7).to(gpu)
    q, s = capi.flatquant_quantize(x, left, right, 0.9, pack)
    routing.on("FQ_GENERIC")
    qg, sg = capi.flatquant_quantize(x, left, right, 0.9, pack)
    routing.off("FQ_GENERIC")
    torch.cuda.synchronize()
    assert torch.equal(s, sg) and torch.equal(q, qg)


# the other instances of the kernel's table (rows rounded up to 16 MBX, columns to 64, 128, 192 or 256)
INSTANCES = [(20, 54), (52, 54), (84, 54), (116, 54), (20, 118), (52, 118), (84, 118), (20, 182), (52, 182), (84, 182),
             (116, 172), (20, 246), (84, 246), (100, 206)]


@pytest.mark.parametrize("m,n,tokens", [(m, n, 300) for m, n in INSTANCES] +
                         [(17, 24, 1537), (17, 24, 2051), (24, 14, 2049), (24, 30, 5000)])   # three and four tokens per workgroup
def test_f32_instances_match_generic_kernel(gpu, m, n, tokens, routing):
    print(f"[gpu-f32] instance {tokens} x {m}x{n}", flush=True)
    x = wl.activations(tokens, m * n, torch.float32, tokens + m, 0.005, 30.0).to(gpu)
    left, right = wl.orthogonal(m, m + 1).to(gpu), wl.orthogonal(n, n + 7).to(gpu)
    for pack in (True, False):
        q, s = capi.flatquant_quantize(x, left, right, 0.9, pack)
        routing.on("FQ_GENERIC")
        qg, sg = capi.flatquant_quantize(x, left, right, 0.9, pack)
        routing.off("FQ_GENERIC")
        torch.cuda.synchronize()
        assert torch.equal(s, sg) and torch.equal(q, qg)


@pytest.mark.parametrize("pack", [True, False])
@pytest.mark.parametrize("m,n,tokens", [(96, 96, 300), (64, 64, 1100), (22, 40, 64)])
def test_f32_codes_at_ties_bit_exact(gpu, m, n, tokens, pack):
    """Permutation matrices as L and R make Y an exact permutation of X. Each
    token's absmax is 7 times a factor, so quotients are half-integers and their
    neighbours up to the rounding of x * factor, for scales of many mantissas
    (all ones among them): the kernel's quotient has to round as y / s does."""
    g = torch.Generator().manual_seed(m + n + tokens)
    half = torch.arange(-7, 7) + 0.5
    vals = torch.cat([half, half * (1 + 2.0 ** -23), half * (1 - 2.0 ** -24), torch.arange(-7, 8).float()]).clamp(-7, 7)
    x = vals[torch.randint(0, vals.numel(), (tokens, m * n), generator=g)]
    x[torch.arange(tokens), torch.randint(0, m * n, (tokens,), generator=g)] = 7.0
    factor = 0.5 + torch.rand(tokens, 1, generator=g)
    factor[::7] = 1.0 - 2.0 ** -24   # an all-ones mantissa
    factor[1::7] = 1.0
    x = x * factor
    left = torch.eye(m)[torch.randperm(m, generator=g)]
    right = torch.eye(n)[torch.randperm(n, generator=g)]
    q, s = capi.flatquant_quantize(x.to(gpu), left.to(gpu), right.to(gpu), 1.0, pack)
    q_ref, s_ref = ofq.flatquant_pytorch(x, left, right, 1.0, pack)
    assert torch.equal(s.cpu(), s_ref) and torch.equal(q.cpu(), q_ref.to(q.dtype))
