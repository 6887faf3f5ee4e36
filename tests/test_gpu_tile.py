"""fq_tile_kernel (fp16 / bf16, every shape without a kernel of its own): against
the generic kernel at the edges of its blocks and pieces, and against the oracle
at rounding ties.

The two kernels sum in float32 in different orders, so a code may differ by one
where a quotient lies within the sums' error of a rounding boundary (the bar of
the parity tests: 0.1 % of the codes). A scale may differ by three units of its
type: max |Y| rounds the other way (one unit), and so may its product with clip
and that by 1/7 (one each; 1.3857 against 1.3877 in fp16 was seen, two units)."""
import pytest
import torch

from quant_ops_amd import capi
from quant_ops_amd import workloads as wl
from oracle import fq_reference as ofq

pytestmark = pytest.mark.gpu

# (M, N): smallest; one row block and one short of it; rows of 8, 4 and 2-element
# pieces; odd M; the last odd row block and column block absent; both largest
SHAPES = [(2, 8), (8, 2), (4, 10), (17, 24), (16, 30), (33, 40), (96, 96), (32, 202), (44, 48), (86, 128), (128, 148),
          (64, 214), (144, 192), (168, 176), (64, 254), (150, 256)]


def _codes(q, pack):
    if not pack:
        return q.int()
    shifts = torch.arange(0, 32, 4, dtype=torch.int32, device=q.device)
    return (((q.unsqueeze(-1) >> shifts) & 15) - 8).reshape(q.shape[0], -1)


@pytest.mark.parametrize("pack", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tokens", [1, 300, 1100])
@pytest.mark.parametrize("m,n", SHAPES)
def test_tile_matches_generic_kernel(gpu, m, n, tokens, dtype, pack, routing):
    print(f"[gpu-tile] {tokens} x {m}x{n} {dtype} pack={pack}", flush=True)
    f = m * n
    x = wl.activations(tokens, f, dtype, tokens + m, 0.005, 30.0)
    special = []
    if tokens > 8:   # an all-zero token, infinities, a NaN, tiny values
        x[tokens // 2].zero_()
        x[3, f // 3] = float("inf")
        x[4, f // 2] = float("nan")
        x[5] *= 1e-6 if dtype == torch.float16 else 1e-9
        special = [tokens // 2, 3, 4]
    wide = torch.full((tokens, f + 24), 7.0, dtype=dtype)   # rows at a stride above their length
    wide[:, :f] = x
    x = wide.to(gpu)[:, :f]
    left, right = wl.orthogonal(m, m + 1, dtype).to(gpu), wl.orthogonal(n, n + 7, dtype).to(gpu)
    q, s = capi.flatquant_quantize(x, left, right, 0.9, pack)
    routing.on("FQ_GENERIC")
    qg, sg = capi.flatquant_quantize(x, left, right, 0.9, pack)
    routing.off("FQ_GENERIC")
    torch.cuda.synchronize()
    assert torch.equal(q[special], qg[special]) and torch.equal(s[special], sg[special])
    # subnormal fp16 scales have an absolute unit of 2^-24
    unit = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7
    fin = torch.isfinite(sg)
    assert ((s - sg).abs()[fin] <= 3 * (sg[fin] * unit + (2.0 ** -24 if dtype == torch.float16 else 0.0))).all()
    same = s == sg
    assert same.float().mean() >= 0.97 or tokens == 1
    d = (_codes(q, pack) - _codes(qg, pack)).abs()
    ok = (same | ~fin) & (sg > 1e-6)   # codes of subnormal scales jump with the scale's unit
    assert d[ok].numel() == 0 or (int(d[ok].max()) <= 1 and (d[ok] > 0).float().mean().item() <= 1e-3)


def _ties(dtype):
    vals = []
    for k in range(-7, 7):
        h = torch.tensor(k + 0.5, dtype=dtype)
        bits = h.view(torch.int16)
        vals += [float(h), float((bits + 1).view(dtype)), float((bits - 1).view(dtype)), float(k)]
    return torch.tensor(vals + [0.0, -0.0, 7.0, -7.0, 6.96875, -6.96875]).clamp(-7, 7)


@pytest.mark.parametrize("pack", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,tokens", [(96, 96, 300), (22, 32, 1100), (64, 214, 40), (128, 148, 600)])
def test_tile_codes_at_ties_bit_exact(gpu, m, n, tokens, dtype, pack):
    """Permutation matrices as L and R make Y an exact permutation of X; with an
    absmax of 7 the scale is 1 and every quotient the element itself."""
    print(f"[gpu-tile] ties {tokens} x {m}x{n} {dtype} pack={pack}", flush=True)
    g = torch.Generator().manual_seed(m + n + tokens)
    vals = _ties(dtype)
    x = vals[torch.randint(0, vals.numel(), (tokens, m * n), generator=g)]
    x[torch.arange(tokens), torch.randint(0, m * n, (tokens,), generator=g)] = 7.0
    x = x.to(dtype)
    left = torch.eye(m)[torch.randperm(m, generator=g)].to(dtype)
    right = torch.eye(n)[torch.randperm(n, generator=g)].to(dtype)
    q, s = capi.flatquant_quantize(x.to(gpu), left.to(gpu), right.to(gpu), 1.0, pack)
    q_ref, s_ref = ofq.flatquant_pytorch(x, left, right, 1.0, pack)
    assert torch.equal(s.cpu(), s_ref.float()) and torch.equal(q.cpu(), q_ref.to(q.dtype))


# one shape per instance of the kernel's table (rows rounded up to 16 MBX, columns to 32 KS), widths of 2-element pieces
_ROWS = {2: 20, 4: 52, 6: 84, 8: 116, 10: 148, 11: 172}
INSTANCES = [(_ROWS[mbx], 32 * ks - 10) for ks, most in ((1, 4), (2, 6), (3, 8), (4, 10), (5, 11), (6, 11), (7, 11), (8, 11))
             for mbx in _ROWS if mbx <= most]


def _exact(x, left, right, clip):
    """Codes and scales of the transform in 64 bits throughout."""
    t, m, n = x.shape[0], left.shape[0], right.shape[0]
    z = (x.double().reshape(t * m, n) @ right.double()).view(t, m, n)
    y = (z.transpose(1, 2).reshape(t * n, m) @ left.double()).view(t, n, m).transpose(1, 2).reshape(t, m * n)
    s = (y.abs().amax(1) * clip / 7.0).clamp(min=1e-8)
    return torch.round(y / s[:, None]).clamp(-8, 7), s


@pytest.mark.parametrize("pack", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n", INSTANCES)
def test_every_instance_no_further_from_64_bits(gpu, m, n, dtype, pack, routing):
    """Codes and scales as close to the 64-bit transform as the generic kernel's: the two share every rounding
    point, so their mean errors differ only by tokens whose sums fall on the other side of a rounding."""
    print(f"[gpu-tile] instance {m}x{n} {dtype} pack={pack}", flush=True)
    tokens = 600
    x = wl.activations(tokens, m * n, dtype, m + n, 0.005, 30.0).to(gpu)
    left, right = wl.orthogonal(m, m + 1, dtype).to(gpu), wl.orthogonal(n, n + 7, dtype).to(gpu)
    q, s = capi.flatquant_quantize(x, left, right, 0.9, pack)
    routing.on("FQ_GENERIC")
    qg, sg = capi.flatquant_quantize(x, left, right, 0.9, pack)
    routing.off("FQ_GENERIC")
    q64, s64 = _exact(x, left, right, 0.9)

    def errors(q, s):
        return ((s.double() - s64).abs() / s64).mean().item(), (_codes(q, pack) != q64).double().mean().item()

    (se, ce), (sge, cge) = errors(q, s), errors(qg, sg)
    print(f"[gpu-tile]   scales {se:.3e} (generic {sge:.3e}), codes {ce:.3e} ({cge:.3e})", flush=True)
    assert se <= 1.02 * sge + 1e-7 and ce <= 1.02 * cge + 1e-6
    d = (_codes(q, pack) - _codes(qg, pack)).abs()[s == sg]
    assert (s == sg).float().mean() >= 0.97 and int(d.max()) <= 1 and (d > 0).float().mean().item() <= 1e-3


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,tokens", [(17, 24, 1537), (17, 24, 2051), (24, 14, 2049), (44, 32, 1790), (24, 30, 5000)])
def test_several_tokens_per_workgroup(gpu, m, n, tokens, dtype, routing):
    """Three and four token slots per workgroup, the last group part empty: each token as in a call of its own kind
    (300 tokens: one slot), bit for bit."""
    print(f"[gpu-tile] slots {tokens} x {m}x{n} {dtype}", flush=True)
    x = wl.activations(tokens, m * n, dtype, tokens + m, 0.005, 30.0).to(gpu)
    left, right = wl.orthogonal(m, m + 1, dtype).to(gpu), wl.orthogonal(n, n + 7, dtype).to(gpu)
    q, s = capi.flatquant_quantize(x, left, right, 0.9, True)
    parts = [capi.flatquant_quantize(x[i:i + 300], left, right, 0.9, True) for i in range(0, tokens, 300)]
    torch.cuda.synchronize()
    assert torch.equal(q, torch.cat([p[0] for p in parts])) and torch.equal(s, torch.cat([p[1] for p in parts]))
