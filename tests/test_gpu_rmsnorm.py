"""GPU parity of the fused RMSNorm -> NVFP4 kernel (C ABI) against the CPU oracle.

Bar: normed output within 2e-3 relative Frobenius error of the oracle (the row mean is summed in
a different order, so single bf16 roundings may flip); codes, scale bytes and unit bit-exact
against the oracle's packing of the kernel's own bf16 normed tensor.
"""
import pytest
import torch

from helpers import rel_fro, synthetic_activation

pytestmark = pytest.mark.gpu

TOL = 2e-3


def _gamma(seed, cols):
    g = torch.Generator().manual_seed(seed)
    return (1 + 0.1 * torch.randn(cols, generator=g)).bfloat16()


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("rows,cols", [(64, 512), (33, 1536), (16, 4096), (5, 8192), (7, 48), (3, 12288), (256, 512), (300, 3584), (257, 4096)])
def test_fused_rmsnorm_quant(rows, cols, mode):
    from metis_hip import ops
    from oracle import metis_oracle as O
    x = synthetic_activation(1002 + rows, rows, cols)
    gamma = _gamma(7, cols)
    normed, p = ops.rmsnorm_quantize(x.cuda(), gamma.cuda(), 1e-6, mode)
    torch.cuda.synchronize()
    want = O.rmsnorm(x, gamma, 1e-6)
    assert rel_fro(normed.cpu(), want) <= TOL
    # elementwise: the row sum is taken in a different order, so rstd may differ in its last bit; a flip of the first
    # bf16 rounding (x * rstd) can carry through the multiplication by gamma and its rounding: at most two bf16 ulps
    d = (normed.cpu().float() - want.float()).abs()
    assert bool((d <= want.float().abs() * 2.0 ** -6 + 1e-30).all())
    assert float((d > 0).float().mean()) < 0.01                  # and that is rare
    mine = normed.cpu()
    codes, scales, unit, _ = O.nvfp4_pack(mine.float() if mode == 0 else mine)
    assert torch.equal(p.codes.cpu(), codes) and torch.equal(p.scales.cpu(), scales)
    assert float(p.unit.cpu()) == float(unit)
    # packed-only variant produces the same integers
    none, p2 = ops.rmsnorm_quantize(x.cuda(), gamma.cuda(), 1e-6, mode, want_normed=False)
    assert none is None and torch.equal(p2.codes, p.codes) and torch.equal(p2.scales, p.scales)


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("rows,cols", [(64, 512), (300, 3584), (16384, 4096), (7, 96)])
def test_fused_rmsnorm_quant_with_deferred_scale_bytes(rows, cols, mode):
    """deferred=True: the main kernel only.  Same normed tensor and codes; scale bytes and unit appear on first access
    with the bytes of the two-launch call, and the tiled expansion forms them itself, bit-equal to the eager tensor's."""
    from metis_hip import ops
    x = synthetic_activation(1100 + rows, rows, cols).cuda()
    gamma = _gamma(8, cols).cuda()
    normed, ref = ops.rmsnorm_quantize(x, gamma, 1e-6, mode)
    normed2, lazy = ops.rmsnorm_quantize(x, gamma, 1e-6, mode, deferred=True)
    assert torch.equal(normed, normed2) and torch.equal(lazy.codes, ref.codes)
    assert lazy.__dict__.get("_scales") is None
    assert torch.equal(ops.expand_tiled(lazy, cache=False, mode=mode), ops.expand_tiled(ref, cache=False, mode=mode))
    assert lazy.__dict__.get("_scales") is None and float(lazy.unit.cpu()) == float(ref.unit.cpu())
    _, lazy2 = ops.rmsnorm_quantize(x, gamma, 1e-6, mode, want_normed=False, deferred=True)
    assert torch.equal(lazy2.scales, ref.scales) and float(lazy2.unit.cpu()) == float(ref.unit.cpu())


def test_fused_rmsnorm_quant_config2_full_size():
    """bf16 [16384, 4096], gamma = 1 + N(0, 0.1^2), eps = 1e-6 (P32)."""
    from metis_hip import ops
    from oracle import c_oracle as C
    x = synthetic_activation(1002, 16384, 4096)
    gamma = _gamma(1002, 4096)
    normed, p = ops.rmsnorm_quantize(x.cuda(), gamma.cuda(), 1e-6, 0)
    torch.cuda.synchronize()
    cn, _, _, _ = C.rmsnorm_nvfp4(x, gamma, 1e-6, 0)
    assert rel_fro(normed.cpu(), cn) <= TOL
    cc, cs, cu, _ = C.nvfp4_pack(normed.cpu().contiguous(), 0)
    assert torch.equal(p.codes.cpu(), cc) and torch.equal(p.scales.cpu(), cs) and float(p.unit.cpu()) == cu


def test_value_error_and_limits():
    from metis_hip import ops
    with pytest.raises(ValueError):
        ops.rmsnorm_quantize(torch.zeros(4, 40, dtype=torch.bfloat16, device="cuda"),
                             torch.ones(40, dtype=torch.bfloat16, device="cuda"), 1e-6)


@pytest.mark.parametrize("rows,cols", [(1, 16), (5, 48), (7, 512), (33, 528), (300, 1040), (2049, 1536), (513, 3584), (9, 4096)])
def test_rmsnorm_backward(rows, cols):
    """Both gradients against the same formula in double precision.  gx carries one rounding to bf16 (eight significant bits: 2^-8 of the value)
    of a difference formed in binary32 (its two terms rounded a few times: 2^-20 of their sizes); ggamma one rounding of a
    binary32 sum whose terms hold bf16(x rstd): a term may round to the neighbouring bf16 value (2^-8 of the term) where
    rstd differs in its last bit, which is rare."""
    from metis_hip import ops
    eps = 1e-6
    x = synthetic_activation(40 + rows, rows, cols).cuda()
    gamma = _gamma(9, cols).cuda()
    g = (torch.randn(rows, cols, generator=torch.Generator().manual_seed(rows)) * 1e-3).bfloat16().cuda()
    xd, gd, md = x.double(), g.double(), gamma.double()
    rstd = (xd.pow(2).mean(-1, keepdim=True) + eps).rsqrt()
    xh = xd * rstd
    gh = gd * md
    mean = (gh * xh).mean(-1, keepdim=True)
    want = rstd * (gh - xh * mean)
    terms = gd * xh.float().bfloat16().double()
    gx, gg = ops.rmsnorm_backward(x, g, gamma, eps)
    assert bool(((gx.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -20 * rstd * (gh.abs() + (xh * mean).abs()) + 1e-30).all())
    want_g = terms.sum(0)
    slack = 2.0 ** -8 * terms.abs().amax(0) * (1 + rows / 2000) + 2.0 ** -20 * terms.abs().sum(0)
    assert bool(((gg.double() - want_g).abs() <= 2.0 ** -8 * want_g.abs() + slack).all())
    # without gamma's gradient, from a gradient that is a strided view, and from one that is not 16-byte aligned: the same bits
    wide = torch.zeros(rows, cols + 8, dtype=torch.bfloat16, device="cuda")
    wide[:, 1:cols + 1] = g
    odd = torch.zeros(rows * cols + 1, dtype=torch.bfloat16, device="cuda")[1:].view(rows, cols).copy_(g)
    assert torch.equal(ops.rmsnorm_backward(x, wide[:, 1:cols + 1], gamma, eps)[0], gx)
    again = ops.rmsnorm_backward(x, odd, gamma, eps)
    assert torch.equal(again[0], gx) and torch.equal(again[1], gg)
    only, none = ops.rmsnorm_backward(x, g, gamma, eps, want_gamma=False)
    assert none is None and torch.equal(only, gx)


def test_rmsnorm_backward_gamma_precision():
    """The binary32 gradient of gamma is no further from double precision than the formula that autograd records with create_graph.
    Its terms hold bf16(x rstd), which is the neighbouring bf16 value where the error of rstd puts x rstd on the other side of a
    midpoint: with rstd to twice binary32 from a sum of squares in binary32, in fewer elements than with rstd rounded."""
    from metis_hip import ops
    from metis_hip._lib import DTYPE_F32, load
    rows, cols, eps = 4096, 3584, 1e-6
    gamma = torch.ones(cols, dtype=torch.bfloat16, device="cuda")
    gx = torch.empty(rows, cols, dtype=torch.bfloat16, device="cuda")
    gg = torch.empty(cols, dtype=torch.float32, device="cuda")
    L = load()
    ws = torch.empty(L.metis_rmsnorm_backward_workspace_bytes(rows, cols), dtype=torch.uint8, device="cuda")
    squares = formula = 0.0
    for seed in range(8):
        gen = torch.Generator("cuda").manual_seed(seed)
        x = torch.randn(rows, cols, device="cuda", generator=gen).bfloat16()
        g = (torch.randn(rows, cols, device="cuda", generator=gen) * 1e-3).bfloat16()
        rc = L.metis_rmsnorm_backward(x.data_ptr(), g.data_ptr(), gamma.data_ptr(), eps, rows, cols, gx.data_ptr(), gg.data_ptr(), DTYPE_F32,
                                      ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        xd = x.double()
        xh = xd * (xd.pow(2).mean(-1, keepdim=True) + eps).rsqrt()
        want = (g.double() * xh.to(torch.bfloat16).double()).sum(0)
        squares += float((gg.double() - want).norm() / want.norm()) ** 2
        xf = x.float()
        recorded = (g.float() * (xf * torch.rsqrt(xf.pow(2).mean(dim=-1, keepdim=True) + eps)).to(torch.bfloat16).float()).double().sum(0)
        formula += float((recorded - want).norm() / want.norm()) ** 2
    assert squares <= formula
    # rows without remainders: zeros (rstd = eps^-1/2), and squares beyond binary32 (rstd = 0)
    one = torch.ones(4, 16, dtype=torch.bfloat16, device="cuda")
    for value, want in ((0.0, 1000.0), (1e30, 0.0)):
        assert torch.equal(ops.rmsnorm_backward(one * value, one, one[0], eps)[0], one * want)
