"""The W4A16 group behind a decoder layer's elementwise step (a mode of paroquant::w4a16_linear_group) on both rotation
paths (split up to 16 rows, row kernel above): the members get exactly the rows the kernel writes, those are torch's
to the last bit of the format, and the module's operands that the kernel does not take still run on torch's operations."""

import numpy as np
import pytest
import torch

import alpamayo_amd  # noqa: F401
from alpamayo_amd import _lib, workloads
from alpamayo_amd.quantization.paroquant_marlin_w4a8 import _rmsnorm_like_module
from tests.gpu_util import to_np
from tests.test_gpu_compile import _operands

pytestmark = pytest.mark.gpu

MODES = {"norm": _lib.PQ_PRO_RMSNORM, "add": _lib.PQ_PRO_ADD, "swiglu": _lib.PQ_PRO_SWIGLU}


def _args(ops_, bf16, out_dt):
    get = lambda key: [o[key] for o in ops_]   # noqa: E731
    return (get("rot_idx"), get("rot_cs"), get("sc"), 8, get("wp16"), get("wm16"), [None] * len(ops_), bf16, out_dt)


@pytest.mark.parametrize("m", [1, 2, 16, 17, 300])
@pytest.mark.parametrize("mode", list(MODES))
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_fused_group(m, mode, dtype):
    print(f"w4a16 fused m={m} {mode} {dtype}", flush=True)
    k = 1152
    ops_ = [_operands(n, k, 9000 + n) for n in (48, 1024)]
    g = workloads.generator(9100 + m)
    x, r = (workloads.activations(m, k, g).to(dtype).cuda() for _ in range(2))
    w = (0.8 + 0.4 * torch.rand(k, generator=g)).to(dtype).cuda() if mode == "norm" else None
    args = _args(ops_, dtype == torch.bfloat16, dtype)
    outs = torch.ops.paroquant.w4a16_linear_group(x, *args, MODES[mode], r, w, 1e-6, mode != "add", mode != "swiglu")
    if mode == "swiglu":
        rows, ref = outs[2], torch.nn.functional.silu(x) * r
    else:
        s = outs[-1]
        assert torch.equal(s, x + r)
        rows, ref = (outs[2], _rmsnorm_like_module(s, w, 1e-6)) if mode == "norm" else (s, s)
    a, b = to_np(rows.float()), to_np(ref.float())
    if dtype == torch.float32:
        np.testing.assert_allclose(a, b, rtol=1e-5, atol=1e-30)
    else:   # at most one unit of the format apart (two roundings of values one float32 ulp apart), and rarely
        ulp = 2.0 ** (-10 if dtype == torch.float16 else -7)
        assert np.all(np.abs(a - b) <= 2 * ulp * np.abs(b) + 2.0 ** -24) and np.mean(a == b) >= 0.995
    for y, yp in zip(outs, torch.ops.paroquant.w4a16_linear_group(rows, *args)):
        assert torch.equal(y, yp)


@pytest.mark.parametrize("m", [1, 40])
def test_module_operands_off_the_fused_path(m):
    """Broadcast operands, a type to promote, views off a 16-byte boundary and rows with a gradient to record."""
    from alpamayo_amd.quantization import RotateLinearInt4, SharedInputRotateLinears
    k, g = 1152, workloads.generator(9200)
    rls = [RotateLinearInt4(k, 64, bias=False, dtype=torch.float16).cuda() for _ in range(2)]
    for rl in rls:
        rl.qlinear.scales.copy_(0.01 * torch.rand(rl.qlinear.scales.shape))
    grp = SharedInputRotateLinears(rls)
    x, r = (workloads.activations(m, k, g).half().cuda() for _ in range(2))
    w = (0.8 + 0.4 * torch.rand(k, generator=g)).half().cuda()
    plain = lambda rows: grp(rows)   # noqa: E731
    off = lambda t: torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape)   # noqa: E731
    # broadcast residual, scalar weight, eps past the kernel's range: torch's own rows
    s = x + r[:1]
    for got, rows in ((grp(x, residual=r[:1], return_sum=True), s),
                      (grp(x, residual=r, norm_weight=w[:1]), _rmsnorm_like_module(x + r, w[:1], 1e-6)),
                      (grp(x, norm_weight=w, eps=2.0), _rmsnorm_like_module(x, w, 2.0)),
                      (grp.forward_swiglu(x, r[:1]), torch.nn.functional.silu(x) * r[:1])):
        for y, yp in zip(got, plain(rows)):
            assert torch.equal(y, yp)
    # views off a 16-byte boundary: the aligned copy's results
    for got, want in ((grp(off(x), residual=off(r), norm_weight=w), grp(x, residual=r, norm_weight=w)),
                      (grp.forward_swiglu(off(x), off(r)), grp.forward_swiglu(x, r))):
        for y, yp in zip(got, want):
            assert torch.equal(y, yp)
    # the sum and the norm are still differentiable
    xg = x.clone().requires_grad_(True)
    out = grp(xg, residual=r, norm_weight=w, return_normed=True, return_sum=True)
    assert out[-1].requires_grad and out[-2].requires_grad


@pytest.mark.parametrize("m", [1, 40])
def test_module_operands_torch_shapes(m):
    """Weights, residuals and eps that torch's operations take in a form of their own: one more leading dimension, a
    column, a number, an eps on the device, one that float32 rounds up to 1, and tangents of forward-mode AD."""
    from torch.autograd import forward_ad

    from alpamayo_amd.quantization import RotateLinearInt4, SharedInputRotateLinears
    k, g = 1152, workloads.generator(9300)
    rls = [RotateLinearInt4(k, 64, bias=False, dtype=torch.float16).cuda() for _ in range(2)]
    for rl in rls:
        rl.qlinear.scales.copy_(0.01 * torch.rand(rl.qlinear.scales.shape))
    grp = SharedInputRotateLinears(rls)
    x, r, t = (workloads.activations(m, k, g).half().cuda() for _ in range(3))
    w = (0.8 + 0.4 * torch.rand(k, generator=g)).half().cuda()
    w3, near1, eps_t = w.view(1, 1, k), 1.0 - 2.0 ** -30, torch.full((), 1e-6, device="cuda")
    for got, rows in ((grp(x, norm_weight=w3), _rmsnorm_like_module(x, w3, 1e-6)),
                      (grp(x, residual=r, norm_weight=w3), _rmsnorm_like_module(x + r, w3, 1e-6)),
                      (grp(x, norm_weight=w, eps=near1), _rmsnorm_like_module(x, w, near1)),
                      (grp(x, norm_weight=w, eps=eps_t), _rmsnorm_like_module(x, w, eps_t)),
                      (grp(x, residual=0.5), x + 0.5),
                      (grp.forward_swiglu(x, 0.5), torch.nn.functional.silu(x) * 0.5)):
        for y, yp in zip(got, grp(rows)):
            assert y.shape == yp.shape and torch.equal(y, yp)
    if m > 1:
        with pytest.raises(RuntimeError):
            grp(x, norm_weight=w.view(k, 1))
    with forward_ad.dual_level():
        xd = forward_ad.make_dual(x, t)
        assert forward_ad.unpack_dual(grp(xd, residual=r, return_sum=True)[-1]).tangent is not None
        act = grp.forward_swiglu(xd, r, return_act=True)[-1]
        assert forward_ad.unpack_dual(act).tangent is not None
