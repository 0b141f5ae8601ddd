"""The W4A16 GEMM on tiled fp16 rows (17 to 512 rows behind the linear entry points) at the edges of its row blocks,
column units and K splits, against float64 products of the rotated rows and the dequantized weights.

Bound: a float32 sum of K products in any order, and one add of the bias: (K + 2) 2^-24 sum |x w| + 2^-23 |y|."""

import zlib

import pytest
import torch

import alpamayo_amd  # noqa: F401
from alpamayo_amd import workloads
from tests.gpu_util import packed_rotation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,ns", [
    (17, 1024, (16,)), (31, 1152, (1040,)), (33, 4096, (4096, 1024, 1024)), (48, 12288, (4096,)), (64, 1408, (12288, 12304)),
    (65, 4096, (4096,)), (97, 2048, (1040, 80)), (129, 4224, (4096,)), (200, 1024, (5120,)), (255, 1152, (4112,)),
    (320, 2048, (4096,)), (512, 1024, (4096, 1040)), (511, 1024, (272,)),
])
def test_tiled_w16_gemm(M, K, ns):
    print(f"tiled W4A16 M={M} K={K} ns={ns}", flush=True)
    x = workloads.activations(M, K, workloads.generator(5000 + M)).half().cuda()
    ops_, refs, bounds = [], [], []
    for i, n in enumerate(ns):
        spec = workloads.linear_spec(f"t{i}", n, K, workloads.generator(zlib.crc32(f"{K}{n}{i}".encode())),
                                     keep_codes=True)
        rot_idx, rot_cs, _, _ = packed_rotation(spec.pairs, spec.theta)
        s, sz = workloads.w16_scales(spec.w)
        wp, wm = torch.ops.paroquant.w4a16_prepack(spec.w.awq_qweight.cuda(), s.cuda(), sz.cuda())
        b = torch.randn(n, generator=workloads.generator(n)).half().cuda() if i == 0 else None
        o = (rot_idx.cuda(), rot_cs.cuda(), spec.channel_scales.float().reshape(-1).cuda(), wp, wm, b)
        ops_.append(o)
        _, _, rows = torch.ops.paroquant.rotate_quant_i8_rot(x, o[0], o[1], o[2], 8, False, True)
        q = spec.w.codes.cuda().double().view(n, K // 128, 128)
        w = (q * s.cuda().double().t()[..., None] + sz.cuda().double().t()[..., None]).half().double().view(n, K)
        r = rows.double()
        bias = b.double() if b is not None else torch.zeros(n, device="cuda").double()
        refs.append(r @ w.t().contiguous() + bias)
        bounds.append((K + 2) * 2.0 ** -24 * (r.abs() @ w.abs().t().contiguous()) + 2.0 ** -23 * (refs[-1].abs() + bias.abs()))
    args = ([o[0] for o in ops_], [o[1] for o in ops_], [o[2] for o in ops_], 8, [o[3] for o in ops_],
            [o[4] for o in ops_], [o[5] for o in ops_], False)
    ys = torch.ops.paroquant.w4a16_linear_group(x, *args, torch.float32)
    y16 = torch.ops.paroquant.w4a16_linear_group(x, *args, torch.float16)
    for y, yh, ref, bound in zip(ys, y16, refs, bounds):
        assert torch.all((y.double() - ref).abs() <= bound)
        assert torch.equal(yh.view(torch.int16), y.half().view(torch.int16))
