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


def _operands(n, K, seed, with_bias):
    spec = workloads.linear_spec("t", n, K, workloads.generator(seed), keep_codes=True)
    rot_idx, rot_cs, _, _ = packed_rotation(spec.pairs, spec.theta)
    s, sz = workloads.w16_scales(spec.w)
    wp, wm = torch.ops.paroquant.w4a16_prepack(spec.w.awq_qweight.cuda(), s.cuda(), sz.cuda())
    b = torch.randn(n, generator=workloads.generator(n)).half().cuda() if with_bias else None
    return (rot_idx.cuda(), rot_cs.cuda(), spec.channel_scales.float().reshape(-1).cuda(), wp, wm, b), spec, s, sz


@pytest.mark.parametrize("M,K,ns", [
    (17, 1024, (16,)), (31, 1152, (1040,)), (33, 4096, (4096, 1024, 1024)), (48, 12288, (4096,)), (64, 1408, (12288, 12304)),
    (65, 4096, (4096,)), (97, 2048, (1040, 80)), (129, 4224, (4096,)), (200, 1024, (5120,)), (255, 1152, (4112,)),
    (320, 2048, (4096,)), (512, 1024, (4096, 1040)), (511, 1024, (272,)),
    # every size of block with one, one or two, and more groups of K per part
    (17, 1024, (8208,)), (30, 1920, (12304,)), (30, 2048, (8208,)), (33, 1024, (4096, 1040)), (47, 1920, (3856, 3840)),
    (49, 1024, (4096, 1040)), (63, 1920, (4112,)), (49, 2176, (3856, 3840)), (511, 4224, (2064,)),
])
def test_tiled_w16_gemm(M, K, ns):
    print(f"tiled W4A16 M={M} K={K} ns={ns}", flush=True)
    x = workloads.activations(M, K, workloads.generator(5000 + M)).half().cuda()
    ops_, refs, bounds = [], [], []
    for i, n in enumerate(ns):
        o, spec, s, sz = _operands(n, K, zlib.crc32(f"{K}{n}{i}".encode()), i == 0)
        b = o[5]
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


@pytest.mark.parametrize("M,K,ns", [
    (17, 1152, (4096, 1040)),
    (33, 1024, (12288, 12304)),          # one group per part of K, on both widths of workgroup
    (33, 1024, (4096, 1040)),
    (49, 1920, (3856, 3840)),            # parts of one and two groups
    (49, 2176, (3856, 3840)),
    (48, 2176, (9728, 9728)),            # 17 groups: parts of two and three
    (64, 1152, (12288, 12288)),          # a lone member this wide asks for another split of K than the pair
    (65, 1024, (16, 8192)),
    (96, 4096, (12288, 12288, 1024)),    # the pair asks for another number of waves than the narrow member
    (130, 1024, (12288, 12288)),
    (320, 2048, (4096, 1024, 1024)),
    (500, 1152, (5120, 1280, 1280)),     # the first member runs the prefill tiles by itself
    (512, 1408, (4096, 5120, 48, 16)),
])
def test_group_returns_its_members_bits(M, K, ns):
    print(f"W4A16 group against its members M={M} K={K} ns={ns}", flush=True)
    x = workloads.activations(M, K, workloads.generator(6000 + M)).half().cuda()
    ops_ = [_operands(n, K, 77 + i, i % 2 == 0)[0] for i, n in enumerate(ns)]
    get = lambda i: [o[i] for o in ops_]   # noqa: E731
    ys = torch.ops.paroquant.w4a16_linear_group(x, get(0), get(1), get(2), 8, get(3), get(4), get(5), False,
                                                torch.float32)
    for o, y in zip(ops_, ys):
        single = torch.ops.paroquant.w4a16_linear(x, *o[:3], 8, *o[3:], False, torch.float32)
        assert torch.equal(y, single)
