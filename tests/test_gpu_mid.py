"""The GEMM on tiled int8 activations (17 rows up to a few hundred) behind the W4A8 linear entry points, at the edges
of its row blocks, column units and K splits: the codes and int32 partials as in test_gpu_intermediates.py, and the
float32 outputs against float64 sums of the same codes.

Bound of the outputs: a sum of G float32 terms s_g * P_g (P_g exact in float32, one fma each), in any order, then one
product with the token scale and one add of the bias, is off by at most (G + 3) 2^-24 sum_g |s_g P_g| * xscale + 2^-24 |y|.
"""

import zlib

import numpy as np
import pytest
import torch

import alpamayo_amd  # noqa: F401
from alpamayo_amd import ops, workloads
from tests.gpu_util import gemm_instances, to_np
from tests.test_gpu_group import _members
from tests.test_gpu_intermediates import _check, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,ns,flags", [
    (17, 1024, (16,), (True, True)),             # one wave per group of K, one ragged column unit
    (31, 1152, (4096,), (True, True)),           # nine groups over eight waves, one column tile per wave
    (32, 4096, (4112, 48), (True, True)),        # odd column tiles in both members
    (33, 4096, (4096, 1024, 1024), (True, True)),
    (47, 12288, (4096,), (True, True)),
    (64, 1408, (8192, 8208), (True, True)),
    (65, 4096, (4096,), (True, True)),           # first size on the row rotate+quant kernel
    (97, 2048, (1040, 80), (False, False)),      # float32 rows
    (128, 4096, (4096, 1024, 1024), (True, True)),
    (200, 4224, (4096,), (True, True)),          # 33 groups: uneven K splits
    (255, 1024, (5120,), (True, True)),
    (511, 1024, (1040,), (True, True)),          # the most rows it takes, less one
    (160, 1152, (12288, 12304), (True, True)),   # too wide: 128 x 256 prefill tiles in four chains of K
    (113, 1408, (24576,), (True, True)),         # one wide member: the widest launch of the tiled kernel itself
    (96, 1152, (16384, 16400), (True, True)),    # a group too wide for one round, each member in less than one
    (113, 1408, (8192,) * 4, (True, True)),
    (500, 1152, (6144, 1280), (True, True)),     # short rows past 384 rows: the prefill tiles in one chain
    (96, 2048, (12288, 48), (True, True)),       # the most rows on eight waves
    (97, 2048, (8192, 8208), (True, True)),      # and the first past them: 64 x 128 tiles in four chains
    (128, 1024, (12288, 4112), (True, True)),
    (256, 4096, (4096, 1040, 1024), (True, True)),
    (257, 3072, (3072, 3088), (True, True)),     # short rows up to 384 rows
    (384, 1024, (5120, 272), (True, True)),
    (320, 6144, (16384, 1040), (True, True)),    # long rows up to 512: 128 x 256 tiles in four chains
    (512, 6144, (4096, 48), (False, True)),
    (513, 6144, (4096, 48), (True, True)),       # the first row count past the mid-size GEMM
])
def test_tiled_gemm(M, K, ns, flags):
    print(f"tiled GEMM M={M} K={K} ns={ns} flags={flags}", flush=True)
    krot = 8
    mbs = _members(ns, K, krot, zlib.crc32(f"mid{ns}-{K}".encode()), with_bias=True)
    x = workloads.activations(M, K, workloads.generator(7 * M + K)).cuda()
    codes, xscale, parts, _, _ = _run(mbs, x, krot, flags)
    rows = np.unique(np.concatenate([np.arange(0, M, max(1, M // 24)), np.arange(max(0, M - 17), M)]))
    _check(mbs, to_np(x), codes, xscale, parts, flags, rows=rows)
    args = ([m["rot_idx"] for m in mbs], [m["rot_cs"] for m in mbs], [m["scales"] for m in mbs], krot,
            [m["wp"] for m in mbs], [m["wm"] for m in mbs], [m["bias"] for m in mbs], *flags)
    ys = torch.ops.paroquant.w4a8_linear_group(x, *args, torch.float32)
    y16 = torch.ops.paroquant.w4a8_linear_group(x, *args, torch.bfloat16)
    for i, (mb, y) in enumerate(zip(mbs, ys)):
        sc = (mb["wm"].cpu().numpy().view(np.uint32) & 0xFFFF).astype(np.uint16).view(np.float16)   # [N/16, G, 16]
        s = sc.transpose(1, 0, 2).reshape(K // 128, -1).astype(np.float64)
        terms = to_np(parts[i]).astype(np.float64) * s[None]
        xs = to_np(xscale[i]).astype(np.float64)[:, None]
        b = to_np(mb["bias"].float()).astype(np.float64) if mb["bias"] is not None else np.zeros(1)
        ref = terms.sum(1) * xs + b
        bound = (K // 128 + 3) * 2.0 ** -24 * np.abs(terms).sum(1) * xs + 2.0 ** -23 * (np.abs(ref) + np.abs(b))
        assert np.all(np.abs(to_np(y).astype(np.float64) - ref) <= bound)
        if M > 64:   # the bits of the member called by itself, whichever kernel that call takes
            single = torch.ops.paroquant.w4a8_linear(x, *(a[i] for a in args[:3]), krot, *(a[i] for a in args[4:7]), *flags,
                                                     torch.float32)
            assert torch.equal(y, single)
        assert torch.equal(y16[i].view(torch.int16), y.to(torch.bfloat16).view(torch.int16))


@pytest.mark.parametrize("M,K,ns", [
    (24, 2048, (4096,)), (80, 2048, (4096, 1040)), (144, 1152, (12288, 12304)), (200, 4096, (8192, 8192)),
    (500, 1152, (6144, 1280)), (500, 6144, (6144, 1280)),
])
def test_parity_form_runs_the_tiles_of_the_product(M, K, ns):
    """pq_w4a8_linear_group_intermediates multiplies on the kernel and tiling that the linear takes: the same template
    arguments but for the partials flag and, of gemm_prefill, the chains of the sum that the partials precede, of
    gemm_mid the cache policy of its weight loads."""
    print(f"instances M={M} K={K} ns={ns}", flush=True)
    mbs = _members(ns, K, 8, 5, with_bias=False)
    x = workloads.activations(M, K, workloads.generator(M)).cuda()
    get = lambda key: [m[key] for m in mbs]   # noqa: E731
    args = (get("rot_idx"), get("rot_cs"), get("scales"), 8, get("wp"), get("wm"), get("bias"), True, True)
    own = {"gemm_prefill": (0, 1, 2, 3, 5, 6), "gemm_mid": (0, 1, 2, 3)}
    got, want = ([(n, tuple(a[i] for i in own[n])) for n, a in gemm_instances(f)] for f in
                 (lambda: _run(mbs, x, 8, (True, True)),
                  lambda: torch.ops.paroquant.w4a8_linear_group(x, *args, torch.bfloat16)))
    assert want and got == want


SKINNY, MID, PREFILL = "gemm_skinny", "gemm_mid", "gemm_prefill"


@pytest.mark.parametrize("M,K,ns,kernel,rows", [
    (16, 4096, (4096,), SKINNY, None), (17, 4096, (4096,), MID, None),
    (24, 1024, (12288,), SKINNY, None), (24, 1536, (4096,), SKINNY, None), (24, 2048, (4096,), MID, None),
    (33, 1024, (4096,), MID, None), (33, 1024, (24576,), SKINNY, None), (33, 1536, (24576,), MID, None),
    (64, 4096, (12288, 12288), MID, None), (65, 4096, (12288, 12288), MID, None),
    (112, 4096, (12288, 12288), PREFILL, 64), (112, 4096, (4096, 1024, 1024), MID, None),
    (144, 4096, (8192, 8192), MID, None), (200, 4096, (12288, 12288), PREFILL, 128), (256, 4096, (4096,), MID, None),
    (257, 4096, (4096,), PREFILL, None), (320, 4096, (12288, 12288), PREFILL, 192),
    (384, 4096, (12288, 12288), PREFILL, 192), (320, 12288, (4096,), MID, None), (500, 1024, (4096,), PREFILL, None),
    (300, 2048, (2048, 512, 512), MID, None), (400, 2048, (2048, 512, 512), PREFILL, None),
    (512, 12288, (4096,), MID, None), (513, 12288, (4096,), PREFILL, None),
])
def test_kernel_by_size(M, K, ns, kernel, rows):
    """The kernel, and of gemm_prefill the rows of a tile, that each range of sizes measured fastest on."""
    print(f"dispatch M={M} K={K} ns={ns}", flush=True)
    dev = "cuda"
    identity = torch.stack([torch.ones(1, K // 2), torch.zeros(1, K // 2)], dim=-1)
    rot_idx, rot_cs = (t.to(dev) for t in ops.pack_rotation(torch.arange(128).repeat(1, K // 128), identity))
    wps = [torch.zeros(n // 16, K // 128, 64, 16, dtype=torch.uint8, device=dev) for n in ns]
    wms = [torch.zeros(n // 16, K // 128, 16, dtype=torch.int32, device=dev) for n in ns]
    c = len(ns)
    x = torch.zeros(M, K, dtype=torch.bfloat16, device=dev)
    found = gemm_instances(lambda: torch.ops.paroquant.w4a8_linear_group(
        x, [rot_idx] * c, [rot_cs] * c, [None] * c, 1, wps, wms, [None] * c, True, True, torch.bfloat16))
    assert [f[0] for f in found] == [kernel] and (rows is None or found[0][1][0] == str(rows))
