"""rotation::rotate and rotate_and_quant_mxfp4 from 4 M elements (the register chain derived on the device; one and two
layers without codes from 6 M) against the
tile kernel that fewer run: the same float32 sequence, so the same bits, for every layer count, group size, odd row
slice and the 64-channel tail; also for indices that pair no proper matching, and for blocks with NaN and infinities."""

import zlib

import numpy as np
import pytest
import torch

import alpamayo_amd  # noqa: F401
from tests.gpu_util import kernel_instances, to_np
from tests.test_gpu_rotate import DT, _params

pytestmark = pytest.mark.gpu


def _both(x, pairs, th, sc, gs):
    rot = torch.ops.rotation.rotate
    mx = torch.ops.rotation.rotate_and_quant_mxfp4
    y, (q, s) = rot(x, pairs, th, sc, gs), mx(x, pairs, th, sc, gs)
    assert x.numel() >= 1 << 22
    few = [c.contiguous() for c in x.split(x.size(0) // 2)]
    assert all(c.numel() < 1 << 22 for c in few)
    yt = torch.cat([rot(c, pairs, th, sc, gs) for c in few])
    parts = [mx(c, pairs, th, sc, gs) for c in few]
    qt, st = (torch.cat([p[i] for p in parts]) for i in range(2))
    bits = torch.int32 if x.dtype == torch.float32 else torch.int16
    assert torch.equal(y.view(bits), yt.view(bits))
    assert torch.equal(q, qt) and torch.equal(s, st)


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("gs,krot,h,rows", [(128, 8, 256, 16385), (64, 1, 64, 65601), (64, 2, 192, 21900),
                                            (128, 4, 384, 10931), (64, 16, 320, 13113), (128, 8, 4096, 1027),
                                            (128, 16, 128, 32773),
                                            # one and two layers without MXFP4 codes: from 6 M elements
                                            (64, 1, 64, 93761), (64, 2, 192, 31261), (128, 2, 640, 9379)])
@pytest.mark.parametrize("with_scale", [True, False])
def test_chain_equals_tile(dt, gs, krot, h, rows, with_scale):
    print(f"chain dt={dt} gs={gs} krot={krot} h={h} rows={rows} scale={with_scale}", flush=True)
    rng = np.random.default_rng(zlib.crc32(f"chain{dt}{gs}{krot}{h}{rows}".encode()))
    pairs, theta, scales = _params(rng, krot, h, gs)
    x = torch.from_numpy(rng.standard_normal((rows, h)).astype(np.float32) * 3).to(DT[dt]).cuda()
    sc = torch.from_numpy(scales).to(DT[dt]).reshape(1, h).cuda() if with_scale else None
    _both(x, torch.from_numpy(pairs).cuda(), torch.from_numpy(theta).to(DT[dt]).cuda(), sc, gs)


@pytest.mark.parametrize("krot,rows,h,chain,mx_chain", [
    (8, 1024, 4096, True, True), (8, 1023, 4096, False, False), (1, 1024, 4096, False, True), (2, 1465, 4096, True, True),
    (8, 31, 262144, False, False), (8, 32, 262144, True, True), (16, 1, 1 << 22, False, False),
])
def test_form_by_size(krot, rows, h, chain, mx_chain):
    """The chain where every workgroup has a step of rows for it and the launch is large, else the tile form."""
    print(f"form krot={krot} {rows}x{h}", flush=True)
    x = torch.randn(rows, h, device="cuda").half()
    pairs = torch.arange(128, dtype=torch.int16).repeat(krot, h // 128).cuda()
    th = torch.rand(krot, h // 2, device="cuda").half()
    for op, want in ((torch.ops.rotation.rotate, chain), (torch.ops.rotation.rotate_and_quant_mxfp4, mx_chain)):
        found = kernel_instances(lambda: op(x, pairs, th, None, 128), r"rotate_\w+")   # noqa: B023
        assert [f[0] for f in found] == ["rotate_chain" if want else "rotate_kernel"]


@pytest.mark.parametrize("krot,rows,h,chain", [
    (8, 192, 4096, True), (8, 191, 4096, False), (8, 31, 65536, False), (8, 32, 65536, True), (4, 1, 1 << 20, False),
    (16, 47, 65536, False), (16, 48, 65536, True), (16, 300, 4096, False),
])
def test_backward_form_by_size(krot, rows, h, chain):
    print(f"backward form krot={krot} {rows}x{h}", flush=True)
    x, gy = torch.randn(2, rows, h, device="cuda").unbind(0)
    pairs = torch.arange(128, dtype=torch.int16).repeat(krot, h // 128).cuda()
    th = torch.rand(krot, h // 2, device="cuda")
    found = kernel_instances(lambda: torch.ops.paroquant.rotate_backward(gy, x, pairs, th, None, 128), "rotate_chain_bwd")
    assert [f[1][3] for f in found] == [str(chain).lower()]


def test_special_values_and_fixed_layers():
    """The identity pairing in every layer (cycles of length two) and pairs that repeat from layer to layer; rows with
    NaN and infinities in single channels."""
    rng = np.random.default_rng(11)
    pairs, theta, _ = _params(rng, 8, 256, 128)
    pairs[2:5] = pairs[1]
    pairs[6] = np.tile(np.arange(128), 2)
    x = rng.standard_normal((16400, 256)).astype(np.float32)
    x[3, 17], x[9, 140], x[77, 0], x[150, 255] = np.nan, np.inf, -np.inf, np.nan
    x[20], x[21, :128] = 0.0, 0.0
    for dt in DT.values():
        _both(torch.from_numpy(x).to(dt).cuda(), torch.from_numpy(pairs).cuda(), torch.from_numpy(theta).to(dt).cuda(),
              None, 128)


def test_pairs_without_a_matching():
    """A layer whose pairs name one channel twice each (its lanes write no channel in common) in one of two groups:
    the tile form's result."""
    rng = np.random.default_rng(12)
    pairs, theta, _ = _params(rng, 4, 256, 128)
    pairs[2, :128] = np.repeat(np.arange(64), 2)
    x = torch.from_numpy(rng.standard_normal((16400, 256)).astype(np.float32)).cuda()
    p, th = torch.from_numpy(pairs).cuda(), torch.from_numpy(theta).cuda()
    _both(x, p, th, None, 128)
    # its backward: the second channel of a pair is the one written
    rows = 3100   # past the size from which the backward looks for a chain
    x = x[:rows].contiguous()
    gy = torch.from_numpy(rng.standard_normal((rows, 256)).astype(np.float32)).cuda()
    gx, gth, _ = torch.ops.paroquant.rotate_backward(gy, x, p, th, None, 128)
    v, outs = to_np(x).astype(np.float64), []
    for r in range(4):
        for g in (0, 128):
            i, j = g + pairs[r, g:g + 128:2], g + pairs[r, g + 1:g + 128:2]
            t = theta[r, g // 2:g // 2 + 64].astype(np.float64)
            a, b = v[:, i].copy(), v[:, j].copy()
            na, nb = a * np.cos(t) + b * np.sin(t), b * np.cos(t) - a * np.sin(t)
            v[:, i] = na
            v[:, j] = nb
            outs.append((r, g, i, j, t, na, nb))
    u = to_np(gy).astype(np.float64)
    ref = np.zeros_like(theta, dtype=np.float64)
    for r, g, i, j, t, na, nb in reversed(outs):
        a, b = u[:, i].copy(), u[:, j].copy()
        ref[r, g // 2:g // 2 + 64] = (a * nb - b * na).sum(0)
        u[:, i] = a * np.cos(t) - b * np.sin(t)
        u[:, j] = b * np.cos(t) + a * np.sin(t)
    assert np.linalg.norm(to_np(gx) - u) <= 1e-5 * np.linalg.norm(u)
    assert np.linalg.norm(to_np(gth) - ref) <= 1e-5 * np.linalg.norm(ref)
