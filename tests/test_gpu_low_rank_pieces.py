"""Matrices with a short side of at most 64 in whole pieces: turned ones of every multiple of four rows, on and off the boundaries that the
pieces need, widths of several kernels in one launch, divisions that a reciprocal cannot stand for."""
import pytest
import torch

from lmms_engine_amd import _abi
from tests.test_gpu_parity import env  # noqa: F401

pytestmark = pytest.mark.gpu

# the edges of pieces of four and of eight, of blocks of 16 rows and of chunks of 32 columns, and a short and a long run of chunks per wave
SHAPES = [(4, 33), (8, 250), (12, 2049), (16, 31), (16, 5632), (20, 264), (24, 1000), (28, 4096), (32, 47), (36, 100), (48, 1025), (60, 2048), (64, 72)]


@pytest.mark.parametrize("offset", [0, 1, 2, 4])
@pytest.mark.parametrize("pdtype", [torch.float32, torch.bfloat16])
def test_turned_parameters_are_bitwise_the_tiled_products(env, pdtype, offset):
    """Parameters `offset` elements behind a 16-byte boundary; one step over all shapes, both ways round, so that matrices of every width
    meet in a launch; nothing around a parameter is written."""
    print(f"turned pieces {pdtype} offset {offset}", flush=True)
    lib, mu, dev = env["lib"], env["mu"], env["dev"]
    gen = torch.Generator().manual_seed(8)
    shapes = [(c, r) for r, c in SHAPES] + SHAPES
    ws = [(0.02 * torch.randn(*s, generator=gen)).to(pdtype) for s in shapes]
    gs = [(1e-3 * torch.randn(*s, generator=gen)).to(pdtype) for s in shapes]
    out = []
    for cfg in (_abi.CFG_AUTO, _abi.CFG_128_PIPE):
        places = [torch.full((w.numel() + offset + 8,), 7.0, dtype=pdtype, device=dev) for w in ws]
        params = [torch.nn.Parameter(b[offset:offset + w.numel()].view(w.shape).copy_(w)) for b, w in zip(places, ws)]
        for p, g in zip(params, gs):
            p.grad = g.to(dev)
        _abi.check(lib.muon_hip_set_gemm_config(cfg))
        try:
            mu.Muon([dict(params=list(params), use_muon=True, lr=0.02, momentum=0.95, nesterov=True, weight_decay=0.01, ns_steps=5, rms_scale=True)]).step()
        finally:
            _abi.check(lib.muon_hip_set_gemm_config(_abi.CFG_AUTO))
        torch.cuda.synchronize()
        for b, w in zip(places, ws):
            assert bool((b[:offset] == 7).all()) and bool((b[offset + w.numel():] == 7).all())
        out.append([p.detach() for p in params])
    for s, p, q in zip(shapes, *out):
        assert torch.equal(p, q), s


@pytest.mark.parametrize("narrow,wide", [(3, 2), (384, 5), (385, 5)])
def test_widths_together_and_apart_are_bitwise_the_tiled_products(env, narrow, wide):
    """The line between one launch for all widths and one per width, on a device of 256 compute units."""
    print(f"{narrow} narrow, {wide} wide", flush=True)
    lib, mu, dev = env["lib"], env["mu"], env["dev"]
    gen = torch.Generator().manual_seed(narrow)
    shapes = [(16, 96)] * (narrow - 1) + [(96, 16)] + [(16, 5000)] * (wide - 1) + [(4100, 16)]
    ws, gs = ([0.02 * torch.randn(*s, generator=gen) for s in shapes] for _ in range(2))
    out = []
    for cfg in (_abi.CFG_AUTO, _abi.CFG_128_PIPE):
        params = [torch.nn.Parameter(w.to(dev)) for w in ws]
        for p, g in zip(params, gs):
            p.grad = g.to(dev)
        _abi.check(lib.muon_hip_set_gemm_config(cfg))
        try:
            mu.Muon([dict(params=list(params), use_muon=True, lr=0.02, momentum=0.95, nesterov=True, weight_decay=0.01, ns_steps=5)]).step()
        finally:
            _abi.check(lib.muon_hip_set_gemm_config(_abi.CFG_AUTO))
        torch.cuda.synchronize()
        out.append([p.detach() for p in params])
    assert all(torch.equal(p, q) for p, q in zip(*out))


@pytest.mark.parametrize("rows,cols", [(16, 96), (64, 128), (20, 61), (128, 256), (101, 259)])
def test_quotients_among_the_subnormal_numbers(env, rows, cols):
    """Elements so far below the norm that X = u / d is no normal number, beside ordinary ones: the quotient itself, of IEEE division, in X
    after no iteration, and the same bits on the chain and on the tiled kernels after one."""
    print(f"subnormal quotients {rows}x{cols}", flush=True)
    lib, mu, dev = env["lib"], env["mu"], env["dev"]
    gen = torch.Generator().manual_seed(rows)
    g = torch.randn(2, rows, cols, generator=gen) * torch.exp2(torch.randint(-130, 8, (2, rows, cols), generator=gen).float())
    g[1] *= 2.0**20
    g = g.bfloat16()
    assert bool(((g[0].float().abs() < 2.0**-126) & (g[0] != 0)).any())
    for x in (g.to(dev), g.mT.contiguous().to(dev)):
        d = (x.float().double().square().sum((1, 2), keepdim=True).sqrt().bfloat16().float() + 1e-7).bfloat16()
        want = (x.float() / d.float()).bfloat16()
        got = mu.fast_newtonschulz(x, 0)
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
        got = mu.fast_newtonschulz(x, 1)
        _abi.check(lib.muon_hip_set_gemm_config(_abi.CFG_128_PIPE))
        try:
            ref = mu.fast_newtonschulz(x, 1)
        finally:
            _abi.check(lib.muon_hip_set_gemm_config(_abi.CFG_AUTO))
        torch.cuda.synchronize()
        assert torch.equal(got, ref)
