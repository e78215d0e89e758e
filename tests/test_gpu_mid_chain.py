"""Matrices with a short side of 65 to 128 and a long one of at most 512, whose whole Newton-Schulz chain runs in one workgroup each as well: the
edges of that range and of its blocks, chunks and pieces, both orientations, special values, and steps in which they meet shorter ones."""
import pytest
import torch

from lmms_engine_amd import _abi
from tests.helpers import rel_fro
from tests.test_gpu_parity import NS_TOL, env  # noqa: F401

pytestmark = pytest.mark.gpu

SHAPES = [(65, 65), (65, 66), (68, 96), (80, 257), (96, 96), (97, 250), (100, 511), (113, 264), (127, 129), (128, 128), (128, 255), (128, 256), (128, 512), (65, 512)]
BEYOND = [(65, 513), (129, 129), (128, 1024)]  # the tiled products


def _named(fn):
    _abi.check(_abi.lib().muon_hip_set_gemm_config(_abi.CFG_128_PIPE))
    try:
        return fn()
    finally:
        _abi.check(_abi.lib().muon_hip_set_gemm_config(_abi.CFG_AUTO))


@pytest.mark.parametrize("rows,cols", SHAPES + BEYOND)
def test_bitwise_the_tiled_products(env, rows, cols):
    print(f"mid chain {rows}x{cols}", flush=True)
    mu, O, dev = env["mu"], env["O"], env["dev"]
    G = torch.randn(3, rows, cols, generator=torch.Generator().manual_seed(rows * 11 + cols))
    G *= torch.logspace(-3, 1, rows).view(1, rows, 1)
    for g in (G.to(dev), G.mT.contiguous().to(dev)):
        for steps in (1, 2, 5):
            got, ref = mu.fast_newtonschulz(g, steps), _named(lambda: mu.fast_newtonschulz(g, steps))
            torch.cuda.synchronize()
            assert bool(torch.isfinite(ref.float()).all()) and torch.equal(got, ref), steps
        assert rel_fro(got[0], O.newton_schulz(g[0].cpu(), 5)) <= NS_TOL


@pytest.mark.parametrize("rows,cols", [(65, 70), (128, 128), (100, 301), (128, 512)])
def test_infinities_zeros_and_nan(env, rows, cols):
    """The same values and the same NaN as on the tiled kernels."""
    print(f"mid chain, special values {rows}x{cols}", flush=True)
    mu, dev = env["mu"], env["dev"]
    G = torch.randn(7, rows, cols, generator=torch.Generator().manual_seed(rows))
    G[0] = 0.0
    G[1, rows // 2, cols // 3] = float("inf")
    G[2, 0, cols - 1] = float("nan")
    G[3] *= 1e30
    G[4] *= 1e-36
    G[5, :, 1:] = 0.0
    for g in (G.to(dev), G.mT.contiguous().to(dev)):
        for steps in (1, 5):
            got, ref = mu.fast_newtonschulz(g, steps), _named(lambda: mu.fast_newtonschulz(g, steps))
            torch.cuda.synchronize()
            assert torch.equal(got.isnan(), ref.isnan()), steps
            assert torch.equal(got.nan_to_num(nan=0.0).view(torch.int16), ref.nan_to_num(nan=0.0).view(torch.int16)), steps


# shorter matrices with no more columns go along in the launch, those with more and larger ones do not; more workgroups than a device of 256
# compute units has at once
@pytest.mark.parametrize("shapes", [
    [(s, 1) for s in SHAPES] + [((64, 128), 2), ((16, 96), 1), ((24, 500), 1), ((16, 2048), 1)], [((128, 384), 4), ((64, 128), 4), ((256, 512), 8)],
    [((128, 128), 200), ((48, 100), 56)], [((128, 128), 200), ((48, 100), 57)], [((128, 128), 385), ((100, 400), 3)],
])
@pytest.mark.parametrize("dtype,offset", [(torch.float32, 0), (torch.bfloat16, 0), (torch.bfloat16, 3)])
def test_steps_are_bitwise_the_tiled_products(env, shapes, dtype, offset):
    print(f"mid chain step {len(shapes)} shapes {dtype} offset {offset}", flush=True)
    mu, dev = env["mu"], env["dev"]
    gen = torch.Generator().manual_seed(len(shapes))
    all_shapes = [s for (r, c), n in shapes for k in range(n) for s in [(r, c) if k % 2 == 0 else (c, r)]]
    ws = [(0.02 * torch.randn(*s, generator=gen)).to(dtype) for s in all_shapes]
    gs = [(1e-3 * torch.randn(*s, generator=gen)).to(dtype) for s in all_shapes]

    def steps():
        places = [torch.full((w.numel() + offset + 8,), 7.0, dtype=dtype, device=dev) for w in ws]
        ps = [torch.nn.Parameter(b[offset:offset + w.numel()].view(w.shape).copy_(w)) for b, w in zip(places, ws)]
        for p, g in zip(ps, gs):
            p.grad = g.to(dev)
        opt = mu.Muon([dict(params=list(ps), use_muon=True, lr=0.02, momentum=0.95, nesterov=True, weight_decay=0.01, ns_steps=5, rms_scale=True)],
                      momentum_dtype=torch.float32)
        opt.step(), opt.step()
        torch.cuda.synchronize()
        assert all(bool((b[:offset] == 7).all()) and bool((b[offset + w.numel():] == 7).all()) for b, w in zip(places, ws))
        return [p.detach() for p in ps]

    for s, p, q in zip(all_shapes, steps(), _named(steps)):
        assert torch.equal(p, q), s


# every number of elements that a row's last piece of eight, or a column's last piece of four, can have, in a wave's first and second chunk
@pytest.mark.parametrize("dtype,offsets", [(torch.float32, (0, 1)), (torch.bfloat16, (0, 1, 4))])
def test_parameters_that_end_inside_a_piece(env, dtype, offsets):
    lib, dev, code = env["lib"], env["dev"], _abi.dtype_code(dtype)
    shapes = [(66, 472 + k) for k in range(1, 8)] + [(66, 240 + k) for k in range(1, 8)] + [(479 - k, 124 + k) for k in range(1, 4)] + [(130 + k, 68 - k) for k in range(1, 4)]
    for rows, cols in shapes:
        print(f"cut pieces {rows}x{cols} {dtype}", flush=True)
        gen = torch.Generator().manual_seed(rows + cols)
        n = rows * cols
        w, g = (torch.randn(2, rows, cols, generator=gen).to(dtype) for _ in range(2))
        ws = torch.empty(lib.muon_hip_workspace_bytes(rows, cols, 2), dtype=torch.uint8, device=dev)
        assert _abi.routes([(rows, cols, 2)], "small_chain")[0][1] == 128
        for by in offsets:
            out = []
            for folded in (True, False):
                place = torch.full((2, -(-n // 8) * 8 + 16), 7.0, dtype=dtype, device=dev)
                p = place[:, by:by + n]
                p.copy_(w.view(2, n))
                gd, m = g.to(dev), torch.zeros(2, rows, cols, dtype=dtype, device=dev)
                table = torch.tensor([t.data_ptr() for x in (p, gd, m) for t in x], dtype=torch.int64, device=dev)
                tp, tg, tm = (table.data_ptr() + 16 * i for i in range(3))
                ns = (3.4445, -4.775, 2.0315)
                if folded:
                    _abi.check(lib.muon_hip_step_grouped(tp, tg, tm, code, code, code, ws.data_ptr(), rows, cols, 2, 0.02, 0.01, 0.95, 1, 5, 0.7, *ns, 0, 0))
                else:
                    _abi.check(lib.muon_hip_momentum_norm(tg, tm, code, code, ws.data_ptr(), rows, cols, 2, 0.95, 1, 0, 0))
                    _abi.check(lib.muon_hip_ns_grouped(ws.data_ptr(), rows, cols, 2, 5, *ns, 0))
                    _abi.check(lib.muon_hip_apply_update(tp, code, ws.data_ptr(), rows, cols, 2, 5, 0.7, 0.02, 0.01, 0))
                torch.cuda.synchronize()
                assert bool((place[:, :by] == 7).all()) and bool((place[:, by + n:] == 7).all())
                out.append(p.clone())
            assert torch.equal(*out) and not torch.equal(out[0].cpu(), w.view(2, n)), (rows, cols, by)


@pytest.mark.parametrize("rows,cols,batch", [(100, 333, 3), (333, 100, 3), (333, 101, 2), (128, 256, 260), (511, 128, 2)])
def test_results_and_stages_bitwise(env, rows, cols, batch):
    """muon_hip_ns_result against muon_hip_ns_grouped and muon_hip_ns_output, on aligned outputs and on others, and nothing around them."""
    print(f"mid chain result {batch} x {rows}x{cols}", flush=True)
    lib, dev = env["lib"], env["dev"]
    G = torch.randn(batch, rows, cols, generator=torch.Generator().manual_seed(rows + cols)).to(dev)
    ws = torch.empty(lib.muon_hip_workspace_bytes(rows, cols, batch), dtype=torch.uint8, device=dev)
    n, ns = G.numel(), (5, 3.4445, -4.775, 2.0315)
    for shift in (8, 4, 1):
        buf = torch.full((n + 16,), 7.0, dtype=torch.bfloat16, device=dev)
        ref = torch.empty(G.shape, dtype=torch.bfloat16, device=dev)
        for direct in (True, False):
            _abi.check(lib.muon_hip_cast_norm(G.data_ptr(), _abi.dtype_code(G.dtype), ws.data_ptr(), rows, cols, batch, 0))
            if direct:
                _abi.check(lib.muon_hip_ns_result(ws.data_ptr(), rows, cols, batch, *ns, buf.data_ptr() + 2 * shift, 0))
            else:
                _abi.check(lib.muon_hip_ns_grouped(ws.data_ptr(), rows, cols, batch, *ns, 0))
                _abi.check(lib.muon_hip_ns_output(ws.data_ptr(), rows, cols, batch, 5, ref.data_ptr(), 0))
        torch.cuda.synchronize()
        assert torch.equal(buf[shift:shift + n].view(G.shape), ref), shift
        assert bool((buf[:shift] == 7).all()) and bool((buf[shift + n:] == 7).all())
