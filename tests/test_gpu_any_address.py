"""Rows that are no whole pieces of 16 bytes, and tensors that start behind such a boundary, go in whole pieces from wherever they start: the
same bits as the stages of their own, and nothing around a tensor is written."""
import pytest
import torch

from lmms_engine_amd import _abi
from tests.test_gpu_parity import env  # noqa: F401

pytestmark = pytest.mark.gpu

NS = (3.4445, -4.775, 2.0315)


# 128-tiles and 256-tiles, both orientations, rows that end inside a piece, at its edge and one element behind it
@pytest.mark.parametrize("rows,cols,batch", [(130, 257, 2), (257, 130, 2), (500, 641, 3), (641, 519, 3), (1024, 1031, 20), (1033, 1024, 20), (67, 65, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_parameters_at_any_address_equal_the_stages_bitwise(env, rows, cols, batch, dtype):
    print(f"update {batch} x {rows}x{cols} {dtype}", flush=True)
    lib, dev, code = env["lib"], env["dev"], _abi.dtype_code(dtype)
    gen = torch.Generator().manual_seed(rows + cols)
    n = rows * cols
    w, g = (torch.randn(batch, rows, cols, generator=gen).to(dtype) for _ in range(2))
    ws = torch.empty(lib.muon_hip_workspace_bytes(rows, cols, batch), dtype=torch.uint8, device=dev)
    for by in (1, 2, 5):  # elements behind a 16-byte boundary
        out = []
        for folded in (True, False):
            place = torch.full((batch, -(-n // 8) * 8 + 16), 7.0, dtype=dtype, device=dev)
            p = place[:, by:by + n]
            p.copy_(w.view(batch, n))
            gd, m = g.to(dev), torch.zeros(batch, rows, cols, dtype=dtype, device=dev)
            table = torch.tensor([t.data_ptr() for x in (p, gd, m) for t in x], dtype=torch.int64, device=dev)
            tp, tg, tm = (table.data_ptr() + 8 * batch * i for i in range(3))
            if folded:
                _abi.check(lib.muon_hip_step_grouped(tp, tg, tm, code, code, code, ws.data_ptr(), rows, cols, batch, 0.02, 0.01, 0.95, 1, 5, 0.7, *NS, 0, 0))
            else:
                _abi.check(lib.muon_hip_momentum_norm(tg, tm, code, code, ws.data_ptr(), rows, cols, batch, 0.95, 1, 0, 0))
                _abi.check(lib.muon_hip_ns_grouped(ws.data_ptr(), rows, cols, batch, 5, *NS, 0))
                _abi.check(lib.muon_hip_apply_update(tp, code, ws.data_ptr(), rows, cols, batch, 5, 0.7, 0.02, 0.01, 0))
            torch.cuda.synchronize()
            assert bool((place[:, :by] == 7).all()) and bool((place[:, by + n:] == 7).all())
            out.append(p.clone())
        assert torch.equal(*out) and not torch.equal(out[0].cpu(), w.view(batch, n)), by


@pytest.mark.parametrize("rows,cols,batch", [(130, 257, 2), (257, 130, 2), (640, 1001, 3), (1001, 640, 3)])
def test_results_at_any_address_and_their_values(env, rows, cols, batch):
    """muon_hip_ns_output after no iteration: bf(u / d) itself, from u's ragged rows into rows that start anywhere."""
    print(f"normalised {batch} x {rows}x{cols}", flush=True)
    lib, dev = env["lib"], env["dev"]
    G = torch.randn(batch, rows, cols, generator=torch.Generator().manual_seed(cols)).bfloat16().to(dev)
    ws = torch.empty(lib.muon_hip_workspace_bytes(rows, cols, batch), dtype=torch.uint8, device=dev)
    want = env["mu"].fast_newtonschulz(G, 0)
    d = (G.double().square().sum((1, 2), keepdim=True).sqrt().bfloat16().float() + 1e-7).bfloat16()
    assert torch.equal(want, (G.float() / d.float()).bfloat16())
    for by in (1, 4):
        buf = torch.full((G.numel() + 16,), 7.0, dtype=torch.bfloat16, device=dev)
        _abi.check(lib.muon_hip_cast_norm(G.data_ptr(), _abi.dtype_code(G.dtype), ws.data_ptr(), rows, cols, batch, 0))
        _abi.check(lib.muon_hip_normalize(ws.data_ptr(), rows, cols, batch, 0))
        _abi.check(lib.muon_hip_ns_output(ws.data_ptr(), rows, cols, batch, 0, buf.data_ptr() + 2 * by, 0))
        torch.cuda.synchronize()
        assert torch.equal(buf[by:by + G.numel()].view(G.shape), want)
        assert bool((buf[:by] == 7).all()) and bool((buf[by + G.numel():] == 7).all())


# one launch for all products, 64-tiles and 128-tiles in launches of their own, 256-tiles (where the result is copied), both orientations
@pytest.mark.parametrize("rows,cols,batch,steps", [(1024, 256, 48, 5), (256, 1024, 48, 2), (130, 701, 64, 1), (701, 130, 33, 2), (896, 4864, 1, 5), (4864, 896, 1, 1),
                                                   (300, 1001, 3, 2), (1001, 299, 3, 2), (640, 2560, 60, 1), (1408, 1408, 16, 1), (1024, 1024, 40, 2), (520, 512, 2, 0)])
def test_results_written_by_the_last_product_equal_the_copy_bitwise(env, rows, cols, batch, steps):
    print(f"result of {batch} x {rows}x{cols}, {steps} steps", flush=True)
    lib, dev = env["lib"], env["dev"]
    G = torch.randn(batch, rows, cols, generator=torch.Generator().manual_seed(rows + cols)).bfloat16().to(dev)
    ws = torch.empty(lib.muon_hip_workspace_bytes(rows, cols, batch), dtype=torch.uint8, device=dev)
    n, ref = G.numel(), torch.empty_like(G)
    for by in (0, 1):
        buf = torch.full((n + 16,), 7.0, dtype=torch.bfloat16, device=dev)
        for direct in (True, False):
            _abi.check(lib.muon_hip_cast_norm(G.data_ptr(), _abi.dtype_code(G.dtype), ws.data_ptr(), rows, cols, batch, 0))
            if direct:
                _abi.check(lib.muon_hip_ns_result(ws.data_ptr(), rows, cols, batch, steps, *NS, buf.data_ptr() + 16 + 2 * by, 0))
            else:
                _abi.check(lib.muon_hip_ns_grouped(ws.data_ptr(), rows, cols, batch, steps, *NS, 0))
                _abi.check(lib.muon_hip_ns_output(ws.data_ptr(), rows, cols, batch, steps, ref.data_ptr(), 0))
        torch.cuda.synchronize()
        at = 8 + by
        assert bool(torch.isfinite(ref.float()).all()) and torch.equal(buf[at:at + n].view(G.shape), ref), by
        assert bool((buf[:at] == 7).all()) and bool((buf[at + n:] == 7).all())
