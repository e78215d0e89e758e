"""Matrices with a short side of at most 64, whose whole Newton-Schulz chain runs in one workgroup each (small_chain.hip): edges
of the 16-row blocks and 32-column chunks, one chunk per wave and less, the longest long side of every kernel and one past it
(which the tiled products take), one row past it, both orientations, ragged sizes."""
import pytest
import torch

from tests.helpers import rel_fro
from tests.test_gpu_parity import NS_TOL, env  # noqa: F401

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (1, 9), (3, 33), (15, 16), (16, 31), (16, 256), (16, 257), (13, 2048), (16, 2049), (16, 4097), (16, 8192), (7, 8185),
          (17, 17), (32, 96), (24, 1024), (32, 1025), (31, 4095), (33, 64), (64, 64), (64, 512), (48, 513), (50, 1025), (64, 2048),
          (16, 8193), (32, 4097), (64, 2049), (65, 128), (65, 513)]


@pytest.mark.parametrize("rows,cols", SHAPES)
def test_small_chain_against_the_oracle(env, rows, cols):
    """One iteration differs from the oracle by the order of its fp32 sums, which a bf16 rounding shows as one unit in the last place
    (2^-8) of the few values next to a rounding point: below 2e-3 in norm, plus 2^-8 where the norm itself, a bf16 value, comes out as its
    neighbour.  More iterations are held to the bound of every shape."""
    print(f"small chain {rows}x{cols}", flush=True)
    mu, O = env["mu"], env["O"]
    G = torch.randn(2, rows, cols, generator=torch.Generator().manual_seed(rows * 7 + cols)) * 1e-3
    for g in (G, G.mT.contiguous()):
        for steps, tol in ((1, 2e-3 + 2**-8), (2, NS_TOL), (5, NS_TOL)):
            got = mu.fast_newtonschulz(g.to(env["dev"]), steps)
            assert got.shape == g.shape
            for i in range(2):
                assert rel_fro(got[i], O.newton_schulz(g[i], steps)) <= tol, (steps, i)


@pytest.mark.parametrize("rows,cols", SHAPES)
def test_small_chain_is_bitwise_the_tiled_products(env, rows, cols):
    """Every fp32 sum of the chain runs in the order of the tiled kernels (ascending k in 32-deep MFMAs), so a configuration named
    for the tiled products gives the same bits."""
    print(f"small chain against tiles {rows}x{cols}", flush=True)
    lib, abi, mu = env["lib"], env["abi"], env["mu"]
    G = torch.randn(3, rows, cols, generator=torch.Generator().manual_seed(rows * 11 + cols))
    G *= torch.logspace(-3, 1, rows).view(1, rows, 1)  # rows of different sizes, as gradients have: small singular values too
    for g in (G.to(env["dev"]), G.mT.contiguous().to(env["dev"])):
        for steps in (1, 2, 5):
            got = mu.fast_newtonschulz(g, steps)
            abi.check(lib.muon_hip_set_gemm_config(abi.CFG_128_PIPE))
            try:
                ref = mu.fast_newtonschulz(g, steps)
            finally:
                abi.check(lib.muon_hip_set_gemm_config(abi.CFG_AUTO))
            torch.cuda.synchronize()
            assert bool(torch.isfinite(ref.float()).all())
            assert torch.equal(got, ref), steps


@pytest.mark.parametrize("rows,cols", [(16, 96), (5, 40), (32, 300), (64, 128)])
def test_small_chain_on_infinities_zeros_and_nan(env, rows, cols):
    """Zero matrices, an infinity, a NaN, sums of squares past fp32 and values near its smallest: the same values and the same NaN."""
    print(f"small chain, special values {rows}x{cols}", flush=True)
    lib, abi, mu = env["lib"], env["abi"], env["mu"]
    G = torch.randn(7, rows, cols, generator=torch.Generator().manual_seed(rows))
    G[0] = 0.0
    G[1, rows // 2, cols // 3] = float("inf")
    G[2, 0, cols - 1] = float("nan")
    G[3] *= 1e30
    G[4] *= 1e-36
    G[5, :, 1:] = 0.0
    for g in (G.to(env["dev"]), G.mT.contiguous().to(env["dev"])):
        for steps in (1, 5):
            got = mu.fast_newtonschulz(g, steps)
            abi.check(lib.muon_hip_set_gemm_config(abi.CFG_128_PIPE))
            try:
                ref = mu.fast_newtonschulz(g, steps)
            finally:
                abi.check(lib.muon_hip_set_gemm_config(abi.CFG_AUTO))
            torch.cuda.synchronize()
            assert torch.equal(got.isnan(), ref.isnan()), steps
            assert torch.equal(got.nan_to_num(nan=0.0).view(torch.int16), ref.nan_to_num(nan=0.0).view(torch.int16)), steps


@pytest.mark.parametrize("pdtype", [torch.float32, torch.bfloat16])
def test_small_chain_in_a_step_is_bitwise_the_tiled_products(env, pdtype):
    """The same through Muon.step, where the chain applies the parameter update itself."""
    print(f"small chain step against tiles {pdtype}", flush=True)
    lib, abi, mu, dev = (env[k] for k in ("lib", "abi", "mu", "dev"))
    gen = torch.Generator().manual_seed(6)
    shapes = SHAPES + [(c, r) for r, c in SHAPES if r != c]
    ws = [(0.02 * torch.randn(*s, generator=gen)).to(pdtype) for s in shapes]
    gs = [(1e-3 * torch.randn(*s, generator=gen)).to(pdtype) for s in shapes]
    out = []
    for cfg in (abi.CFG_AUTO, abi.CFG_128_PIPE):
        params = [torch.nn.Parameter(w.to(dev)) for w in ws]
        for p, g in zip(params, gs):
            p.grad = g.to(dev)
        abi.check(lib.muon_hip_set_gemm_config(cfg))
        try:
            mu.Muon([dict(params=list(params), use_muon=True, lr=0.02, momentum=0.95, nesterov=True, weight_decay=0.01, ns_steps=5,
                          rms_scale=True)]).step()
        finally:
            abi.check(lib.muon_hip_set_gemm_config(abi.CFG_AUTO))
        torch.cuda.synchronize()
        out.append([p.detach() for p in params])
    for s, p, q in zip(shapes, *out):
        assert torch.equal(p, q), s


@pytest.mark.parametrize("pdtype", [torch.float32, torch.bfloat16])
def test_small_chain_in_a_step_equals_the_stages_bitwise(env, pdtype):
    """One call over all the shapes (several kernels and the tiled products in one launch sequence, parameters updated by the
    chain) against momentum, iterations and update as calls of their own, for parameters on a 16-byte boundary and off it."""
    print(f"small chain step {pdtype}", flush=True)
    lib, abi, mu, O, dev = (env[k] for k in ("lib", "abi", "mu", "O", "dev"))
    gen = torch.Generator().manual_seed(5)
    shapes = SHAPES + [(c, r) for r, c in SHAPES if r != c]
    hp = dict(lr=0.02, momentum=0.95, nesterov=True, weight_decay=0.01, ns_steps=5, rms_scale=True)

    def off(t, by):  # the same values, `by` elements past an aligned address
        buf = torch.zeros(t.numel() + 8, dtype=t.dtype, device=dev)
        buf[by:by + t.numel()] = t.reshape(-1).to(dev)
        return buf[by:by + t.numel()].view(t.shape)

    ws = [(0.02 * torch.randn(*s, generator=gen)).to(pdtype) for s in shapes]
    gs = [(1e-3 * torch.randn(*s, generator=gen)).to(pdtype) for s in shapes]
    params = [torch.nn.Parameter(off(w, i % 2)) for i, w in enumerate(ws)]
    for p, g in zip(params, gs):
        p.grad = g.to(dev)
    mu.Muon([dict(params=list(params), use_muon=True, **hp)]).step()
    a, b, c = O.NS_COEFFS
    code = abi.dtype_code(pdtype)
    for s, p, w, g in zip(shapes, params, ws, gs):
        q, gd, m = w.to(dev), g.to(dev), torch.zeros(s, dtype=pdtype, device=dev)
        area = torch.empty(abi.workspace_bytes(*s, 1), dtype=torch.uint8, device=dev)
        table = torch.tensor([t.data_ptr() for t in (q, gd, m)], dtype=torch.int64, device=dev)
        tp, tg, tm = (table.data_ptr() + 8 * i for i in range(3))
        abi.check(lib.muon_hip_momentum_norm(tg, tm, code, code, area.data_ptr(), *s, 1, hp["momentum"], 1, 0, 0))
        abi.check(lib.muon_hip_ns_grouped(area.data_ptr(), *s, 1, 5, a, b, c, 0))
        abi.check(lib.muon_hip_apply_update(tp, code, area.data_ptr(), *s, 1, 5, mu.scale_factor(*s, True), hp["lr"], hp["weight_decay"], 0))
        torch.cuda.synchronize()
        assert torch.equal(p.detach(), q), s


@pytest.mark.parametrize("rows,cols,batch", [(16, 2048, 3), (13, 333, 2), (13, 2049, 2), (64, 2048, 1), (64, 520, 200), (333, 7, 2), (2048, 64, 3),
                                             (2048, 64, 192), (515, 33, 193), (1, 1, 1), (4096, 32, 192)])
def test_small_chain_writes_its_result_where_the_copy_would(env, rows, cols, batch):
    """muon_hip_ns_result against muon_hip_ns_grouped and muon_hip_ns_output: the same bits, on aligned outputs and on others, and nothing
    around them."""
    print(f"small chain result {batch} x {rows}x{cols}", flush=True)
    lib, abi, dev = env["lib"], env["abi"], env["dev"]
    G = torch.randn(batch, rows, cols, generator=torch.Generator().manual_seed(rows + cols)).to(dev)
    ws = torch.empty(lib.muon_hip_workspace_bytes(rows, cols, batch), dtype=torch.uint8, device=dev)
    n = G.numel()
    for shift in (8, 1):
        buf = torch.full((n + 16,), 7.0, dtype=torch.bfloat16, device=dev)
        ref = torch.empty(G.shape, dtype=torch.bfloat16, device=dev)
        for direct in (True, False):
            abi.check(lib.muon_hip_cast_norm(G.data_ptr(), abi.dtype_code(G.dtype), ws.data_ptr(), rows, cols, batch, 0))
            if direct:
                abi.check(lib.muon_hip_ns_result(ws.data_ptr(), rows, cols, batch, 5, 3.4445, -4.775, 2.0315, buf.data_ptr() + 2 * shift, 0))
            else:
                abi.check(lib.muon_hip_ns_grouped(ws.data_ptr(), rows, cols, batch, 5, 3.4445, -4.775, 2.0315, 0))
                abi.check(lib.muon_hip_ns_output(ws.data_ptr(), rows, cols, batch, 5, ref.data_ptr(), 0))
        torch.cuda.synchronize()
        assert torch.equal(buf[shift:shift + n].view(G.shape), ref), shift
        assert bool((buf[:shift] == 7).all()) and bool((buf[shift + n:] == 7).all())
