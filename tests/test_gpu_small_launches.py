"""Launches that do not fill the machine: the 64-tile kernel and the choice of smaller tiles.  Every configuration sums the
products of an element in ascending k, so all of them agree bit for bit; the two-stage 128-tile kernel, which
tests/test_gpu_parity.py holds to the fp64 product, is the reference."""
from collections import Counter

import pytest
import torch

from tests.test_gpu_parity import _blocked_nan, _pack, env  # noqa: F401

pytestmark = pytest.mark.gpu


def _products(env, M, K, batch, cfg):
    lib, abi, dev, O = env["lib"], env["abi"], env["dev"], env["O"]
    g = torch.Generator().manual_seed(M + 3 * K + batch)
    X = _pack(env, (torch.randn(batch, M, K, generator=g) / 16).bfloat16().to(dev))
    A, B, Xo = _blocked_nan(env, batch, M, M), _blocked_nan(env, batch, M, M), _blocked_nan(env, batch, M, K)
    a, b, c = O.NS_COEFFS
    abi.check(lib.muon_hip_syrk_bf16(X.data_ptr(), A.data_ptr(), M, K, batch, cfg, env["ctr_ptr"], 0))
    abi.check(lib.muon_hip_sympoly_bf16(A.data_ptr(), B.data_ptr(), M, batch, b, c, cfg, env["ctr_ptr"], 0))
    abi.check(lib.muon_hip_bx_axpy_bf16(B.data_ptr(), X.data_ptr(), Xo.data_ptr(), M, K, batch, a, cfg, env["ctr_ptr"], 0))
    torch.cuda.synchronize()
    # as bit patterns: rows of a block that the padded matrix does not reach keep the NaN they were filled with
    return [t.view(torch.int16) for t in (A, B, Xo)]


# reductions of 2, 4, 6, 8, 10 and 18 k-tiles of 64 (the pipeline is eight deep), one tile row and several, more than one
# block of 256 rows, tile counts that are no multiple of the eight XCDs
@pytest.mark.parametrize("M,K,batch", [(128, 128, 1), (128, 256, 3), (256, 384, 1), (128, 512, 5), (384, 640, 2), (640, 1152, 1),
                                       (1024, 128, 1)])
def test_64_tiles_are_bitwise_the_two_stage_kernel(env, M, K, batch):
    print(f"64-tiles M={M} K={K} batch={batch}", flush=True)
    ref = _products(env, M, K, batch, env["abi"].CFG_128_PIPE)
    for name, r, got in zip(("syrk", "sympoly", "bx"), ref, _products(env, M, K, batch, env["abi"].CFG_64_DEEP)):
        assert torch.equal(r, got), name


# around the two limits of the choice: 64-tiles up to one per compute unit, 128-tiles up to two
@pytest.mark.parametrize("M,K,batch", [(512, 512, 7), (512, 512, 8), (1408, 256, 1), (1408, 256, 2), (1024, 1024, 14), (1024, 1024, 15)])
def test_the_choice_by_tile_count_does_not_change_the_result(env, M, K, batch):
    print(f"auto M={M} K={K} batch={batch}", flush=True)
    ref = _products(env, M, K, batch, env["abi"].CFG_128_PIPE)
    for name, r, got in zip(("syrk", "sympoly", "bx"), ref, _products(env, M, K, batch, env["abi"].CFG_AUTO)):
        assert torch.equal(r, got), name


# one call over many shapes: more shapes than a call takes, a bucket that runs the persistent kernel beside small ones, both
# orientations, ragged edges, the norms of matrices above and below the limit of the inline sums, bf16 momentum
# lists: for a.X + B.X, how many shapes share one persistent launch, by tile height
@pytest.mark.parametrize("name,shapes,dtype,mdtype,lists", [
    ("17 shapes", [(64 + 8 * i, 100 + 16 * i) for i in range(17)], torch.float32, None, {}),
    ("persistent beside small", [(512, 1024)] * 40 + [(256, 384)] * 3 + [(300, 100)] * 2 + [(33, 47), (1024, 1100)], torch.bfloat16,
     torch.float32, {256: 2}),
    ("persistent lists of every tile height", [(896, 1000)] * 20 + [(1100, 900)] * 20 + [(650, 640)] * 60 + [(1000, 1024)] * 9 +
     [(1030, 990)] * 9 + [(1160, 1152)] * 24 + [(384, 700)] * 32, torch.float32, None, {256: 3, 224: 2, 192: 2}),
    ("tall and wide", [(1408, 256), (256, 1408), (1, 9), (200, 200)], torch.bfloat16, None, {}),
])
def test_one_call_over_many_shapes_equals_one_call_per_matrix(env, name, shapes, dtype, mdtype, lists):
    print(f"many shapes: {name}", flush=True)
    mu, dev, abi = env["mu"], env["dev"], env["abi"]
    if len(set(shapes)) <= abi.MAX_BUCKETS:
        routes = abi.routes([(*s, shapes.count(s)) for s in sorted(set(shapes), reverse=True)], "bx_axpy")
        persistent = Counter((launch, height) for cfg, height, launch in routes if cfg == abi.CFG_256_PERSIST)
        assert {height: n for (_, height), n in persistent.items()} == lists
    g = torch.Generator().manual_seed(len(shapes))
    ws = [(0.02 * torch.randn(*s, generator=g)).to(dtype) for s in shapes]
    gs = [(1e-3 * torch.randn(*s, generator=g)).to(dtype) for s in shapes]
    hp = dict(lr=0.02, momentum=0.95, nesterov=True, weight_decay=0.01, ns_steps=5, rms_scale=True)
    pa, pb = ([torch.nn.Parameter(w.clone().to(dev)) for w in ws] for _ in range(2))
    for p, q, gr in zip(pa, pb, gs):
        p.grad, q.grad = gr.to(dev), gr.to(dev)
    opt = mu.Muon([dict(params=list(pa), use_muon=True, **hp)], momentum_dtype=mdtype)
    opt.step()
    for q in pb:
        st = {"momentum_buffer": torch.zeros_like(q, dtype=mdtype or dtype)}
        mu.SingelDeviceWork(q, st, dict(opt.param_groups[0]), 0).start()
    torch.cuda.synchronize()
    for s, p, q, w in zip(shapes, pa, pb, ws):
        assert torch.equal(p.detach(), q.detach()), s
        assert not torch.equal(p.detach().cpu(), w), s


# a.X + B.X on tiles of the matrix's own height: 224, 192 and 256 rows, short sides that end inside the last 128 rows, long
# sides whose last 256-tile overhangs, more than one row block, and rounds that are filled enough and not
@pytest.mark.parametrize("rows,cols,batch,height", [
    (896, 1000, 40, 224), (900, 640, 90, 224), (384, 520, 100, 128), (384, 520, 255, 192), (1160, 1152, 24, 192), (1290, 1408, 12, 128),
    (1290, 1408, 14, 256), (1000, 1100, 30, 256), (1000, 1000, 17, 256), (896, 1000, 20, 128), (2700, 1930, 8, 256)])
def test_odd_short_sides_do_not_change_the_result(env, rows, cols, batch, height):
    print(f"odd short side {batch} x {rows} x {cols}", flush=True)
    lib, abi, mu = env["lib"], env["abi"], env["mu"]
    assert abi.routes([(rows, cols, batch)], "bx_axpy")[0][1] == height
    g = torch.randn(batch, rows, cols, generator=torch.Generator().manual_seed(rows + cols)).bfloat16().to(env["dev"])
    got = mu.fast_newtonschulz(g, 5)
    abi.check(lib.muon_hip_set_gemm_config(abi.CFG_128_PIPE))
    try:
        ref = mu.fast_newtonschulz(g, 5)
    finally:
        abi.check(lib.muon_hip_set_gemm_config(abi.CFG_AUTO))
    torch.cuda.synchronize()
    assert bool(torch.isfinite(ref.float()).all())
    assert torch.equal(got, ref)


# the single product where the short side is padded to whole 256-tiles and the long one is not
@pytest.mark.parametrize("M,K", [(1000, 640), (400, 130), (1930, 1000)])
def test_matmul_transpose_of_padded_short_sides(env, M, K):
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).bfloat16()
    got = env["mu"].matmul_transpose(x.to(env["dev"])).cpu().double()
    ref = x.double() @ x.double().T
    # one rounding to bf16 and an fp32 sum of K products
    assert ((got - ref).abs() <= ref.abs() * 2.0**-8 + K * 2.0**-24 * (x.double().abs() @ x.double().abs().T)).all()
    assert torch.equal(got, got.T)


# configurations that the caller names, on short sides of one 256-tile and long sides that end inside a 256-tile, in batches: a
# tile past the end of a matrix would write the next one
@pytest.mark.parametrize("rows,cols,batch", [(100, 300, 5), (256, 640, 3), (640, 200, 4), (300, 700, 3)])
def test_named_configurations_agree_bitwise(env, rows, cols, batch):
    lib, abi, mu = env["lib"], env["abi"], env["mu"]
    g = torch.randn(batch, rows, cols, generator=torch.Generator().manual_seed(rows + cols)).bfloat16().to(env["dev"])
    out = []
    for cfg in (abi.CFG_128_PIPE, abi.CFG_256_PIPE, abi.CFG_256_PINGPONG, abi.CFG_128_PINGPONG, abi.CFG_256_PERSIST, abi.CFG_64_DEEP):
        print(f"named configuration {cfg}: {batch} x {rows} x {cols}", flush=True)
        abi.check(lib.muon_hip_set_gemm_config(cfg))
        try:
            out.append(mu.fast_newtonschulz(g, 5))
        finally:
            abi.check(lib.muon_hip_set_gemm_config(abi.CFG_AUTO))
        torch.cuda.synchronize()
    assert bool(torch.isfinite(out[0].float()).all())
    for i, o in enumerate(out[1:], 1):
        assert torch.equal(o, out[0]), i


# 64 workgroups of the normalisation per 200 x 512 matrix: 256 matrices are the most whose workgroups add the norm's partial sums
# themselves, one more takes the launch that adds them; turned matrices have no such limit, up to 256 partial sums of 4096 elements each
@pytest.mark.parametrize("rows,cols,batch", [(200, 512, 256), (200, 512, 257), (512, 200, 600), (1025, 1024, 3), (1024, 1025, 3), (1024, 1024, 3)])
def test_norms_of_large_and_small_batches_agree_bitwise(env, rows, cols, batch):
    print(f"norms {batch} x {rows} x {cols}", flush=True)
    assert env["abi"].routes([(rows, cols, batch)], "syrk")[0][2] >= 0  # (matrices that a workgroup holds do not come that way)
    g = torch.randn(batch, rows, cols, generator=torch.Generator().manual_seed(batch)).bfloat16().to(env["dev"])
    got = env["mu"].fast_newtonschulz(g, 1)
    for lo in (0, batch // 2, batch - 3):
        assert torch.equal(got[lo:lo + 3], env["mu"].fast_newtonschulz(g[lo:lo + 3], 1)), lo
    d = (g.double().square().sum((1, 2), keepdim=True).sqrt().bfloat16().float() + 1e-7).bfloat16()
    x = env["mu"].fast_newtonschulz(g, 0)
    want = (g.float() / d.float()).bfloat16()
    # the norm itself is a bf16 value, whose neighbour it may come out as: at most 2^-7 away, and both quotients are rounded by up to 2^-9
    assert bool(((x.float() - want.float()).abs() <= 3 * 2.0**-8 * want.float().abs()).all())
