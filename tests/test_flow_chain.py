"""The iterations of many small matrices in one launch: which tiles there are and in which order they are taken (host side), and the
results against a launch per product, bit for bit (every kernel sums an element's products in ascending k)."""
import random

import pytest
import torch

from lmms_engine_amd import _abi
from tests.test_gpu_parity import env  # noqa: F401

MIXED = [(512, 512, 16), (256, 512, 16), (1408, 512, 16), (512, 1408, 8)]
# the 64-row matrices run in a workgroup each; those of 128 rows would, were they alone
TINY = [(384, 256, 2), (128, 128, 4), (64, 128, 4), (256, 384, 2)]
ALONE = [(384, 128, 4), (128, 128, 4), (64, 128, 4), (128, 384, 2)]


def _check_order(shapes, steps, update, xcds):
    tiles = _abi.flow_tiles(shapes, steps, update, xcds)
    products = {_abi.K_SYRK: 0, _abi.K_SYMPOLY: 1, _abi.K_BX: 2}
    done, group_of, groups = {}, {}, []
    for t in tiles:
        assert t.group < xcds and t.group >= (groups[-1] if groups else 0)
        groups.append(t.group)
        m = (t.bucket, t.matrix)
        assert 0 <= t.matrix < shapes[t.bucket][2]
        assert group_of.setdefault(m, t.group) == t.group
        mine = done.setdefault(m, [])
        # everything that this tile waits for has been taken before it, and it waits for every tile of the products before
        stage = (t.iteration, products[t.product])
        assert all(s <= stage for s, _ in mine)
        assert t.before == sum(s < stage for s, _ in mine)
        mine.append((stage, t.tile))
    for i, (rows, cols, n) in enumerate(shapes):
        tm, tn = -(-min(rows, cols) // 128), -(-max(rows, cols) // 128)
        want = sorted(((it, s), k) for it in range(steps) for s in range(3) for k in range(tm * tn if s == 2 else tm * (tm + 1) // 2))
        for k in range(n if tiles and min(rows, cols) > 64 else 0):
            assert sorted(done.pop((i, k))) == want
    assert not done
    return tiles


@pytest.mark.parametrize("xcds", [1, 2, 4, 8])
@pytest.mark.parametrize("shapes,steps,update,not_on", [
    (MIXED, 5, True, (1, 2)),  # there a launch of its own per product is full
    (TINY, 5, True, ()), ([(256, 1024, 48)], 1, False, ()), ([(130, 700, 64)], 3, False, ()),
    ([(130, 700, 33)], 3, False, (8,)),  # 33 matrices: one XCD has a quarter more than the others
])
def test_every_tile_once_and_after_what_it_waits_for(shapes, steps, update, not_on, xcds):
    assert bool(_check_order(shapes, steps, update, xcds)) == (xcds not in not_on)


def test_every_tile_once_for_drawn_calls():
    rng, taken = random.Random(3), 0
    for _ in range(60):
        shapes = [(rng.randint(65, 700), rng.randint(65, 1500), rng.randint(1, 40)) for _ in range(rng.randint(1, 5))]
        taken += bool(_check_order(shapes, rng.randint(1, 3), rng.random() < 0.5, rng.choice([1, 2, 4, 8])))
    assert taken > 20


def test_calls_that_stay_with_a_launch_per_product():
    assert not _abi.flow_tiles([(896, 4864, 1)], 5, False)  # one matrix: one XCD
    assert not _abi.flow_tiles([(896, 4864, 72), (896, 896, 48)], 5, True)  # large
    assert not _abi.flow_tiles([(256, 1024, 48)], 0, False)
    assert not _abi.flow_tiles([(16, 2048, 48)], 5, True)  # a workgroup per matrix
    assert not _abi.flow_tiles(ALONE, 5, True) and not _abi.flow_tiles([(128, 512, 48)], 5, False)
    for kind in ("syrk", "sympoly", "bx_axpy", "bx_axpy_update"):
        assert [launch for _, _, launch in _abi.routes(ALONE, kind)] == [-1] * 4
        assert [launch >= 0 for _, _, launch in _abi.routes(TINY, kind)] == [True, True, False, True]
    assert _abi.flow_tiles([(256, 1024, 48)], 5, False)
    for cfg in (_abi.CFG_STAGED, _abi.CFG_128_PINGPONG):
        _abi.check(_abi.lib().muon_hip_set_gemm_config(cfg))
        try:
            assert not _abi.flow_tiles([(256, 1024, 48)], 5, False)
        finally:
            _abi.check(_abi.lib().muon_hip_set_gemm_config(_abi.CFG_AUTO))


def test_a_recorded_step_over_very_little_keeps_its_launches():
    """The one launch is the slower one on the device there; it saves the caller of an eager step his own launches, which a replay has not."""
    assert _abi.flow_tiles(TINY, 5, True) and not _abi.flow_tiles(TINY, 5, True, recorded=True)
    assert len(_abi.flow_tiles(MIXED, 5, True, recorded=True)) == len(_abi.flow_tiles(MIXED, 5, True)) > 0
    assert _abi.flow_tiles([(256, 1024, 48)], 5, False, recorded=True)


def _steps(mu, dev, shapes, dtype, mdtype, config, steps=2, offset=0):
    g = torch.Generator().manual_seed(len(shapes))
    ws = [(0.02 * torch.randn(r, c, generator=g)).to(dtype) for r, c, n in shapes for _ in range(n)]
    gs = [(1e-3 * torch.randn(w.shape, generator=g)).to(dtype) for w in ws]
    places = [torch.full((w.numel() + offset + 8,), 7.0, dtype=dtype, device=dev) for w in ws]
    ps = [torch.nn.Parameter(b[offset:offset + w.numel()].view(w.shape).copy_(w)) for b, w in zip(places, ws)]
    for p, gr in zip(ps, gs):
        p.grad = gr.to(dev)
    opt = mu.Muon([dict(params=list(ps), use_muon=True, lr=0.02, momentum=0.95, nesterov=True, weight_decay=0.01, ns_steps=5, rms_scale=True)],
                  momentum_dtype=mdtype)
    _abi.check(_abi.lib().muon_hip_set_gemm_config(config))
    try:
        for _ in range(steps):
            opt.step()
        torch.cuda.synchronize()
    finally:
        _abi.check(_abi.lib().muon_hip_set_gemm_config(_abi.CFG_AUTO))
    for b, w in zip(places, ws):  # nothing around a parameter has been written
        assert bool((b[:offset] == 7).all()) and bool((b[offset + w.numel():] == 7).all())
    return ps, ws, opt


# both orientations, ragged edges, odd numbers of tiles, odd column counts, parameters of whole 16-byte pieces that lie one element
# behind a 16-byte boundary
@pytest.mark.gpu
@pytest.mark.parametrize("name,shapes,dtype,mdtype,offset", [
    ("mixed", MIXED, torch.bfloat16, torch.float32, 0),
    ("tiny", TINY, torch.float32, None, 0),
    ("ragged", [(200, 333, 24), (333, 200, 16), (130, 130, 16), (901, 257, 8)], torch.bfloat16, None, 0),
    ("ragged fp32", [(70, 129, 40), (500, 411, 32), (129, 1000, 8)], torch.float32, None, 0),
    ("unaligned", MIXED, torch.bfloat16, torch.float32, 1),
    ("unaligned fp32", [(256, 384, 24), (384, 256, 24), (128, 512, 8)], torch.float32, None, 1),
])
def test_steps_equal_a_launch_per_product_bitwise(env, name, shapes, dtype, mdtype, offset):
    print(f"one launch: {name}", flush=True)
    assert _abi.flow_tiles(sorted(shapes, reverse=True), 5, True)
    mu, dev = env["mu"], env["dev"]
    a, ws, _ = _steps(mu, dev, shapes, dtype, mdtype, _abi.CFG_AUTO, offset=offset)
    b, _, _ = _steps(mu, dev, shapes, dtype, mdtype, _abi.CFG_STAGED)
    assert all(p.data_ptr() % 16 for p in a) if offset else not any(p.data_ptr() % 16 for p in a)
    for p, q, w in zip(a, b, ws):
        assert bool(torch.isfinite(p.detach().float()).all())
        assert torch.equal(p.detach(), q.detach()) and not torch.equal(p.detach().cpu(), w), tuple(p.shape)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,batch,steps", [(1024, 256, 48, 5), (256, 1024, 48, 1), (130, 700, 64, 2), (512, 512, 40, 3)])
def test_stacks_equal_a_launch_per_product_bitwise(env, rows, cols, batch, steps):
    print(f"one launch: {batch} x {rows} x {cols}, {steps} steps", flush=True)
    assert _abi.flow_tiles([(rows, cols, batch)], steps, False)
    g = torch.randn(batch, rows, cols, generator=torch.Generator().manual_seed(rows)).bfloat16().to(env["dev"])
    got = env["mu"].fast_newtonschulz(g, steps)
    _abi.check(_abi.lib().muon_hip_set_gemm_config(_abi.CFG_STAGED))
    try:
        ref = env["mu"].fast_newtonschulz(g, steps)
    finally:
        _abi.check(_abi.lib().muon_hip_set_gemm_config(_abi.CFG_AUTO))
    torch.cuda.synchronize()
    assert bool(torch.isfinite(ref.float()).all())
    assert torch.equal(got, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [MIXED, TINY])
def test_replays_and_two_streams_equal_eager_steps_bitwise(env, shapes):
    """A recorded step replayed beside eager steps of another optimizer on a second stream, four times."""
    mu, dev = env["mu"], env["dev"]
    assert _abi.flow_tiles(sorted(shapes, reverse=True), 5, True)
    assert bool(_abi.flow_tiles(sorted(shapes, reverse=True), 5, True, recorded=True)) == (shapes is MIXED)
    want, _, _ = _steps(mu, dev, shapes, torch.bfloat16, torch.float32, _abi.CFG_STAGED, steps=6)
    pa, _, oa = _steps(mu, dev, shapes, torch.bfloat16, torch.float32, _abi.CFG_AUTO, steps=2)
    pb, _, ob = _steps(mu, dev, shapes, torch.bfloat16, torch.float32, _abi.CFG_AUTO, steps=2)
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph):
        oa.step()
    for _ in range(4):
        with torch.cuda.stream(side):
            ob.step()
        graph.replay()
        torch.cuda.synchronize()
    for p, q, w in zip(pa, pb, want):
        assert torch.equal(p.detach(), w.detach()) and torch.equal(q.detach(), w.detach()), tuple(p.shape)


@pytest.mark.gpu
def test_an_abandoned_chain_stores_nothing_unfinished_and_is_reported(env):
    """A wait that gives up at its second poll: every workgroup leaves, no element of a parameter is computed from operands that were not
    there, and the next call says what happened, once."""
    mu, dev, lib = env["mu"], env["dev"], env["lib"]
    assert _abi.flow_tiles(sorted(MIXED, reverse=True), 5, True)
    ps, ws, opt = _steps(mu, dev, MIXED, torch.bfloat16, torch.float32, _abi.CFG_AUTO, steps=1)
    want, _, _ = _steps(mu, dev, MIXED, torch.bfloat16, torch.float32, _abi.CFG_STAGED, steps=2)
    before = [p.detach().clone() for p in ps]
    moms = [opt.state[p]["momentum_buffer"].clone() for p in ps]
    assert lib.muon_hip_chain_status() == 0
    print("an abandoned chain", flush=True)
    _abi.check(lib.muon_hip_set_chain_polls(1))
    try:
        opt.step()
    finally:
        _abi.check(lib.muon_hip_set_chain_polls(-1))
    torch.cuda.synchronize()
    left = [p.detach().clone() for p in ps]
    changed = 0
    for p, b, w in zip(left, before, want):
        same = p == b
        assert bool((same | (p == w.detach())).all()), tuple(p.shape)
        changed += int(not bool(same.all()))
    assert changed < len(ps)
    with pytest.raises(_abi.MuonHipError, match="gave up waiting"):
        opt.step()
    torch.cuda.synchronize()
    assert lib.muon_hip_chain_status() == 0
    for p, q in zip(ps, left):
        assert torch.equal(p.detach(), q)
    # as a program goes on from its last checkpoint
    for p, b, m in zip(ps, before, moms):
        p.detach().copy_(b)
        opt.state[p]["momentum_buffer"].copy_(m)
    opt.step()
    torch.cuda.synchronize()
    assert lib.muon_hip_chain_status() == 0
    for p, w in zip(ps, want):
        assert torch.equal(p.detach(), w.detach())


# the lists of the persistent kernel that calls of these sizes run when every product has a launch of its own
@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [[(512, 1024, 40), (256, 384, 3), (300, 100, 2), (1024, 1100, 1)], [(512, 1408, 24), (512, 512, 16)]])
def test_launches_per_product_equal_named_configurations_bitwise(env, shapes):
    print(f"a launch per product: {shapes}", flush=True)
    assert any(cfg == _abi.CFG_256_PERSIST for cfg, _, _ in _abi.routes(shapes, "bx_axpy"))
    a, _, _ = _steps(env["mu"], env["dev"], shapes, torch.bfloat16, torch.float32, _abi.CFG_STAGED)
    b, _, _ = _steps(env["mu"], env["dev"], shapes, torch.bfloat16, torch.float32, _abi.CFG_128_PIPE)
    for p, q in zip(a, b):
        assert torch.equal(p.detach(), q.detach()), tuple(p.shape)
