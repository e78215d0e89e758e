"""Matrices of one row of 256-tiles beside large ones: in the launches of those up to an eighth of their tiles, on 128-tiles beyond; the same bits."""
import random

import pytest
import torch

from lmms_engine_amd import _abi
from tests.test_gpu_parity import env  # noqa: F401

LARGE = [(1000, 1000, 20)]  # 16 tiles a product, 10 of the symmetric ones


def _cfg(shapes, kind):
    return [r[0] for r in _abi.routes(shapes, kind)]


@pytest.mark.parametrize("kind,most", [("syrk", 25), ("sympoly", 25), ("bx_axpy", 10), ("bx_axpy_update", 10)])
def test_an_eighth_of_the_tiles_goes_along(kind, most):
    small = lambda n: LARGE + [(200, 1000, n)]  # noqa: E731
    for n in (1, most):
        large, along = _cfg(small(n), kind)
        assert large == along != _abi.CFG_128_PINGPONG, n
    assert _cfg(small(most + 1), kind)[1] == _abi.CFG_128_PINGPONG


def test_what_stays_on_128_tiles():
    assert set(_cfg([(200, 1000, 300)], "syrk")) == {_abi.CFG_128_PINGPONG}  # nothing to go along with
    assert _cfg(LARGE + [(100, 1000, 2)], "sympoly")[1] == _abi.CFG_128_PINGPONG  # 128 rows of storage
    assert _cfg(LARGE + [(200, 600, 2)], "bx_axpy")[1] == _abi.CFG_128_PINGPONG  # 640 columns of storage, no whole 256-tiles
    assert _cfg(LARGE + [(384, 1000, 2)], "sympoly")[1] == _abi.CFG_128_PINGPONG


# The persistent symmetric products take reductions of at most 2048 columns: with large matrices on one side of that line and short ones on the
# other they end in launches of their own.
@pytest.mark.parametrize("shapes,along", [
    ([(1024, 2048, 100), (256, 12288, 4)], False), ([(768, 2048, 384), (256, 4096, 4)], False), ([(1024, 2048, 100), (256, 2049, 4)], False),
    ([(1024, 2048, 100), (256, 2048, 4)], True), ([(1024, 4096, 100), (256, 12288, 4)], True), ([(1024, 4096, 100), (256, 2048, 4)], True),
    # some of each: those beyond the line keep their tiles where the large ones beyond it are too few
    ([(1024, 2048, 100), (1024, 4096, 3), (256, 4096, 4)], False), ([(1024, 2048, 100), (1024, 4096, 4), (256, 4096, 4)], True),
])
def test_nothing_goes_along_in_a_launch_without_large_ones(shapes, along):
    routes = _abi.routes(shapes, "syrk")
    assert (routes[-1][0] != _abi.CFG_128_PINGPONG) == along, routes
    assert (routes[-1][2] in [r[2] for r in routes[:-1]]) == along, routes


def test_what_goes_along_shares_its_launch_for_drawn_calls():
    """Every 256-tile of a matrix of one row of them lies in a launch with eight times as many of larger matrices."""
    rng, taken = random.Random(5), 0
    for _ in range(3000):
        side = lambda: rng.choice([rng.randint(129, 256), 128 * rng.randint(3, 12), rng.randint(257, 2000)])  # noqa: E731
        shapes = [(side(), rng.choice([512, 1000, 2048, 2049, 4096, 12288]), rng.randint(1, 120)) for _ in range(rng.randint(2, 5))]
        for kind in ("syrk", "sympoly", "bx_axpy", "bx_axpy_update"):
            own, along = {}, {}
            for (r, c, n), (cfg, height, launch) in zip(shapes, _abi.routes(shapes, kind)):
                if cfg == _abi.CFG_128_PINGPONG or launch < 0 or height != 256:
                    continue
                t, tn = -(-min(r, c) // 256), -(-max(r, c) // 256)
                tiles = n * (t * tn if kind.startswith("bx") else t * (t + 1) // 2)
                d = along if t == 1 else own
                d[launch] = d.get(launch, 0) + tiles
            for launch, tiles in along.items():
                taken += 1
                assert 8 * tiles <= own.get(launch, 0), (kind, shapes)
    assert taken > 100


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shapes", [
    [(1000, 1000, 20), (200, 1000, 9), (1000, 200, 1)], [(1000, 1000, 20), (129, 257, 2), (600, 256, 3), (256, 256, 2)],
    [(1024, 2731, 6), (2731, 1024, 6), (250, 1024, 8)],
])
def test_steps_are_bitwise_the_two_stage_kernel(env, shapes, dtype):
    print(f"along {shapes} {dtype}", flush=True)
    mu, dev = env["mu"], env["dev"]
    gen = torch.Generator().manual_seed(len(shapes))
    ws = [(0.02 * torch.randn(r, c, generator=gen)).to(dtype) for r, c, n in shapes for _ in range(n)]
    gs = [(1e-3 * torch.randn(w.shape, generator=gen)).to(dtype) for w in ws]
    out = []
    for cfg in (_abi.CFG_AUTO, _abi.CFG_STAGED, _abi.CFG_128_PIPE):
        ps = [torch.nn.Parameter(w.to(dev)) for w in ws]
        for p, g in zip(ps, gs):
            p.grad = g.to(dev)
        opt = mu.Muon([dict(params=list(ps), use_muon=True, lr=0.02, momentum=0.95, nesterov=True, weight_decay=0.01, ns_steps=5, rms_scale=True)],
                      momentum_dtype=torch.float32)
        _abi.check(_abi.lib().muon_hip_set_gemm_config(cfg))
        try:
            opt.step(), opt.step()
            torch.cuda.synchronize()
        finally:
            _abi.check(_abi.lib().muon_hip_set_gemm_config(_abi.CFG_AUTO))
        out.append([p.detach() for p in ps])
    for a, b, c in zip(*out):
        assert bool(torch.isfinite(a.float()).all()) and torch.equal(a, b) and torch.equal(a, c), tuple(a.shape)
