"""Launches that do not fill the machine: the 64-tile kernel and the choice of smaller tiles.  Every configuration sums the
products of an element in ascending k, so all of them agree bit for bit; the two-stage 128-tile kernel, which
tests/test_gpu_parity.py holds to the fp64 product, is the reference."""
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
