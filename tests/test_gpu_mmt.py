"""X Xt of row-major matrices: read where they lie or packed first, on every kernel that takes them, the same bits either way."""
import pytest
import torch

from lmms_engine_amd import _abi
from tests.test_gpu_parity import env  # noqa: F401

pytestmark = pytest.mark.gpu


def _mmt(lib, x, out=None):
    M, K = x.shape
    out = torch.full((M, M), float("nan"), dtype=torch.bfloat16, device=x.device) if out is None else out
    n = lib.muon_hip_mmt_scratch_elems(x.data_ptr(), out.data_ptr(), M, K)
    scratch = torch.full((max(n, 1),), float("nan"), dtype=torch.bfloat16, device=x.device)
    _abi.check(lib.muon_hip_mmt_bf16(x.data_ptr(), out.data_ptr(), M, K, scratch.data_ptr() if n else None, 0))
    return out, n


# 64-tiles (whole tiles past the last row among them), 128-tiles, 256-tiles, 256-tiles with a last round in quarters; rows that end at
# the last element of the buffer; results whose rows are no whole number of 16-byte pieces
@pytest.mark.parametrize("M,K", [(1, 128), (7, 128), (129, 256), (200, 384), (1030, 128), (1000, 640), (2040, 256), (2048, 1024), (3000, 128),
                                 (3072, 384), (5893, 128), (6136, 256)])
def test_read_in_place_equals_packed_bitwise(env, M, K):
    print(f"mmt {M} x {K}", flush=True)
    lib, dev = env["lib"], env["dev"]
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).bfloat16()
    guard = torch.full((M * K + 16,), float("nan"), dtype=torch.bfloat16, device=dev)  # nothing in front of X or behind it is taken
    direct = guard[8:8 + M * K].view(M, K).copy_(x)
    odd = guard.new_full((M * K + 16,), float("nan"))[1:1 + M * K].view(M, K).copy_(x)  # not 16-byte aligned
    got, n = _mmt(lib, direct)
    ref, m = _mmt(lib, odd)
    torch.cuda.synchronize()
    assert n == 0 and m > 0
    assert torch.equal(got, ref) and torch.equal(got, got.T)
    exact = x.double() @ x.double().T
    # one rounding to bf16 and an fp32 sum of K products
    assert ((got.cpu().double() - exact).abs() <= exact.abs() * 2.0**-8 + K * 2.0**-24 * (x.double().abs() @ x.double().abs().T)).all()


# aligned operands that are packed because of their size
@pytest.mark.parametrize("M,K", [(2048, 5632), (3072, 3072), (1536, 6144), (1700, 3200)])
def test_large_operands_on_128_tiles_are_packed(env, M, K):
    print(f"mmt {M} x {K}", flush=True)
    lib, dev = env["lib"], env["dev"]
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).bfloat16().to(dev)
    out = torch.empty(M, M, dtype=torch.bfloat16, device=dev)
    assert lib.muon_hip_mmt_scratch_elems(x.data_ptr(), out.data_ptr(), M, K) >= M * K
    assert lib.muon_hip_mmt_bf16(x.data_ptr(), out.data_ptr(), M, K, None, 0) < 0  # scratch that the caller has not brought
    got, n = _mmt(lib, x, out)
    torch.cuda.synchronize()
    assert n > 0 and torch.equal(got, got.T)
    exact, bound = x.double() @ x.double().T, x.double().abs() @ x.double().abs().T
    assert ((got.double() - exact).abs() <= exact.abs() * 2.0**-8 + K * 2.0**-24 * bound).all()


# 64-tiles, 128-tiles, 256-tiles
@pytest.mark.parametrize("M,K,line", [(896, 4864, 128), (2048, 2048, 64), (4096, 4096, 64)])
def test_rows_that_straddle_cache_lines_are_packed(env, M, K, line):
    """Read in place from such an address 896 x 32768 takes 139 us instead of 117, 4096 x 12288 300 instead of 213."""
    print(f"mmt {M} x {K}", flush=True)
    lib, dev = env["lib"], env["dev"]
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).bfloat16()
    buf, out = torch.empty(M * K + 128, dtype=torch.bfloat16, device=dev), []
    assert buf.data_ptr() % 512 == 0
    for at in (0, 8, 16, 32, 64):
        got, n = _mmt(lib, buf[at:at + M * K].view(M, K).copy_(x))
        assert (n > 0) == (2 * at % line != 0), at
        out.append(got)
    torch.cuda.synchronize()
    assert all(torch.equal(out[0], o) for o in out)


def test_result_stays_inside_its_rows(env):
    lib, dev = env["lib"], env["dev"]
    for M, K in [(130, 128), (1030, 128), (2047, 256), (3001, 100)]:
        x = torch.randn(M, K, device=dev).bfloat16()
        buf = torch.full((M * M + 64,), 7.0, dtype=torch.bfloat16, device=dev)
        out, _ = _mmt(lib, x, buf[32:32 + M * M].view(M, M))
        torch.cuda.synchronize()
        assert bool((buf[:32] == 7).all()) and bool((buf[32 + M * M:] == 7).all()) and bool(torch.isfinite(out.float()).all()), (M, K)


def test_a_result_over_its_own_input(env):
    mu, dev = env["mu"], env["dev"]
    x = torch.randn(512, 512, generator=torch.Generator().manual_seed(1)).bfloat16().to(dev)
    ref = mu.matmul_transpose(x)
    mu.matmul_transpose_assign(x, x)
    flat = torch.randn(3 * 256 * 256, generator=torch.Generator().manual_seed(2)).bfloat16().to(dev)
    a, b = flat[:2 * 256 * 256].view(256, 512), flat[256 * 256:2 * 256 * 256].view(256, 256)
    ref2 = mu.matmul_transpose(a)
    mu.matmul_transpose_assign(a, b)
    torch.cuda.synchronize()
    assert torch.equal(x, ref) and torch.equal(b, ref2)


@pytest.mark.parametrize("M,K", [(100, 130), (512, 384), (896, 128), (1030, 256), (2048, 1024)])
def test_a_named_configuration_multiplies(env, M, K):
    """muon_hip_set_gemm_config holds for matmul_transpose: the same bits on each kernel, an error where its tiles do not divide the padded
    matrix."""
    print(f"mmt {M} x {K} on named configurations", flush=True)
    mu, lib, dev = env["mu"], env["lib"], env["dev"]
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).bfloat16().to(dev)
    ref = mu.matmul_transpose(x)
    whole256 = -(-M // 128) % 2 == 0 and M > 384
    for cfg in (*_abi.GEMM_CONFIGS, _abi.CFG_256_PERSIST, _abi.CFG_64_DEEP):
        refused = not whole256 and cfg in (_abi.CFG_256_PIPE, _abi.CFG_256_PINGPONG, _abi.CFG_256_PERSIST)
        _abi.check(lib.muon_hip_set_gemm_config(cfg))
        try:
            if refused:
                with pytest.raises(_abi.MuonHipError, match="multiples of the 256 tile"):
                    mu.matmul_transpose(x)
            else:
                assert lib.muon_hip_mmt_scratch_elems(x.data_ptr(), ref.data_ptr(), M, K) > 0
                assert torch.equal(mu.matmul_transpose(x), ref), cfg
        finally:
            _abi.check(lib.muon_hip_set_gemm_config(_abi.CFG_AUTO))
