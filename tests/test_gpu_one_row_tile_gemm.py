"""ops.gemm_tall for 129 .. 256 rows (UnquantizedLinearMethod.apply, layers/linear.py:165-172): tiles of 256 rows x 128 columns and its choice of K slices."""
import pytest
import torch

from test_gpu_share_of_cus import _share

pytestmark = pytest.mark.gpu


@pytest.fixture
def ops():
    from semi_pd_amd import ops
    return ops


def _inputs(M, N, K, dtype):
    g = torch.Generator(device="cpu").manual_seed(M * 7 + N + K)
    return torch.randn(M, K, generator=g).to(dtype).cuda(), (torch.randn(N, K, generator=g) * K ** -0.5).to(dtype).cuda()


# (ragged rows and columns, one K step and several, slices that are not as long as the others; columns of one tile, of a tile and a rest)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(129, 16, 64), (256, 128, 128), (200, 144, 192), (255, 272, 1088), (192, 1536, 2048), (206, 4096, 4096), (1, 112, 64), (300, 400, 576)])
def test_narrow_tiles_match_fp32(ops, monkeypatch, dtype, M, N, K):
    x, w = _inputs(M, N, K, dtype)
    want = x.float() @ w.float().t()
    rtol = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)             # one rounding of the result is half of it
    for geo in ("256", "0"):
        monkeypatch.setenv("SEMIPD_G8_XH", geo)
        for ks in ("0", "1", "2", "5", "16"):
            monkeypatch.setenv("SEMIPD_G8_KS", ks)
            # (sums of K products of size K^-1/2 in another order: K^1/2 2^-24 times a few)
            torch.testing.assert_close(ops.gemm_tall(x, w).float(), want, rtol=rtol, atol=1e-4)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,I,K", [(129, 64, 64), (256, 80, 192), (200, 1408, 2048), (140, 8192, 1024)])
def test_narrow_tiles_with_silu_equal_the_unfused_pair(ops, monkeypatch, dtype, M, I, K):
    x, w = _inputs(M, 2 * I, K, dtype)
    for geo in ("256", "0"):
        monkeypatch.setenv("SEMIPD_G8_XH", geo)
        for ks in ("0", "1", "3"):
            monkeypatch.setenv("SEMIPD_G8_KS", ks)
            assert torch.equal(ops.gemm_tall(x, w, fuse_silu_mul=True), ops.silu_and_mul(ops.gemm_tall(x, w)))


# (a last row tile of which one quarter of the rows is there, one row more, three quarters, one row more, all but one)
@pytest.mark.parametrize("silu", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [257, 320, 321, 384, 385, 448, 449, 767])
def test_last_row_tiles_of_the_eight_wave_form(ops, monkeypatch, dtype, M, silu):
    x, w = _inputs(M, 2 * 144, 640, dtype)
    monkeypatch.setenv("SEMIPD_G8_XH", "128")
    ops.gemm_tall_set_form(8)
    try:
        plain = ops.gemm_tall(x, w)
        got = ops.gemm_tall(x, w, fuse_silu_mul=True) if silu else plain
    finally:
        ops.gemm_tall_set_form(0)
    if silu:
        assert torch.equal(got, ops.silu_and_mul(plain))
    else:
        torch.testing.assert_close(got.float(), x.float() @ w.float().t(), rtol=2.0 ** (-8 if dtype == torch.bfloat16 else -11), atol=1e-4)


def _slices(ops, rows, n, k):
    """How many slices of K a plain product is cut into, and the product."""
    x, w = _inputs(rows, n, k, torch.bfloat16)
    got = ops.gemm_tall_planes(x, w)
    if isinstance(got, torch.Tensor):
        return 1, got, x, w
    # (planes are fp32: their sum is the product before its rounding)
    return got.ksplit, got.planes.view(torch.float32)[: got.ksplit * rows * n].view(got.ksplit, rows, n).sum(0), x, w


# (the choice of 256-column tiles alone stands where the planes' way is the share's: the slices that it takes)
@pytest.mark.parametrize("cus,rows,n,k,slices", [(64, 140, 6144, 4096, 2), (64, 206, 4096, 4096, 4), (48, 206, 28672, 4096, 1), (128, 206, 4096, 4096, 4),
                                                 (192, 140, 28672, 4096, 1), (208, 129, 28672, 4096, 1), (224, 129, 32000, 4096, 1)])
def test_slices_on_a_share_of_the_cus(ops, cus, rows, n, k, slices):
    with _share(cus):
        took, got, x, w = _slices(ops, rows, n, k)
        out = ops.gemm_tall(x, w)
    assert took == slices
    want = x.float() @ w.float().t()
    # (a rounding of the result to bf16 and sums of K products of size K^-1/2 in another order, as above)
    torch.testing.assert_close(got.float(), want, rtol=2.0 ** -8, atol=1e-4)
    torch.testing.assert_close(out.float(), want, rtol=2.0 ** -8, atol=1e-4)


# (one slice of narrow tiles on most of the CUs over a long K is left to the wide ones in two: x does not stay in an L2 beside the weight's stream)
@pytest.mark.parametrize("rows,n,k,slices", [(160, 32768, 6144, 2), (206, 32768, 6144, 2), (240, 30720, 5120, 2), (192, 30720, 5120, 1), (256, 24576, 5120, 1),
                                             (206, 28672, 8192, 2), (206, 28672, 4096, 1)])
def test_slices_of_a_long_k(ops, rows, n, k, slices):
    took, got, x, w = _slices(ops, rows, n, k)
    assert took == slices
    torch.testing.assert_close(got.float(), x.float() @ w.float().t(), rtol=2.0 ** -8, atol=1e-4)
