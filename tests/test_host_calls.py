"""CPU-only checks of what the native half's callables accept and which route a size query announces: nothing here
launches a kernel."""

import pytest
import torch


@pytest.mark.parametrize("scale,zp", [(0.25, 7), (0.25, 7.0), (torch.tensor(0.25), torch.tensor(7.0)), (1, True)])
def test_lut_callables_take_any_real_scale_and_zero_point(scale, zp):
    """dimq_amd._C.linear_lut / conv2d_lut convert the scale with float() and the zero point with int(), so a float
    zero point read from a checkpoint reaches the op's own checks (here: that its tensors are on the GPU)."""
    from dimq_amd import _C
    pw, cb = torch.zeros(2, dtype=torch.uint8), torch.zeros(16)
    with pytest.raises(RuntimeError, match="linear_lut expects CUDA input"):
        _C.linear_lut(torch.zeros(1, 4), pw, cb, scale, zp, None, 1, 4)
    with pytest.raises(RuntimeError, match="conv2d_lut expects CUDA input"):
        _C.conv2d_lut(torch.zeros(1, 4, 1, 1), pw, cb, scale, zp, None, 1, 4, 1, 1, 1, 1, 0, 0, 1, 1, 1)


def _conv_ws(x_dtype, layout, B, C, H, W, OC, ks, groups, bits=4):
    from dimq_amd import _C
    return _C.lib.dimq_conv2d_codebook_workspace_bytes(x_dtype, layout, B, C, H, W, bits, 0, 0, OC, 1 << bits, OC, ks, ks,
                                                       1, 1, ks // 2, ks // 2, 1, 1, groups, x_dtype, layout, 0, 0, 0)


def test_general_path_workspace_is_bounded():
    """Laid-out activations and flags take at most 256 MiB however large the input: a depthwise layer's would be 8 to 10
    times its fp16 input (2.87 GiB for the first)."""
    from dimq_amd import _C
    limit, weights = 256 << 20, 1 << 20
    for dt in (_C.F32, _C.F16, _C.BF16):
        for layout in (_C.NCHW, _C.NHWC):
            assert 0 < _conv_ws(dt, layout, 128, 96, 112, 112, 96, 3, 96) <= limit + weights
    lut = _C.lib.dimq_conv2d_lut_full_workspace_bytes
    assert 0 < lut(_C.F32, 128, 96, 112, 112, 96, 1, 3, 3, 1, 1, 1, 1, 1, 1, 96, _C.F32) <= limit + weights
    lin = _C.lib.dimq_linear_codebook_full_workspace_bytes
    assert 0 < lin(20_000_000, 3, 16, 4, _C.F32) <= limit + weights
    # one image beyond the bound goes by itself
    assert limit < _conv_ws(_C.F32, _C.NCHW, 2, 64, 640, 640, 64, 3, 64) <= 640 * 640 * 64 * 20 + weights


@pytest.mark.parametrize("M,K,N,bits,general", [
    (17, 2048, 2048, 4, True), (17, 2048, 3072, 4, False), (17, 1024, 8192, 4, False), (48, 2048, 4096, 3, False),
    (64, 2048, 3072, 4, True), (64, 2048, 3200, 4, False), (64, 1024, 4096, 4, False),
    (17, 1536, 1536, 2, True), (17, 1536, 2048, 2, False), (49, 1536, 2048, 2, True), (64, 1024, 8192, 2, False),
    (17, 384, 3072, 4, False), (32, 3072, 768, 4, True), (17, 8192, 1024, 4, True), (64, 2112, 8192, 4, True),
    (17, 4096, 4096, 8, True), (17, 1000, 4096, 4, True), (16, 1000, 4096, 8, False)])
def test_general_path_on_few_rows(M, K, N, bits, general):
    """Up to 64 rows with K % 128 == 0 the general path takes only the layers of few outputs: laying the weights of wider
    ones out costs more than the register-codebook tiles take."""
    from dimq_amd import _C
    need = _C.lib.dimq_linear_codebook_full_workspace_bytes(M, K, N, bits, _C.BF16)
    assert (need >= N * K * 2) == general


@pytest.mark.parametrize("M,K,N,general", [(17, 2048, 3072, True), (17, 2048, 3200, False), (64, 1024, 8192, False)])
def test_general_path_on_few_w4a4_rows(M, K, N, general):
    from dimq_amd import _C
    assert (_C.lib.dimq_linear_lut_full_workspace_bytes(_C.F32, M, N, K, _C.F16) >= N * K * 2) == general


@pytest.mark.parametrize("M,K,N,general", [
    (1, 4096, 4096, True), (16, 8192, 8192, True), (128, 8192, 8192, True), (512, 8192, 8192, False),
    (512, 4096, 4096, True), (768, 4096, 4096, True), (1024, 4096, 4096, False), (4096, 4096, 4096, False),
    (4096, 1024, 4096, True), (4096, 3072, 768, True), (4096, 4000, 4096, True)])
def test_general_path_on_w4a4_codebooks_that_are_not_fp16(M, K, N, general):
    """Their generic tiles keep the products that fill the chip."""
    from dimq_amd import _C
    assert (_C.lib.dimq_linear_lut_full_workspace_bytes(_C.F32, M, N, K, _C.F32) >= N * K * 4) == general


@pytest.mark.parametrize("M,K,N,general", [
    (500, 4000, 4096, True), (1500, 4000, 4096, False), (2047, 4000, 4096, True), (500, 8160, 8192, False),
    (1000, 8160, 8192, True), (1500, 4001, 4096, True), (1500, 928, 4096, True), (2047, 4000, 2048, True)])
def test_general_path_off_the_large_tiles_k_steps(M, K, N, general):
    """K % 32 == 0: the register-codebook tiles keep the products that fill the chip on their smaller form."""
    from dimq_amd import _C
    assert (_C.lib.dimq_linear_codebook_full_workspace_bytes(M, K, N, 4, _C.F16) >= N * K * 2) == general
    assert (_C.lib.dimq_linear_lut_full_workspace_bytes(_C.F32, M, N, K, _C.F16) >= N * K * 2) == general


def test_general_path_leaves_products_beyond_one_launch():
    """2^24 work-groups of 256 threads exceed a launch dimension: those calls keep the larger tiles."""
    from dimq_amd import _C
    lin = _C.lib.dimq_linear_codebook_full_workspace_bytes
    assert lin(4 << 20, 448, 16384, 8, _C.F16) == 0
    assert lin(4 << 20, 448, 16320, 8, _C.F16) > 0
