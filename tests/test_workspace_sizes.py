"""CPU checks of the workspace queries: pure functions of the sizes, which any
program may ask before it has data, sizes of zero included."""
import pytest

from ml_engine_amd import hip


@pytest.mark.parametrize("zero", range(4))
def test_queries_take_empty_products(zero):
    sizes = [300, 520, 700, 2]
    sizes[zero] = 0
    assert hip.lib().mle_gemm_ws_bytes(*sizes) == 0
    if zero < 3:  # rows, in, out; a layer there is always
        for layers in (1, 3):
            dx = hip.lib().mle_gemm_sum_ws_bytes(sizes[0], sizes[1], layers)
            assert hip.lib().mle_linear_bwd_ws_bytes(*sizes[:3], layers) == dx


@pytest.mark.parametrize("rows", [65536, 1_000_000])
def test_narrow_weight_gradient_workspace(rows):
    """256 -> 10 over many rows: what the plan's splits need (the gradient's own
    10 KB a split), not a split per 32 rows (21 MB and 321 MB)."""
    assert hip.lib().mle_linear_bwd_ws_bytes(rows, 256, 10, 1) <= 4e6
    assert hip.lib().mle_gemm_ws_bytes(64, 10, rows, 1) <= 4e6


@pytest.mark.parametrize("n,cin,side,cout,limit_mb", [(32, 1024, 32, 1024, 152), (16, 256, 128, 256, 20)])
def test_weight_gradient_workspace_follows_the_chip_not_the_pixels(n, cin, side, cout, limit_mb):
    """At most four partial gradients, or what fills the chip."""
    assert hip.lib().mle_conv2d_wgrad_ws_bytes(n, cin, side, side, cout, 3, 3, 1, 1) <= limit_mb * 1e6
