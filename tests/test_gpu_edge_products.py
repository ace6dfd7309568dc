"""The decoder's edge products of the split and 16-bit modes (tiles of 32 slots, three layers per tile)."""
import numpy as np
import pytest

from hikoboshi_amd import _lib, backbone

from .test_gpu_parity import _fp32_on_trajectory

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision, tol", [(_lib.PRECISION_BF16X3, 2e-3), (_lib.PRECISION_FP16, 2e-2)])
@pytest.mark.parametrize("L", [1, 2, 6, 17, 33, 50, 67])
def test_edge_products_at_tile_edges(gpu_ctx, L, precision, tol):
    """L * min(48, L) slots around multiples of 32 (1, 4, 36, 289, 1089, 2400, 3216): log-probs at T = 1 against the
    fp32 path on the same trajectory. The bounds are the modes' own: split bf16 within 2e-3 at T = 0.1 as measured, a
    tenth of it at T = 1; fp16 operands carry 3 bits more than bf16's, whose error is 0.2-0.4 at T = 0.1, so 0.005 at
    T = 1. A slot's row left out or doubled moves log-probs by 0.1 and more."""
    bb = backbone.single_chain(L, 70 + L)
    order = _lib.decode_order(bb.atom_sources, 3)
    print(f"design L={L} precision={precision}", flush=True)
    gpu_ctx.set_precision(precision)
    try:
        res = gpu_ctx.design(bb.coords, bb.atom_sources, 2, np.arange(2, dtype=np.uint64),
                             order_mode=_lib.ORDER_INPUT_SHARED, orders=order, temperature=1.0)
    finally:
        gpu_ctx.set_precision(_lib.PRECISION_FP32)
    for b in range(2):
        ref = _fp32_on_trajectory(gpu_ctx, bb, res["tokens"][b], order, 1.0)
        assert np.abs(res["log_probs"][b] - ref).max() <= tol
