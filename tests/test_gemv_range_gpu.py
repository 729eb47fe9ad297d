"""GPU parity of the dequant matmuls on values far outside ordinary activations,
on every kernel that a row count selects, against the CPU oracle."""
import numpy as np
import pytest

import oracle_lib as O
from floyd_amd import native
from floyd_amd.native import DeviceBuffer

pytestmark = pytest.mark.gpu


# one row (gemv_kernel), the batch kernel, and the GEMM tiles
@pytest.mark.parametrize("fmt", [1, 2])
@pytest.mark.parametrize("rows,kernel", [(1, "gemv"), (6, "gemv_batch"), (330, "qgemm_kernel")])
def test_swiglu_over_the_range_of_fp32(device, fmt, rows, kernel):
    """silu(g) * u is formed as the oracle forms it wherever it is finite: with a
    product g u beyond fp32, a saturated silu, infinite u.

    The gate and up weights are 1 in column 0 and x is 1 there and 0 elsewhere,
    so an output's g and u are its two scales.  Tolerance: expf, a division and
    two products, each within 2 ulp: 8 * 2^-24 < 1e-6.
    """
    print(f"[gpu] swiglu range fmt={fmt} rows={rows}", flush=True)
    gs = [-np.inf, -1e38, -200.0, -100.0, -88.0, -87.0, -86.5, -50.0, -5.0, -1e-3, -1e-30, 0.0,
          1e-30, 1e-3, 5.0, 50.0, 1e20, 2.5e38, 3.4e38, np.inf]
    us = [-np.inf, -1e38, -1e37, -3.0, -1e-20, 0.0, 1e-20, 3.0, 1e37, 1e38, np.inf]
    g, u = (np.repeat(v.ravel(), 8).astype(np.float32) for v in np.meshgrid(gs, us))
    width, in_width = g.size, 192
    assert kernel in native.gemv_kernel_name(fmt, width, in_width, rows, swiglu=True)
    if fmt == 1:
        q = np.zeros((width, in_width), np.uint8)
        q[:, 0] = 1
    else:
        q = np.full((width, in_width // 2), 0x88, np.uint8)
        q[:, 0] = 0x89
    x = np.zeros((rows, in_width), np.float32)
    x[:, 0] = 1.0
    dq, dg, du, dx = (DeviceBuffer.from_array(a) for a in (q, g, u, x))
    dh = DeviceBuffer(rows * width * 4)
    native.gemv_swiglu(fmt, dq, dg, dq, du, dx, dh, width, in_width, rows)
    got = dh.download(np.float32).reshape(rows, width)
    expect = np.array([O.lib().orc_silu_mul(a, b) for a, b in zip(g, u)], np.float32)
    ordinary = np.isfinite(expect)
    for r in range(rows):
        np.testing.assert_array_equal(got[r][~ordinary], expect[~ordinary])
        # results below fp32's normal range count as zero
        np.testing.assert_allclose(got[r][ordinary], expect[ordinary], rtol=1e-6, atol=1.2e-38)
