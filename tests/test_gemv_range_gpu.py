"""GPU parity of the dequant matmuls on values far outside ordinary activations,
on every kernel that a row count selects, against the CPU oracle."""
import numpy as np
import pytest

import oracle_lib as O
from conftest import rel_l2
from floyd_amd import native
from floyd_amd.native import DeviceBuffer
from test_gemv_batch_gpu import shifted
from test_gemv_gpu import make_weights

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


def unpacked(fmt, q, in_width):
    """The stored integers [out, in] in 64 bits."""
    if fmt == 1:
        return q.view(np.int8).astype(np.float64)
    return (np.stack([q & 15, q >> 4], 2).reshape(q.shape[0], -1)[:, :in_width]).astype(np.float64) - 8


def store(fmt, q, column, value):
    """Sets one column of packed weights."""
    if fmt == 1:
        q.view(np.int8)[:, column] = value
    elif column % 2:
        q[:, column // 2] = q[:, column // 2] & 15 | (value + 8) << 4
    else:
        q[:, column // 2] = q[:, column // 2] & 240 | (value + 8)


def normed(x, nw):
    x = x.astype(np.float64)
    return x / np.sqrt((x * x).mean(1, keepdims=True) + 1e-5) * nw


# (out, in, rows, byte offset of w, of x): widths that are no multiple of a
# 16-byte weight chunk, operands at any address, rows wider than the vector
# kernel's LDS
@pytest.mark.parametrize("fmt", [1, 2])
@pytest.mark.parametrize("out_width,in_width,rows,w_off,x_off", [
    (50, 999, 1, 0, 0), (2000, 999, 1, 0, 0), (50, 999, 6, 0, 0), (333, 4111, 40, 0, 0), (70, 95, 17, 0, 0),
    (60, 40, 3, 0, 0), (40, 15, 2, 0, 0), (3, 2113, 700, 0, 0), (70, 2112, 1, 1, 0),
    (70, 2112, 20, 0, 4), (1500, 2112, 900, 3, 12), (40, 45056, 6, 0, 0), (4096, 45056, 70, 0, 0)])
def test_small_columns_beside_large_ones_keep_fp32(device, fmt, out_width, in_width, rows, w_off,
                                                   x_off):
    """Calls outside the vector kernel's shapes hold x in fp32: columns 1e5 times
    the rest whose weights are 0 take nothing from the others' precision.

    Tolerance: fp32 roundings of products, norm and sums that are added pairwise,
    about 25 of them one after the other at the widest row, 2^-24 each and none
    larger than the result's rms times a few: 1e-6.
    """
    print(f"[gpu] large columns fmt={fmt} O={out_width} I={in_width} rows={rows} "
          f"+{w_off} +{x_off}", flush=True)
    if not (w_off or x_off):
        name = native.gemv_kernel_name(fmt, out_width, in_width, rows)
        assert "gemv_generic" in name or "gemv_batch_kernel" in name and name.endswith("true>")
    q, s = make_weights(fmt, out_width, in_width, seed=out_width + in_width)
    q = q.reshape(out_width, -1)
    x = O.fill_normal(rows * in_width, 7 + rows).reshape(rows, in_width)
    for c in {3, in_width // 2, in_width - 1}:
        x[:, c] *= 1e5
        store(fmt, q, c, 0)
    nw = O.fill_normal(in_width, 4, mean=1.0, std=0.1)
    ds, dn = DeviceBuffer.from_array(s), DeviceBuffer.from_array(nw)
    dy = DeviceBuffer(rows * out_width * 4)
    keep_w, w = shifted(q, w_off)
    keep_x, xp = shifted(x, x_off)
    wt = (unpacked(fmt, q, in_width) * s.astype(np.float64)[:, None]).T
    for norm in (None, dn):
        native.gemv(fmt, w, ds, xp, dy, out_width, in_width, rows, norm_w=norm, eps=1e-5)
        expect = (normed(x, nw) if norm else x.astype(np.float64)) @ wt
        assert rel_l2(dy.download(np.float32).reshape(rows, out_width), expect) < 1e-6
    native.gemv_swiglu(fmt, w, ds, w, ds, xp, dy, out_width, in_width, rows, norm_w=dn, eps=1e-5)
    g = normed(x, nw) @ wt
    # silu(g) g moves by up to 2.1 |g| of g's error, and g here is small
    assert rel_l2(dy.download(np.float32).reshape(rows, out_width), g / (1 + np.exp(-g)) * g) < 4e-6


@pytest.mark.parametrize("fmt", [1, 2])
@pytest.mark.parametrize("out_width,in_width,rows", [
    (100, 2048, 3), (100, 2080, 7), (64, 6144, 40), (2048, 4160, 210), (11264, 2048, 130)])
def test_limbs_hold_30_bits_of_the_largest(device, fmt, out_width, in_width, rows):
    """The limb kernels (the batch kernel in all its token tiles, the GEMM tiles
    whole and split) on rows with columns 1e4 times the rest.

    Bound of one output: an element is cut by less than 2^-29 of the row's
    largest, so its sum by that times the sum of its weights' magnitudes; the
    integer sums are exact, their conversions and the at most 30 additions of
    ranges round 2^-24 of the sum of the products' magnitudes each.
    """
    print(f"[gpu] limbs fmt={fmt} O={out_width} I={in_width} rows={rows}", flush=True)
    name = native.gemv_kernel_name(fmt, out_width, in_width, rows)
    assert "qgemm_kernel" in name or name.endswith("false>")
    q, s = make_weights(fmt, out_width, in_width, seed=out_width + in_width)
    q = q.reshape(out_width, -1)
    x = O.fill_normal(rows * in_width, 7 + rows).reshape(rows, in_width)
    x[:, ::301] *= 1e4
    dw, ds, dx = (DeviceBuffer.from_array(a) for a in (q, s, x))
    dy = DeviceBuffer(rows * out_width * 4)
    native.gemv(fmt, dw, ds, dx, dy, out_width, in_width, rows)
    wt = (unpacked(fmt, q, in_width) * s.astype(np.float64)[:, None]).T
    x = x.astype(np.float64)
    bound = 2.0 ** -29 * np.abs(x).max(1)[:, None] * np.abs(wt).sum(0) + \
        32 * 2.0 ** -24 * (np.abs(x) @ np.abs(wt))
    assert (np.abs(dy.download(np.float32).reshape(rows, out_width) - x @ wt) <= bound).all()
