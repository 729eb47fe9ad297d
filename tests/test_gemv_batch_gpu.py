"""GPU parity of the matmuls of several token rows (gemv_batch.hip: q8 / q4, any
width, from 2 token rows where the one-pass kernels of gemv_mfma.hip do not take
the shape; gemv_f32_batch.hip; the GEMM tiles of larger batches) against the CPU
oracle, at the edges of their tiles.

Tolerance: x is cut to 30 bits of the largest of its range (ragged widths and
unaligned operands: fp32) and the limbs' products are exact, so the difference is
the oracle's own serial fp32 sum: at most I * 2^-24 relative, in practice sqrt(I) *
2^-24 = 6e-6 at the widest row here.
"""
import numpy as np
import pytest

import oracle_lib as O
from conftest import rel_l2
from floyd_amd import native
from floyd_amd.native import DeviceBuffer
from test_gemv_gpu import TOL, make_weights

pytestmark = pytest.mark.gpu


def shifted(array, offset):
    """A device copy of `array` that starts `offset` bytes into its allocation."""
    array = np.ascontiguousarray(array)
    buf = DeviceBuffer(array.nbytes + offset)
    buf.upload(array.view(np.uint8).reshape(-1), offset)
    return buf, buf.ptr + offset


# (out, in, rows): token tiles of 4, 8 and 16 with remainders; weight tiles of
# 16, 32 and 64 rows with remainders; one, two and three 2048-column chunks (in
# one workgroup and split over several), ranges that end inside a wave's 256
# columns and inside a 64-column step; widths cut at 16 or 32 columns
SHAPES = [
    (1, 16, 3), (17, 32, 4), (33, 64, 5), (130, 96, 8), (64, 272, 9), (100, 2048, 16),
    (65, 2080, 17), (31, 4096, 33), (2048, 2304, 16), (2048, 1408, 40), (4200, 2048, 6),
    (17000, 64, 16), (576, 11264, 3), (3000, 4160, 20), (40, 6144, 70),
    (33, 15, 3), (20, 33, 5), (50, 999, 2), (64, 2049, 17), (3, 4111, 4),
]


@pytest.mark.parametrize("fmt", [1, 2])
@pytest.mark.parametrize("out_width,in_width,rows", SHAPES)
def test_batch_matches_oracle(device, fmt, out_width, in_width, rows):
    print(f"[gpu] batch fmt={fmt} O={out_width} I={in_width} rows={rows}", flush=True)
    assert "gemv_batch_kernel" in native.gemv_kernel_name(fmt, out_width, in_width, rows)
    check(fmt, out_width, in_width, rows)


# the four-limb GEMM tiles (qgemm.hip) that larger batches take: row tiles of 64
# and column tiles of 256 with remainders, widths that end inside a 128-wide
# slice; reductions in 2 shares, the last of them ending inside a slice, and in 5
# (rows past one launch's scratch: test_gemm_tiles.py)
@pytest.mark.parametrize("fmt", [1, 2])
@pytest.mark.parametrize("out_width,in_width,rows", [
    (11264, 2048, 97), (4100, 64, 300), (3001, 2112, 321), (900, 192, 1100), (5000, 16448, 260),
    (2048, 4160, 210), (300, 11264, 701)])
def test_tiles_match_oracle(device, fmt, out_width, in_width, rows):
    print(f"[gpu] tiles fmt={fmt} O={out_width} I={in_width} rows={rows}", flush=True)
    assert "qgemm_kernel" in native.gemv_kernel_name(fmt, out_width, in_width, rows)
    check(fmt, out_width, in_width, rows)


def check(fmt, out_width, in_width, rows):
    q, s = make_weights(fmt, out_width, in_width, seed=out_width + in_width)
    x = O.fill_normal(rows * in_width, 31 + rows).reshape(rows, in_width)
    nw = O.fill_normal(in_width, 4, mean=1.0, std=0.1)
    res = O.fill_normal(rows * out_width, 9).reshape(rows, out_width)
    xn = np.empty_like(x)
    O.lib().orc_rmsnorm(O.fptr(x), O.fptr(nw), O.fptr(xn), rows, in_width, 1e-5)
    dw, ds, dx, dn, dr = (DeviceBuffer.from_array(a) for a in (q, s, x, nw, res))
    dy = DeviceBuffer(rows * out_width * 4)
    for norm, resid in ((None, None), (dn, dr)):
        native.gemv(fmt, dw, ds, dx, dy, out_width, in_width, rows, norm_w=norm, eps=1e-5,
                    resid=resid)
        expect = O.matmul(fmt, q, s, xn if norm else x, out_width, in_width)
        got = dy.download(np.float32).reshape(rows, out_width)
        assert rel_l2(got, res + expect if resid else expect) < TOL


# f32 matrices of many rows on either side of the line between the batch and the
# vector kernel (narrow ones and 17 rows: vector; the batch kernel's tiles and
# its line: test_f32_batch.py)
@pytest.mark.parametrize("out_width,in_width,rows,norm", [
    (4096, 2048, 3, True), (4099, 4, 4, True), (8200, 252, 5, False), (8193, 260, 8, False),
    (9001, 516, 9, True), (8192, 2048, 17, False), (4100, 4096, 12, True), (4097, 9216, 4, True)])
def test_f32_batch_matches_oracle(device, out_width, in_width, rows, norm):
    print(f"[gpu] f32 batch O={out_width} I={in_width} rows={rows}", flush=True)
    w, _ = make_weights(0, out_width, in_width, seed=out_width + in_width)
    x = O.fill_normal(rows * in_width, 31 + rows).reshape(rows, in_width)
    nw = O.fill_normal(in_width, 4, mean=1.0, std=0.1)
    res = O.fill_normal(rows * out_width, 9).reshape(rows, out_width)
    xn = np.empty_like(x)
    O.lib().orc_rmsnorm(O.fptr(x), O.fptr(nw), O.fptr(xn), rows, in_width, 1e-5)
    dw, dx, dn, dr = (DeviceBuffer.from_array(a) for a in (w, x, nw, res))
    dy = DeviceBuffer(rows * out_width * 4)
    expect = O.matmul(0, w, None, xn if norm else x, out_width, in_width)
    for resid in (None, dr):
        native.gemv(0, dw, None, dx, dy, out_width, in_width, rows, norm_w=dn if norm else None,
                    eps=1e-5, resid=resid)
        got = dy.download(np.float32).reshape(rows, out_width)
        assert rel_l2(got, res + expect if resid else expect) < TOL


@pytest.mark.parametrize("fmt", [1, 2])
@pytest.mark.parametrize("width,in_width,rows", [
    (40, 96, 3), (100, 2048, 7), (1408, 4096, 16), (9000, 64, 17), (33, 999, 6),
    (2816, 192, 200)])  # GEMM tiles
def test_batch_swiglu(device, fmt, width, in_width, rows):
    print(f"[gpu] batch swiglu fmt={fmt} W={width} I={in_width} rows={rows}", flush=True)
    (qg, sg), (qu, su) = (make_weights(fmt, width, in_width, seed=k) for k in (21, 22))
    x = O.fill_normal(rows * in_width, 23).reshape(rows, in_width)
    nw = O.fill_normal(in_width, 24, mean=1.0, std=0.1)
    xn = np.empty_like(x)
    O.lib().orc_rmsnorm(O.fptr(x), O.fptr(nw), O.fptr(xn), rows, in_width, 1e-5)
    g, u = (O.matmul(fmt, q, s, xn, width, in_width).astype(np.float64)
            for q, s in ((qg, sg), (qu, su)))
    bufs = [DeviceBuffer.from_array(a) for a in (qg, sg, qu, su, x, nw)]
    dh = DeviceBuffer(rows * width * 4)
    native.gemv_swiglu(fmt, *bufs[:5], dh, width, in_width, rows, norm_w=bufs[5], eps=1e-5)
    assert rel_l2(dh.download(np.float32), g / (1.0 + np.exp(-g)) * u) < TOL


@pytest.mark.parametrize("fmt,rows", [(1, 3), (2, 20)])
@pytest.mark.parametrize("w_off,x_off", [(1, 0), (0, 4), (3, 12)])
def test_batch_unaligned_operands(device, fmt, rows, w_off, x_off):
    """Weights at any byte and x at any float give the aligned call's result."""
    out_width, in_width = 70, 2112
    q, s = make_weights(fmt, out_width, in_width, seed=3)
    x = O.fill_normal(rows * in_width, 5).reshape(rows, in_width)
    ds, dy = DeviceBuffer.from_array(s), DeviceBuffer(rows * out_width * 4)
    keep_w, w = shifted(q, w_off)
    keep_x, xp = shifted(x, x_off)
    native.gemv(fmt, w, ds, xp, dy, out_width, in_width, rows)
    expect = O.matmul(fmt, q, s, x, out_width, in_width)
    assert rel_l2(dy.download(np.float32).reshape(rows, out_width), expect) < TOL


@pytest.mark.parametrize("fmt,out_width,in_width,rows", [
    (1, 48, 2048, 6), (2, 48, 4103, 6), (1, 9000, 1024, 110)])  # the last: GEMM tiles
def test_batch_nonfinite_inputs(device, fmt, out_width, in_width, rows):
    """A NaN or infinity anywhere in a token row, the cut end included, leaves
    no finite output in it and the other rows untouched."""
    q, s = make_weights(fmt, out_width, in_width, seed=8)
    x = O.fill_normal(rows * in_width, 6).reshape(rows, in_width)
    x[0, 3], x[2, in_width - 1], x[3, 1000] = np.inf, np.nan, -np.inf
    dw, ds, dx = (DeviceBuffer.from_array(a) for a in (q, s, x))
    dy = DeviceBuffer(rows * out_width * 4)
    native.gemv(fmt, dw, ds, dx, dy, out_width, in_width, rows)
    got = dy.download(np.float32).reshape(rows, out_width)
    fine = [r for r in range(rows) if r not in (0, 2, 3)]
    assert not np.isfinite(got[[0, 2, 3]]).any()
    assert rel_l2(got[fine], O.matmul(fmt, q, s, x[fine], out_width, in_width)) < TOL
