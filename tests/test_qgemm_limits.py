"""Shapes at the ends of the int8 GEMM tiles' integer ranges (qgemm.h): byte
offsets inside a tile and int32 sums, which the dispatch has to keep in range.
No GPU but for the test that runs the call."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from floyd_amd import native
from floyd_amd.native import DeviceBuffer

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def host_values(tmp_path, *expressions):
    """Integer expressions over qgemm.h, evaluated by a host program."""
    src, exe = tmp_path / "values.cpp", tmp_path / "values"
    prints = "".join('printf("%%ld\\n", (long)(%s));' % e for e in expressions)
    src.write_text('#include <cstdio>\n#include "qgemm.h"\n'
                   "using namespace mlh;\nint main() { %s }\n" % prints)
    subprocess.run([HIPCC, "-std=c++17", "--cuda-host-only", "-x", "hip",
                    "-I" + os.path.join(ROOT, "floyd_amd", "csrc"),
                    "-I" + os.path.join(ROOT, "include"), str(src), "-o", str(exe)],
                   check=True, capture_output=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    return [int(v) for v in out.split()]


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_reductions_stay_within_int32(tmp_path):
    """A limb of -128 against a weight of -128 (q8, or 16 times a q4 weight of -8)
    in every column adds up to 2^14 a column: 2^31 at 131072 columns."""
    at = (64, 131008, 131072, 131136, 1 << 20)
    got = host_values(tmp_path, *["qgemm_shape_ok(%s, %d)" % (f, k)
                                  for f in ("kQ8", "kQ4") for k in at])
    assert got == 2 * [int(k * 2 ** 14 < 2 ** 31) for k in at]


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_gathered_rows_stay_within_32_bit_offsets(tmp_path):
    """The MoE tiles reach a gathered row's limbs by a 32-bit offset from row 0,
    of which kQgGatherBytes and more mean a row that is not there: the largest
    batch's last row ends below, and ordinary batches are not cut (16384 rows
    route at most)."""
    widths = (64, 2048, 7168, 16384, 81920, 81984, 131008)
    rows = host_values(tmp_path, *["moe_gemm_max_rows(%d)" % w for w in widths])
    ends = host_values(tmp_path, "kQgGatherBytes", *["limb_bytes(moe_gemm_max_rows(%d), %d)" % (w, w)
                                                     for w in widths])
    assert ends[0] + 16 * 1024 * 1024 < 2 ** 32  # and a slice's offset on top
    assert all(e <= ends[0] for e in ends[1:])
    assert [r >= 16384 for r in rows] == [w <= 81920 for w in widths] and min(rows) > 8192


@pytest.mark.parametrize("fmt", [1, 2])
@pytest.mark.parametrize("swiglu", [False, True])
def test_tile_rows_stay_within_31_bit_offsets(fmt, swiglu):
    """A tile addresses its output rows by 31-bit byte offsets from its first one:
    64 rows of more than 2^23 floats (128 rows of the widest tile: 2^22) reach
    past them, so such a matrix is left to the batch kernel."""
    name = {o: native.gemv_kernel_name(fmt, o, 64, 64, swiglu)
            for o in (4194303, 4194304, 8388700, 16777300)}
    assert "qgemm_kernel" in name.pop(4194303)
    assert all("gemv_batch_kernel" in n for n in name.values()), name


@pytest.mark.gpu
@pytest.mark.parametrize("in_width", [16, 19])
def test_more_rows_than_one_grid(device, in_width):
    """The batch kernel's grid holds 65535 token tiles of 16: more rows run in
    slices, each with its own rows of x, y and the residual."""
    rows, out_width = 16 * 65535 + 21, 3
    print(f"[gpu] O={out_width} I={in_width} rows={rows}", flush=True)
    assert "gemv_batch" in native.gemv_kernel_name(1, out_width, in_width, rows)
    rng = np.random.default_rng(4)
    q = rng.integers(-127, 128, (out_width, in_width), dtype=np.int8)
    s = np.full(out_width, 1.0 / 127, np.float32)
    x = rng.standard_normal((rows, in_width)).astype(np.float32)
    res = rng.standard_normal((rows, out_width)).astype(np.float32)
    dq, ds, dx, dr = (DeviceBuffer.from_array(a) for a in (q.view(np.uint8), s, x, res))
    dy = DeviceBuffer(rows * out_width * 4)
    native.gemv(1, dq, ds, dx, dy, out_width, in_width, rows, resid=dr)
    expect = x.astype(np.float64) @ q.T.astype(np.float64) / 127 + res
    # at most 24 roundings, of sums below 100
    assert np.abs(dy.download(np.float32).reshape(rows, out_width) - expect).max() < 24 * 100 * 2.0 ** -24


@pytest.mark.gpu
def test_outputs_of_over_2_gib(device):
    """64 token rows of 8,388,700 outputs, every output against numpy's fp32
    product (64 columns: at most 64 roundings of 2^-24 each of the sum of the
    products' magnitudes)."""
    out_width, in_width, rows = 8388700, 64, 64
    print(f"[gpu] O={out_width} I={in_width} rows={rows}", flush=True)
    rng = np.random.default_rng(3)
    q = rng.integers(-127, 128, (out_width, in_width), dtype=np.int8)
    s = np.full(out_width, 1.0 / 127, np.float32)
    x = rng.standard_normal((rows, in_width)).astype(np.float32)
    dq, ds, dx = (DeviceBuffer.from_array(a) for a in (q.view(np.uint8), s, x))
    dy = DeviceBuffer(rows * out_width * 4)
    native.gemv(1, dq, ds, dx, dy, out_width, in_width, rows)
    step = 1 << 20
    for r in (0, 31, 62, 63):
        got = dy.download(np.float32, out_width, r * out_width * 4)
        for o in range(0, out_width, step):
            w = q[o:o + step].astype(np.float32)
            bound = 64 * 2.0 ** -23 * (np.abs(w) @ np.abs(x[r])) / 127
            assert (np.abs(got[o:o + step] - (w @ x[r]) / 127) <= bound).all(), (r, o)
