"""The f32 batch matmul (gemv_f32_batch.hip): where the dispatch takes it (no GPU),
and parity with the CPU oracle at the edges of its tiles."""
import os

import numpy as np
import pytest

import oracle_lib as O
from conftest import rel_l2
from floyd_amd import native
from floyd_amd.native import DeviceBuffer
from test_gemv_gpu import TOL, make_weights
from test_qgemm_limits import HIPCC, host_values

# (weight rows, columns, token rows, norm, token rows of a workgroup or 0 for the
# vector kernel)
RULE = [
    (163840, 2048, 2, 1, 0), (163840, 2048, 3, 1, 4), (163840, 2048, 8, 1, 8),
    (163840, 2048, 4, 0, 0), (163840, 2048, 6, 0, 8), (20000, 5120, 6, 0, 0),
    # narrow matrices, where a pass of a few weight rows costs more than their bytes
    (70000, 64, 3, 1, 0), (20000, 256, 16, 1, 0), (9000, 348, 8, 1, 0), (9000, 352, 8, 1, 8),
    (9000, 352, 9, 1, 0), (70000, 64, 8, 0, 0), (20490, 352, 9, 0, 0), (20000, 704, 8, 0, 0),
    (9000, 1024, 8, 0, 8),
    # padded token rows and the last round of workgroups
    (9000, 2048, 9, 0, 0), (9000, 2048, 16, 0, 16), (20000, 1024, 9, 0, 16),
    (9000, 1024, 17, 0, 0), (9000, 512, 16, 1, 16), (9000, 512, 17, 1, 0)]


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_rule(tmp_path):
    got = host_values(tmp_path, *["f32_batch_rows(%d, %d, %d, %d)" % case[:4] for case in RULE])
    assert got == [case[4] for case in RULE]
    for o, i, rows, norm, b in RULE:
        if not norm:
            name = native.gemv_kernel_name(0, o, i, rows)
            assert name.endswith("gemv_f32_batch_kernel<%d>" % b) if b else "gemv_kernel" in name


# token tiles of 4, 8 and 16 with remainders, weight tiles of 64 and 32 with
# remainders, rows that end inside a wave's two loads, rows that fill the LDS
@pytest.mark.gpu
@pytest.mark.parametrize("out_width,in_width,rows,norm,tokens", [
    (4096, 352, 3, 1, 4), (4099, 356, 4, 1, 4), (4100, 9212, 4, 1, 4), (4097, 516, 7, 1, 8),
    (8200, 1028, 5, 0, 8), (8193, 1024, 8, 0, 8), (4100, 4096, 12, 1, 8), (9001, 916, 9, 1, 16),
    (16401, 1028, 9, 0, 16), (8200, 1300, 30, 0, 16), (4100, 2048, 17, 1, 16)])
def test_matches_oracle(device, tmp_path, out_width, in_width, rows, norm, tokens):
    print(f"[gpu] f32 batch O={out_width} I={in_width} rows={rows} norm={norm}", flush=True)
    if os.path.exists(HIPCC):
        assert host_values(tmp_path, "f32_batch_rows(%d, %d, %d, %d)" %
                           (out_width, in_width, rows, norm)) == [tokens]
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
