"""GPU parity of the absorbed prefill attention of many rows against the CPU
oracle: the form that keys past the expanded copy take, here at a head shape that
the expanded form has no kernel for (nope 64, rope 16, value 64; latent 512), so
that short caches reach it.  Up to 256 rows attend one to an 8-wave workgroup,
more in pairs on 4 waves (an odd last row alone); from 65 rows the value
projection is the head GEMM.

Tolerance: split-f16 products (22 bits each) in fp32 sums over 512 dims, as in the
few-row test: 1e-5.
"""
import numpy as np
import pytest

import container_util as CU
import oracle_lib as O
from conftest import rel_l2
from floyd_amd import session as S

pytestmark = pytest.mark.gpu
CFG = dict(CU.TINY, layer_count=1, kv_lora_rank=512, qk_nope_dim=64, qk_rope_dim=16, value_dim=64)


@pytest.mark.parametrize("bits", [8, 4])
def test_many_rows(device, tmp_path, bits):
    tensors = CU.build_tensors(CFG, ebits=bits, dbits=bits, seed=50 + bits)
    model = S.Model.open(CU.write_container(str(tmp_path), CFG, tensors))
    sess = S.Session(model, 1300, 512)
    orc = CU.oracle_model(CFG, tensors, 1300)
    O.lib().orc_set_threads(16)
    pos = 0
    for rows in (65, 257, 258, 200, 256, 64):
        print(f"[gpu] absorbed attention q{bits}: {rows} rows at {pos}", flush=True)
        x = O.fill_normal(rows * 256, 60 + rows).reshape(rows, 256)
        got = sess.test_attention(0, x, pos)
        assert got is not None
        expect = np.empty_like(x)
        assert O.lib().orc_attention(orc.handle, 0, O.fptr(x), rows, pos, O.fptr(expect))
        assert rel_l2(got, expect) < 1e-5, rows
        pos += rows
    sess.close()
    orc.close()
    model.close()
