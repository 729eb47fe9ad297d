"""GPU parity of the prefill attention of few rows at the Moonlight shape (16
heads, latent 512) against the CPU oracle: the value projection of 16-row and
16-output workgroups (up to 63 rows) and the expansion of few keys (64 rows or
more, a quarter of a head's outputs per workgroup), q8 and q4 kv_b.

Tolerance: split-f16 products (22 bits each) in fp32 sums over 512 dims,
1.3e-6 to 1.6e-6 in the larger prefills; 1e-5 leaves the oracle's serial sums.
"""
import numpy as np
import pytest

import oracle_lib as O
from conftest import rel_l2
from floyd_amd import session as S
from test_moonlight_scale_gpu import attention_names, oracle_with

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[8, 4])
def one_layer(request, device):
    model = S.Model.synthetic(layer_count=1, first_dense_layer_count=0, vocab_size=512,
                              expert_bits=8, dense_bits=request.param, seed=5)
    yield model
    model.close()


# rows at position 0 then rows after them: 16-row groups whole and cut, then the
# expansion of one, two and five 64-key blocks
@pytest.mark.parametrize("first,then", [(2, 15), (17, 48), (63, 3), (64, 0), (70, 65), (200, 120)])
def test_attention_of_few_rows(one_layer, first, then):
    print(f"[gpu] MLA few rows {first} + {then}", flush=True)
    sess = S.Session(one_layer, 512, 256)
    orc = oracle_with(one_layer, attention_names(0), 512)
    x = O.fill_normal((first + then) * 2048, first + then).reshape(-1, 2048)
    pos = 0
    for rows in (first, then):
        if not rows:
            continue
        part = np.ascontiguousarray(x[pos:pos + rows])
        got = sess.test_attention(0, part, pos)
        expect = np.empty_like(part)
        assert O.lib().orc_attention(orc.handle, 0, O.fptr(part), rows, pos, O.fptr(expect))
        assert rel_l2(got, expect) < 1e-5
        pos += rows
    sess.close()
    orc.close()
