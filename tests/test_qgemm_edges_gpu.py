"""GPU parity of the int8 GEMM (qgemm.hip) at the edges of its k slices and row
tiles, through the session's MoE block, against the CPU oracle:
reductions that end inside a 128-wide slice (hidden 192 and 320, expert width
64 and 192) or are whole slices (256, 128), 8-row limb blocks that a task
starts or ends inside, one and several row tiles.

Tolerance: activations are held to 2^-23 of their row's largest value, in two
projections one after the other; 1e-5 is ten times that at these widths' ratio
of largest value to rms.
"""
import numpy as np
import pytest

import container_util as CU
import oracle_lib as O
from conftest import rel_l2
from floyd_amd import session as S

pytestmark = pytest.mark.gpu
TOL = 1e-5


# (hidden, expert width, bits): expert reductions of 64 and 192 end inside a
# slice, of 128 and 320 + 64 are whole slices and a part
@pytest.fixture(scope="module", params=[(192, 64, 8), (320, 192, 4), (256, 128, 8), (256, 128, 4)],
                ids=lambda p: "h%d_i%d_q%d" % p)
def edge(request, device, tmp_path_factory):
    hidden, inter, bits = request.param
    cfg = dict(CU.TINY, hidden_size=hidden, moe_intermediate_size=inter, layer_count=2)
    tensors = CU.build_tensors(cfg, ebits=bits, dbits=bits, seed=hidden + inter + bits)
    model = S.Model.open(CU.write_container(str(tmp_path_factory.mktemp("edge")), cfg, tensors))
    yield cfg, tensors, model, bits
    model.close()


# streaming tile (k a multiple of 128) or 32-row tile, 32-row tiles with one
# and several row tiles per expert, and for q8 64-row tiles (400 rows: over 32 rows
# per expert) and 128-row tiles (1000 rows: over 64); q4 stays on 32 rows here
@pytest.mark.parametrize("rows", [3, 17, 61, 400, 1000])
def test_moe_block_edges(edge, rows):
    cfg, tensors, model, bits = edge
    hidden = cfg["hidden_size"]
    print(f"[gpu] MoE edges hidden={hidden} rows={rows} q{bits}", flush=True)
    x = O.fill_normal(rows * hidden, rows).reshape(rows, hidden)
    sess = S.Session(model, 1024, 1024)
    got = sess.test_moe(1, x)
    orc = CU.oracle_model(cfg, tensors, 8)
    e = {k: np.empty_like(x) for k in ("routed", "shared", "out")}
    ids, w = np.empty((rows, 6), np.int32), np.empty((rows, 6), np.float32)
    logits = np.empty((rows, 64), np.float32)
    assert O.lib().orc_moe_layer(orc.handle, 1, O.fptr(x), rows, O.iptr(ids), O.fptr(w),
                                 O.fptr(logits), O.fptr(e["routed"]), O.fptr(e["shared"]),
                                 O.fptr(e["out"]))
    same = (got["ids"] == ids).all(axis=1)  # a near-tie may fall the other way
    assert same.mean() > 0.99
    for k, v in e.items():
        assert rel_l2(got[k][same], v[same]) < TOL, k
    sess.close()
