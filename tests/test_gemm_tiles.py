"""The int8 GEMM tiles (qgemm.hip) in every size that the dispatch chooses: which
tile a session's projections and a gemv() of many rows run on (no GPU), and parity
of each with 64-bit products or the CPU oracle.

A three-limb tile holds an activation to half of 2^-22 of its row's largest value,
a four-limb tile cuts less than 2^-29; the integer sums are exact, and their
conversions and the epilogue round at most 32 times by 2^-24 of the sum of the
products' magnitudes.
"""
import os

import numpy as np
import pytest

import container_util as CU
import oracle_lib as O
from conftest import rel_l2
from floyd_amd import native
from floyd_amd import session as S
from floyd_amd.native import DeviceBuffer
from test_gemv_gpu import make_weights
from test_gemv_range_gpu import normed, unpacked
from test_moonlight_scale_gpu import moe_layer_names, oracle_with
from test_prefill_gpu import outlier_rows
from test_qgemm_limits import HIPCC, host_values

Q, DOWN = "model.layers.0.self_attn.q_proj.weight", "model.layers.0.mlp.down_proj.weight"
# (weight, columns, outputs, token rows, token rows of the tile): rows and outputs
# that end inside tiles
DENSE = [(Q, 2048, 3072, 511, 32), (Q, 2048, 3072, 701, 64), (Q, 2048, 3072, 1399, 128),
         (DOWN, 11264, 2048, 331, 32)]
# a model of one dense layer, (token rows, tile of o_proj and down, residual added)
RESID = [(511, 32), (1100, 64), (2100, 128)]
RESID_CFG = dict(layer_count=1, first_dense_layer_count=1, dense_intermediate_size=1024,
                 vocab_size=512)
# the SwiGLU pair of 11264 outputs
SWIGLU = [(50, 32), (100, 64), (300, 128)]
# gemv() of more rows than one launch's scratch: (outputs, columns, rows)
CHUNKED = [(300, 192, 8500), (700, 38400, 500)]


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_rules(tmp_path):
    """The cases below run on the tiles they name."""
    cases = [(o, r, i, 0, t) for _, i, o, r, t in DENSE]
    cases += [(2048, r, i, 0, t) for r, t in RESID for i in (2048, 1024)]
    cases += [(11264, r, 2048, 1, t) for r, t in SWIGLU]
    got = host_values(tmp_path, *[e for o, r, i, d, _ in cases for e in
                                  ("gemv_batch_fits(%d, %d, %d)" % (o * (d + 1), r, i),
                                   "tile_bm(dense_tile(%d, true, %d, %d))" % (r, o, d))])
    assert got == [v for *_, t in cases for v in (0, t)]
    chunks = host_values(tmp_path, *["tiles_chunk(%d, %d)" % (r, i) for _, i, r in CHUNKED])
    for (o, i, r), chunk in zip(CHUNKED, chunks):
        assert chunk < r and chunk % 8 == 0
        for fmt in (1, 2):
            assert "qgemm_kernel" in native.gemv_kernel_name(fmt, o, i, r)


@pytest.fixture(scope="module", params=[8, 4], ids=["q8", "q4"])
def moon(request, device):
    model = S.Model.synthetic(layer_count=2, vocab_size=3072, expert_bits=request.param,
                              dense_bits=request.param, seed=6)
    O.lib().orc_set_threads(16)
    yield model, 1 if request.param == 8 else 2
    model.close()


def matrix(model, fmt, name, out, width):
    q = model.read_tensor(name, np.uint8).reshape(out, -1)
    s = model.read_tensor(name + ".qs", np.float32)
    return (unpacked(fmt, q, width) * s.astype(np.float64)[:, None]).T


@pytest.mark.gpu
@pytest.mark.parametrize("name,width,out,rows,tile", DENSE,
                         ids=["%s-%d" % (d[0].split(".")[-2], d[3]) for d in DENSE])
def test_projections(moon, name, width, out, rows, tile):
    model, fmt = moon
    print(f"[gpu] dense tile {tile}: {name} T={rows}", flush=True)
    w = matrix(model, fmt, name, out, width)
    sess = S.Session(model, 2048, 2048)
    for x in (O.fill_normal(rows * width, 500 + rows).reshape(rows, width),
              outlier_rows(rows, width, 600 + rows)):
        got = sess.test_matmul(name, x, out)
        assert got is not None
        x = x.astype(np.float64)
        bound = 2.0 ** -23 * np.abs(x).max(1)[:, None] * np.abs(w).sum(0) + \
            32 * 2.0 ** -24 * (np.abs(x) @ np.abs(w))
        assert (np.abs(got - x @ w) <= bound).all()
    sess.close()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,tile", SWIGLU)
def test_swiglu_pair(moon, rows, tile):
    """gate / up on the tile, then the down projection (batch kernel)."""
    model, fmt = moon
    print(f"[gpu] SwiGLU tile {tile}: T={rows}", flush=True)
    p = "model.layers.0.mlp."
    g, u = (matrix(model, fmt, p + m + "_proj.weight", 11264, 2048) for m in ("gate", "up"))
    x = O.fill_normal(rows * 2048, 800 + rows).reshape(rows, 2048)
    sess = S.Session(model, 512, 512)
    got = sess.test_dense_mlp(0, x)
    assert got is not None
    gate = x @ g
    expect = (gate / (1 + np.exp(-gate)) * (x @ u)) @ matrix(model, fmt, DOWN, 2048, 11264)
    # two projections one after the other, each 1e-6 at N(0, 1) rows of these widths
    assert rel_l2(got, expect) < 4e-6
    sess.close()


@pytest.mark.gpu
@pytest.mark.parametrize("bits", [8, 4])
def test_residual_outputs(device, bits):
    """o_proj and the down projection added to the residual stream, on all three
    tiles, through a prefill of one dense layer."""
    model = S.Model.synthetic(expert_bits=bits, dense_bits=bits, seed=8, **RESID_CFG)
    cfg = dict(CU.TINY, hidden_size=2048, head_count=16, kv_lora_rank=512, qk_nope_dim=128,
               qk_rope_dim=64, value_dim=128, **RESID_CFG)
    O.lib().orc_set_threads(16)
    for rows, tile in RESID:
        print(f"[gpu] residual tile {tile}: T={rows} q{bits}", flush=True)
        orc = O.Model(cfg, rows)
        for name, *_ in CU.tensor_specs(cfg):
            for n in (name, name + ".qs"):
                info = model.tensor_info(n)
                if info is not None:
                    orc.add(n, model.read_tensor(n, np.uint8 if info[0] == 3 else np.float32),
                            dtype=info[0])
        ids = np.random.default_rng(rows).integers(0, 512, rows).astype(np.int32)
        expect = np.empty((1, rows, 2048), np.float32)
        trace = np.empty((1, rows, 6), np.int32)
        logits = np.empty(512, np.float32)
        assert O.lib().orc_forward(orc.handle, O.iptr(ids), rows, 0, O.fptr(expect), O.iptr(trace),
                                   O.fptr(logits))
        sess = S.Session(model, rows, rows)
        layers, got = sess.prefill_layers(ids)
        # the oracle's serial fp32 sums: 2048 * 2^-24 at most, sqrt of that in practice
        assert rel_l2(layers, expect) < 1e-5 and rel_l2(got, logits) < 1e-5
        sess.close()
        orc.close()
    model.close()


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [1, 2])
@pytest.mark.parametrize("out_width,in_width,rows", CHUNKED)
def test_rows_past_the_scratch(device, fmt, out_width, in_width, rows):
    """gemv() on the four-limb tiles in two launches: the second one's rows of x,
    y and the residual, its own number of shares, the scratch used again."""
    print(f"[gpu] tiles in chunks fmt={fmt} O={out_width} I={in_width} rows={rows}", flush=True)
    q, s = make_weights(fmt, out_width, in_width, seed=out_width + in_width)
    w = (unpacked(fmt, q.reshape(out_width, -1), in_width) * s.astype(np.float64)[:, None]).T
    x = O.fill_normal(rows * in_width, 31 + rows).reshape(rows, in_width)
    nw = O.fill_normal(in_width, 4, mean=1.0, std=0.1)
    res = O.fill_normal(rows * out_width, 9).reshape(rows, out_width)
    dq, ds, dx, dn, dr = (DeviceBuffer.from_array(a) for a in (q, s, x, nw, res))
    dy = DeviceBuffer(rows * out_width * 4)
    for norm, resid in ((None, None), (dn, dr)):
        native.gemv(fmt, dq, ds, dx, dy, out_width, in_width, rows, norm_w=norm, eps=1e-5,
                    resid=resid)
        xs = normed(x, nw) if norm else x.astype(np.float64)
        expect = xs @ w + (res if resid else 0.0)
        # a norm adds the roundings of its sum (at most 64 in one chain)
        bound = 2.0 ** -29 * np.abs(xs).max(1)[:, None] * np.abs(w).sum(0) + \
            (96 if norm else 32) * 2.0 ** -24 * (np.abs(xs) @ np.abs(w)) + 2.0 ** -22 * np.abs(expect)
        got = dy.download(np.float32).reshape(rows, out_width)
        assert (np.abs(got - expect) <= bound).all()


# reductions shared by several workgroups, whose counters and shares are the
# library's own: the batch kernel (limbs and fp32) and the tiles
@pytest.mark.gpu
@pytest.mark.parametrize("fmt,out_width,in_width,rows", [
    (1, 576, 11264, 20), (2, 40, 6145, 20), (1, 2048, 4160, 210)])
def test_replays_repeat_the_eager_call(device, fmt, out_width, in_width, rows):
    print(f"[gpu] graph replays fmt={fmt} O={out_width} I={in_width} rows={rows}", flush=True)
    q, s = make_weights(fmt, out_width, in_width, seed=out_width + in_width)
    x = O.fill_normal(rows * in_width, 31 + rows)
    dq, ds, dx = (DeviceBuffer.from_array(a) for a in (q, s, x))
    eager, dy = DeviceBuffer(rows * out_width * 4), DeviceBuffer(rows * out_width * 4)
    native.gemv(fmt, dq, ds, dx, eager, out_width, in_width, rows)
    expect = eager.download(np.float32)
    for launches in (1, 4):  # per replay; each graph is replayed twice
        dy.zero()
        native.time_gemv(fmt, [dq], [ds], dx, dy, out_width, in_width, rows, 1, launches)
        np.testing.assert_array_equal(dy.download(np.float32), expect)
        native.gemv(fmt, dq, ds, dx, eager, out_width, in_width, rows)
        np.testing.assert_array_equal(eager.download(np.float32), expect)


@pytest.mark.gpu
def test_moe_128_row_tile(moon):
    """Experts of more than 140 rows each on average (1601 rows of 6 experts): the
    largest tile for q4 too."""
    model, _ = moon
    rows = 1601
    print(f"[gpu] MoE T={rows}", flush=True)
    ids = O.zipf_routes(rows, 64, 6, seed=4)
    x = O.fill_normal(rows * 2048, 12).reshape(rows, 2048)
    sess = S.Session(model, rows, rows)
    sess.fix_routes(ids)
    got = sess.test_moe(1, x)
    assert got is not None and np.array_equal(got["ids"], ids)
    orc = oracle_with(model, moe_layer_names(1), 8)
    expect, w = np.empty_like(x), np.empty((rows, 6), np.float32)
    assert O.lib().orc_moe_layer_fixed(orc.handle, 1, O.fptr(x), rows, O.iptr(ids), O.fptr(w),
                                       O.fptr(expect))
    assert rel_l2(got["out"], expect) < 1e-5
    sess.fix_routes(None)
    sess.close()
    orc.close()
