"""The work this library is timed on: what a program asks of it through its
public entry points, from one projection of one token to a 2048-token prompt
through the whole model.

A case is a dict of plain values.  `kind` says which entry point it takes:

  proj    one projection, RMSNorm'ed input or residual output (mlk_gemv)
  mlp     a dense SwiGLU block with its norm and residual (mlk_gemv_swiglu and
          mlk_gemv)
  head    the final norm and an f32 output head (mlk_gemv)
  host    the fm_matmul_q8 / _q4 call on host buffers, weights cached
  layer   a prompt through a model of one MoE layer (embedding, attention,
          routed and shared experts, head; moonlight_session_prefill, and
          moonlight_test_prefill_layers where every row's output is asked for)
  prefill a prompt through the 27-layer model (moonlight_session_prefill)
  decode  one more token of a running generation on the 27-layer model
          (moonlight_session_decode)

Matrix shapes are those of the Moonlight-16B-A3B configuration, and in the
drawn cases ragged ones as well.  Weights are N(0, 0.02) packed per row as the
container packs them, activations N(0, 1), as in bench.py.
"""
import numpy as np
import torch

from floyd_amd import native
from floyd_amd.session import Model, Session

FORMATS = {"f32": native.MLK_F32, "q8": native.MLK_Q8, "q4": native.MLK_Q4}
HIDDEN, DENSE, INTER, EXPERTS, TOP_K, SHARED = 2048, 11264, 1408, 64, 6, 2816
HEADS, NOPE, ROPE, VALUE, LATENT, LAYERS, VOCAB = 16, 128, 64, 128, 512, 27, 163840
ROUTED_SCALE, THETA, EPS = 2.446, 50000.0, 1e-5
# (out, in) of the configuration's matrices
SHAPES = [(3072, 2048), (576, 2048), (3648, 2048), (2048, 2048), (11264, 2048), (2048, 11264),
          (1408, 2048), (2048, 1408), (2816, 2048), (2048, 2816)]
LAYER_VOCAB = 4096  # the one-layer models' vocabulary: their head stays a small part
LAYER_TRACE = 64    # prompts up to this many tokens ask for every row's output
DECODE_ROOM = 4096  # positions a running generation goes on for before it starts over
# fm_matmul caches weights by their host address for the life of the process, so
# a program keeps them as long
HOST_WEIGHTS = []


def listed():
    return [
        # the query projection of one token: the smallest call, a launch and its latency
        dict(name="proj_q8_1", kind="proj", fmt="q8", out=3072, inp=2048, rows=1, norm=True),
        # o_proj of a short chunk, added to the residual stream
        dict(name="proj_q4_23", kind="proj", fmt="q4", out=2048, inp=2048, rows=23, norm=False),
        # the dense FFN of one decoded token
        dict(name="mlp_q8_1", kind="mlp", fmt="q8", hidden=HIDDEN, inter=DENSE, rows=1),
        # a handful of streams or of drafted tokens through the dense FFN
        dict(name="mlp_q4_6", kind="mlp", fmt="q4", hidden=HIDDEN, inter=DENSE, rows=6),
        # a long prompt through the dense FFN
        dict(name="mlp_q8_777", kind="mlp", fmt="q8", hidden=HIDDEN, inter=DENSE, rows=777),
        # the output head of a few streams
        dict(name="head_3", kind="head", vocab=VOCAB, hidden=HIDDEN, rows=3),
        # the host-buffer matmul, as the reference's CPU engine calls it
        dict(name="host_q8_16", kind="host", fmt="q8", out=2048, inp=2048, rows=16),
        # a decode batch's worth of rows through one MoE layer
        dict(name="layer_q8_8", kind="layer", bits=8, rows=8),
        # a short user turn through one MoE layer
        dict(name="layer_q8_64", kind="layer", bits=8, rows=64),
        # a paragraph through one MoE layer of the 4-bit packing
        dict(name="layer_q4_600", kind="layer", bits=4, rows=600),
        # one token of a generation that stands at 4096 tokens
        dict(name="decode_q8_4096", kind="decode", bits=8, context=4096),
        # a full prompt
        dict(name="prefill_q8_2048", kind="prefill", bits=8, rows=2048),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["proj", "proj", "mlp", "mlp", "head", "host", "layer", "layer", "layer",
                       "prefill", "decode"])
    fmt = rng.choice(["q8", "q4"])
    bits = 8 if fmt == "q8" else 4
    if kind == "proj" or kind == "host":
        out, inp = rng.choice(SHAPES)
        if rng.random() < 0.3:  # other models' widths, most of them no multiple of a tile
            out, inp = _log_int(rng, 100, 12000), _log_int(rng, 100, 12000)
        if kind == "host":
            return dict(kind=kind, fmt=fmt, out=out, inp=inp, rows=_log_int(rng, 1, 200))
        return dict(kind=kind, fmt=fmt, out=out, inp=inp, rows=_log_int(rng, 1, 1200),
                    norm=rng.random() < 0.5)
    if kind == "mlp":
        inter = rng.choice([DENSE, SHARED, INTER, 16 * _log_int(rng, 16, 700)])
        return dict(kind=kind, fmt=fmt, hidden=HIDDEN, inter=inter, rows=_log_int(rng, 1, 1200))
    if kind == "head":
        return dict(kind=kind, vocab=rng.choice([VOCAB, _log_int(rng, 4000, VOCAB)]),
                    hidden=HIDDEN, rows=_log_int(rng, 1, 16))
    if kind == "decode":
        return dict(kind=kind, bits=bits, context=_log_int(rng, 64, 16384))
    return dict(kind=kind, bits=bits, rows=_log_int(rng, 2 if kind == "layer" else 16, 2048))


# ---- inputs -------------------------------------------------------------------


class State:
    """What the program holds: tensors, and for the session cases the model and
    its session, closed with it."""

    def __init__(self, **fields):
        self.__dict__.update(fields)

    def __del__(self):
        for field in ("session", "model"):
            if self.__dict__.get(field) is not None:
                self.__dict__.pop(field).close()


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape, std=1.0):
    return torch.randn(shape, generator=g, device="cuda") * std


def _pack(w, fmt):
    """Rows packed as the container packs them: (bytes, scales)."""
    if fmt == "f32":
        return w, None
    top = 127.0 if fmt == "q8" else 7.0
    s = (w.abs().amax(1) / top).clamp(min=1e-8)
    q = torch.round(w / s[:, None]).clamp(-top - 1, top).to(torch.int32)
    if fmt == "q8":
        return q.to(torch.int8), s
    if q.shape[1] % 2:
        q = torch.nn.functional.pad(q, (0, 1))
    u = q + 8
    return (u[:, 0::2] | (u[:, 1::2] << 4)).to(torch.uint8), s


def _matrix(g, out, inp, fmt):
    return _pack(_normal(g, out, inp, std=0.02), fmt)


def _unpacked(packed, inp):
    """The matrix that packed rows stand for, in 64 bits."""
    w, s = packed
    if s is None:
        return w.double()
    if w.dtype == torch.uint8:
        u = w.to(torch.int16)
        w = torch.stack([u & 15, u >> 4], 2).reshape(w.shape[0], -1)[:, :inp] - 8
    return w.double() * s.double()[:, None]


def _config(case):
    whole = case["kind"] != "layer"
    cfg = dict(expert_bits=case["bits"], dense_bits=case["bits"])
    if not whole:
        cfg.update(layer_count=1, first_dense_layer_count=0, vocab_size=LAYER_VOCAB)
    return cfg


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("layer", "prefill", "decode"):
        model = Model.synthetic(seed=seed % 100003 + 1, **_config(case))
        vocab = LAYER_VOCAB if kind == "layer" else VOCAB
        count = DECODE_ROOM if kind == "decode" else case["rows"]
        ids = np.random.default_rng(seed).integers(0, vocab, count).astype(np.int32)
        if kind == "decode":
            session = Session(model, case["context"] + DECODE_ROOM, 64)
            session.fill_kv(case["context"], seed)
        else:
            session = Session(model, max(case["rows"], 64), max(case["rows"], 64))
        return State(kind=kind, model=model, session=session, ids=ids, seed=seed,
                     context=case.get("context", 0))
    g = _generator(seed)
    if kind == "host":
        w, s = _matrix(g, case["out"], case["inp"], case["fmt"])
        x = _normal(g, case["rows"], case["inp"])
        w, s = w.cpu().numpy(), s.cpu().numpy()
        HOST_WEIGHTS.append((w, s))
        return State(kind=kind, fmt=case["fmt"], w=w, s=s, x=x.cpu().numpy(),
                     y=np.empty((case["rows"], case["out"]), np.float32))
    if kind == "mlp":
        hidden, inter, rows = case["hidden"], case["inter"], case["rows"]
        st = State(kind=kind, fmt=case["fmt"], gate=_matrix(g, inter, hidden, case["fmt"]),
                   up=_matrix(g, inter, hidden, case["fmt"]),
                   down=_matrix(g, hidden, inter, case["fmt"]),
                   norm=1.0 + _normal(g, hidden, std=0.1), x=_normal(g, rows, hidden))
        st.h = torch.empty(rows, inter, device="cuda")
        st.y = torch.empty(rows, hidden, device="cuda")
        return st
    out, inp = (case["vocab"], case["hidden"]) if kind == "head" else (case["out"], case["inp"])
    fmt = "f32" if kind == "head" else case["fmt"]
    st = State(kind=kind, fmt=fmt, w=_matrix(g, out, inp, fmt), x=_normal(g, case["rows"], inp),
               norm=None, resid=None, y=torch.empty(case["rows"], out, device="cuda"))
    if kind == "head" or case["norm"]:
        st.norm = 1.0 + _normal(g, inp, std=0.1)
    else:
        st.resid = _normal(g, case["rows"], out)
    return st


# ---- one pass -----------------------------------------------------------------


def _p(t):
    return None if t is None else t.data_ptr()


def run(state):
    s = state
    if s.kind == "decode":
        at = s.session.position() - s.context
        if at >= DECODE_ROOM:  # the generation has ended: the next one starts
            s.session.fill_kv(s.context, s.seed)
            at = 0
        return s.session.decode(s.ids[at])
    if s.kind == "layer" and s.ids.size <= LAYER_TRACE:
        s.session.reset()
        return s.session.prefill_layers(s.ids)
    if s.kind in ("layer", "prefill"):
        s.session.reset()
        return s.session.prefill(s.ids)
    fmt = FORMATS[s.fmt]
    if s.kind == "host":
        lib = native.load()
        call = lib.fm_matmul_q8 if s.fmt == "q8" else lib.fm_matmul_q4
        call(s.y.ctypes.data, s.x.ctypes.data, s.w.ctypes.data, s.s.ctypes.data, s.y.shape[1],
             s.x.shape[1], s.x.shape[0], 1)
        return s.y
    rows, inp = s.x.shape
    if s.kind == "mlp":
        inter = s.h.shape[1]
        native.gemv_swiglu(fmt, _p(s.gate[0]), _p(s.gate[1]), _p(s.up[0]), _p(s.up[1]), _p(s.x),
                           _p(s.h), inter, inp, rows, norm_w=_p(s.norm), eps=EPS)
        native.gemv(fmt, _p(s.down[0]), _p(s.down[1]), _p(s.h), _p(s.y), inp, inter, rows,
                    resid=_p(s.x))
        return s.y
    native.gemv(fmt, _p(s.w[0]), _p(s.w[1]), _p(s.x), _p(s.y), s.y.shape[1], inp, rows,
                norm_w=_p(s.norm), eps=EPS, resid=_p(s.resid))
    return s.y


# ---- what a pass cannot do without ---------------------------------------------


def _weight_bytes(out, inp, fmt):
    per_row = {"f32": 4 * inp, "q8": inp + 4, "q4": (inp + 1) // 2 + 4}[fmt]
    return out * per_row


def _layer_work(rows, past, fmt, dense):
    """Bytes and operations of one layer for `rows` tokens after `past` cached ones."""
    q, kv, kvb = HEADS * (NOPE + ROPE), LATENT + ROPE, HEADS * (NOPE + VALUE)
    mats = [(q, HIDDEN), (kv, HIDDEN), (kvb, LATENT), (HIDDEN, HEADS * VALUE)]
    macs = sum(o * i for o, i in mats) * rows
    macs += HEADS * (NOPE + ROPE + VALUE) * (rows * past + rows * (rows + 1) // 2)
    nbytes = sum(_weight_bytes(o, i, fmt) for o, i in mats) + 4 * kv * (past + rows)
    if dense:
        mats = 2 * [(DENSE, HIDDEN)] + [(HIDDEN, DENSE)]
        return (nbytes + sum(_weight_bytes(o, i, fmt) for o, i in mats),
                2 * (macs + rows * sum(o * i for o, i in mats)))
    expert = 2 * _weight_bytes(INTER, HIDDEN, fmt) + _weight_bytes(HIDDEN, INTER, fmt)
    shared = 2 * _weight_bytes(SHARED, HIDDEN, fmt) + _weight_bytes(HIDDEN, SHARED, fmt)
    used = EXPERTS * (1 - (1 - TOP_K / EXPERTS) ** rows)
    nbytes += used * expert + shared + 4 * EXPERTS * HIDDEN
    macs += rows * (3 * HIDDEN * (TOP_K * INTER + SHARED) + EXPERTS * HIDDEN)
    return nbytes, 2 * macs


def work(case):
    kind, rows = case["kind"], case.get("rows", 1)
    if kind in ("layer", "prefill", "decode"):
        fmt = "q8" if case["bits"] == 8 else "q4"
        layers, vocab = (1, LAYER_VOCAB) if kind == "layer" else (LAYERS, VOCAB)
        nbytes, flops = 4 * vocab * (HIDDEN + 1) + 4 * rows * HIDDEN, 2 * vocab * HIDDEN
        for layer in range(layers):
            b, f = _layer_work(rows, case.get("context", 0), fmt, layers > 1 and layer == 0)
            nbytes, flops = nbytes + b, flops + f
        if kind == "layer" and rows <= LAYER_TRACE:
            nbytes += 4 * rows * HIDDEN
        return {"bytes": nbytes, "flops": flops}
    if kind == "mlp":
        hidden, inter, fmt = case["hidden"], case["inter"], case["fmt"]
        return {"bytes": 2 * _weight_bytes(inter, hidden, fmt) + _weight_bytes(hidden, inter, fmt) +
                8 * rows * hidden, "flops": 6 * rows * hidden * inter}
    out, inp = (case["vocab"], case["hidden"]) if kind == "head" else (case["out"], case["inp"])
    fmt = "f32" if kind == "head" else case["fmt"]
    resid = out if kind == "proj" and not case["norm"] else 0
    return {"bytes": _weight_bytes(out, inp, fmt) + 4 * rows * (inp + out + resid),
            "flops": 2 * rows * out * inp}


def tolerance(case):
    kind = case["kind"]
    if kind in ("proj", "mlp", "head", "host"):
        # 32-bit sums: 3e-7 to 1e-6 off 64 bits
        return {"rel": 4e-6, "max": 1e-4}
    if kind == "layer":
        # one layer in 32 bits, its split products and its head
        return {"rel": 2e-5, "max": 5e-4}
    # 27 layers, where a near-tie of two experts may fall the other way for a
    # token far from the last one
    return {"rel": 1e-2, "max": 5e-2}


# ---- the same in 64 bits --------------------------------------------------------


def _rmsnorm(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _layer_exact(model, ids, rows_out):
    """The one-layer model on `ids`: the last `rows_out` rows' hidden state and the
    last row's logits."""
    def tensor(name, dtype, shape):
        return torch.from_numpy(model.read_tensor(name, dtype).copy()).cuda().reshape(shape)

    def matrix(name, out, inp):
        name = "model.layers.0." + name + ".weight"
        raw = tensor(name, np.uint8, (out, -1))
        return _unpacked((raw.view(torch.int8) if raw.shape[1] == inp else raw,
                          tensor(name + ".qs", np.float32, (out,))), inp)

    n = ids.size
    embed = tensor("model.embed_tokens.weight", np.float32, (LAYER_VOCAB, HIDDEN))
    x = embed[torch.from_numpy(ids).long().cuda()].double()
    ones = torch.ones(1, dtype=torch.float64, device="cuda")  # the synthetic norms
    xn = _rmsnorm(x, ones)
    # attention: the last rows_out queries over every key
    q = (xn[n - rows_out:] @ matrix("self_attn.q_proj", HEADS * (NOPE + ROPE), HIDDEN).T)
    q = q.reshape(rows_out, HEADS, NOPE + ROPE)
    kv = xn @ matrix("self_attn.kv_a_proj_with_mqa", LATENT + ROPE, HIDDEN).T
    kvb = (_rmsnorm(kv[:, :LATENT], ones) @
           matrix("self_attn.kv_b_proj", HEADS * (NOPE + VALUE), LATENT).T)
    kvb = kvb.reshape(n, HEADS, NOPE + VALUE)

    def rotate(v, at):  # pairs (2 i, 2 i + 1) to halves
        p = torch.arange(ROPE // 2, device="cuda", dtype=torch.float64)
        inv = (torch.tensor(THETA, device="cuda", dtype=torch.float64) ** (-2 * p / ROPE))
        angle = at.double()[:, None] * inv
        c, s = angle.cos(), angle.sin()
        if v.dim() == 3:
            c, s = c[:, None], s[:, None]
        a, b = v[..., 0::2], v[..., 1::2]
        return torch.cat([a * c - b * s, b * c + a * s], -1)

    at = torch.arange(n, device="cuda")
    q_rope, k_rope = rotate(q[..., NOPE:], at[n - rows_out:]), rotate(kv[:, LATENT:], at)
    ctx = torch.empty(rows_out, HEADS, VALUE, dtype=torch.float64, device="cuda")
    hidden = at[None, :] > at[n - rows_out:, None]
    for h in range(HEADS):
        scores = q[:, h, :NOPE] @ kvb[:, h, :NOPE].T + q_rope[:, h] @ k_rope.T
        scores = (scores / (NOPE + ROPE) ** 0.5).masked_fill(hidden, float("-inf"))
        ctx[:, h] = torch.softmax(scores, -1) @ kvb[:, h, NOPE:]
    x = x[n - rows_out:] + ctx.reshape(rows_out, -1) @ matrix("self_attn.o_proj", HIDDEN,
                                                               HEADS * VALUE).T
    # routed and shared experts
    xn = _rmsnorm(x, ones)
    router = tensor("model.layers.0.mlp.gate.weight", np.float32, (EXPERTS, HIDDEN)).double()
    bias = tensor("model.layers.0.mlp.gate.e_score_correction_bias", np.float32, (EXPERTS,))
    score = torch.sigmoid(xn @ router.T)
    top = torch.topk(score + bias.double(), TOP_K, dim=1).indices
    weight = torch.gather(score, 1, top)
    weight = weight / (weight.sum(1, keepdim=True) + 1e-20) * ROUTED_SCALE

    def ffn(name, v, width):
        g = v @ matrix(name + ".gate_proj", width, HIDDEN).T
        u = v @ matrix(name + ".up_proj", width, HIDDEN).T
        return (g * torch.sigmoid(g) * u) @ matrix(name + ".down_proj", HIDDEN, width).T

    out = x + ffn("mlp.shared_experts", xn, SHARED)
    for e in range(EXPERTS):
        row, slot = torch.nonzero(top == e, as_tuple=True)
        if row.numel():
            out.index_add_(0, row, ffn("mlp.experts.%d" % e, xn[row], INTER) *
                           weight[row, slot][:, None])
    head = tensor("lm_head.weight", np.float32, (LAYER_VOCAB, HIDDEN)).double()
    return out, _rmsnorm(out[-1:], ones)[0] @ head.T


def exact(case, seed):
    kind = case["kind"]
    if kind in ("prefill", "decode"):
        return None
    s = prepare(case, seed)
    if kind == "layer":
        whole = s.ids.size <= LAYER_TRACE
        hidden, logits = _layer_exact(s.model, s.ids, s.ids.size if whole else 1)
        return (hidden[None], logits) if whole else logits
    if kind == "host":
        w, scale, x = (torch.from_numpy(v).cuda() for v in (s.w, s.s, s.x))
        return (x.double() @ _unpacked((w, scale), case["inp"]).T).cpu()
    x = s.x.double()
    if kind == "mlp":
        v = _rmsnorm(x, s.norm.double())
        g = v @ _unpacked(s.gate, case["hidden"]).T
        u = v @ _unpacked(s.up, case["hidden"]).T
        return x + (g * torch.sigmoid(g) * u) @ _unpacked(s.down, case["inter"]).T
    y = (x if s.norm is None else _rmsnorm(x, s.norm.double())) @ _unpacked(s.w, s.x.shape[1]).T
    return y if s.resid is None else y + s.resid.double()
