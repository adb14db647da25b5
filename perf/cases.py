"""The work that users of the codec have it do, as measurable cases.

Two ways of calling it are in use and both are here.  A program that only changes the import keeps the reference's
calls, one parameter at a time (`encode` and `compress`; `decompress` or `batch_decompress` and `decode`); a program
written for this package hands over a whole gradient set at once (`TensorBatch`, `RowBatch`, `PayloadStage`).
Settings: the default ones (64x64 chunks through the transform, top 32, values sent as fp32) and the production ones
(chunks not transformed, top 64, values sent as the codes of a four-bin quantiser, 20 peers).

Gradients are heavy-tailed (Student t with three degrees of freedom) with a scale of their own per row; the peers'
gradients of one parameter share half of their signal, so that their selections overlap as they do in training.
"""
import math
from types import SimpleNamespace

import torch

import templar_amd.compress as tc

DECAY = 0.95     # the miner's momentum decay
LR = 0.4         # the outer step's learning rate
BINS = 4         # the production quantiser
RANGE = 6

_M1B = dict(layers=16, hidden=2048, kv=2048, inter=8192, vocab=32000)
_M150M = dict(layers=12, hidden=768, kv=768, inter=3072, vocab=32000)
_BLOCK72B = dict(layers=1, hidden=8192, kv=1024, inter=29568, vocab=0)


# ---------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # a norm vector through the reference's calls: the smallest call there is, nothing but latency
        dict(name="vector_send", kind="send", rows=0, cols=2048, k=32, dct=True, bins=0),
        # an attention projection of a 1B model, sent with the default settings
        dict(name="param_send", kind="send", rows=2048, cols=2048, k=32, dct=True, bins=0),
        # the miner's loop body for an up-projection with the production settings: what is sent is also taken back
        # out (decompress, decode) to be subtracted from the error feedback
        dict(name="param_send_codes", kind="send_back", rows=8192, cols=2048, k=64, dct=False, bins=BINS),
        # the outer step's loop body for one projection, fifteen peers, default settings
        dict(name="param_receive", kind="receive", rows=2048, cols=2048, k=32, peers=15, dct=True, bins=0),
        # the same for a down-projection with the production settings: twenty peers' codes
        dict(name="param_receive_codes", kind="receive", rows=2048, cols=8192, k=64, peers=20, dct=False, bins=BINS),
        # a parameter whose dimensions 64 does not divide (chunks of 60 x 50), there and back
        dict(name="param_ragged", kind="send_back", rows=3000, cols=1000, k=32, dct=True, bins=0),
        # whole gradient sets, sent: a small model, and a 1B model
        dict(name="set_send_150m", kind="set_send", k=32, dct=True, **_M150M),
        dict(name="set_send_1b", kind="set_send", k=32, dct=True, **_M1B),
        # the window's aggregate of a 1B model from fifteen peers, clip factors included
        dict(name="set_receive_1b", kind="set_receive", k=32, peers=15, dct=True, **_M1B),
        # the miner's whole step on one block of a 72B model (its largest matrices, top 64)
        dict(name="set_miner_step_72b", kind="set_miner_step", k=64, dct=True, bins=0, **_BLOCK72B),
        # the outer step of a 1B model with the production settings, straight from twenty peers' codes
        dict(name="set_outer_step_1b", kind="set_outer_step", k=64, peers=20, dct=False, bins=BINS, **_M1B),
        # the validator's evaluation of one peer: its decoded, clipped update taken off every parameter
        dict(name="set_eval_update_1b", kind="set_eval", k=32, dct=True, **_M1B),
    ]


def draw(rng):
    """One more case: any kind, sizes over the range between the small and the large listed ones."""

    def spread(lo, hi):  # evenly over the logarithm
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["vector", "send", "send_back", "receive", "ragged", "set_send", "set_receive", "set_miner_step",
                       "set_outer_step", "set_eval"])
    production = rng.random() < 0.5
    k = 64 if production else rng.choice([16, 32, 32, 48])
    dct, bins = not production, BINS if production else 0
    peers = rng.randint(16, 24) if production else rng.randint(1, 15)
    if kind == "vector":
        return dict(kind="send", rows=0, cols=64 * spread(2, 256), k=min(k, 64), dct=dct, bins=bins)
    if kind in ("send", "send_back", "receive"):
        case = dict(kind=kind, rows=64 * spread(4, 160), cols=64 * spread(4, 160), k=k, dct=dct, bins=bins)
        if kind == "receive":
            case["peers"] = peers
        return case
    if kind == "ragged":  # chunk edges below 64: the largest divisor up to 64 of each dimension
        edge = lambda: rng.choice([20, 24, 30, 40, 45, 48, 50, 52, 56, 60, 63])  # noqa: E731
        return dict(kind=rng.choice(["send", "send_back"]), rows=edge() * spread(4, 96), cols=edge() * spread(4, 96),
                    k=32, dct=True, bins=0)
    hidden = 64 * spread(6, 40)
    inter = 64 * spread(16, 128)
    per_layer = 2 * hidden * hidden * 2 + 3 * hidden * inter
    vocab = 64 * spread(16, 500)
    layers = max(1, min(spread(1, 24), int((1.0e9 - 2 * vocab * hidden) / per_layer)))
    case = dict(kind=kind, k=k, dct=dct, layers=layers, hidden=hidden, kv=64 * rng.randint(1, hidden // 64), inter=inter,
                vocab=vocab)
    if kind == "set_receive":
        case.update(dct=True, k=min(k, 48) if peers > 15 else k, peers=min(peers, 20))
    elif kind == "set_outer_step":
        case.update(peers=peers, bins=bins)
    elif kind == "set_miner_step":
        case.update(bins=bins)
    elif kind == "set_eval":
        case.update(dct=True)
    return case


# ---------------------------------------------------------------------------------------- sizes
def _shapes(case):
    h, kv, i, v = case["hidden"], case["kv"], case["inter"], case["vocab"]
    two, one = [], []
    for _ in range(case["layers"]):
        two += [(h, h), (kv, h), (kv, h), (h, h), (i, h), (i, h), (h, i)]
        one += [(h,), (h,)]
    if v:
        two += [(v, h), (v, h)]
        one += [(h,)]
    return two, one


def _edges(case):
    """(chunk rows, chunk columns) of a parameter."""
    h = tc._get_smaller_split(case["rows"], 64) if case["rows"] else 1
    return h, tc._get_smaller_split(case["cols"], 64)


def _param(case):
    """(elements, payload entries) of a parameter."""
    h, w = _edges(case)
    n = (case["rows"] or 1) * case["cols"]
    k = max(min(case["k"], h * w), 2)
    return n, n // (h * w) * (k - k % 2)


def work(case):
    """Bytes: every input read once, every output written once.  Operations: a 64-point transform of a row takes
    about 540 of them factorised (8.4 per value and direction of the chunk), a selection one comparison per value, an
    entry received a multiplication and an addition."""
    bins, P = case.get("bins", 0), case.get("peers", 1)
    entry = 1.5 + (1 if bins else 4)
    kind = case["kind"]
    if kind in ("send", "send_back", "receive"):
        n, sent = _param(case)
        one = 0
    else:
        two, vec = _shapes(case)
        n = sum(r * c for r, c in two)
        sent = n // 4096 * case["k"]
        one = sum(s[0] for s in vec)
        sent1 = one // 64 * min(case["k"], 64)
    transform = 2 * 8.4 * n if case["dct"] else 0
    if kind == "send":
        return {"bytes": 4 * n + entry * sent, "flops": transform + n}
    if kind == "send_back":
        return {"bytes": 8 * n + entry * sent, "flops": 2 * transform + n}
    if kind == "receive":
        return {"bytes": 4 * n + P * entry * sent, "flops": transform + 2 * P * sent}
    if kind == "set_send":
        return {"bytes": 4 * (n + one) + entry * (sent + sent1), "flops": transform + n + one}
    if kind == "set_receive":
        return {"bytes": 4 * (n + one) + P * entry * (sent + sent1), "flops": transform + 2 * P * (sent + sent1)}
    if kind == "set_miner_step":
        return {"bytes": 12 * n + entry * sent, "flops": 2 * transform + 4 * n}
    # the outer step and the evaluation update: parameters read and written
    return {"bytes": 8 * n + P * entry * sent, "flops": transform + 2 * n + 2 * P * sent}


# ---------------------------------------------------------------------------------------- inputs
def _gradient(shape, gen, dev):
    z = torch.randn((4,) + tuple(shape), generator=gen, device=dev)
    g = z[0].mul_(1e-3).div_(torch.sqrt_((z[1].square_() + z[2].square_() + z[3].square_()).div_(3.0)))
    if len(shape) == 2:
        g.mul_(torch.exp_(0.5 * torch.randn((shape[0], 1), generator=gen, device=dev)))
    return g.clone()


def _transformer(shapes, dev):
    params = [SimpleNamespace(requires_grad=True, shape=tuple(s), dtype=torch.float32, device=dev) for s in shapes]
    model = SimpleNamespace(named_parameters=lambda: ((f"p{i}", p) for i, p in enumerate(params)))
    return tc.ChunkingTransformer(model, target_chunk=64)


def _compressor(bins):
    if not bins:
        return tc.TopKCompressor()
    return tc.TopKCompressor(use_quantization=True, quantization_bins=bins, quantization_range=RANGE)


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    state = _prepare_set(case, gen, dev) if case["kind"].startswith("set_") else _prepare_param(case, gen, dev)
    state.update(kind=case["kind"], k=case["k"], dct=case["dct"])
    return state


def _prepare_param(case, gen, dev):
    shape = (case["rows"], case["cols"]) if case["rows"] else (case["cols"],)
    tr, comp = _transformer([shape], dev), _compressor(case["bins"])
    state = dict(transformer=tr, compressor=comp, quantised=bool(case["bins"]), x=_gradient(shape, gen, dev))
    if case["kind"] == "receive":
        idxs, vals, qps, norms = [], [], [], []
        for _ in range(case["peers"]):
            g = _gradient(shape, gen, dev).add_(state["x"], alpha=0.5)
            sent = comp.compress(tr.encode(g, use_dct=case["dct"]), case["k"])
            idxs.append(sent[0])
            vals.append(sent[1])
            if case["bins"]:
                qps.append(sent[4])
            norms.append(torch.linalg.vector_norm(comp._dequantize_values(sent[1], sent[4]) if case["bins"] else sent[1]))
        # the outer step has the peers' norms in hand: it logs them before it aggregates
        state.update(idxs=idxs, vals=vals, qps=qps, norms=torch.stack(norms), xshape=sent[2], totalk=sent[3])
    return state


def _flat(shapes, dev):
    """A set's tensors as views of one buffer, as a sharded optimiser holds them: (buffer, views)."""
    buf = torch.empty(sum(math.prod(s) for s in shapes), device=dev)
    return buf, [v.view(s) for v, s in zip(buf.split([math.prod(s) for s in shapes]), shapes)]


def _prepare_set(case, gen, dev):
    kind, k, dct = case["kind"], case["k"], case["dct"]
    two, one = _shapes(case)
    base = [_gradient(s, gen, dev) for s in two]
    batch = tc.TensorBatch(base)
    if kind == "set_send":
        return dict(batch=batch, rows=tc.RowBatch([_gradient(s, gen, dev) for s in one]) if one else None)
    if kind == "set_miner_step":
        # error feedback carries several steps of what was not sent
        flat, views = _flat(two, dev)
        for v in views:
            v.copy_(_gradient(v.shape, gen, dev)).mul_(2.0)
        return dict(batch=tc.TensorBatch(views), flat=flat, grad=batch, compressor=_compressor(case["bins"]))
    bins, peers = case.get("bins", 0), case.get("peers", 1)
    stage = tc.PayloadStage(batch, k, peers, quantized=bool(bins)) if kind != "set_eval" else None
    idxs, vals, tables = [], [], []
    base1 = [_gradient(s, gen, dev) for s in one] if kind == "set_receive" else []
    idxs1, vals1 = [], []
    flat, views = _flat(two, dev)
    own = tc.TensorBatch(views)
    for p in range(peers):
        for t, b in zip(own.tensors, base):
            t.copy_(_gradient(b.shape, gen, dev).add_(b, alpha=0.5))
        idx, val = tc.encode_compress_batch(own, k, use_dct=dct)
        if bins:
            val, shift, _, lookup = tc.quantize_batch(own, val, k, bins, RANGE)
            tables.append((lookup + shift[:, None]).float())
        if stage is not None:  # the window as it is staged: the peers' payloads equally spaced
            ri, rv = stage.regions(p)
            ri.copy_(idx)
            rv.copy_(val)
            idx, val = ri, rv
        idxs.append(idx)
        vals.append(val)
        if base1:
            rows = tc.RowBatch([_gradient(b.shape, gen, dev).add_(b, alpha=0.5) for b in base1])
            i1, v1 = tc.encode_compress_rows_batch(rows, k, use_dct=dct)
            idxs1.append(i1)
            vals1.append(v1)
    state = dict(batch=own, flat=flat, idxs=idxs, vals=vals, stage=stage, rows=None)
    if kind == "set_receive":
        if base1:
            flat1, views1 = _flat(one, dev)
            state.update(rows=tc.RowBatch(views1), flat1=flat1, idxs1=idxs1, vals1=vals1)
        return state
    for t, b in zip(own.tensors, base):  # the parameters to be updated
        t.copy_(b).mul_(20.0)
    if bins:
        state["tables"] = (torch.stack(tables, dim=1).contiguous(), bins)
    if kind == "set_eval":  # the window's clip norms: this peer is clipped in about half of the parameters
        norms = torch.stack([torch.linalg.vector_norm(own.payload_slice(i, idxs[0], vals[0], k)[1]) for i in range(len(own))])
        state["clip_norm"] = norms * torch.exp(0.1 * torch.randn(len(own), generator=gen, device=dev))
    return state


# ---------------------------------------------------------------------------------------- one pass
def run(state):
    kind, k, dct = state["kind"], state["k"], state["dct"]
    if kind in ("send", "send_back"):
        tr, comp, x = state["transformer"], state["compressor"], state["x"]
        sent = comp.compress(tr.encode(x, use_dct=dct), k)
        out = [sent[0], sent[1]]
        if state["quantised"]:
            out += [sent[4][0], sent[4][3]]
        if kind == "send_back":
            out.append(tr.decode(comp.decompress(x, *sent), use_dct=dct))
        return out
    if kind == "receive":
        tr, comp, x = state["transformer"], state["compressor"], state["x"]
        vals = state["vals"]
        if state["quantised"]:
            vals = comp.maybe_dequantize_values(vals, state["qps"], x.device)
        dense = comp.batch_decompress(x, state["idxs"], vals, state["xshape"], state["totalk"], quantize_params=None,
                                      block_norms=state["norms"], normalise=False, clip_norm=True)
        return tr.decode(dense, use_dct=dct)
    if kind == "set_send":
        out = list(tc.encode_compress_batch(state["batch"], k, use_dct=dct))
        if state["rows"] is not None:
            out += tc.encode_compress_rows_batch(state["rows"], k, use_dct=dct)
        return out
    if kind == "set_receive":
        tc.batch_decompress_decode_batch(state["batch"], state["idxs"], state["vals"], k, use_dct=dct)
        out = [state["flat"]]
        if state["rows"] is not None:
            tc.batch_decompress_decode_rows_batch(state["rows"], state["idxs1"], state["vals1"], k, use_dct=dct)
            out.append(state["flat1"])
        return out
    if kind == "set_miner_step":
        idx, val, quant = tc.error_feedback_step_batch(state["batch"], state["grad"], DECAY, k, use_dct=dct,
                                                       compressor=state["compressor"])
        if quant is not None:  # what is sent per parameter: its codes and its table
            val = [torch.cat([q.reshape(-1) for q, _ in quant]), torch.stack([qp[3] for _, qp in quant])]
        return {"idx": idx, "val": val, "error_feedback": state["flat"]}
    if kind == "set_outer_step":
        if "tables" in state:
            stats, skipped = tc.outer_step_codes_batch(state["batch"], state["idxs"], state["vals"], None, k, LR,
                                                       tables=state["tables"])
        else:
            stats, skipped = tc.outer_step_batch(state["batch"], state["idxs"], state["vals"], k, LR, use_dct=dct)
        return [stats, state["flat"]]
    tc.apply_decoded_batch(state["batch"], state["idxs"][0], state["vals"][0], k, alpha=LR, clip_norm=state["clip_norm"],
                           use_dct=dct)
    return state["flat"]


def tolerance(case):
    """Measured: every case against itself with all inputs times three, so that every product and sum rounds
    differently, scaled back.  What is received, decoded or updated then differs by at most 2.2e-7 (largest single
    difference 5.8e-6 of the value).  What is selected after a transform differs where two magnitudes are equal up to
    rounding and change places: 2.3e-5 of the index bytes, and, because such a pair often differs in sign, 7e-3 of
    the values in the 2-norm.  In a small parameter a single such pair (six bytes) is a larger share.  Selections from
    untransformed values involve no rounding; a code may fall on the edge of its bin."""
    kind = case["kind"]
    if kind not in ("send", "send_back", "set_send", "set_miner_step"):
        return {"rel": 1e-6, "max": 2.5e-5}
    if kind in ("send", "send_back"):
        sent = _param(case)[1]
    else:
        sent = sum(r * c for r, c in _shapes(case)[0]) // 4096 * case["k"]
    if case["dct"]:
        # one exchanged pair in a small parameter: two of `sent` values with the other's sign
        return {"rel": max(3e-2, 2.0 / math.sqrt(sent)), "differ": max(1e-4, 6.0 / (1.5 * sent))}
    return {"rel": 1e-6, "differ": max(1e-5, 4.0 / sent) if case.get("bins") else 0.0}
