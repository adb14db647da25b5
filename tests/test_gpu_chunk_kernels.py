"""Kernels that take one chunk per wave: sets of any make-up, and payloads at the edges of their peer counts."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from oracle import codec as orc  # noqa: E402  (the checker)
import templar_amd.compress as tc  # noqa: E402
from templar_amd import _lib  # noqa: E402


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "these tests need an MI355X"
    return torch.device("cuda:0")


def _randn(shape, rng, dev):
    return torch.empty(shape, device=dev).copy_(torch.from_numpy(rng.standard_normal(shape).astype(np.float32)))


def _sizes(n, rng):
    """(rows, columns) of n tensors of 0 .. 3 chunks, an empty one first, last and in between."""
    out = [(64 * int(rng.integers(0, 3)), 64 * int(rng.integers(1, 3))) for _ in range(n)]
    out[0] = out[-1] = (0, 64)
    out[n // 2] = (64, 192)
    return out


@pytest.mark.parametrize("k", [2, 32, 34, 64, 128])
@pytest.mark.parametrize("n", [1, 3, 8, 9, 64, 65, 513])
def test_untransformed_sets_of_any_make_up(dev, n, k):
    rng = np.random.default_rng(n)
    x = [_randn(s, rng, dev) for s in _sizes(n, rng)]
    batch = tc.TensorBatch(x)
    idx, val = tc.encode_compress_batch(batch, k, use_dct=False)
    want = [orc.topk_rows(orc.encode2d(t.cpu().numpy(), use_dct=False).reshape(-1, 4096), k) for t in x if t.numel()]
    assert np.array_equal(idx.cpu().numpy(), np.concatenate([orc.pack12(i) for i, _ in want]))
    assert np.array_equal(val.cpu().numpy(), np.concatenate([v for _, v in want]))
    ef = [0.5 * t for t in x]
    own, prev = tc.TensorBatch([t.clone() for t in ef]), tc.TensorBatch([t - 0.475 * t for t in x])
    i2, v2 = torch.empty_like(idx), torch.empty_like(val)
    st = _lib.load().tplr_ef_encode_topk_pack_batch(
        ctypes.c_void_p(own.table.data_ptr()), ctypes.c_void_p(prev.table.data_ptr()), n, batch.total_chunks, 0.95, k, 0,
        ctypes.c_void_p(i2.data_ptr()), ctypes.c_void_p(v2.data_ptr()), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert st == 0
    for got, e, g in zip(own.tensors, ef, prev.tensors):
        assert torch.equal(got, e * 0.95 + g)
    i3, v3 = tc.encode_compress_batch(own, k, use_dct=False)
    assert torch.equal(i2, i3) and torch.equal(v2, v3)


# Sets with the transform are walked by one resident round of waves up to a chunk for each, and again from five rounds (k <= 32) or
# twenty on; between, every wave takes one chunk, as all of them do for a single tensor.
@pytest.mark.parametrize("rounds,over,k", [(1, -1, 32), (1, 1, 32), (1, 0, 64), (2, 0, 64), (5, 0, 32), (5, 1, 32), (5, 1, 34), (7, 5, 32),
                                           (20, 0, 64), (20, 1, 64)])
def test_transformed_sets_alike_in_both_forms(dev, rounds, over, k):
    resident = torch.cuda.get_device_properties(dev).multi_processor_count * 12  # three waves a SIMD
    chunks = rounds * resident + over
    rng, gen = np.random.default_rng(chunks), torch.Generator(device=dev).manual_seed(chunks)
    small = [_sizes(n, rng) for n in (150, 150)]  # of 0 to 4 chunks: a wave's range crosses several
    rest = chunks - sum(r * c // 4096 for s in small for r, c in s) - 7 * 17
    shapes = [*small[0], (64 * 7, 64 * 17), (64, 64 * (rest // 2)), *small[1], (64 * (rest - rest // 2), 64)]
    x = [torch.randn(s, device=dev, generator=gen) for s in shapes]
    batch = tc.TensorBatch(x)
    assert batch.total_chunks == chunks
    idx, val = tc.encode_compress_batch(batch, k, use_dct=True)
    for t, one in enumerate(x):
        if one.numel():
            si, sv = batch.payload_slice(t, idx, val, k)
            i1, v1, _, _ = tc.encode_compress(one, k, use_dct=True)
            assert torch.equal(si, i1) and torch.equal(sv.reshape(-1), v1.reshape(-1)), t


@pytest.mark.parametrize("use_dct", [True, False])
@pytest.mark.parametrize("k", [32, 64])
@pytest.mark.parametrize("chunks", [5, 1023, 1024, 1029])  # single waves, and teams of four from a chunk for every SIMD on
def test_momentum_update_and_encode(dev, chunks, k, use_dct):
    gen = torch.Generator(device=dev).manual_seed(chunks)
    shapes = [(64, 64 * 2), (64, 64 * (chunks - 3)), (64, 64)]
    ef, grad = ([torch.randn(s, device=dev, generator=gen) for s in shapes] for _ in range(2))
    want = [e * 0.9 + g for e, g in zip(ef, grad)]
    own, from_ = tc.TensorBatch(ef), tc.TensorBatch(grad)
    idx, val = torch.empty(chunks * k * 3 // 2, dtype=torch.uint8, device=dev), torch.empty(chunks, k, device=dev)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    assert _lib.load().tplr_ef_encode_topk_pack_batch(ptr(own.table), ptr(from_.table), 3, chunks, 0.9, k, int(use_dct), ptr(idx), ptr(val),
                                                      ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    assert all(torch.equal(e, w) for e, w in zip(ef, want))
    i2, v2 = tc.encode_compress_batch(own, k, use_dct=use_dct)
    assert torch.equal(idx, i2) and torch.equal(val, v2)


def _payloads(dev, batch, P, k, rng, repeat):
    """P payloads that share half of their coefficients; `repeat`: some rows name one twice."""
    n = batch.total_chunks
    shared = np.stack([rng.permutation(4096)[: k // 2] for _ in range(n)])
    idxs, vals = [], []
    for _ in range(P):
        own = np.stack([rng.permutation(np.setdiff1d(rng.permutation(4096)[: 3 * k], s))[: k - k // 2] for s in shared])
        idx = rng.permuted(np.concatenate([shared, own], 1), axis=1)
        if repeat:
            idx[:: max(1, n // 3), -1] = idx[:: max(1, n // 3), 0]
        idxs.append(torch.from_numpy(orc.pack12(idx)).to(dev))
        vals.append(torch.from_numpy(rng.standard_normal((n, k)).astype(np.float32)).to(dev))
    return idxs, vals


# (the last: more chunks than waves that can be resident at a time)
@pytest.mark.parametrize("shapes,repeat", [([(64, 64)], False), ([(64, 64)], True), ([(0, 64), (128, 192), (64, 64), (64, 320), (0, 64)], False),
                                           ([(0, 64), (128, 192), (64, 64), (64, 320), (0, 64)], True),
                                           ([(2048, 8192), (2048, 320)], False)])
@pytest.mark.parametrize("P,k", [(1, 64), (2, 32), (3, 32), (4, 64), (5, 64), (6, 16), (7, 4), (8, 34), (9, 32), (12, 64), (13, 4),
                                 (15, 32), (15, 64)])
def test_payloads_with_the_transform(dev, shapes, P, k, repeat):
    rng = np.random.default_rng(1000 * P + k)
    params = [_randn(s, rng, dev) for s in shapes]
    before = [p.clone() for p in params]
    out = tc.TensorBatch([torch.full_like(p, 7.0) for p in params])
    batch = tc.TensorBatch(params)
    idxs, vals = _payloads(dev, batch, P, k, rng, repeat)
    scale = torch.from_numpy(rng.uniform(0.5, 1.0, (len(batch), P)).astype(np.float32)).to(dev)
    n = batch.total_chunks
    lib, stream = _lib.load(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    lists = [(ctypes.c_void_p * P)(*[t.data_ptr() for t in ts]) for ts in (idxs, vals)]
    flags = torch.zeros(len(batch), dtype=torch.int32, device=dev)
    chunk_stats, stats = torch.zeros(2 * n, device=dev), torch.zeros(4 * len(batch), device=dev)
    assert lib.tplr_decode_aggregate_batch(*lists, ptr(scale), P, k, ptr(out.table), len(batch), n, 0, 0, 1, None, stream) == 0
    assert lib.tplr_outer_step_batch(*lists, ptr(scale), P, k, ptr(batch.table), len(batch), n, ptr(chunk_stats), ptr(stats), ptr(flags),
                                     stream) == 0
    assert not bool(flags.any())
    for t in range(len(batch)):
        if params[t].numel() == 0:
            continue
        # the step subtracts exactly what the aggregate leaves
        assert torch.equal(params[t], before[t] - out.tensors[t]), t
        if params[t].numel() <= 1 << 20:
            sl = [batch.payload_slice(t, i, v, k) for i, v in zip(idxs, vals)]
            Y, X = batch.xshape(t)[:2]
            coef = orc.batch_decompress([i.cpu().numpy() for i, _ in sl],
                                        [(v * scale[t, p]).cpu().numpy().reshape(Y, X, k) for p, (_, v) in enumerate(sl)],
                                        batch.xshape(t), 4096, clip_norm=False)
            want = orc.decode2d(coef)
            assert np.abs(out.tensors[t].cpu().numpy() - want).max() <= 1e-5 * np.abs(want).max()
    ss = torch.stack([o.double().square().sum() for o in out.tensors if o.numel()])
    got = torch.stack([stats[4 * t + 3].double() for t in range(len(batch)) if params[t].numel()])
    assert bool((got - ss).abs().le(4e-5 * ss).all())
    # a chunk whose result is not finite is left as it is, and its tensor flagged
    last = max(t for t in range(len(batch)) if params[t].numel())
    vals[P - 1][-1, 0] = float("nan")
    kept = params[last].clone()
    assert lib.tplr_outer_step_batch(*lists, ptr(scale), P, k, ptr(batch.table), len(batch), n, None, None, ptr(flags), stream) == 0
    assert flags.cpu().tolist() == [int(t == last) for t in range(len(batch))]
    assert torch.equal(params[last][-64:, -64:], kept[-64:, -64:])


def _crowded(dev, n, k, seed, repeat):
    """A payload of n rows whose entries lie among 256 coefficients of the chunk (so that peers meet in them); `repeat`: every fifth
    row names one twice."""
    gen = torch.Generator(device=dev).manual_seed(seed)
    idx = torch.rand((n, 256), device=dev, generator=gen).topk(k, dim=1).indices * 16 + 5
    if repeat:
        idx[::5, k - 1] = idx[::5, 0]
    return tc.pack_12bit_indices(idx.reshape(-1)), torch.randn((n, k), device=dev, generator=gen)


@pytest.mark.parametrize("staged", [False, True])
@pytest.mark.parametrize("repeat", [False, True])
@pytest.mark.parametrize("P,k", [(2, 64), (3, 32), (4, 2), (7, 64), (8, 32), (9, 32), (12, 64), (15, 32), (15, 64)])
def test_aggregates_with_the_transform_alike_in_both_forms(dev, P, k, repeat, staged):
    # Up to 8192 chunks a wave takes one (k_decode_chunk), beyond resident waves take several in turn (k_decode_aggregate): the same
    # payload rows give the same bits, chunks on the exact path and chunks that are not finite among them.
    shapes = [(64 * 40, 64 * 100), (0, 64), (64 * 33, 64 * 64), (64, 64 * 2080)]
    extra = (64, 64)
    n = sum(r * c // 4096 for r, c in shapes)
    assert n == 8192
    pays = [_crowded(dev, n + 1, k, 10 * P + p, repeat) for p in range(P)]
    pays[P - 1][1][77, 0], pays[0][1][8000, 1], pays[P // 2][1][4100, 0] = float("nan"), float("inf"), float("-inf")
    if staged:
        ib, vb = (torch.stack([p[i].reshape(-1) for p in pays]) for i in (0, 1))
        pays = [(ib[p], vb[p].view(n + 1, k)) for p in range(P)]
    scale = torch.rand((len(shapes) + 1, P), device=dev) + 0.5
    got = []
    for last in ([], [extra]):
        out = tc.TensorBatch([torch.full(s, 7.0, device=dev) for s in shapes + last])
        m = out.total_chunks
        ss = torch.zeros(m, device=dev)
        tc.batch_decompress_decode_batch(out, [i[: m * k * 3 // 2] for i, _ in pays], [v[:m] for _, v in pays], k,
                                         scale=scale[: len(out)].contiguous(), use_dct=True, sumsq=ss)
        got.append((out.tensors, ss))
    for a, b in zip(got[0][0], got[1][0]):
        assert bool(((a.view(torch.int32) == b.view(torch.int32)) | (a.isnan() & b.isnan())).all())
    a, b = got[0][1], got[1][1][:n]
    assert bool(((a == b) | (a.isnan() & b.isnan()) | ((a - b).abs() <= 1e-5 * a)).all())


@pytest.mark.parametrize("T,P", [(1, 1), (3, 20), (65, 64), (130, 65), (7, 128)])
def test_factors_of_updates(dev, T, P):
    rng = np.random.default_rng(T)
    lib, stream = _lib.load(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    scale = torch.from_numpy(rng.uniform(0.1, 1.0, (T, P)).astype(np.float32)).to(dev)
    for t, bad in zip(range(1, T), [0.0, -1.0, float("nan"), float("inf"), float("-inf")]):
        scale[t, P - 1 - t % P] = bad
    want = torch.where((torch.isfinite(scale) & (scale > 0)).all(1, keepdim=True), scale * 0.4, float("nan"))
    got = torch.empty_like(scale)
    for code in (None, torch.zeros(1, dtype=torch.int32, device=dev), torch.full((1,), 9, dtype=torch.int32, device=dev)):
        assert lib.tplr_outer_factors(ptr(scale), T, P, 0.4, None if code is None else ptr(code), ptr(got), stream) == 0
        refused = code is not None and int(code)
        assert torch.equal(got.isnan(), torch.ones_like(want, dtype=torch.bool) if refused else want.isnan())
        assert refused or torch.equal(got.nan_to_num(-1.0), want.nan_to_num(-1.0))
    # one peer's: the norm from P partial sums
    ss, clip = scale.nan_to_num(1.0, 1.0, 1.0).abs(), torch.from_numpy(rng.uniform(0.0, 2.0 * P**0.5, T).astype(np.float32)).to(dev)
    clip[T // 2] = float("nan")
    f = torch.empty(T, device=dev)
    assert lib.tplr_update_factors(ptr(ss), P, ptr(clip), -0.5, T, ptr(f), stream) == 0
    torch.testing.assert_close(f.double(), -0.5 * (clip.double() / (ss.double().sum(1).sqrt() + 1e-8)).clamp(max=1), rtol=3e-7, atol=0,
                               equal_nan=True)  # (three roundings of a single precision)
    assert lib.tplr_update_factors(None, 0, ptr(clip), -0.5, T, ptr(f), stream) == 0
    torch.testing.assert_close(f, -0.5 * clip, rtol=0, atol=0, equal_nan=True)
    for lr, squares in ((-0.4, 0.16), (0.7, 0.49), (1e-23, 1e-30)):
        lr = float(np.float32(lr))
        stats = torch.from_numpy(rng.uniform(1.0, 2.0, (T, 4)).astype(np.float32) * np.float32([abs(lr), lr, 1.0, squares])).to(dev)
        want = stats.cpu().double() / torch.tensor([abs(lr), lr, 1.0, lr * lr], dtype=torch.float64)
        assert lib.tplr_outer_stats(ptr(stats), T, lr, stream) == 0
        assert torch.equal(stats.cpu(), want.float())  # the quotients, rounded once


_PEERS = [(1, 64), (2, 2), (3, 32), (4, 64), (5, 64), (8, 32), (9, 34), (12, 64), (13, 16), (15, 64), (16, 64), (20, 64), (21, 32), (24, 64)]


# (47 x 48: more than a resident round of workgroups per chunk; 64 x 128: the last of the rows, and of one or two peers past it)
@pytest.mark.parametrize("repeat", [False, True])
@pytest.mark.parametrize("Y,X,P,k", [(*s, *p) for s in ((47, 48), (64, 128)) for p in _PEERS] +
                         [(128, 192, 1, 32), (129, 191, 1, 64), (96, 128, 2, 64), (97, 127, 2, 32)])
def test_parameter_of_a_chunk_per_wave(dev, Y, X, P, k, repeat):
    n, rng = Y * X, np.random.default_rng(100 * P + k)
    unit = tc.TensorBatch([torch.empty(64, 64 * 41, device=dev)])
    idx, val = _payloads(dev, unit, P, k, rng, repeat)
    over = -(-n // 41)  # the payload rows over and over
    idx = [i.repeat(over)[: n * k * 3 // 2].contiguous() for i in idx]
    val = [v.repeat(over, 1)[:n].contiguous() for v in val]
    val[-1][3, 0], val[0][5, 1] = float("inf"), float("nan")
    lib, stream = _lib.load(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    lists = [(ctypes.c_void_p * P)(*[t.data_ptr() for t in ts]) for ts in (idx, val)]
    norms = torch.from_numpy(rng.gamma(2.0, 1.0, P).astype(np.float32)).to(dev)
    scale, scratch = torch.empty(P, device=dev), torch.empty(P, device=dev)
    assert lib.tplr_clip_scales(ptr(norms), P, 0, ptr(scale), None, stream) == 0
    for factors in ("norms", "factors", "none"):
        for ld in (X * 64, X * 64 + 12, 0):
            got, want = torch.full((2, n * 4096 + 12 * 64 * Y), 7.0, device=dev)
            given = ptr(norms) if factors == "norms" else None
            own = {"norms": ptr(scratch), "factors": ptr(scale), "none": None}[factors]
            assert lib.tplr_aggregate_param(*lists, given, P if given else 0, own, P, k, Y * 64, X * 64, ptr(got), ld, stream) == 0
            assert lib.tplr_decode_aggregate(*lists, None if factors == "none" else ptr(scale), P, k, Y * 64, X * 64, 0, 0, 0, ptr(want), ld,
                                             None, stream) == 0
            same = (got.view(torch.int32) == want.view(torch.int32)) | (got.isnan() & want.isnan())
            assert bool(same.all()), (factors, ld)


def _decoder(shape, dev):
    from types import SimpleNamespace

    p = SimpleNamespace(requires_grad=True, shape=shape, dtype=torch.float32, device=dev)
    return tc.ChunkingTransformer(SimpleNamespace(named_parameters=lambda: [("p", p)]), 64)


@pytest.mark.parametrize("Y,X", [(1, 1), (3, 1), (1, 2), (5, 3), (2, 4), (7, 5), (1, 65), (130, 9)])
def test_untransformed_decode(dev, Y, X):
    tr, base = _decoder((Y * 64, X * 64), dev), torch.randn(Y * X * 4096 + 8, device=dev)
    for at in (0, 1, 4):  # aligned for wide loads or not
        x = base[at: at + Y * X * 4096].view(Y, X, 64, 64)
        out = tr.decode(x, use_dct=False)
        assert out.is_contiguous() and torch.equal(out, x.permute(0, 2, 1, 3).reshape(Y * 64, X * 64))
        assert (out.data_ptr() == x.data_ptr()) == (X == 1)


def test_untransformed_decode_under_transforms_and_modes(dev):
    from torch.utils._python_dispatch import TorchDispatchMode

    tr, x = _decoder((128, 192), dev), torch.randn(4, 2, 3, 64, 64, device=dev)
    want = torch.stack([tr.decode(c, use_dct=False) for c in x])
    assert torch.equal(torch.func.vmap(lambda c: tr.decode(c, use_dct=False))(x), want)
    out, tangent = torch.func.jvp(lambda c: tr.decode(c, use_dct=False), (x[0],), (x[1],))
    assert torch.equal(out, want[0]) and torch.equal(tangent, want[1])
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x[0], x[2])
        out, tangent = torch.autograd.forward_ad.unpack_dual(tr.decode(dual, use_dct=False))
        assert torch.equal(out, want[0]) and torch.equal(tangent, want[2])
    seen = []

    class Log(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with Log():
        assert tr.decode(x[0], use_dct=False).shape == (128, 192)
    assert any("permute" in s for s in seen)


@pytest.mark.parametrize("n_rows,k", [(1, 2), (1, 6), (5, 6), (3, 64), (1025, 64), (4099, 34)])
@pytest.mark.parametrize("n_words", [1, 3, 64])
def test_check_of_indices(dev, n_rows, k, n_words):
    rng, lib = np.random.default_rng(n_rows), _lib.load()
    pairs = n_rows * k // 2
    for where in (None, 0, pairs - 1, int(rng.integers(0, pairs))):
        for length, worst in ((4095, 4095), (100, 100), (1, 1)):
            idx = rng.integers(0, length, (n_rows, k))
            if where is not None:
                idx.reshape(-1)[2 * where + int(rng.integers(0, 2))] = worst
            for shift in (0, 1):  # payload bytes that do not begin on a word
                buf = torch.zeros(pairs * 3 + 1, dtype=torch.uint8, device=dev)
                buf[shift: shift + pairs * 3] = torch.from_numpy(orc.pack12(idx)).to(dev)
                words = torch.full((n_words,), -1, dtype=torch.int32).pin_memory()
                assert lib.tplr_check_rows(buf.data_ptr() + shift, n_rows, k, length, words.data_ptr(), n_words,
                                           torch.cuda.current_stream().cuda_stream) == 0
                torch.cuda.synchronize()
                want = [int(where is not None and pairs * i // n_words <= where < pairs * (i + 1) // n_words) for i in range(n_words)]
                assert words.tolist() == want
    assert lib.tplr_check_rows(buf.data_ptr(), n_rows, k, 4097, words.data_ptr(), n_words, None) == _lib.TPLR_E_TOOMANY
