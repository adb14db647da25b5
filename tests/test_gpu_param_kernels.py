"""Kernels behind the reference's per-parameter calls, at the sizes where their tilings can go wrong."""
import ctypes
import os
import subprocess
import sys
import threading
import time

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


@pytest.mark.parametrize("h,w", [(1, 1), (1, 17), (1, 50), (1, 64), (2, 2), (7, 1), (16, 16), (16, 17), (17, 16), (15, 48),
                                 (31, 64), (33, 5), (48, 33), (49, 32), (60, 50), (63, 63), (64, 49), (64, 64)])
@pytest.mark.parametrize("Y,X", [(1, 1), (3, 5), (37, 41)])
def test_dense_transform_at_tile_edges(dev, h, w, Y, X):
    rng = np.random.default_rng(h * 100 + w)
    x = rng.standard_normal((Y * h, X * w)).astype(np.float32)
    bh, bw = rng.standard_normal((h, h)).astype(np.float32), rng.standard_normal((w, w)).astype(np.float32)
    chunks = x.reshape(Y, h, X, w).transpose(0, 2, 1, 3)
    x64 = chunks.astype(np.float64)
    want = bh.T.astype(np.float64) @ x64 @ bw.astype(np.float64)
    # h terms, then w terms, every product and sum rounded once: (h + w) 2^-24 of the sum of magnitudes, doubled
    bound = (h + w + 2) * 2.0 ** -23 * (np.abs(bh.T) @ np.abs(x64) @ np.abs(bw))
    rows = lambda a: a.transpose(0, 2, 1, 3).reshape(Y * h, X * w)  # noqa: E731
    for in_chunked, out_chunked in ((False, True), (True, False), (True, True), (False, False)):
        src = torch.from_numpy(np.ascontiguousarray(chunks) if in_chunked else x).to(dev)
        got = tc.ChunkingTransformer._dense(src, Y * h, X * w, h, w, torch.from_numpy(bh).to(dev),
                                            torch.from_numpy(bw).to(dev), in_chunked, out_chunked).cpu().numpy()
        ref, tol = (want, bound) if out_chunked else (rows(want), rows(bound))
        assert (np.abs(got - ref) <= tol).all(), (in_chunked, out_chunked)


@pytest.mark.parametrize("h,w", [(2, 1), (7, 3), (17, 18), (60, 50), (63, 63), (64, 49), (1, 50)])
def test_dense_contraction_with_an_infinite_matrix(dev, h, w):
    # an infinity in either matrix reaches the results that depend on it, and no padding of the tiles turns it into NaN
    rng = np.random.default_rng(h + w)
    x, b, d = (rng.random(s).astype(np.float32) + 0.5 for s in ((3, 2, h, w), (h, h), (w, w)))
    b[h // 2, h - 1] = np.inf
    d2 = d.copy()
    d2[w - 1, 0] = -np.inf
    tr = tc.ChunkingTransformer(torch.nn.Linear(1, 1, bias=False), 64)
    for second in (d, d2):
        with np.errstate(invalid="ignore"):
            want = b.T.astype(np.float64) @ x.astype(np.float64) @ second
        got = tr.einsum_2d(*(torch.from_numpy(a).to(dev) for a in (x, b, second))).cpu().numpy()
        assert np.array_equal(np.isnan(got), np.isnan(want))
        assert np.allclose(got, want, rtol=1e-4, equal_nan=True)


def _rows(kind, n_rows, n, rng):
    if kind == "normal":
        return rng.standard_normal((n_rows, n)).astype(np.float32)
    if kind == "levels":  # ties everywhere, zeros and both signs among them
        return rng.integers(-3, 4, (n_rows, n)).astype(np.float32)
    x = np.where(rng.random((n_rows, n)) < 0.01, rng.standard_normal((n_rows, n)), 0.0).astype(np.float32)
    x[0] = 0.0  # fewer non-zero values than are selected: zeros of the row itself have to follow, lowest index first
    x[-1, -1] = np.nan
    return x


@pytest.mark.parametrize("kind", ["normal", "levels", "sparse"])
@pytest.mark.parametrize("n,k", [(2, 2), (37, 6), (63, 62), (64, 32), (64, 64), (65, 64), (100, 10), (127, 126), (128, 128),
                                 (129, 32), (129, 128), (400, 32), (1000, 64), (2500, 32), (3000, 128), (4032, 2), (4033, 32),
                                 (4095, 64), (4096, 32)])
def test_rows_select_at_every_length(dev, n, k, kind):
    rows = _rows(kind, 7, n, np.random.default_rng(n * 131 + k))
    idx12, val = tc._topk_rows(torch.from_numpy(rows).to(dev), k)
    want_i, want_v = orc.topk_rows(rows, k)
    assert np.array_equal(idx12.cpu().numpy(), orc.pack12(want_i))
    assert np.array_equal(val.cpu().numpy().view(np.uint32), np.asarray(want_v, np.float32).view(np.uint32))


@pytest.mark.parametrize("repeats", [False, True])
@pytest.mark.parametrize("n,k", [(2, 2), (37, 6), (64, 64), (1001, 32), (3000, 32), (4093, 64), (4096, 2)])
def test_scatter_into_rows(dev, n, k, repeats):
    rng = np.random.default_rng(n + k)
    n_rows = 6
    idx = np.stack([rng.permutation(n)[:k] for _ in range(n_rows)]).astype(np.int64)
    if repeats:
        idx[1] = idx[1, 0]  # one element named by every entry
        idx[4, k // 2:] = idx[4, :k - k // 2]
    val = rng.standard_normal((n_rows, k)).astype(np.float32)
    got = tc._scatter_rows(torch.from_numpy(orc.pack12(idx)).to(dev), torch.from_numpy(val).to(dev), n_rows, k, n)
    # entries of one element added in entry order, divided by their number
    want = np.zeros((n_rows, n), np.float32)
    count = np.zeros((n_rows, n), np.float32)
    for r in range(n_rows):
        for j in range(k):
            want[r, idx[r, j]] += val[r, j]
            count[r, idx[r, j]] += 1
    want = np.where(count > 1, want / np.maximum(count, 1), want)
    assert np.array_equal(got.cpu().numpy(), want)


def test_scatter_into_more_rows_than_one_launch_takes(dev):
    # a workgroup of 256 threads per row: 2^24 rows are 2^32 threads
    n = (1 << 24) + 21
    val = torch.arange(2.0 * n, device=dev).view(n, 2)  # (exact: below 2^26, rounded alike on both sides)
    idx = torch.from_numpy(orc.pack12(np.array([[3, 1]]))).to(dev).repeat(n)
    want = torch.zeros(n, 5, device=dev)
    want[:, 3], want[:, 1] = val[:, 0], val[:, 1]
    assert torch.equal(tc.TopKCompressor().decompress(val, idx, val, (n, 5), 5), want)
    assert torch.equal(tc._scatter_rows(idx, val, n, 2, 5), want)
    idx.view(-1, 3)[-1] = torch.from_numpy(orc.pack12(np.array([[3, 7]]))).to(dev)
    for call in (lambda: tc._scatter_rows(idx, val, n, 2, 5), lambda: tc.TopKCompressor().decompress(val, idx, val, (n, 5), 5)):
        with pytest.raises(RuntimeError, match="index 7 is out of bounds"):
            call()


@pytest.mark.parametrize("use_dct", [True, False])
def test_rows_of_a_set_of_more_groups_than_one_launch_takes(dev, use_dct):
    # four workgroups of 256 threads per 64 rows: 2^22 groups are 2^32 threads; the same tensor over and over
    rows, times = 1 << 16, (1 << 12) + 1
    x = torch.randn(rows * 64, generator=torch.Generator(device=dev).manual_seed(5), device=dev)
    want_i, want_v = tc.encode_compress_rows_batch(tc.RowBatch([x]), 2, use_dct=use_dct)
    table = torch.tensor([[x.data_ptr(), 64, t * rows, rows | (1 << 32)] for t in range(times)], dtype=torch.int64, device=dev)
    idx = torch.zeros(times, rows * 3, dtype=torch.uint8, device=dev)
    val = torch.zeros(times, rows, 2, device=dev)
    _lib.check(_lib.load().tplr_encode_rows_batch(table.data_ptr(), times, times * (rows // 64), 2, int(use_dct), idx.data_ptr(),
                                                  val.data_ptr(), torch.cuda.current_stream(dev).cuda_stream), "tplr_encode_rows_batch")
    assert bool((idx == want_i).all()) and bool((val == want_v).all())


@pytest.mark.parametrize("use_dct", [True, False])
@pytest.mark.parametrize("groups", [8, 16, 17, 255, 256, 257, 383, 384, 1023, 1024])
def test_rows_of_a_set_alike_in_both_forms(dev, groups, use_dct):
    # the launch changes form with the set's groups of 64 rows and with k, at k = 64 never: its leading entries are the others'
    rows = [1, 63, 65, 64 * 70 + 1, 3] if groups > 80 else [1, 63, 65, 30, 3]
    rows.append(64 * (groups - sum((r + 63) // 64 for r in rows)) - 5)
    rng = np.random.default_rng(groups)
    many = [rng.standard_normal(r * 64).astype(np.float32) for r in rows]
    many[3][:640] = 0.0
    many[3][640:1280] = rng.integers(-2, 3, 640)  # ties
    many[4][70] = np.nan
    if not use_dct:
        many[4][[3, 90]] = np.inf, -np.inf
    batch = tc.RowBatch([torch.from_numpy(m).to(dev) for m in many])
    assert batch.total_groups == groups
    idx64, val64 = tc.encode_compress_rows_batch(batch, 64, use_dct=use_dct)
    for k in (2, 24, 26, 32, 34, 48, 50):
        idx, val = tc.encode_compress_rows_batch(batch, k, use_dct=use_dct)
        assert torch.equal(idx.view(-1, 3 * k // 2), idx64.view(-1, 96)[:, :3 * k // 2])
        want = val64[:, :k]
        assert bool(((val.view(torch.int32) == want.contiguous().view(torch.int32)) | (val.isnan() & want.isnan())).all())


@pytest.mark.parametrize("inverse", [0, 1])
@pytest.mark.parametrize("n_vec", [1, 3, 4, 5, 32, 63, 16384, 16385])
def test_vectors_transform_alike_in_both_forms(dev, n_vec, inverse):
    # the launch changes form past 16384 vectors; every vector's bits are the same in either
    x = torch.from_numpy(np.random.default_rng(n_vec).standard_normal((n_vec, 64)).astype(np.float32)).to(dev)
    lib = _lib.load()

    def run(a):
        out = torch.full_like(a, float("nan"))
        assert lib.tplr_dct1d(a.data_ptr(), a.shape[0], inverse, out.data_ptr(), None) == 0
        torch.cuda.synchronize()
        return out

    many = torch.zeros((16384 + 64 + n_vec, 64), device=dev)
    many[:n_vec] = x
    assert torch.equal(run(x), run(many)[:n_vec])


@pytest.mark.parametrize("bins", [2, 4, 5, 8, 9, 256])
@pytest.mark.parametrize("n", [4, 8, 1020, 1028, 65540, 270336])
def test_quantiser_at_slice_and_bin_edges(dev, n, bins):
    # the first value far out (values arrive in descending magnitude): the moments are taken about it
    rng = np.random.default_rng(n + bins)
    v = (rng.standard_t(3, n) * 1e-3 + 2e-4).astype(np.float32)
    v[0] = 0.05
    comp = tc.TopKCompressor(use_quantization=True, quantization_bins=bins, quantization_range=6)
    q, (shift, scale, half, lut, _) = comp._quantize_values(torch.from_numpy(v).to(dev))
    x = v.astype(np.float64)
    # both figures are sums in double rounded once to fp32 (and a product and a quotient in fp32 for the scale)
    assert abs(float(shift) - x.mean()) <= 2.0 ** -23 * abs(x.mean()) + 1e-12 * abs(x).max()
    assert abs(scale / (6 * np.sqrt(((x - float(shift)) ** 2).sum() / (n - 1)) / bins) - 1) <= 2.0 ** -21
    # with the device's own shift and scale every code and table entry is determined
    c = v - np.float32(shift.item())
    want = np.clip(np.rint(c / np.float32(scale) + np.float32(half)), 0, bins - 1).astype(np.uint8)
    assert np.array_equal(q.cpu().numpy(), want)
    for b in range(bins):
        mine = c[want == b].astype(np.float64)
        mean = mine.mean() if mine.size else 0.0
        assert abs(float(lut[b]) - mean) <= 2.0 ** -23 * abs(mean) + 1e-12
    const = torch.full((n,), 0.125, device=dev)
    q, (shift, scale, _, _, _) = comp._quantize_values(const)
    assert float(shift) == 0.125 and scale == 1.0 and (q == bins // 2).all()


def test_per_parameter_calls_agree_for_plain_and_converted_inputs(dev):
    # plain tensors take the native host path, everything else is converted first: the same bits either way
    from types import SimpleNamespace

    params = [SimpleNamespace(requires_grad=True, shape=s, dtype=torch.float32, device=dev) for s in [(128, 192), (100, 60), (640,)]]
    tr = tc.ChunkingTransformer(SimpleNamespace(named_parameters=lambda: ((str(i), p) for i, p in enumerate(params))), 64)
    comp = tc.TopKCompressor(use_quantization=True, quantization_bins=4)
    g = torch.Generator(device=dev).manual_seed(3)
    for p in params:
        x = torch.randn(p.shape, generator=g, device=dev)
        wide = torch.randn(tuple(p.shape[:-1]) + (2 * p.shape[-1],), generator=g, device=dev)
        wide[..., ::2] = x
        results = []
        for other in (x, torch.nn.Parameter(x.clone()), wide[..., ::2]):
            enc = tr.encode(other, use_dct=True)
            idx, q, xshape, totalk, qp = comp.compress(enc, 32)
            dense = comp.decompress(x, idx, q, xshape, totalk, qp)
            dec = tr.decode(dense, use_dct=True)
            assert not dec.requires_grad and not enc.requires_grad
            slow = tr.decode(comp.decompress(x, idx.reshape(1, -1), q, list(xshape), totalk, list(qp)), use_dct=True)
            assert torch.equal(dec, slow)
            results.append((idx, q, qp[0], torch.tensor(qp[1]), qp[3], dec))
        for r in results[1:]:
            assert all(torch.equal(a.reshape(-1), b.reshape(-1)) for a, b in zip(results[0], r))


# (a process of its own: the limits bound what the allocator takes from the device, and the free rests of segments that other
# tests keep partly in use would serve the requests whatever the limit)
OUT_OF_MEMORY = """
import torch
import templar_amd.compress as tc

dev = torch.device("cuda:0")
comp = tc.TopKCompressor(use_quantization=True, quantization_bins=4)
qp = (torch.tensor(0.5, device=dev), 1.0, 2, torch.arange(4.0, device=dev), torch.float32)
codes = [torch.zeros(1 << 25, dtype=torch.uint8, device=dev)] * 16  # 16 results of 128 MiB each
x = torch.zeros(1 << 19, 64, device=dev)  # 128 MiB of values, 32 MiB of codes and 48 MiB of indices
total = torch.cuda.get_device_properties(dev).total_memory
before = torch.cuda.memory_allocated(dev)


def refused(call, mib):
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    room = torch.cuda.memory_reserved(dev) + (mib << 20)
    assert room - before < (mib + 40) << 20  # (two pools, segments of 20 MiB at most for what is small)
    torch.cuda.set_per_process_memory_fraction(room / total, dev)
    try:
        call()
    except torch.OutOfMemoryError:
        pass
    else:
        raise SystemExit("was not refused")
    assert torch.cuda.memory_allocated(dev) == before


for _ in range(2):
    refused(lambda: comp.maybe_dequantize_values(codes, [qp] * 16, dev), 1024)
refused(lambda: comp.compress(x, 64), 180)
torch.cuda.set_per_process_memory_fraction(1.0, dev)
assert comp.maybe_dequantize_values(codes[:2], [qp] * 2, dev)[1].numel() == 1 << 25
print("nothing left")
"""


def test_running_out_of_memory_leaves_nothing_allocated():
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    run = subprocess.run([sys.executable, "-c", OUT_OF_MEMORY], cwd=root, capture_output=True, text=True, timeout=100)
    assert run.returncode == 0 and "nothing left" in run.stdout, run.stderr[-2000:] + run.stdout


def test_decompress_names_the_index_outside_its_row(dev):
    comp = tc.TopKCompressor()
    idx = np.array([[1, 2, 3, 9], [4, 5, 11, 0]], np.int64)
    val = torch.ones(2, 4, device=dev)
    with pytest.raises(RuntimeError, match="index 11 is out of bounds for dimension -1 with size 9"):
        comp.decompress(val, torch.from_numpy(orc.pack12(idx)).to(dev), val, (2, 9), 9)


@pytest.mark.parametrize("k", [2, 32, 64])
def test_scatter_of_rows_flags_an_index_outside_its_row(dev, k):
    # tplr_decompress_rows by itself: the flag is set where an index lies outside its row, that entry is dropped
    lib, stream = _lib.load(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rng, n, length = np.random.default_rng(k), 517, 100
    idx = np.stack([rng.permutation(length)[:k] for _ in range(n)])
    val = rng.standard_normal((n, k)).astype(np.float32)
    dv = torch.from_numpy(val).to(dev)
    for where in (None, (0, 0), (n - 1, k - 1), (200, k // 2)):
        sent, kept = idx.copy(), val.copy()
        if where:
            sent[where], kept[where] = length + 7, 0.0
        di, out = torch.from_numpy(orc.pack12(sent)).to(dev), torch.full((n, length), 7.0, device=dev)
        flag = torch.zeros(1, dtype=torch.int32, device=dev)
        assert lib.tplr_decompress_rows(di.data_ptr(), dv.data_ptr(), n, k, length, out.data_ptr(), flag.data_ptr(), stream) == 0
        assert bool(flag.item()) == (where is not None)
        want = np.zeros((n, length), np.float32)
        np.put_along_axis(want, idx, kept, 1)
        assert np.array_equal(out.cpu().numpy(), want)


def test_decompress_of_many_rows_waits_once_for_the_interpreter(dev):
    # 64 words tell whether the indices lie in their rows.  Beside a busy thread every release of the interpreter may cost a switch
    # interval; the call releases it once for all words, and the rest of it another time at most.
    comp, interval = tc.TopKCompressor(), sys.getswitchinterval()
    x = torch.randn(32768, 100, device=dev)
    sent = comp.compress(x, 64)
    comp.decompress(x, *sent)
    stop = threading.Event()

    def busy():
        while not stop.is_set():
            pass

    thread, took = threading.Thread(target=busy), []
    sys.setswitchinterval(0.01)
    thread.start()
    try:
        for _ in range(40):
            t = time.perf_counter()
            comp.decompress(x, *sent)
            took.append(time.perf_counter() - t)
    finally:
        stop.set()
        thread.join()
        sys.setswitchinterval(interval)
    assert sum(t > 0.025 for t in took) <= 1, took


@pytest.mark.parametrize("bins", [4, 256])
@pytest.mark.parametrize("n", [4, 70000])
@pytest.mark.parametrize("at,what", [(0, "inf"), (0, "-inf"), (0, "nan"), (3, "inf"), (-1, "-inf"), (-1, "nan")])
def test_quantiser_of_values_that_are_not_finite(dev, bins, n, at, what):
    # the reference's mean is the infinity (or NaN), and its scale, NaN, becomes one (:594-600); wherever it stands
    v = torch.randn(n, device=dev)
    v[at] = float(what)
    comp = tc.TopKCompressor(use_quantization=True, quantization_bins=bins)
    q, (shift, scale, half, lut, _) = comp._quantize_values(v)
    b = tc.TensorBatch([torch.empty(64, 64, device=dev) for _ in range(2)])
    pair = torch.randn(2, 4, device=dev)
    pair[1, at] = float(what)
    _, shifts, scales, _ = tc.quantize_batch(b, pair, 4, bins)
    for got, sc in ((shift, scale), (shifts[1], float(scales[1]))):
        assert float(got) == float(what) or (what == "nan" and bool(got.isnan()))
        assert sc == 1.0
    assert bool(torch.isfinite(shifts[0])) and float(scales[0]) != 1.0
    # a finite value lies infinitely far below an infinite mean, or above (codes of NaN are not defined)
    if what != "nan":
        finite = torch.isfinite(v)
        assert bool((q[finite] == (0 if what == "inf" else bins - 1)).all())


@pytest.mark.parametrize("bins", [0, -4])
@pytest.mark.parametrize("shape", [(2, 3, 64, 64), (4, 100), (3, 50), (64,)])
def test_quantiser_without_bins_is_refused(dev, bins, shape):
    comp = tc.TopKCompressor(use_quantization=True, quantization_bins=bins)
    x = torch.randn(shape, device=dev)
    for other in (x, x.to(torch.bfloat16)):
        with pytest.raises(RuntimeError, match=f"quantiser of {bins} bins"):
            comp.compress(other, 10)
    with pytest.raises(RuntimeError):
        comp._quantize_values(x)


@pytest.mark.parametrize("bins", [4, 256])
def test_quantiser_queued_behind_other_work(dev, bins):
    # the host watches for the scale for half a millisecond, and then waits for the stream
    comp = tc.TopKCompressor(use_quantization=True, quantization_bins=bins)
    v = torch.randn(262144, device=dev)
    codes, (shift, scale, _, lookup, _) = comp._quantize_values(v)
    a = torch.randn(4096, 4096, device=dev)
    torch.mm(a, a)
    torch.cuda.synchronize()
    for _ in range(3):
        events = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        events[0].record()
        for _ in range(8):
            torch.mm(a, a)
        events[1].record()
        late = comp._quantize_values(v)
        assert events[1].query() and events[0].elapsed_time(events[1]) > 2.0
        assert torch.equal(late[0], codes) and torch.equal(late[1][0], shift) and late[1][1] == scale
        assert torch.equal(late[1][3], lookup) if bins <= 8 else torch.allclose(late[1][3], lookup, rtol=2.0 ** -22, atol=1e-9)


def test_quantisers_of_two_threads_do_not_meet(dev):
    # each thread on a stream of its own: the scale travels through pinned memory of its own call
    import threading

    comp = tc.TopKCompressor(use_quantization=True, quantization_bins=4)
    vals = [torch.randn(64 * 1024, device=dev) * (1 + 9 * t) for t in range(2)]
    want = [comp._quantize_values(v)[1][1] for v in vals]
    torch.cuda.synchronize()
    wrong = []

    def work(t):
        with torch.cuda.stream(torch.cuda.Stream(dev)):
            for _ in range(200):
                if comp._quantize_values(vals[t])[1][1] != want[t]:
                    wrong.append(t)

    threads = [threading.Thread(target=work, args=(t,)) for t in range(2)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not wrong


@pytest.mark.parametrize("Y,X", [(1, 1), (1, 3), (3, 1), (2, 5)])
def test_decode_of_row_major_and_chunked_coefficients(dev, Y, X):
    tr = tc.ChunkingTransformer(torch.nn.Linear(64 * X, 64 * Y, bias=False, device=dev), 64)
    flat = torch.from_numpy(np.random.default_rng(Y * 7 + X).standard_normal((64 * Y, 64 * X + 64)).astype(np.float32)).to(dev)
    for rows in (flat[:, :64 * X].contiguous(), flat[:, :64 * X]):  # without and with a gap between the rows
        view = rows.reshape(Y, 64, X, 64).permute(0, 2, 1, 3) if rows.is_contiguous() else \
            torch.as_strided(rows, (Y, X, 64, 64), (64 * rows.stride(0), 64, rows.stride(0), 1))
        for use_dct in (True, False):
            assert torch.equal(tr.decode(view, use_dct=use_dct), tr.decode(view.contiguous(), use_dct=use_dct))


@pytest.mark.parametrize("Y,X", [(1, 1), (1, 3), (3, 1), (2, 5), (40, 64)])
@pytest.mark.parametrize("k,P", [(4, 1), (32, 3), (64, 15), (66, 2), (32, 25)])
def test_dense_results_are_contiguous_on_every_route(dev, Y, X, k, P):
    """Plain payloads, from codes, converted ones: contiguous chunks, and decode without the transform of them a copy."""
    rng, n = np.random.default_rng(Y * 100 + X + k), Y * X
    idx = torch.from_numpy(orc.pack12(np.stack([rng.permutation(4096)[:k] for _ in range(n)]).astype(np.int64))).to(dev)
    vals = [torch.from_numpy(rng.standard_normal((Y, X, k)).astype(np.float32)).to(dev) for _ in range(P)]
    shape, p = torch.Size((Y, X, 64, 64)), torch.empty(Y * 64, X * 64, device=dev)
    tr = tc.ChunkingTransformer(torch.nn.Linear(64 * X, 64 * Y, bias=False, device=dev), 64)
    plain, coder = tc.TopKCompressor(), tc.TopKCompressor(use_quantization=True, quantization_bins=4)
    codes, qp = coder._quantize_values(vals[0])
    norms = torch.rand(P, device=dev) + 0.5
    groups = [[plain.decompress(p, idx, vals[0], shape, 4096), plain.decompress(p, idx, vals[0], list(shape), 4096)],
              [coder.decompress(p, idx, codes, shape, 4096, qp), coder.decompress(p, idx, codes, shape, 4096, list(qp))]]
    for kw in (dict(clip_norm=False), dict(block_norms=norms), dict()):
        groups.append([plain.batch_decompress(p, [idx] * P, vals, shape, 4096, **kw),
                       plain.batch_decompress(p, tuple([idx] * P), tuple(vals), list(shape), 4096, **kw)])
    for same in groups:
        for dense in same:
            assert dense.shape == shape and dense.is_contiguous() and dense.view(-1).numel() == n * 4096
            assert torch.equal(dense, same[0])
            before, grad = dense.clone(), tr.decode(dense, use_dct=False)
            assert torch.equal(grad, before.permute(0, 2, 1, 3).reshape(Y * 64, X * 64))
            if X > 1:  # (a single column of chunks lies as the tensor does: the reference's rearrange is a view there too)
                grad.mul_(0.5).add_(1.0)
                assert torch.equal(dense, before)


def test_parameter_of_more_columns_than_a_row_stride_holds(dev):
    """Chunked results have no row stride, and so none of its limit of 2^23 floats."""
    X = (1 << 17) + 2
    shape, p = (1, X, 64, 64), torch.empty(1, device=dev)
    idx = torch.from_numpy(orc.pack12(np.array([[5, 4094]]))).to(dev).repeat(X)
    val = torch.arange(1.0, 2 * X + 1, device=dev).view(1, X, 2)
    plain, coder = tc.TopKCompressor(), tc.TopKCompressor(use_quantization=True, quantization_bins=4)
    codes, qp = torch.tensor([1, 3], dtype=torch.uint8, device=dev).expand(1, X, 2).contiguous(), \
        (torch.tensor(0.5, device=dev), 1.0, 2, torch.arange(4.0, device=dev), torch.float32)
    for call, want in ((lambda: plain.decompress(p, idx, val, shape, 4096), val),
                       (lambda: plain.batch_decompress(p, [idx] * 2, [val] * 2, shape, 4096, clip_norm=False), val),
                       (lambda: coder.decompress(p, idx, codes, shape, 4096, qp), torch.tensor([1.5, 3.5], device=dev))):
        flat = call().view(X, 4096)
        assert bool((flat[:, [5, 4094]] == want).all()) and int(torch.count_nonzero(flat)) == 2 * X


def _payloads(dev, P, n, k, rng, repeats=False):
    idx, val = [], []
    for _ in range(P):
        i = np.stack([rng.permutation(4096)[:k] for _ in range(n)]).astype(np.int64)
        i[:, : k // 2] = np.arange(k // 2) * 61 % 4096  # shared by all peers (61 is odd: distinct)
        if repeats:
            i[n - 1, : max(2, k // 4)] = 4095
        else:
            for r in range(n):  # the other half distinct from it
                rest = np.setdiff1d(rng.permutation(4096)[: 2 * k], i[r, : k // 2])
                i[r, k // 2:] = rng.permutation(rest)[: k - k // 2]
        idx.append(torch.from_numpy(orc.pack12(i)).to(dev))
        val.append(torch.from_numpy(rng.standard_normal((n, k)).astype(np.float32)).to(dev))
    return idx, val


@pytest.mark.parametrize("repeats", [False, True])
@pytest.mark.parametrize("P,k,Y,X", [(1, 2, 1, 1), (1, 64, 3, 5), (4, 32, 1, 9), (5, 32, 3, 3), (8, 64, 1, 1), (9, 2, 2, 3), (15, 32, 3, 5),
                                     (16, 64, 2, 2), (17, 32, 1, 3), (24, 64, 3, 3), (25, 32, 2, 2), (3, 66, 2, 2)])
def test_param_aggregate_is_the_two_launches(dev, P, k, Y, X, repeats):
    """tplr_aggregate_param leaves the bits of tplr_clip_scales and tplr_decode_aggregate, in either layout."""
    lib, rng, n = _lib.load(), np.random.default_rng(P * 100 + k), Y * X
    idx, val = _payloads(dev, P, n, k, rng, repeats)
    ptrs = lambda ts: (ctypes.c_void_p * P)(*[t.data_ptr() for t in ts])  # noqa: E731
    ip, vp = ptrs(idx), ptrs(val)
    stream = torch.cuda.current_stream(dev).cuda_stream
    norms = rng.gamma(2.0, 1.0, P + 3).astype(np.float32)
    cases = {"plain": norms[:P], "more": norms, "ties": np.round(norms[:P]) + 1.0, "nan": np.where(np.arange(P) == P // 2, np.nan, norms[:P]),
             "inf": np.where(np.arange(P) == 0, np.inf, norms[:P]), "zero": np.zeros(P), "negative": norms[:P] - 2.0, "factors": None,
             "none": None}
    for name, given in cases.items():
        for ld in (X * 64, 0):
            scale = torch.from_numpy(norms[:P].copy()).to(dev) if name != "none" else None
            got, want = torch.full((2, n * 4096), 7.0, device=dev)
            gn, m = None, 0
            if given is not None:
                gn = torch.from_numpy(np.asarray(given, np.float32)).to(dev)
                m = gn.numel()
                scale = torch.empty(m, device=dev)
            sp = scale.data_ptr() if scale is not None else None
            _lib.check(lib.tplr_aggregate_param(ip, vp, gn.data_ptr() if m else None, m, sp, P, k, Y * 64, X * 64, got.data_ptr(), ld,
                                                stream), "tplr_aggregate_param")
            if m:
                _lib.check(lib.tplr_clip_scales(gn.data_ptr(), m, 0, sp, None, stream), "tplr_clip_scales")
            _lib.check(lib.tplr_decode_aggregate(ip, vp, sp, P, k, Y * 64, X * 64, 0, 0, 0, want.data_ptr(), ld, None, stream),
                       "tplr_decode_aggregate")
            same = (got.view(torch.int32) == want.view(torch.int32)) | (got.isnan() & want.isnan())
            assert bool(same.all()), (name, ld)


@pytest.mark.parametrize("bins,k,Y,X", [(1, 2, 1, 1), (4, 64, 3, 5), (8, 32, 1, 9), (255, 62, 2, 3), (256, 64, 5, 1)])
def test_decompress_from_codes_is_the_two_launches(dev, bins, k, Y, X):
    lib, rng, n = _lib.load(), np.random.default_rng(bins + k), Y * X
    (idx,), _ = _payloads(dev, 1, n, k, rng)
    codes = torch.from_numpy(rng.integers(0, 256, (n, k)).astype(np.uint8)).to(dev)  # codes past the table among them
    lookup, shift = torch.randn(bins, device=dev), torch.randn((), device=dev)
    stream = torch.cuda.current_stream(dev).cuda_stream
    one = lambda t: (ctypes.c_void_p * 1)(t.data_ptr())  # noqa: E731
    val = lookup[codes.long().clamp(max=bins - 1)] + shift
    for ld in (X * 64, 0):
        got, want = torch.full((2, n * 4096), 7.0, device=dev)
        _lib.check(lib.tplr_decompress_codes(idx.data_ptr(), codes.data_ptr(), lookup.data_ptr(), shift.data_ptr(), bins, k, Y * 64,
                                             X * 64, got.data_ptr(), ld, stream), "tplr_decompress_codes")
        _lib.check(lib.tplr_decode_aggregate(one(idx), one(val), None, 1, k, Y * 64, X * 64, 0, 0, 0, want.data_ptr(), ld, None,
                                             stream), "tplr_decode_aggregate")
        assert torch.equal(got.view(torch.int32), want.view(torch.int32)), ld


@pytest.mark.parametrize("n,bins,slices", [(4, 4, 1), (1020, 1, 1), (2052, 8, 2), (65536, 4, 64), (262144, 4, 256), (70000, 256, 68)])
def test_quantiser_of_one_tensor_is_the_batch_of_one(dev, n, bins, slices):
    """The table made by the workgroup that finishes last, or past eight bins by a launch: the bits of the batch's launches."""
    lib = _lib.load()
    stream = torch.cuda.current_stream(dev).cuda_stream
    v = torch.from_numpy(np.random.default_rng(n).standard_t(3, n).astype(np.float32)).to(dev)
    desc = torch.tensor([0, 0, 0, (n // 4) | (1 << 32)], dtype=torch.int64, device=dev)  # rows of four values: n / 4 x 1 of them
    size = slices * (2 + 2 * bins)
    outs = []
    for one in (True, False) * 3:
        work = torch.full((size + 1,), -1.0, dtype=torch.float64, device=dev)
        codes, out = torch.empty(n, dtype=torch.uint8, device=dev), torch.empty(2 + bins, device=dev)
        ptr = [t.data_ptr() for t in (codes, out, out[1:], out[2:])]
        if one:
            _lib.check(lib.tplr_quantize(v.data_ptr(), n, bins, 6.0, slices, work.data_ptr(), *ptr, stream), "tplr_quantize")
        else:
            _lib.check(lib.tplr_quantize_batch(v.data_ptr(), 4, desc.data_ptr(), 1, bins, 6.0, slices, work.data_ptr(), *ptr, stream),
                       "tplr_quantize_batch")
        outs.append((codes, out))
    for codes, out in outs[1:]:
        assert torch.equal(codes, outs[0][0])
        # the sums in LDS of more than eight bins are added in no fixed order: sums in double, one rounding to fp32
        assert torch.equal(out, outs[0][1]) if bins <= 8 else torch.allclose(out, outs[0][1], rtol=2.0 ** -22, atol=1e-9)


@pytest.mark.parametrize("repeats", [False, True])
@pytest.mark.parametrize("P,k", [(6, 64), (13, 32), (24, 64)])
def test_large_param_aggregate_is_the_two_launches(dev, P, k, repeats):
    """The same where the parameter is large for a chunk per workgroup: the persistent launch makes the factors itself."""
    Y, X = 64, 130
    assert Y * X * P > 24576
    lib, n = _lib.load(), Y * X
    idx, val = _payloads(dev, P, 65, k, np.random.default_rng(P), repeats)
    idx = [i.reshape(65, -1).repeat(n // 65, 1).reshape(-1) for i in idx]  # the rows over and over
    val = [v.repeat(n // 65, 1) for v in val]
    ptrs = lambda ts: (ctypes.c_void_p * P)(*[t.data_ptr() for t in ts])  # noqa: E731
    ip, vp = ptrs(idx), ptrs(val)
    stream = torch.cuda.current_stream(dev).cuda_stream
    norms = torch.rand(P + 2, device=dev) + 0.1
    for m, ld in ((P, X * 64), (P + 2, X * 64), (P, 0), (P + 2, 0)):
        scale, (got, want) = torch.empty(m, device=dev), torch.full((2, n * 4096), 7.0, device=dev)
        _lib.check(lib.tplr_aggregate_param(ip, vp, norms.data_ptr(), m, scale.data_ptr(), P, k, Y * 64, X * 64, got.data_ptr(), ld,
                                            stream), "tplr_aggregate_param")
        _lib.check(lib.tplr_clip_scales(norms.data_ptr(), m, 0, scale.data_ptr(), None, stream), "tplr_clip_scales")
        _lib.check(lib.tplr_decode_aggregate(ip, vp, scale.data_ptr(), P, k, Y * 64, X * 64, 0, 0, 0, want.data_ptr(), ld, None,
                                             stream), "tplr_decode_aggregate")
        assert torch.equal(got.view(torch.int32), want.view(torch.int32)), (m, ld)
