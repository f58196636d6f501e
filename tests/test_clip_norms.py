"""``dmuon_clip_norms``: norms, coefficients and flags of a job table in two to four launches."""
import ctypes
import math
import time

import pytest
import torch

import dmuon_amd as dmuon
from dmuon_amd import _C, fast_clip
from dmuon_amd.fast_clip import GradClipBucket, clip_grad_norm_buckets_


def test_workspace_and_refusals():
    lib, need = _C.lib(), ctypes.c_int64()
    size = lambda *a: lib.dmuon_clip_workspace_size(*a, ctypes.byref(need))  # noqa: E731
    assert size(1, 262144, 1) == 0 and need.value == 8 + 4 * 32     # pieces of at least 8192
    assert size(10000, 262144, 3) == 0 and need.value == 24 + 4 * 10000
    assert size(0, 16, 2) == 0 and need.value == 16
    assert size(-1, 16, 2) != 0 and size(1, 0, 2) != 0
    q, ws = 4096, 1 << 20
    call = lambda **k: lib.dmuon_clip_norms(  # noqa: E731
        q, q, q, q, q, q, k.get("first", q), 1, 16, k.get("n", 1), 1, 1.0, q, k.get("coefs", q), q,
        q, k.get("ws", 8), k.get("bytes", ws), None)
    for bad in (dict(n=0), dict(first=None), dict(coefs=None), dict(ws=None), dict(ws=12),
                dict(bytes=4)):
        assert call(**bad) != 0, bad


def _grads(sizes, dtypes, gpu, seed):
    gen = torch.Generator(device=gpu).manual_seed(seed)
    return [torch.randn(n, device=gpu, generator=gen).to(dt) for n, dt in zip(sizes, dtypes)]


DT = [torch.float32, torch.bfloat16, torch.float16]
# empty and single-element tensors, sizes around a piece and a job, more tensors and segments than
# the finishing block has waves, jobs enough that a piece is a whole job
CASES = [([1], None), ([0, 5], None), ([8191, 8192, 8193, 262144, 262145], None),
         (list(range(1, 40)), None), ([3_000_000, 17, 70_001], None),
         ([4096 * 257], 256)]


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,chunk", CASES)
@pytest.mark.parametrize("max_norm", [None, 0.5, 1e6])
def test_segments_against_float64(gpu, sizes, chunk, max_norm):
    dts = [DT[i % 3] for i in range(len(sizes))]
    grads = _grads(sizes, dts, gpu, len(sizes))
    before = [g.double() for g in grads]
    buckets = tuple(GradClipBucket(str(i), [g], reduce=False) for i, g in enumerate(grads))
    first = [s.total_norm.clone() for s in
             clip_grad_norm_buckets_(buckets, None, chunk_size=chunk).bucket_stats]
    res = clip_grad_norm_buckets_(buckets, max_norm, chunk_size=chunk)
    total = 0.0
    for s, f, g, b in zip(res.bucket_stats, first, grads, before):
        norm = float(b.norm())
        total += norm * norm
        assert torch.equal(s.total_norm, f)                     # the same bits on every call
        assert float(s.total_norm) == pytest.approx(norm, rel=1e-6, abs=1e-30)
        coef = 1.0 if max_norm is None else min(1.0, max_norm / (norm + 1e-6))
        assert float(s.clip_coef) == pytest.approx(coef, rel=1e-6)
        assert bool(s.clipped) == (max_norm is not None and norm > max_norm)
        assert not bool(s.found_inf)
        want = b if max_norm is None else b.float() * s.clip_coef
        assert torch.equal(g, want.to(g.dtype))
    assert float(res.total_norm) == pytest.approx(math.sqrt(total), rel=1e-6, abs=1e-30)


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_one_norm_over_all_rounds_each_to_its_dtype(gpu, bad):
    sizes = [70_001, 33, 262_145, 8192] * 5
    grads = _grads(sizes, [DT[i % 3] for i in range(len(sizes))], gpu, 3)
    table = fast_clip._JobTable(grads, list(range(len(grads))), gpu, 262144)
    norms, coefs, clipped, found = table.norms(0, 1.0)
    want = math.sqrt(sum(float(g.double().norm().to(g.dtype)) ** 2 for g in grads))
    assert float(norms[0]) == pytest.approx(want, rel=1e-6)
    assert float(coefs[0]) == pytest.approx(1.0 / (want + 1e-6), rel=1e-6)
    assert bool(clipped[0]) and not bool(found[0])
    assert float(table.norms(0, None)[1][0]) == 1.0 and not bool(table.norms(0, None)[2][0])
    grads[3][5] = bad
    norms, coefs, clipped, found = table.norms(0, 1.0)
    assert not math.isfinite(float(norms[0])) and bool(found[0]) and not bool(clipped[0])
    want = 0.0 if bad == float("inf") else bad
    assert float(coefs[0]) == want or math.isnan(want) and math.isnan(float(coefs[0]))


@pytest.mark.gpu
def test_a_nan_limit_is_a_limit(gpu):
    """max_norm=nan gives NaN coefficients and gradients, as min(nan / norm, 1) does; only None is
    no limit."""
    nan = float("nan")
    for dt in DT:
        grads = _grads([33, 9000], [dt, dt], gpu, 5)
        norms = [float(g.double().norm()) for g in grads]
        buckets = tuple(GradClipBucket(str(i), [g], reduce=False) for i, g in enumerate(grads))
        res = clip_grad_norm_buckets_(buckets, nan)
        for s, g, n in zip(res.bucket_stats, grads, norms):
            assert math.isnan(float(s.clip_coef)) and not bool(s.clipped)
            assert float(s.total_norm) == pytest.approx(n, rel=1e-6) and not bool(s.found_inf)
            assert g.isnan().all()
        grads = _grads([33, 9000], [dt, dt], gpu, 6)
        model = torch.nn.Module()
        model.mats = torch.nn.ParameterList(
            [torch.nn.Parameter(torch.zeros(g.numel() // 3, 3, dtype=dt, device=gpu)) for g in grads])
        dmuon.dedicate_params(model, None, lambda name, p: True)
        dmuon.replicate(model)
        for p, g in zip(model.mats, grads):
            p.grad = g.view(p.shape)
        stats = dmuon.Muon(model).clip_grad_norm_(nan)
        assert math.isnan(float(stats.clip_coef)) and not bool(stats.clipped)
        assert all(g.isnan().all() for g in grads)


@pytest.mark.gpu
def test_a_cached_table_waits_for_its_upload_on_another_stream(gpu):
    """The device table is uploaded in the order of the stream that built it: a later call on
    another stream waits for that before its kernels read the table."""
    grads = _grads([33, 9000], [torch.float32, torch.bfloat16], gpu, 9)
    # no earlier work is left to wait for, and the first upload's own allocations exist
    fast_clip._job_table(grads[:1], [0], gpu, 4096)
    torch.cuda.synchronize()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(a):
        torch.cuda._sleep(200_000_000)                # about 0.1 s
        table = fast_clip._job_table(grads, [0, 1], gpu, 4096)
    with torch.cuda.stream(b):
        assert fast_clip._job_table(grads, [0, 1], gpu, 4096) is table
        assert table._stream() == b.cuda_stream        # what each of its kernels is launched on
        reached = torch.cuda.Event()
        reached.record()
    time.sleep(0.01)                                  # an event with nothing before it is done
    waits, asleep = not reached.query(), not a.query()
    torch.cuda.synchronize()
    assert asleep and waits
    with torch.cuda.stream(b):                         # now there is nothing to wait for
        norms = table.norms(2, None)[0]
    for n, g in zip(norms.tolist(), grads):
        assert n == pytest.approx(float(g.double().norm()), rel=1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_segments", [(256, 256), (257, 1), (257, 257), (2000, 3), (40, 700)])
def test_many_tensors_and_segments(gpu, n, n_segments):
    """On both sides of what one finishing block takes: norms, total, coefficients and flags, for
    segments (some of them empty) and for one norm over all tensors."""
    sizes = [1 + (7 * i) % 300 for i in range(n)]
    sizes[n // 2] = 40_000
    dts = [DT[i % 3] for i in range(n)]
    grads = _grads(sizes, dts, gpu, n)
    of = [(5 * i) % n_segments for i in range(n)]
    sq = [0.0] * n_segments
    for g, s in zip(grads, of):
        sq[s] += float(g.double().square().sum())
    table = fast_clip._JobTable(grads, of, gpu, 4096)
    norms, coefs, clipped, found = table.norms(n_segments, 6.0)
    want = torch.tensor(sq, dtype=torch.float64).sqrt()
    torch.testing.assert_close(norms[:-1].cpu().double(), want, rtol=1e-6, atol=1e-30)
    assert float(norms[-1]) == pytest.approx(float(want.norm()), rel=1e-6)
    torch.testing.assert_close(coefs.cpu().double(), (6.0 / (want + 1e-6)).clamp(max=1.0),
                               rtol=1e-6, atol=0.0)
    assert clipped.tolist() == (want > 6.0).tolist() and not found.any()
    one = table.norms(0, 6.0)
    total = math.sqrt(sum(float(g.double().norm().to(g.dtype)) ** 2 for g in grads))
    assert float(one[0][0]) == pytest.approx(total, rel=1e-6)
    assert float(one[1][0]) == pytest.approx(min(1.0, 6.0 / (total + 1e-6)), rel=1e-6)
    assert bool(one[2][0]) == (total > 6.0) and not bool(one[3][0])
    for a, b in zip((*table.norms(n_segments, 6.0), *table.norms(0, 6.0)),
                    (norms, coefs, clipped, found, *one)):
        assert torch.equal(a[:1], b[:1])               # the same bits on every call
    grads[n - 1][0] = float("nan")
    found = table.norms(n_segments, 6.0)[3]
    assert found.tolist() == [s == of[n - 1] for s in range(n_segments)]
    assert bool(table.norms(0, 6.0)[3][0])


@pytest.mark.gpu
def test_a_captured_call_reads_the_kept_table(gpu):
    """After one eager call a clip can be captured: the capture's own stream finds the kept table and
    waits for nothing outside the graph; every replay clips what the gradients then hold."""
    grads = _grads([70_001, 33, 9000], DT, gpu, 8)
    buckets = (GradClipBucket("a", grads[:2], reduce=False), GradClipBucket("b", grads[2:], reduce=False))
    values = [[g * (k + 1) for g in grads] for k in range(3)]
    want = []
    for v in values:
        for g, x in zip(grads, v):
            g.copy_(x)
        res = clip_grad_norm_buckets_(buckets, 3.0)
        want.append(([g.clone() for g in grads], res.total_norm.clone()))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        res = clip_grad_norm_buckets_(buckets, 3.0)
    for v, (after, total) in zip(values, want):
        for g, x in zip(grads, v):
            g.copy_(x)
        graph.replay()
        assert all(torch.equal(g, a) for g, a in zip(grads, after))
        assert torch.equal(res.total_norm, total)
        clip_grad_norm_buckets_(buckets, None)          # eager work between the replays
        torch.cuda.synchronize()
