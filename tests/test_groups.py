"""Several oriented shapes in one call (``dmuon_muon_stage_groups`` / ``_apply_groups``): every
product is one launch over all of the groups, and each matrix gets the bits of its own call."""
import ctypes

import pytest
import torch

from dmuon_amd import _C
from dmuon_amd.optim.newton_schulz import (KELLER_COEFFICIENTS, POLAR_EXPRESS_COEFFICIENTS,
                                           _coeff_array)

LR, MU, WD, EPS = 0.02, 0.95, 0.1, 1e-7


def _descs(sizes):
    out = (_C.MuonGroup * len(sizes))()
    for d, (rows, cols, batch, n_t) in zip(out, sizes):
        d.rows, d.cols, d.batch, d.n_transposed = rows, cols, batch, n_t
    return out


@pytest.mark.parametrize("backend", [_C.NS_DIRECT, _C.NS_GRAM])
def test_plan_of_one_group_is_the_single_plan_and_of_several_their_sum(backend):
    sizes = [(1000, 300, 1), (512, 2048, 12), (4096, 4096, 2), (130, 250, 3)]
    for rows, cols, L in sizes:
        tile, ws, us = _C.plan_groups([(rows, cols, L)], backend=backend)
        assert (tile, ws) == (lambda p: (p[0], p[3]))(_C.plan(rows, cols, L, 0, 0, backend))
        assert us > 0
    for tile in (128, 256):
        got = _C.plan_groups(sizes, tile, backend=backend)
        assert got[:2] == (tile, sum(_C.plan(r, c, L, tile, 0, backend)[3] for r, c, L in sizes))
    assert _C.plan_groups(sizes, backend=backend)[0] in (128, 256)


def test_small_shapes_are_worth_joining_and_a_long_one_beside_a_large_one_is_not():
    def joined(a, b):
        return (_C.plan_groups([a, b], backend=_C.NS_GRAM)[2]
                < sum(_C.plan_groups([s], backend=_C.NS_GRAM)[2] for s in (a, b)))
    assert joined((1000, 300, 1), (333, 1025, 2))
    assert joined((4096, 4096, 8), (4096, 14336, 12))
    # the long X X^T (K = 16384) of one small m would run as a few 256-tiles
    assert not joined((16384, 512, 1), (4096, 4096, 1))


def test_refusals():
    fn = _C.lib().dmuon_muon_stage_groups
    ok = _descs([(64, 128, 1, 0)] * 9)
    ws = ctypes.create_string_buffer(64)
    for n, tile, word in ((0, 128, b"groups"), (9, 128, b"groups"), (2, 0, b"buf_ptrs")):
        assert fn(ok, n, MU, 1, _C.NS_GRAM, EPS, ws, 64, tile, None) != 0
        assert word in _C.lib().dmuon_last_error()
    for d in ok:
        d.buf_ptrs = d.g_ptrs = 4096       # never read: refused on the sizes
    assert fn(ok, 2, MU, 1, _C.NS_GRAM, EPS, ws, 64, 0, None) != 0      # a plan's tile is needed
    assert b"tile" in _C.lib().dmuon_last_error()
    with pytest.raises(RuntimeError):
        _C.plan_groups([(64, 64, 1)] * 9)


# (shapes: rows, cols, batch, transposed members), tile -> every kernel of a joined launch: 64-
# and 128-tiles (one and two blocks per CU), 256-tiles, 128-tiles promoted to 256; each staging
# kernel (flat, tall, padded) in one call; ragged sides and pitches
CASES = [
    ([(130, 250, 1, 0), (64, 64, 2, 0), (70, 33, 1, 1)], 128),
    ([(256, 768, 3, 1), (300, 1000, 2, 1), (512, 512, 2, 0)], 128),
    ([(512, 1024, 12, 4), (384, 640, 4, 4), (130, 250, 2, 1)], 128),
    ([(512, 1024, 24, 8), (1024, 1024, 8, 0), (256, 512, 8, 3)], 128),
    ([(256, 1024, 2, 1), (700, 500, 1, 0), (512, 768, 2, 1)], 256),
    # five groups: too many to spread a Q update over other launches, which their own calls do
    ([(256, 768, 3, 1), (300, 1000, 2, 1), (512, 512, 2, 0), (128, 128, 1, 0), (64, 640, 1, 0)], 128),
    ([(512, 2048, 12, 4), (1024, 1024, 3, 0), (384, 640, 4, 4), (130, 250, 2, 1), (64, 64, 1, 0)], 128),
    ([(512, 768, 2, 1), (256, 1024, 2, 1), (700, 500, 1, 0), (300, 300, 1, 0), (256, 256, 3, 0)], 256),
    # one matrix with more partial sums than the joined norm and staging launch takes
    ([(256, 768, 3, 1), (2048, 2112, 1, 0)], 128),
]


@pytest.mark.gpu
@pytest.mark.parametrize("backend", ["gram", "direct"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_joined_groups_give_the_bits_of_their_own_calls(gpu, case, backend):
    sizes, tile = CASES[case]
    code = _C.NS_GRAM if backend == "gram" else _C.NS_DIRECT
    coeff, T = _coeff_array(POLAR_EXPRESS_COEFFICIENTS if backend == "gram"
                            else KELLER_COEFFICIENTS)
    rst, n_rst = _C.restart_array([2] if backend == "gram" else [])
    gen = torch.Generator(device=gpu).manual_seed(case)
    stream = torch.cuda.current_stream().cuda_stream

    def normal(shape, dtype):
        return torch.empty(shape, device=gpu, dtype=dtype).normal_(0.0, 0.02, generator=gen)

    tables = []

    def ptrs(ts):
        tables.append(torch.tensor([t.data_ptr() for t in ts], dtype=torch.int64, device=gpu))
        return tables[-1].data_ptr()

    start = []
    for k, (rows, cols, L, n_t) in enumerate(sizes):
        shapes = [(rows, cols)] * (L - n_t) + [(cols, rows)] * n_t
        dtype = torch.float32 if k % 2 else torch.bfloat16
        start.append(dict(g=[normal(s, dtype) for s in shapes],
                          b=[normal(s, torch.float32) for s in shapes],
                          w=[normal(s, torch.float32) for s in shapes]))

    def run(joined):
        state = [dict(g=s["g"], b=[t.clone() for t in s["b"]], w=[t.clone() for t in s["w"]],
                      p=[torch.empty_like(t, dtype=torch.bfloat16) for t in s["w"]],
                      e=[torch.zeros(1, device=gpu) for _ in s["w"]]) for s in start]
        for call in ([range(len(sizes))] if joined else [[i] for i in range(len(sizes))]):
            descs = _descs([sizes[i] for i in call])
            for d, i in zip(descs, call):
                s = state[i]
                d.g_ptrs, d.buf_ptrs, d.est_ptrs = ptrs(s["g"]), ptrs(s["b"]), ptrs(s["e"])
                d.w_ptrs, d.pub_ptrs = ptrs(s["w"]), ptrs(s["p"])
                d.g_dtype = _C.DTYPE_F32 if i % 2 else _C.DTYPE_BF16
                d.w_dtype, d.pub_dtype = _C.DTYPE_F32, _C.DTYPE_BF16
            _, nbytes, _ = _C.plan_groups([s[:3] for s in (sizes[i] for i in call)], tile,
                                          backend=code)
            ws = torch.empty(nbytes, dtype=torch.uint8, device=gpu)
            for _ in range(2):      # the second step stages with the kept scale
                _C.call("dmuon_muon_stage_groups", descs, len(descs), MU, 1, code, EPS,
                        ws.data_ptr(), ws.numel(), tile, stream)
                _C.call("dmuon_muon_apply_groups", descs, len(descs), LR, WD, coeff, T, code,
                        rst, n_rst, ws.data_ptr(), ws.numel(), tile, stream)
            torch.cuda.synchronize()
        return state

    for one, many in zip(run(False), run(True)):
        for key in "bwpe":
            for a, b in zip(one[key], many[key]):
                assert torch.isfinite(a).all() and torch.equal(a, b), key
