"""Tables that travel as launch arguments: AdamW buckets of up to and past one launch's 80 tensors,
stand-alone Newton-Schulz of more matrices than one table launch holds."""
import ctypes

import numpy as np
import pytest
import torch

import dmuon_amd as dmuon
from dmuon_amd import _C
from oracle import adamw_oracle as ao


def test_entry_points_refuse_bad_tables():
    lib, scal = _C.lib(), (1, 0.99, 0.9, 0.1, 0.999, 0.001, 0.5, 1e-8, -1e-3, None)
    row = (ctypes.c_int64 * 6)(4096, 4096, 4096, 0, 0, 8)
    assert lib.dmuon_adamw_tensors(row, 1, 0, 0, 0, *scal) != 0 and b"NULL" in lib.dmuon_last_error()
    row[3], row[5] = 4096, -1
    assert lib.dmuon_adamw_tensors(row, 1, 0, 0, 0, *scal) != 0 and b"size" in lib.dmuon_last_error()
    row[5] = 8
    assert lib.dmuon_adamw_tensors(row, 1, 9, 0, 0, *scal) != 0 and b"dtype" in lib.dmuon_last_error()
    assert lib.dmuon_adamw_tensors(None, 1, 0, 0, 0, *scal) != 0
    assert lib.dmuon_adamw_tensors(None, 0, 0, 0, 0, *scal) == 0
    g = (ctypes.c_void_p * 2)(4096, None)
    coeff = (ctypes.c_float * 3)(1, 0, 0)
    ws = ctypes.create_string_buffer(4096)
    addr = (ctypes.addressof(ws) + 255) // 256 * 256
    call = lib.dmuon_newton_schulz_matrices
    assert call(g, 0, g, 0, 64, 64, 2, coeff, 1, 0, None, 0, 1e-7, addr, 512, 0, None) != 0
    assert b"NULL" in lib.dmuon_last_error()
    assert call(g, 0, g, 0, 64, 64, 1, coeff, 1, 0, None, 0, 1e-7, addr, 16, 0, None) != 0
    assert b"workspace" in lib.dmuon_last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("n,most", [(1, 1), (3, 5000), (80, 70), (81, 3000), (161, 2049), (12, 300000)])
@pytest.mark.parametrize("publish", [False, True])
def test_adamw_bucket_sizes_bit_exact(gpu, n, most, publish):
    rng = np.random.default_rng(n)
    sizes = [int(s) for s in rng.integers(1, most + 1, n)]
    ps, gs, ms, vs = ([torch.from_numpy(f(rng, s)).to(gpu) for s in sizes] for f in (
        lambda r, s: (r.standard_normal(s) * 0.02).astype(np.float32),
        lambda r, s: (r.standard_normal(s) * 0.02).astype(np.float32),
        lambda r, s: (r.standard_normal(s) * 0.005).astype(np.float32),
        lambda r, s: (r.standard_normal(s) ** 2 * 4e-4).astype(np.float32)))
    kw = dict(step=7, lr=1e-3, betas=(0.9, 0.999), weight_decay=0.01, eps=1e-8)
    want = [ao.adamw_step(*(t.cpu().numpy() for t in row), kw["step"], kw["lr"], betas=kw["betas"],
                          wd=kw["weight_decay"], eps=kw["eps"]) for row in zip(ps, gs, ms, vs)]
    qs = [torch.empty(s, dtype=torch.bfloat16, device=gpu) if i % 3 else None
          for i, s in enumerate(sizes)] if publish else None
    dmuon.fused_adamw_(ps, gs, ms, vs, publish=qs, **kw)
    torch.cuda.synchronize()
    for i, (p, m, v) in enumerate(want):
        for got, exp in ((ps[i], p), (ms[i], m), (vs[i], v)):
            assert np.array_equal(got.cpu().numpy(), np.asarray(exp, dtype=np.float32)), i
        if publish and qs[i] is not None:
            assert torch.equal(qs[i], ps[i].to(torch.bfloat16))


@pytest.mark.gpu
@pytest.mark.parametrize("L", [1, 240, 241])
def test_newton_schulz_of_many_matrices(gpu, L):
    gen = torch.Generator().manual_seed(L)
    Gs = [torch.randn(24, 40, generator=gen).to(gpu) for _ in range(L)]
    outs = dmuon.newton_schulz_batched(Gs, dmuon.KELLER_COEFFICIENTS, tile=128)
    one = dmuon.newton_schulz_batched([Gs[-1]], dmuon.KELLER_COEFFICIENTS, tile=128)[0]
    assert torch.equal(outs[-1], one)
    assert all(torch.isfinite(u).all() for u in outs)
