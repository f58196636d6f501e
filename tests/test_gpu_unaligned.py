"""Rows of any pitch and bases of any element alignment: the step's staging, the final update and
the forward copy, and the SYRK seam's padded copies."""
import pytest
import torch

import dmuon_amd as dmuon
from dmuon_amd import _C
from dmuon_amd.optim.newton_schulz import _coeff_array
from dmuon_amd.optim.syrk_dispatch import syrk_or_cublas

LR, MU, WD = 0.02, 0.95, 0.1


class _Off:
    """``t`` at ``off`` elements past an aligned base, between margins of a known value."""

    def __init__(self, t, off):
        self.off, self.n = off, t.numel()
        self.base = torch.full((off + self.n + 64,), 7.0, dtype=t.dtype, device=t.device)
        self.t = self.base[off:off + self.n].view(t.shape)
        self.t.copy_(t)

    def margins_are_whole(self):
        return bool((self.base[:self.off] == 7.0).all()
                    and (self.base[self.off + self.n:] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("wdt,pdt", [(torch.float32, torch.bfloat16), (torch.bfloat16, None),
                                     (torch.float32, None)])
@pytest.mark.parametrize("gdt", [torch.float32, torch.bfloat16])
# padded shapes (the 64x64 staging tiles) and whole ones (the flat and, with a kept scale, the tall
# staging kernel)
@pytest.mark.parametrize("rows,cols", [(65, 131), (131, 65), (64, 7), (257, 300), (300, 257),
                                       (128, 256), (512, 256)])
@pytest.mark.parametrize("kept", [False, True])
def test_step_at_any_element_alignment(gpu, rows, cols, kept, gdt, wdt, pdt):
    gen = torch.Generator(device=gpu).manual_seed(rows)
    g = torch.randn(rows, cols, device=gpu, generator=gen).mul_(0.02).to(gdt)
    b = torch.randn(rows, cols, device=gpu, generator=gen).mul_(0.02)
    w = torch.randn(rows, cols, device=gpu, generator=gen).mul_(0.02).to(wdt)
    coeff, T = _coeff_array(dmuon.POLAR_EXPRESS_COEFFICIENTS)
    rst, n_rst = _C.restart_array([2])
    code = {torch.float32: _C.DTYPE_F32, torch.bfloat16: _C.DTYPE_BF16}
    _, nbytes, _ = _C.plan_groups([(rows, cols, 1)], 128, backend=_C.NS_GRAM)
    runs = []
    momentum = b * MU + g.float()
    scale = 1.0 / float((g.double() + MU * momentum.double()).norm())
    for off in (0, 1, 3, 5):
        held = [_Off(x, off) for x in (g, b, w)]
        if pdt is not None:
            held.append(_Off(torch.zeros(rows, cols, dtype=pdt, device=gpu), off))
        t = [h.t for h in held]
        p = None if pdt is None else t[3]
        est = torch.tensor([scale], device=gpu)
        ptr = torch.tensor([x.data_ptr() for x in t] + [0] * (4 - len(t)) + [est.data_ptr()],
                           dtype=torch.int64, device=gpu)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=gpu)
        base = ptr.data_ptr()
        _C.call("dmuon_muon_step_group", base, code[gdt], base + 8,
                base + 32 if kept else None, base + 16, code[wdt],
                None if p is None else base + 24, 0 if p is None else code[pdt], rows, cols, 1, 0,
                LR, MU, WD, 1, 0, coeff, T, _C.NS_GRAM, rst, n_rst, 1e-7, ws.data_ptr(), nbytes,
                128, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert all(h.margins_are_whole() for h in held)
        runs.append([t[1].clone(), t[2].clone()] + ([] if p is None else [p.clone()]))
        assert torch.equal(t[0], g)
    # the momentum in the reference's two roundings, the forward copy one rounding of the weight
    assert torch.equal(runs[0][0], momentum)
    if pdt is not None:
        assert torch.equal(runs[0][2], runs[0][1].to(pdt))
    for r in runs[1:]:
        for x, y in zip(runs[0], r):
            assert torch.equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,L", [(7, 3, 1), (65, 129, 2), (129, 1001, 1), (1001, 65, 3)])
def test_padded_copies_of_odd_operands(gpu, M, K, L):
    gen = torch.Generator(device=gpu).manual_seed(M)
    X = torch.randn(L, M, K, device=gpu, generator=gen).mul_(0.1).to(torch.float16)
    big = torch.full((L, M + 1, K + 3), float("nan"), dtype=torch.float16, device=gpu)
    big[:, :M, 1:K + 1] = X
    D = torch.full((L * M * M + 2,), 7.0, dtype=torch.float16, device=gpu)
    view = D[1:-1].view(L, M, M)
    syrk_or_cublas(big[:, :M, 1:K + 1], view)
    Mp, Kp = -(-M // 128) * 128, -(-K // 64) * 64
    Xp = torch.zeros(L, Mp, Kp, dtype=torch.float16, device=gpu)
    Xp[:, :M, :K] = X
    want = torch.empty(L, Mp, Mp, dtype=torch.float16, device=gpu)
    syrk_or_cublas(Xp, want, tile=128)
    assert torch.equal(view, want[:, :M, :M])
    assert float(D[0]) == 7.0 and float(D[-1]) == 7.0
