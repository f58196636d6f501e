"""``dmuon_syrk`` on ragged operands read and written in place: the bits of the zero-padded product,
no value past the operands read or written."""
import ctypes

import pytest
import torch

from dmuon_amd import _C
from dmuon_amd.optim.syrk_dispatch import syrk_or_cublas

# sides around the 8-value chunk, the 64-wide slice and the 64- and 128-tiles; a batch that runs
# on each of the 64-tile and the two 128-tile kernels
CASES = [(8, 8, 1), (56, 72, 2), (72, 56, 1), (120, 1000, 1), (136, 64, 3), (200, 128, 40),
         (328, 328, 30), (1000, 3000, 1), (1000, 1000, 1), (1016, 1016, 4), (1928, 520, 1)]


def _strided(t, pad, fill):
    """``t`` (L, M, N) in a larger tensor of ``fill``: rows N + pad long, and a row between."""
    big = torch.full((t.shape[0], t.shape[1] + 1, t.shape[2] + pad), fill, dtype=t.dtype,
                     device=t.device)
    big[:, :t.shape[1], :t.shape[2]] = t
    return big


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,code", [(torch.float16, _C.DTYPE_F16),
                                        (torch.bfloat16, _C.DTYPE_BF16)])
@pytest.mark.parametrize("M,K,L", CASES)
@pytest.mark.parametrize("other,addend", [(False, False), (False, True), (True, True)])
def test_edges_equal_the_padded_product(gpu, dtype, code, M, K, L, other, addend):
    gen = torch.Generator(device=gpu).manual_seed(M + K + L)
    A = (torch.randn(L, M, K, device=gpu, generator=gen) * 0.1).to(dtype)
    B = (2.0 * A.float()).to(dtype) if other else A             # A B^T stays symmetric
    C = torch.randn(L, M, M, device=gpu, generator=gen).to(dtype)
    C = (C.float() + C.float().transpose(1, 2).contiguous()).to(dtype)
    stream = torch.cuda.current_stream().cuda_stream

    def syrk(a, b, c, d, m, k):
        row = lambda t: (t.data_ptr(), t.stride(1), t.stride(0))  # noqa: E731
        args = (*row(a), *(row(b) if other else (None, 0, 0)),
                *(row(c) if addend else (None, 0, 0)), *row(d), m, k, L)
        _C.call("dmuon_syrk", code, *args, 0.75, 0.5 if addend else 0.0, 0.25, None, 128, None, 0,
                stream)

    # NaN around every operand and a known value around D
    nan = float("nan")
    a, b, c = (_strided(t, p, nan) for t, p in ((A, 8), (B, 16), (C, 24)))
    d = _strided(torch.zeros_like(C), 8, 7.0)
    syrk(a, b, c, d, M, K)
    # the same product on whole tiles
    Mp, Kp = -(-M // 128) * 128, -(-K // 64) * 64
    pad = lambda t, r, w: torch.nn.functional.pad(  # noqa: E731
        t, (0, w - t.shape[2], 0, r - t.shape[1])).contiguous()
    want = torch.empty(L, Mp, Mp, dtype=dtype, device=gpu)
    syrk(pad(A, Mp, Kp), pad(B, Mp, Kp), pad(C, Mp, Mp), want, Mp, Kp)
    torch.cuda.synchronize()
    assert torch.equal(d[:, :M, :M], want[:, :M, :M])
    assert (d[:, M:] == 7.0).all() and (d[:, :, M:] == 7.0).all()
    ref = 0.75 * torch.matmul(A.float(), B.float().transpose(1, 2).contiguous()) \
        + 0.25 * torch.eye(M, device=gpu)
    if addend:
        ref = ref + 0.5 * C.float()
    # one rounding of a result accumulated in fp32
    eps = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    assert (d[:, :M, :M].float() - ref).abs().max() <= 2 * eps * ref.abs().max()


def test_what_needs_copies_still_asks_for_a_workspace():
    lib, p = _C.lib(), 1 << 20
    run = lambda M, K, lda, a=p: lib.dmuon_syrk(  # noqa: E731
        _C.DTYPE_F16, a, lda, M * lda, None, 0, 0, None, 0, 0, 1 << 30, M, M * M, M, K, 1, 1.0, 0.0,
        0.0, None, 0, None, 0, None)
    for args in ((1000, 3001, 3001), (1001, 3000, 3000), (1000, 3000, 3004), (1000, 3000, 3000, p + 2),
                 (4000, 3000, 3000)):
        assert run(*args) != 0 and b"workspace" in lib.dmuon_last_error(), args
    need = ctypes.c_int64()
    assert lib.dmuon_syrk_workspace_size(_C.DTYPE_F16, p, 3000, 0, None, 0, 0, None, 0, 0, 1 << 30,
                                         1000, 0, 1000, 3000, 1, 0, ctypes.byref(need)) == 0


def _need(M, K, L=1, a=1 << 24, c=None, d=1 << 30, lda=0, ldd=0, b=None):
    lib, need = _C.lib(), ctypes.c_int64(-1)
    lda, ldd = lda or K, ldd or M
    assert lib.dmuon_syrk_workspace_size(
        _C.DTYPE_F16, a, lda, M * lda, b, 0 if b is None else lda, 0 if b is None else M * lda, c,
        0 if c is None else M, 0 if c is None else M * M, d, ldd, M * ldd, M, K, L, 0,
        ctypes.byref(need)) == 0, lib.dmuon_last_error()
    return need.value


def test_operands_used_in_place_ask_for_no_workspace():
    assert _need(1024, 3072) == 0                                # whole tiles
    for M, K, L in CASES:
        if M % 128 or K % 64:
            assert _need(M, K, L) == 0 and _need(M, K, L, c=1 << 28) == 0, (M, K, L)
    # padded copies of A (1024 x 3008) and D
    assert _need(1001, 3000) == 2 * (1024 * 3008 + 1024 * 1024)


def test_a_result_inside_the_operands_memory_takes_the_copies():
    """In place, a block may store D before another has read its operands: memory they share (also
    with no value in common) keeps the padded copies, whose result is stored last."""
    M, K = 200, 328
    a = 1 << 24
    end = a + 2 * M * K
    copies = 2 * (256 * 384 + 256 * 256)
    assert _need(M, K, a=a, d=end) == 0                              # D right behind A
    assert _need(M, K, a=a, d=end - 16) == copies
    assert _need(M, K, a=a, d=a - 2 * M * M + 16) == copies
    assert _need(M, K, a=a, d=a - 2 * M * M) == 0
    assert _need(M, K, a=a, d=a + 2 * K, lda=K + M, ldd=K + M) == copies   # columns of one tensor
    c = 1 << 28
    assert _need(M, K, c=c, d=c + 2 * M * M) == 0 and _need(M, K, c=c, d=c + 16) > copies
    assert _need(M, K, L=3, b=1 << 29, d=(1 << 29) + 2 * 2 * M * K + 16) > 3 * copies


@pytest.mark.gpu
@pytest.mark.parametrize("over", ["A", "C"])
def test_a_result_over_its_operands(gpu, over):
    M, K, L = 200, 328, 2
    gen = torch.Generator(device=gpu).manual_seed(4)
    A = (torch.randn(L, M, K, device=gpu, generator=gen) * 0.1).to(torch.float16)
    C = torch.randn(L, M, M, device=gpu, generator=gen).to(torch.float16)
    C = (C.float() + C.float().transpose(1, 2).contiguous()).to(torch.float16)
    want = torch.empty_like(C)
    syrk_or_cublas(A, want, C=C, alpha=0.5, beta=0.25)
    flat = torch.zeros(8 + L * M * K, dtype=torch.float16, device=gpu)
    src = A if over == "A" else C
    x, d = flat[:src.numel()].view_as(src), flat[8:8 + L * M * M].view(L, M, M)
    x.copy_(src)
    syrk_or_cublas(x if over == "A" else A, d, C=C if over == "A" else x, alpha=0.5, beta=0.25)
    assert torch.equal(d, want)
