"""Launches whose 64-tiles are one to two per CU: the bits of the other kernels of a 128-tile
plan, at both ends of that range, and the fp32 product."""
import pytest
import torch

from dmuon_amd import _C

DTYPES = [(torch.float16, _C.DTYPE_F16), (torch.bfloat16, _C.DTYPE_BF16)]


def _close(got, ref, dtype):
    # one rounding to 16 bits: with p significant bits (11 in fp16, 8 in bf16) half an ulp is at
    # most 2^-p of the value; and fp32 sums in another order than the reference's, at most
    # (K + 2) 2^-24 of the sum of the terms' sizes: 2e-4 for the rows of length one of the
    # triangles (K <= 4096), 1.2e-3 for K = 1152 terms whose sizes sum to at most 34 / 2, both
    # under 4e-4 of a largest value above 3
    eps = 2.0 ** (-11 if dtype == torch.float16 else -8)
    assert (got.float() - ref).abs().le(eps * ref.abs() + 4e-4 * ref.abs().max()).all()


def _batches(per_matrix, cus):
    """One matrix, the last batch of one tile per CU, the first and last of two, and one more."""
    one, two = cus // per_matrix, 2 * cus // per_matrix
    return sorted({1, max(one, 1), one + 1, max(two, 1), two + 1})


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,code", DTYPES)
@pytest.mark.parametrize("m,k", [(256, 64), (128, 192), (512, 1088), (256, 4096), (248, 1000)])
def test_triangle_products(gpu, dtype, code, m, k):
    """248 x 1000 is read and written in place on ragged edges."""
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    t = -(-m // 128) * 2
    stream = torch.cuda.current_stream().cuda_stream
    sizes = _batches(t * (t + 1) // 2, cus)
    gen = torch.Generator(device=gpu).manual_seed(m + k)
    A = (torch.randn(sizes[-1], m, k, device=gpu, generator=gen) * k ** -0.5).to(dtype)
    C = torch.randn(sizes[-1], m, m, device=gpu, generator=gen)
    C = (C + C.transpose(1, 2)).to(dtype).contiguous()
    first = None
    for L in sizes:
        D = torch.empty(L, m, m, dtype=dtype, device=gpu)
        _C.call("dmuon_syrk", code, A.data_ptr(), k, m * k, None, 0, 0, C.data_ptr(), m, m * m,
                D.data_ptr(), m, m * m, m, k, L, 0.75, 0.5, 0.25, None, 128, None, 0, stream)
        torch.cuda.synchronize()
        if first is None:
            first = D[:1].clone()
            ref = 0.75 * (A[0].float() @ A[0].float().t()) + 0.5 * C[0].float() \
                + 0.25 * torch.eye(m, device=gpu)
            _close(first[0], ref, dtype)
        assert torch.equal(D[:1], first), L
        last = D
    # every other matrix of the largest batch against its own call
    for l in {1, sizes[-1] // 2, sizes[-1] - 1}:
        D = torch.empty(1, m, m, dtype=dtype, device=gpu)
        _C.call("dmuon_syrk", code, A[l].data_ptr(), k, m * k, None, 0, 0, C[l].data_ptr(), m,
                m * m, D.data_ptr(), m, m * m, m, k, 1, 0.75, 0.5, 0.25, None, 128, None, 0,
                stream)
        torch.cuda.synchronize()
        assert torch.equal(D[0], last[l]), l


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,code", DTYPES)
@pytest.mark.parametrize("kmajor", [False, True])
@pytest.mark.parametrize("m,n", [(128, 256), (512, 384), (1152, 128)])
def test_full_products(gpu, dtype, code, kmajor, m, n):
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    stream = torch.cuda.current_stream().cuda_stream
    sizes = _batches((m // 64) * (n // 64), cus)
    gen = torch.Generator(device=gpu).manual_seed(m + n)
    P = (torch.randn(sizes[-1], m, m, device=gpu, generator=gen) * m ** -0.5).to(dtype)
    X = torch.randn(sizes[-1], m, n, device=gpu, generator=gen).to(dtype)
    XT = X.transpose(1, 2).contiguous()
    first = None
    for L in sizes:
        O = torch.empty(L, m, n, dtype=dtype, device=gpu)
        OT = torch.empty(L, n, m, dtype=dtype, device=gpu)
        _C.call("dmuon_ns_gemm", code, P.data_ptr(), m, m * m,
                *((None, 0, 0) if kmajor else (XT.data_ptr(), m, m * n)),
                X.data_ptr(), n, m * n, O.data_ptr(), n, m * n, OT.data_ptr(), m, m * n, m, n, L,
                0.5, 1.5, None, 128, stream)
        torch.cuda.synchronize()
        assert torch.equal(OT.transpose(1, 2), O)
        if first is None:
            first = O[:1].clone()
            _close(first[0], 0.5 * (P[0].float() @ X[0].float() + 1.5 * X[0].float()), dtype)
        assert torch.equal(O[:1], first), L
    for l in {1, sizes[-1] - 1}:
        one = torch.empty(1, m, n, dtype=dtype, device=gpu)
        _C.call("dmuon_ns_gemm", code, P[l].data_ptr(), m, m * m,
                *((None, 0, 0) if kmajor else (XT[l].data_ptr(), m, m * n)),
                X[l].data_ptr(), n, m * n, one.data_ptr(), n, m * n, None, 0, 0, m, n, 1,
                0.5, 1.5, None, 128, stream)
        torch.cuda.synchronize()
        assert torch.equal(one[0], O[l]), l
