"""Gram Newton-Schulz of matrices of at most 128 rows: the one-workgroup form of a segment's
m x m products (128-tile plans) gives the bits of the NT products (256-tile plans)."""
import pytest
import torch

import dmuon_amd as dmuon
from dmuon_amd import _C
from oracle import ns_oracle as o

PE = list(dmuon.POLAR_EXPRESS_COEFFICIENTS)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,L", [((1, 1), 1), ((3, 50), 2), ((16, 40), 3), ((63, 64), 1),
                                     ((64, 64), 1), ((65, 200), 2), ((200, 65), 1), ((100, 128), 5),
                                     ((127, 129), 1), ((128, 128), 1), ((128, 512), 2),
                                     ((2000, 128), 2)])
@pytest.mark.parametrize("coeffs,restarts", [(PE, (2,)), (PE, ()), (PE, (1, 3)), (PE, (0, 4)),
                                             (PE[:1], ()), (PE[:2], (1,)), (PE[:3], (1, 2))])
def test_same_bits_as_the_tiled_products(gpu, shape, L, coeffs, restarts):
    gen = torch.Generator(device=gpu).manual_seed(shape[0] + shape[1])
    Gs = [torch.randn(shape, device=gpu, generator=gen) for _ in range(L)]
    run = lambda tile: dmuon.newton_schulz_batched(  # noqa: E731
        Gs, coeffs, tile=tile, backend="gram", restart_iterations=restarts)
    for a, b in zip(run(128), run(256)):
        assert torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.gpu
def test_more_matrices_than_compute_units(gpu):
    gen = torch.Generator(device=gpu).manual_seed(9)
    Gs = [torch.randn(96, 160, device=gpu, generator=gen) for _ in range(700)]
    outs = dmuon.newton_schulz_batched(Gs, PE, tile=128, backend="gram", restart_iterations=(2,))
    for i in (0, 255, 256, 699):
        assert torch.equal(outs[i], dmuon.gram_newton_schulz(Gs[i]))


@pytest.mark.gpu
@pytest.mark.parametrize("T", [16, 17])
def test_longest_segment_and_one_past_it(gpu, T):
    gen = torch.Generator(device=gpu).manual_seed(T)
    G = torch.randn(96, 160, device=gpu, generator=gen)
    coeffs = [(1.5, -0.5, 0.0)] * T
    a, b = (dmuon.newton_schulz_batched([G], coeffs, tile=t, backend="gram",
                                        restart_iterations=())[0] for t in (128, 256))
    assert torch.equal(a, b)


@pytest.mark.gpu
def test_against_float64(gpu):
    G = torch.randn(128, 512, generator=torch.Generator().manual_seed(1))
    u = dmuon.gram_newton_schulz(G.to(gpu)).cpu().numpy()
    # fp16 products five steps deep, as the tiled form's bound
    assert o.rel_fro(u, o.closed_form_ns(G.numpy(), o.POLAR_EXPRESS)) < 5e-3


def test_estimate_keeps_small_matrices_out_of_tiled_calls_only_when_it_pays():
    one = _C.plan_groups([(128, 512, 1)], backend=_C.NS_GRAM)
    many = _C.plan_groups([(128, 512, 1), (64, 640, 1)], backend=_C.NS_GRAM)
    assert one[0] == many[0] == 128 and many[2] < 2 * one[2]
