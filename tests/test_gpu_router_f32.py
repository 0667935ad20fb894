"""The fp32 router kernels (logits, softmax / exp weights, dz, drouter) at the
edges of their tiles, against the products in 64 bits, and the fp32 layer that
runs on them against torch's router."""
import pytest
import torch

import moc
from moc import MoC, ops
from moc._lib import ROUTE_EXP, ROUTE_SOFTMAX
from tests._parity import gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _close(got, ref, terms):
    # fp32 sums of `terms` products in some order: the error of one is at most
    # terms 2^-24 of the sum of magnitudes, its rms about sqrt(terms) 2^-24 of
    # the result's rms; 8 of those and one rounding
    ref = ref.double().cpu()
    rms = ref.pow(2).mean().sqrt()
    err = (got.double().cpu() - ref).abs().max()
    assert err <= (8 * terms ** 0.5 + 8) * 2.0 ** -24 * max(rms, ref.abs().max() / 8), (err, rms)


@pytest.mark.parametrize("N,Z,K", [(1, 64, 4), (15, 64, 16), (16, 128, 12), (17, 192, 20),
                                   (63, 320, 32), (65, 512, 16), (1000, 1024, 28), (4097, 64, 8)])
def test_router_f32_edges(N, Z, K):
    g = gen(N + Z + K)
    z, r, dl = (randn(g, N, Z).to(DEV), randn(g, K, Z, scale=0.05).to(DEV),
                randn(g, N, K, scale=0.1).to(DEV))
    assert ops.router_f32_supported(z, r)
    logits = z.double() @ r.double().T
    _close(ops.router_forward(z, r), logits, Z)
    for code, ref in ((ROUTE_SOFTMAX, logits.softmax(-1)), (ROUTE_EXP, logits.exp())):
        # a relative error of the logits' absolute one, and of exp itself (2^-21)
        w = ops.router_forward(z, r, routing=code)
        tol = (8 * Z ** 0.5 + 8) * 2.0 ** -24 * logits.abs().max() + 2.0 ** -20
        assert ((w.double() - ref).abs() <= tol * ref).all()
    dz, dr = ops.router_backward(z, r, dl, True, True)
    _close(dz, dl.double() @ r.double(), K)
    _close(dr, dl.double().T @ z.double(), N)
    assert torch.equal(ops.router_backward(z, r, dl, True, False)[0], dz)
    assert torch.equal(ops.router_backward(z, r, dl, False, True)[1], dr)


# each workgroup form of the forward at its first and last token count (256 CUs): eight waves
# up to 256 blocks of 16 tokens from Z 512, routes past 16 halved (no softmax) up to 128 blocks
@pytest.mark.parametrize("N,Z,K", [(4096, 512, 16), (4097, 512, 20), (4096, 448, 4), (2048, 512, 28), (2049, 576, 32),
                                   (5, 1088, 24), (1, 4096, 32), (33, 64, 20)])
def test_router_f32_workgroup_forms(N, Z, K):
    test_router_f32_edges(N, Z, K)


@pytest.mark.parametrize("route", ["softmax", "exp"])
@pytest.mark.parametrize("K,S", [(4, 4), (16, 4), (16, 6), (32, 3)])
def test_layer_f32_matches_torch_router(K, S, route):
    torch.manual_seed(K + S)
    D, Z, B, T = 66, 128, 2, 70
    m = MoC(D, Z, S, K, activation="silu", init_std=0.3, router_activation=route).to(DEV)
    g = gen(K)
    with torch.no_grad():
        m.router.copy_(randn(g, K, Z, scale=0.05))
    x, z, dy = randn(g, B, T, D).to(DEV), randn(g, B, T, Z).to(DEV), randn(g, B, T, D).to(DEV)
    x.requires_grad_(), z.requires_grad_()
    wrt = [x, z, m.router, m.conv_bases]
    y, _ = m(x, z)
    assert type(y.grad_fn).__name__.startswith("_MoCLayerFunction")
    got = [y, *torch.autograd.grad(y, wrt, dy)]
    a = torch.nn.functional.linear(z, m.router)
    a = a.softmax(-1) if route == "softmax" else a.exp()
    y2, _ = moc.moc_triton(x, a, m.conv_bases, activation="silu")
    for u, v in zip(got, [y2, *torch.autograd.grad(y2, wrt, dy)]):
        # both within the 1e-5 rule of the same result
        assert ((u - v).abs() <= 2e-5 * (v.pow(2).mean().sqrt() + v.abs())).all()


def test_layer_f32_under_autocast_keeps_torch_router():
    m = MoC(64, 64, 4, 16).to(DEV)
    x, z = torch.randn(1, 9, 64, device=DEV), torch.randn(1, 9, 64, device=DEV)
    with torch.autocast("cuda", torch.bfloat16):
        assert not ops.router_f32_supported(z, m.router)
        y, _ = m(x, z)
        a = torch.nn.functional.linear(z, m.router)
        assert a.dtype == torch.bfloat16
        ref, _ = moc.moc_triton(x, torch.softmax(a, -1), m.conv_bases)
    assert ((y - ref).abs() <= 1e-2 * ref.pow(2).mean().sqrt() + 1.6e-2 * ref.abs()).all()
