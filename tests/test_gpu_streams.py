"""The stream form of the fused backward (2 to 8 taps; bf16 up to 32 routes, fp32
up to 16, and 32 with up to 5 taps):
ranges of one and of several steps, token counts around a step and a range, a
ragged last channel group, segment starts at every place of a stream (between
streams, steps and ranges included), against the oracle."""
import pytest
import torch

from moc import moc_triton
from oracle import moc_oracle as O
from tests._parity import assert_close, gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16
F32 = torch.float32


def _check(x, a, b, dy, act, lengths=None, dt=BF):
    xx, aa, bb = (t.to(DEV, dt).requires_grad_() for t in (x, a, b))
    if lengths is None:
        y, _ = moc_triton(xx, aa, bb, activation=act)
    else:
        cu = torch.tensor([0, *lengths]).cumsum(0).to(DEV, torch.int32)
        y, _ = moc_triton(xx, aa, bb, activation=act, cu_seqlens=cu, max_seqlen=max(lengths))
    y.backward(dy.to(DEV, dt).expand_as(y))
    rx, ra, rb = (t.detach().clone().requires_grad_() for t in O.reference_inputs(x.to(dt), a.to(dt), b.to(dt), dt))
    if lengths is None:
        ry = O.moc_ref(rx, ra, rb, act)
    else:
        ry = O.moc_varlen_ref(rx, ra, rb, cu.cpu(), act)
    ry.backward(dy.to(dt).float().expand_as(ry))
    for n, u, r in zip(("y", "dx", "dalpha", "dbasis"), (y, xx.grad, aa.grad, bb.grad),
                       (ry, rx.grad, ra.grad, rb.grad)):
        assert_close(n, u, r, dt)


@pytest.mark.parametrize("S,K,act", [(2, 16, "silu"), (3, 7, None), (4, 16, "silu"), (4, 32, None),
                                     (5, 12, None), (6, 20, "silu"), (7, 16, "silu"), (8, 32, "silu"),
                                     (8, 17, None)])
@pytest.mark.parametrize("B,T,D", [(1, 1, 2), (1, 28, 16), (1, 29, 18), (1, 30, 126), (1, 32, 128),
                                   (2, 33, 130), (1, 64, 254), (3, 5, 66)])
def test_stream_edges_fixed(S, K, act, B, T, D):
    g = gen(100 * S + T)
    _check(randn(g, B, T, D, scale=0.5), torch.softmax(randn(g, B, T, K), -1),
           randn(g, K, S, D, scale=0.3), randn(g, B, T, D), act)


@pytest.mark.parametrize("S,K,act", [(2, 12, None), (3, 12, "silu"), (4, 12, "silu"), (4, 12, None),
                                     (4, 32, "silu"), (6, 16, "silu"), (7, 32, None), (8, 16, "silu"),
                                     (8, 32, None)])
@pytest.mark.parametrize("longest", [3, 45, 700])
def test_stream_ranges_packed(S, K, act, longest):
    # on 256 CUs 172 to 249 ranges of the two 128-channel groups, one to three steps each,
    # in the four-wave form, 103 to 120 of four or five in the two-wave form
    g = gen(S * 10 + longest)
    N, D = 256 * 29 * 2 + 77, 130
    lengths, left = [], N
    while left:
        n = min(left, int(torch.randint(1, longest + 1, (1,), generator=g)))
        lengths.append(n)
        left -= n
    _check(randn(g, N, D, scale=0.5), torch.softmax(randn(g, N, K), -1),
           randn(g, K, S, D, scale=0.3), randn(g, N, D), act, lengths)


@pytest.mark.parametrize("S,K,act", [(2, 12, "silu"), (2, 16, None), (3, 12, "silu"), (4, 12, None),
                                     (4, 16, "silu")])
@pytest.mark.parametrize("longest", [0, 3, 700])
def test_stream_two_tiers(S, K, act, longest):
    # on 256 CUs two workgroups per CU of the two channel groups exactly: 256 ranges, the
    # first half of them longer (0: one sequence)
    g = gen(S * 20 + longest)
    N, D = 512 * (33 - S) - 5, 130
    lengths, left = [], N
    while left:
        n = min(left, int(torch.randint(1, longest + 1, (1,), generator=g))) if longest else N
        lengths.append(n)
        left -= n
    _check(randn(g, N, D, scale=0.5), torch.softmax(randn(g, N, K), -1),
           randn(g, K, S, D, scale=0.3), randn(g, N, D), act, lengths)


@pytest.mark.parametrize("form", ["one", "row"])
@pytest.mark.parametrize("S,K", [(4, 16), (8, 32), (7, 8)])
def test_stream_broadcast_dy(form, S, K):
    g = gen(7)
    B, T, D = 1, 256 * 29 + 1, 258
    dy = randn(g, 1, 1, 1) if form == "one" else randn(g, 1, 1, D)
    _check(randn(g, B, T, D, scale=0.5), torch.softmax(randn(g, B, T, K), -1),
           randn(g, K, S, D, scale=0.3), dy, "silu")


@pytest.mark.parametrize("S,K,act", [(2, 16, "silu"), (3, 7, None), (4, 16, "silu"), (4, 4, None),
                                     (5, 12, None), (6, 16, "silu"), (7, 9, "silu"), (8, 16, "silu"),
                                     (8, 16, None), (2, 32, "silu"), (3, 20, None), (4, 32, "silu"),
                                     (5, 24, None), (5, 32, "silu")])
@pytest.mark.parametrize("B,T,D", [(1, 1, 2), (1, 28, 16), (1, 29, 18), (1, 32, 128), (2, 33, 130),
                                   (1, 64, 254), (3, 5, 66)])
def test_stream_edges_fixed_f32(S, K, act, B, T, D):
    g = gen(100 * S + T)
    _check(randn(g, B, T, D, scale=0.5), torch.softmax(randn(g, B, T, K), -1),
           randn(g, K, S, D, scale=0.3), randn(g, B, T, D), act, dt=F32)


@pytest.mark.parametrize("S,K,act", [(2, 12, None), (4, 16, "silu"), (4, 12, None), (8, 16, "silu"),
                                     (4, 32, "silu"), (5, 20, None)])
@pytest.mark.parametrize("longest", [3, 700])
def test_stream_ranges_packed_f32(S, K, act, longest):
    # on 256 CUs 97 to 121 ranges of the two channel groups, two to four steps each
    g = gen(S * 10 + longest)
    N, D = 128 * 29 * 3 + 77, 130
    lengths, left = [], N
    while left:
        n = min(left, int(torch.randint(1, longest + 1, (1,), generator=g)))
        lengths.append(n)
        left -= n
    _check(randn(g, N, D, scale=0.5), torch.softmax(randn(g, N, K), -1),
           randn(g, K, S, D, scale=0.3), randn(g, N, D), act, lengths, dt=F32)


@pytest.mark.parametrize("form", ["one", "row"])
@pytest.mark.parametrize("S,K,act", [(4, 16, "silu"), (8, 7, None), (4, 32, None)])
def test_stream_broadcast_dy_f32(form, S, K, act):
    g = gen(7)
    B, T, D = 1, 128 * 29 + 1, 258
    dy = randn(g, 1, 1, 1) if form == "one" else randn(g, 1, 1, D)
    _check(randn(g, B, T, D, scale=0.5), torch.softmax(randn(g, B, T, K), -1),
           randn(g, K, S, D, scale=0.3), dy, act, dt=F32)
