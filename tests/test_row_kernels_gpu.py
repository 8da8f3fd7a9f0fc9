"""Row kernels in whole 16-byte pieces against the same kernels number by number (operands that do
not lie at multiples of 16 bytes): the same sums in the same order, so the same bits."""
import pytest
import torch

import util

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    from ninfer_amd.kernels import load_ops
    return load_ops()


def shifted(x):
    """The same numbers one element behind a multiple of 16 bytes."""
    buf = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)
    y = buf[1:].view(x.shape)
    y.copy_(x)
    return y


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("width", [4, 1028])
@pytest.mark.parametrize("seqs", [[(0, 1)], [(0, 1), (7, 1), (2, 1)], [(0, 2), (3, 1), (0, 5)], [(5, 255), (0, 2)],
                                  [(0, 254), (9, 1), (0, 6)],
                                  # (1,028 wide, four rows to a thread: one row per request, and a last one of three)
                                  [(3, 1)] * 1600, [(5, 1597), (0, 2)]])
def test_short_conv(ops, dtype, taps, width, seqs):
    g = torch.Generator(DEV).manual_seed(taps * width + len(seqs))
    ctx = util.make_context(ops, dtype, seqs)
    x = torch.randn(ctx.T, width, generator=g, device=DEV)
    w = torch.randn(width, taps, generator=g, device=DEV)
    first = torch.randn(len(seqs) + 1, (taps - 1) * width, generator=g, device=DEV)
    states, outs = [first.clone(), shifted(first)], []
    for state, xs in zip(states, (x, shifted(x))):
        outs.append(torch.empty(ctx.T, width, dtype=dtype, device=DEV))
        ops.short_conv(xs, w, state, ctx, outs[-1])
    assert torch.equal(outs[0], outs[1])
    assert torch.equal(states[0], states[1]) and torch.equal(states[0][-1], first[-1])


@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("seqs", [[(i, 1 + i % 5) for i in range(10)], [(i, 1 + i % 5) for i in range(540)]])
def test_short_conv_of_requests_that_start_anywhere(ops, taps, seqs):
    """The thread that holds a request's first row moves its state on: requests of one to five rows
    that start at every place of a thread's rows (one row; four rows from 540 requests on)."""
    test_short_conv(ops, torch.float32, taps, 1028, seqs)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [4, 1028])
@pytest.mark.parametrize("k", [0, 1, 5])
@pytest.mark.parametrize("t", [9, 300])   # (from 2^18 numbers on the gated sum goes in pieces)
def test_sums(ops, dtype, width, k, t):
    from ninfer_amd.parts import PendingRows
    g = torch.Generator(DEV).manual_seed(width + k)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    x, s1, s2, wts, gate = rnd(t, width), rnd(width), rnd(width), rnd(t, max(k, 1)), rnd(t)
    a, sh, dense, g1, g2 = (rnd(t, width).to(dtype) for _ in range(5))
    y = rnd(t * max(k, 1), width).to(dtype)
    got = []
    for at in (lambda v: v, shifted):
        f = PendingRows(at(y), wts, at(sh), gate) if k else at(dense)
        res = at(x.clone())
        ops.scaled_sum_add(res, at(a), at(s1), f, at(s2))
        gated = at(x.clone())
        ops.gated_sum_add(gated, at(a), at(g1), at(s1), PendingRows(at(y), wts) if k else at(dense), at(g2), at(s2), 0.7)
        got.append((res, gated))
    for u, v in zip(*got):
        assert torch.equal(u, v) and not torch.equal(u, x)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [2048, 1022, 7])
@pytest.mark.parametrize("center", [False, True])
def test_two_norms_of_the_same_rows(ops, dtype, width, center):
    """Bit for bit what the two norms give one after the other, with a sum before the first."""
    gen = torch.Generator(device="cuda").manual_seed(width)
    x = torch.randn(5, width, generator=gen, device="cuda")
    gains = torch.randn(2, width, generator=gen, device="cuda")
    delta = torch.randn(5, width, generator=gen, device="cuda").to(dtype)
    once, twice = x.clone(), x.clone()
    want, got = ([torch.empty(5, width, dtype=dtype, device="cuda") for _ in range(2)] for _ in range(2))
    ops.rmsnorm(once, gains[0].contiguous(), 1e-6, want[0], delta=delta, center=center)
    ops.rmsnorm(once, gains[1].contiguous(), 1e-6, want[1], center=center)
    ops.rmsnorm_two(twice, gains[0].contiguous(), 1e-6, got[0], gains[1].contiguous(), got[1], delta=delta,
                    center=center)
    assert torch.equal(once, twice) and torch.equal(want[0], got[0]) and torch.equal(want[1], got[1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [2048, 1022])
@pytest.mark.parametrize("shared", [False, True])
def test_two_norms_of_the_same_rows_behind_a_weighted_sum(ops, dtype, width, shared):
    """The same where the sum before the first is that of a sparse feed-forward's rows."""
    from ninfer_amd.parts import PendingRows
    gen = torch.Generator(device="cuda").manual_seed(width)
    draw = lambda *size: torch.randn(*size, generator=gen, device="cuda")
    x, gains, logits = draw(5, width), draw(2, width), draw(5, 7)
    rows = PendingRows(draw(15, width).to(dtype), draw(5, 3).abs(), draw(5, width).to(dtype) if shared else None,
                       logits[:, 6] if shared else None)
    once, twice = x.clone(), x.clone()
    want, got = ([torch.empty(5, width, dtype=dtype, device="cuda") for _ in range(2)] for _ in range(2))
    ops.rmsnorm(once, gains[0].contiguous(), 1e-6, want[0], rows_sum=rows)
    ops.rmsnorm(once, gains[1].contiguous(), 1e-6, want[1])
    ops.rmsnorm_two(twice, gains[0].contiguous(), 1e-6, got[0], gains[1].contiguous(), got[1], rows_sum=rows)
    assert not torch.equal(once, x) and torch.equal(once, twice)
    assert torch.equal(want[0], got[0]) and torch.equal(want[1], got[1])
