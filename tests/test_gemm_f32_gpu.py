"""The 32-bit products on the matrix cores: against 64-bit sums at the edges of rows, features and
K, dense and grouped, and a row's bits whatever the number of rows beside it."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from ninfer_amd.kernels import load_ops
    return load_ops()


@pytest.fixture()
def gen():
    return torch.Generator(device="cuda").manual_seed(77)


def within(got, x, w, want):
    """A sum of K products in 32-bit is off by at most K units of 2^-24 of the sum of their sizes
    (each product and each addition rounds once); twice that leaves room for the bias."""
    k = x.shape[-1]
    bound = 2 * k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 1e-6
    assert ((got.double() - want).abs() <= bound).all(), (got.double() - want).abs().max()


@pytest.mark.parametrize("m", [1, 15, 16, 17, 33, 64, 65, 200])
@pytest.mark.parametrize("n,k", [(1, 4), (15, 60), (17, 128), (60, 132), (130, 2048), (2048, 1408)])
def test_linear(ops, gen, m, n, k):
    x, w = (torch.randn(r, k, generator=gen, device="cuda") for r in (m, n))
    bias = torch.randn(n, generator=gen, device="cuda")
    want = x.double() @ w.double().T + bias.double()
    more = torch.full((m + 2, n), 7.0, device="cuda")      # rows behind the product's
    ops.linear(x, w, more[:m], bias=bias)
    within(more[:m], x, w, want)
    assert (more[m:] == 7.0).all()
    one = torch.empty(1, n, device="cuda")
    ops.linear(x[m - 1:], w, one, bias=bias)
    assert torch.equal(one[0], more[m - 1])


# One shape for each tile that a launch may choose (eight waves of 1 x 1, 1 x 2 and 2 x 2 tiles, four of 1 x 2,
# 2 x 2 and 3 x 2); K whose segments are an odd number of chunks, so that a stage holds the end of one segment
# and the start of the next, and K that ends inside a chunk.
@pytest.mark.parametrize("m,n,k", [(17, 2048, 1412), (16, 6144, 1408), (17, 6130, 1408), (70, 6160, 1412),
                                   (150, 6144, 1424), (40, 6130, 1412)])
def test_every_tile(ops, gen, m, n, k):
    x, w = (torch.randn(r, k, generator=gen, device="cuda") for r in (m, n))
    out, one = torch.empty(m, n, device="cuda"), torch.empty(1, n, device="cuda")
    ops.linear(x, w, out)
    within(out, x, w, x.double() @ w.double().T)
    ops.linear(x[m - 1:], w, one)
    assert torch.equal(one[0], out[m - 1])


# Operands that end beyond 4 GB, in rows of 32 KB: weights (gate rows and, as far behind again, their up rows), rows
# of A and rows of A that an index gathers.
K_FAR, N_FAR = 8192, 131120


def test_weights_beyond_4_gb(ops, gen):
    x, w = (torch.randn(r, K_FAR, generator=gen, device="cuda") for r in (3, 2 * N_FAR))
    w *= K_FAR ** -0.5
    out, gated = torch.empty(3, 2 * N_FAR, device="cuda"), torch.empty(3, N_FAR, device="cuda")
    ops.linear(x, w, out)
    ops.swiglu_linear(x, w, gated)
    ends = torch.tensor([0, 1, N_FAR - 33, N_FAR - 1, N_FAR, 2 * N_FAR - 2, 2 * N_FAR - 1], device="cuda")
    within(out[:, ends], x, w[ends], x.double() @ w[ends].double().T)
    # a feature's bits are those of a product of its rows alone
    part = torch.empty(3, 64, device="cuda")
    ops.linear(x, w[-64:].contiguous(), part)
    assert torch.equal(out[:, -64:], part)
    ops.swiglu_linear(x, torch.cat([w[N_FAR - 64:N_FAR], w[-64:]]), part)
    assert torch.equal(gated[:, -64:], part)


def test_rows_beyond_4_gb(ops, gen):
    x, w = (torch.randn(r, K_FAR, generator=gen, device="cuda") for r in (N_FAR, 34))
    out, gated, one = torch.empty(N_FAR, 34, device="cuda"), torch.empty(N_FAR, 17, device="cuda"), torch.empty(5, 34, device="cuda")
    ends = torch.tensor([0, 7, N_FAR // 2, N_FAR - 2, N_FAR - 1], device="cuda")
    ops.linear(x, w, out)
    within(out[ends], x[ends], w, x[ends].double() @ w.double().T)
    ops.linear(x[ends], w, one)
    assert torch.equal(out[ends], one)
    # rows dealt to two groups in an order of their own: each row's product is that of the row alone
    w2 = torch.randn(2, 34, K_FAR, generator=gen, device="cuda")
    order = torch.randperm(N_FAR, generator=gen, device="cuda").int()
    cut = N_FAR // 3
    offsets = torch.tensor([0, cut, N_FAR], device="cuda", dtype=torch.int32)
    ops.grouped_swiglu(x, w2, offsets, order, 1, gated)
    for place in (0, cut - 1, cut, N_FAR - 1, int((order == N_FAR - 1).nonzero()), int((order == 0).nonzero())):
        want = torch.empty(1, 17, device="cuda")
        ops.swiglu_linear(x[order[place].long()][None], w2[int(place >= cut)], want)
        assert torch.equal(gated[place], want[0])


@pytest.mark.parametrize("m,n,k", [(1, 17, 64), (40, 100, 200), (70, 1408, 256)])
def test_gated_rows_alone_and_together(ops, gen, m, n, k):
    x, w = torch.randn(m, k, generator=gen, device="cuda"), torch.randn(2 * n, k, generator=gen, device="cuda")
    w *= k ** -0.5
    out, one = torch.empty(m, n, device="cuda"), torch.empty(1, n, device="cuda")
    ops.swiglu_linear(x, w, out)
    g, u = (x.double() @ w.double().T).chunk(2, 1)
    torch.testing.assert_close(out.double(), g * torch.sigmoid(g) * u, atol=1e-5, rtol=1e-5)
    ops.swiglu_linear(x[:1], w, one)
    assert torch.equal(one[0], out[0])


@pytest.mark.parametrize("counts", [[0, 1, 0, 15, 16, 17], [3], [70, 0, 129, 33], [1] * 9])
def test_grouped(ops, gen, counts):
    """Experts with no rows, with one, with a tile more or less a row."""
    e, h, inner, m = len(counts), 96, 72, sum(counts)
    w = torch.randn(e, 2 * inner, h, generator=gen, device="cuda") * h ** -0.5
    down = torch.randn(e, h, inner, generator=gen, device="cuda") * inner ** -0.5
    x = torch.randn(m, h, generator=gen, device="cuda")
    ids = torch.repeat_interleave(torch.arange(e), torch.tensor(counts))
    order = torch.randperm(m, generator=torch.Generator().manual_seed(1))
    of_row = torch.empty(m, dtype=torch.long)
    of_row[order] = ids                                        # row order[i] belongs to expert ids[i]
    offsets = torch.zeros(e + 1, dtype=torch.int32)
    offsets[1:] = torch.cumsum(torch.tensor(counts), 0)
    act, y = torch.empty(m, inner, device="cuda"), torch.empty(m, h, device="cuda")
    order, offsets = order.to("cuda", torch.int32), offsets.cuda()
    ops.grouped_swiglu(x, w, offsets, order, 1, act)
    ops.grouped_down(act, down, offsets, order, y)
    for i in range(m):
        at = int(order[i])
        g, u = (x[at].double() @ w[of_row[at]].double().T).chunk(2)
        a = g * torch.sigmoid(g) * u
        torch.testing.assert_close(act[i].double(), a, atol=1e-5, rtol=1e-5)
        torch.testing.assert_close(y[at].double(), act[i].double() @ down[of_row[at]].double().T, atol=1e-5, rtol=1e-5)
