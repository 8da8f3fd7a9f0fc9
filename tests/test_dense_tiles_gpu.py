"""Dense products of many rows whose 256-row tiles do not fill the last round: that round's tiles cut
into blocks of 64 or 128 rows, with rows and features that end inside a block."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from ninfer_amd.kernels import load_ops
    return load_ops()


# tiles of 256 x 256 on 256 CUs: 264 (a last round of 8, cut in four), 16 x 17 = 272 rows of tiles that end early,
# 352 (96, cut in two), 450 (194: whole), 256 and 240 (one round), 306 (50, cut in four), 257 (1, cut in four)
@pytest.mark.parametrize("m,n", [(1531, 11264), (4000, 4200), (2048, 11264), (2300, 12800), (4096, 4096), (4000, 3840),
                                 (1281, 13056), (65537, 256)])
def test_last_round(ops, m, n):
    k = 64
    g = torch.Generator("cuda").manual_seed(m)
    x, w = (torch.randn(r, k, generator=g, device="cuda").bfloat16() for r in (m, n))
    out = torch.full((m + 1, n), 7.0, device="cuda")
    with ops.tuned(force_kernel=3):
        ops.linear(x, w, out[:m])
    want = x.float() @ w.float().T
    # exact products, 64 of them added in 32-bit in any order
    bound = 64 * 2.0 ** -24 * (x.float().abs() @ w.float().abs().T) + 1e-6
    assert ((out[:m] - want).abs() <= 2 * bound).all()
    assert (out[m:] == 7.0).all()


# (K in tiles of 64: one, three, four and five, where the loop's steady part begins, and 32 of a model's width)
@pytest.mark.parametrize("k", [64, 192, 256, 320, 2048])
@pytest.mark.parametrize("m,n", [(1531, 11264), (2000, 11264), (2300, 12800), (4000, 3840)])
def test_last_round_cut_and_whole_have_the_same_bits(ops, m, n, k):
    """A tile's parts walk K as the whole tile does, so a launch with its last round cut in four, in two or
    not at all gives the bits of one that is not cut (as beside another stream's products)."""
    g = torch.Generator("cuda").manual_seed(m + k)
    x, w = (torch.randn(r, k, generator=g, device="cuda").bfloat16() for r in (m, n))
    cut, whole = (torch.full((m + 1, n), 7.0, device="cuda") for _ in range(2))
    with ops.tuned(force_kernel=3):
        ops.linear(x, w, cut[:m])
        ops._side_inside = True
        try:
            ops.linear(x, w, whole[:m])
        finally:
            ops._side_inside = False
    assert torch.equal(cut, whole) and (cut[m:] == 7.0).all()
    rows = list(range(0, m, 97)) + list(range(m - 5, m))
    want = x[rows].double() @ w.double().T
    bound = 2 * k * 2.0 ** -24 * (x[rows].double().abs() @ w.double().abs().T) + 1e-6
    assert ((cut[rows].double() - want).abs() <= bound).all()


def test_gated_last_round(ops):
    m, n, k = 1700, 5632, 128
    g = torch.Generator("cuda").manual_seed(5)
    x, w = (torch.randn(r, k, generator=g, device="cuda").bfloat16() for r in (m, 2 * n))
    w *= 0.1
    whole, out = torch.empty(m, n, device="cuda", dtype=torch.bfloat16), torch.empty(m, n, device="cuda", dtype=torch.bfloat16)
    with ops.tuned(force_kernel=3):
        ops.swiglu_linear(x, w, out)
    with ops.tuned(force_kernel=1):
        ops.swiglu_linear(x, w, whole)
    torch.testing.assert_close(out.float(), whole.float(), atol=1e-3, rtol=2.0 ** -7)


@pytest.mark.parametrize("force", [1, 2, 3])
def test_gated_weights_beyond_4_gb(ops, force):
    """Up rows 4 GB behind their gate rows: the bits are those of a product of the same rows alone."""
    m, n, k = 40, 262200, 8192
    g = torch.Generator("cuda").manual_seed(9)
    x, w = (torch.randn(r, k, generator=g, device="cuda", dtype=torch.bfloat16) for r in (m, 2 * n))
    w *= k ** -0.5
    out, part = (torch.empty(m, f, device="cuda", dtype=torch.bfloat16) for f in (n, 160))   # (129 features and more run here)
    with ops.tuned(force_kernel=force):
        ops.swiglu_linear(x, w, out)
        for first in (0, n // 2, n - 160):
            ops.swiglu_linear(x, torch.cat([w[first:first + 160], w[n + first:n + first + 160]]), part)
            assert torch.equal(out[:, first:first + 160], part)
    last = torch.cat([w[n - 40:n], w[2 * n - 40:]]).double()
    gate, up = (x.double() @ last.T).split(40, 1)
    torch.testing.assert_close(out[:, -40:].double(), gate * torch.sigmoid(gate) * up, atol=1e-2, rtol=2.0 ** -7)


def test_gathered_rows_beyond_4_gb(ops):
    """Rows that an index gathers from more than 4 GB: the bits of the same rows gathered from a few."""
    t, e, h, inner = 524400, 2, 4096, 72
    g = torch.Generator("cuda").manual_seed(11)
    x = torch.randn(t, h, generator=g, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(e, 2 * inner, h, generator=g, device="cuda", dtype=torch.bfloat16) * h ** -0.5
    order, cut = torch.randperm(t, generator=g, device="cuda").int(), t // 3
    i32 = lambda *v: torch.tensor(v, device="cuda", dtype=torch.int32)
    out, few = (torch.empty(r, inner, device="cuda", dtype=torch.bfloat16) for r in (t, 60))
    ops.grouped_swiglu(x, w, i32(0, cut, t), order, 1, out)
    last = (order == t - 1).nonzero().flatten()   # the place of A's last row, at one end of its group's choice
    places = torch.cat([torch.arange(0, 20, device="cuda"), torch.arange(cut - 10, cut + 10, device="cuda"),
                        torch.arange(t - 19, t, device="cuda"), last]).sort().values
    with ops.tuned(force_kernel=2):
        ops.grouped_swiglu(x[order[places].long()], w, i32(0, int((places < cut).sum()), 60),
                           torch.arange(60, device="cuda", dtype=torch.int32), 1, few)
    assert torch.equal(out[places], few)
    rows = x[order[places[-8:]].long()].double()
    gate, up = (rows @ w[1].double().T).split(inner, 1)
    torch.testing.assert_close(out[places[-8:]].double(), gate * torch.sigmoid(gate) * up, atol=1e-2, rtol=2.0 ** -7)
