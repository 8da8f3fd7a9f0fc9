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
