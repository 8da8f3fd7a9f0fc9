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
# 352 (96, cut in two), 450 (194: whole), 256 and 255 (one round)
@pytest.mark.parametrize("m,n", [(1531, 11264), (4000, 4200), (2048, 11264), (2300, 12800), (4096, 4096),
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
