"""Dense products that are one round of tiles, at the edges of every tile: rows and features that end inside a
block, K of one k tile, of fewer than a stage's, of a last stage that K does not fill and of more stages than the ring holds, every
epilogue; and which products come to them."""
import ctypes

import pytest
import torch

BF16 = 1


def _args(m, n, k, **more):
    from ninfer_amd.kernels.ops import _GemmArgs
    return _GemmArgs(A=4096, W=4096, C=4096, M=m, N=n, K=k, lda=k, ldc=n, groups=1, a_div=1, in_dtype=BF16, out_dtype=BF16, **more)


# (256 CUs, as the library assumes without a GPU: both sides of a round of each tile; what no round holds, too few
# rows or features, an index or a K that is not whole k tiles)
@pytest.mark.parametrize("m,n,k,gated,tile", [
    (64, 8192, 2048, 0, 32064), (65, 8193, 2048, 0, 96064), (64, 16384, 2048, 0, 64064), (96, 16384, 2048, 0, 96064),
    (64, 16385, 2048, 0, 64096), (129, 16384, 2048, 0, 192064), (129, 16385, 2048, 0, 192128), (128, 16384, 64, 0, 128064), (256, 8192, 64, 1, 128128),
    (512, 2048, 2048, 0, 64064), (513, 2048, 2048, 0, 96064), (1024, 6144, 2048, 0, 128192), (1025, 6144, 2048, 0, 0),
    (1536, 4096, 2048, 0, 192128), (1537, 4096, 2048, 0, 0), (1536, 2048, 2048, 1, 192128), (1024, 3072, 2048, 1, 0),
    (32, 2048, 2048, 0, 0), (33, 2048, 2048, 0, 32064), (512, 63, 2048, 0, 0), (512, 2048, 2080, 0, 0)])
def test_which_tile(m, n, k, gated, tile):
    from ninfer_amd.kernels.build import ensure_built
    lib = ctypes.CDLL(ensure_built())
    assert lib.ninfer_gemm_mid_tile(ctypes.byref(_args(m, n, k, epilogue=gated))) == tile
    assert lib.ninfer_gemm_mid_tile(ctypes.byref(_args(m, n, k, epilogue=gated, a_index=16, offsets=16))) == 0


# Both sides of where tiles of 64 x 128, two a CU, are the faster ones (256 CUs): 192 x 64 that leaves CUs without a block, 128 rows for up to
# 64, tiles of 128 rows that fill the GPU for few more.
@pytest.mark.parametrize("m,n,k,gated,tile", [
    (144, 4296, 1280, 1, 0), (144, 4296, 7168, 1, 0), (160, 10432, 1792, 0, 0), (315, 3152, 2048, 1, 0), (305, 2904, 4800, 1, 192064), (257, 6000, 2112, 0, 192064), (257, 6000, 2048, 0, 0),
    (130, 10944, 1792, 0, 192064), (144, 11008, 1280, 0, 192064), (33, 32000, 1024, 0, 0), (64, 32000, 4096, 0, 0), (64, 16000, 2048, 1, 0),
    (65, 32000, 1536, 0, 0), (72, 30721, 1024, 0, 0), (72, 30592, 1024, 0, 128128), (73, 32000, 1024, 0, 128128), (65, 32000, 1600, 0, 128128),
    (64, 46144, 1024, 0, 0), (64, 45888, 1024, 0, 128192), (48, 46144, 1600, 0, 128192), (100, 14000, 1024, 0, 128064)])
def test_what_lower_tiles_run_faster_stays_with_them(m, n, k, gated, tile):
    from ninfer_amd.kernels.build import ensure_built
    lib = ctypes.CDLL(ensure_built())
    assert lib.ninfer_gemm_mid_tile(ctypes.byref(_args(m, n, k, epilogue=gated))) == tile
    if tile == 0:
        assert lib.ninfer_gemm_kernel(ctypes.byref(_args(m, n, k, epilogue=gated))) == 4 and lib.ninfer_gemm_tile_rows(ctypes.byref(_args(m, n, k, epilogue=gated))) == 64


SHAPES = [(33, 8192, 64), (64, 2056, 192), (64, 16384, 320), (130, 2050, 64), (512, 2048, 2048), (700, 2047, 192), (760, 2048, 320),
          (250, 6100, 128), (129, 8190, 448), (900, 2304, 192), (1500, 2040, 64), (1140, 2900, 576), (1500, 4090, 128),
          (1020, 6100, 256), (2048, 136, 704)]
EPILOGUES = ["none", "f32", "relu2", "bias", "gated", "gated bias"]
CASES = [(*s, e) for s in SHAPES for e in EPILOGUES if not (e.startswith("gated") and s in SHAPES[-2:])]   # (not a round of gated tiles)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,epilogue", CASES)
def test_products(m, n, k, epilogue):
    from ninfer_amd.kernels import load_ops
    ops = load_ops()
    gated = epilogue.startswith("gated")
    g = torch.Generator("cuda").manual_seed(m + n)
    rows = 2 * (n // 2) if gated else n
    x, w = (torch.randn(r, k, generator=g, device="cuda").bfloat16() for r in (m, rows))
    inner = rows // 2 if gated else n
    bias = torch.randn(rows, generator=g, device="cuda") if "bias" in epilogue else None
    dtype = torch.float32 if epilogue == "f32" else torch.bfloat16
    whole = torch.full((m + 1, inner), 7.0, device="cuda", dtype=dtype)
    out = whole[:m]
    args = _args(m, inner, k, epilogue=int(gated))
    assert ops.lib.ninfer_gemm_mid_tile(ctypes.byref(args)) and ops.lib.ninfer_gemm_kernel(ctypes.byref(args)) == 4
    with ops.tuned(split_min_bytes=1 << 40):   # (nothing is cut along K)
        if gated:
            w = w * 0.1
            ops.swiglu_linear(x, w, out, bias=bias)
        else:
            ops._gemm(x, w, out, m=m, n=n, k=k, bias=bias, epilogue=3 if epilogue == "relu2" else 0)
    sums = x.double() @ w.double().T
    # exact products, k of them added in 32-bit in any order
    bound = 2 * k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 1e-6
    if bias is not None:
        sums = sums + bias.double()
        bound = bound + 2.0 ** -23 * sums.abs()
    if gated:
        a, u = sums[:, :inner], sums[:, inner:]
        want = a * torch.sigmoid(a) * u
        # |d silu| <= 1.1 |d a|; the hardware's exponential and reciprocal, 1 ulp each, and two products
        bound = 1.1 * bound[:, :inner] * u.abs() + a.abs() * bound[:, inner:] + 2.0 ** -20 * want.abs() + 1e-6
    elif epilogue == "relu2":
        want = sums.clamp(min=0) ** 2
        bound = 2 * sums.abs() * bound + bound * bound + 2.0 ** -23 * want
    else:
        want = sums
    if dtype == torch.bfloat16:
        bound = bound + 2.0 ** -8 * (want.abs() + bound)
    assert ((out.double() - want).abs() <= bound).all()
    assert (whole[m:] == 7.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(65, 4096, 2048), (512, 2048, 5632), (700, 1024, 1024), (1024, 6144, 2048)])
def test_plain_products_of_one_round_stay_out_of_the_library(monkeypatch, m, n, k):
    from ninfer_amd.kernels import load_ops
    ops = load_ops()
    g = torch.Generator("cuda").manual_seed(m)
    x, w = (torch.randn(r, k, generator=g, device="cuda").bfloat16() for r in (m, n))
    want = torch.matmul(x.double(), w.double().T)
    out = torch.empty(m, n, device="cuda", dtype=torch.bfloat16)
    monkeypatch.setattr(torch, "matmul", None)
    ops.linear(x, w, out)
    assert float((out.double() - want).norm() / want.norm()) < 2.0 ** -8


# (rows, features, K: cut along K, one round of tiles, more rows than are cut, more than a round)
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,taken", [(100, 3584, 20480, True), (256, 2048, 2048, True), (513, 2048, 1024, True),
                                         (4096, 8192, 512, False)])
def test_one_call_runs_what_the_questions_one_by_one_would(m, n, k, taken):
    from ninfer_amd.kernels import load_ops
    ops = load_ops()
    gen = torch.Generator("cuda").manual_seed(m)
    x, w = (torch.randn(*s, generator=gen, device="cuda").to(torch.bfloat16) for s in ((m, k), (n, k)))
    one, each = (torch.zeros(m, n, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    assert ops._gemm_cut_or_mid(x, w, one, m=m, n=n, k=k, cut=m <= ops.split_max_rows) == taken
    asked = m <= ops.split_max_rows and ops._gemm(x, w, each, m=m, n=n, k=k, only_if_split=True) or \
        ops._gemm(x, w, each, m=m, n=n, k=k, only_if_mid=True)
    assert asked == taken and torch.equal(one, each)
    # products exact, k of them added in 32 bits in any order, rounded to bfloat16
    want = x.double() @ w.double().T
    bound = k * 2.0 ** -23 * (x.double().abs() @ w.double().abs().T)
    assert not taken or ((one.double() - want).abs() <= bound + 2.0 ** -8 * (want.abs() + bound)).all()
    ops.linear(x, w, each)
    assert not taken or torch.equal(one, each)
    with pytest.raises(Exception, match="lda"):
        ops._gemm_cut_or_mid(x[:, :64].contiguous(), w, one, m=m, n=n, k=k, cut=True)


# Plain products that blocks of 32 rows or the few-row kernels would take, more slowly than the library; two that are not one round of whole k
# tiles; and those of a long K that are slower in one round of tiles than in the library.
NOT_OURS = [(80, 4096, 5632), (112, 4096, 5632), (112, 3072, 5632), (100, 4096, 4096), (64, 512, 5632), (512, 129, 8192),
            (2048, 64, 2048), (700, 128, 704), (4096, 8192, 512), (512, 2048, 2080),
            (768, 320, 5376), (45, 1344, 7616), (110, 192, 7616), (180, 8448, 1792),
            (276, 1600, 5120), (140, 2688, 7168), (384, 2176, 6144), (1294, 1600, 5120), (1482, 1920, 5632), (512, 6400, 4608), (1043, 576, 8256)]


@pytest.mark.parametrize("m,n,k,ours", [(*s, 0) for s in NOT_OURS] + [
    (96, 8192, 2048, 1), (513, 2048, 1024, 1), (700, 129, 704, 1), (1294, 1600, 4032, 1), (142, 2688, 4096, 1), (338, 1472, 5632, 1),
    (720, 320, 5056, 1), (1010, 576, 5568, 1), (380, 7296, 3072, 1),
    (512, 2048, 5632, 1), (513, 6400, 4608, 1), (900, 2048, 5632, 1), (2048, 2048, 8192, 1)])
def test_which_plain_products_leave_the_library(m, n, k, ours):
    from ninfer_amd.kernels.build import ensure_built
    lib = ctypes.CDLL(ensure_built())
    assert lib.ninfer_gemm_plain_mid(ctypes.byref(_args(m, n, k))) == ours


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", NOT_OURS)
def test_what_the_library_runs_faster_stays_with_it(monkeypatch, m, n, k):
    from ninfer_amd.kernels import load_ops
    ops = load_ops()
    g = torch.Generator("cuda").manual_seed(m)
    x, w = (torch.randn(r, k, generator=g, device="cuda").bfloat16() for r in (m, n))
    out, calls, matmul = torch.empty(m, n, device="cuda", dtype=torch.bfloat16), [], torch.matmul
    monkeypatch.setattr(torch, "matmul", lambda *a, **b: (calls.append(1), matmul(*a, **b)))
    ops.linear(x, w, out)
    assert calls and torch.equal(out, matmul(x, w.t()))


@pytest.mark.parametrize("n,k", [(0, 256), (256, 0), (0, 0)])
def test_products_of_nothing_are_the_librarys(n, k):
    from ninfer_amd.kernels.build import ensure_built
    lib = ctypes.CDLL(ensure_built())
    assert lib.ninfer_gemm_cut_or_mid(ctypes.byref(_args(600, n, k)), None) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("n,k", [(0, 256), (256, 0), (0, 0)])
def test_linear_over_nothing(n, k):
    from ninfer_amd.kernels import load_ops
    x, w = (torch.ones(r, k, device="cuda", dtype=torch.bfloat16) for r in (600, n))
    out = torch.full((600, n), 7.0, device="cuda", dtype=torch.bfloat16)
    load_ops().linear(x, w, out)
    assert (out == 0).all()


# Each tile at a K whose stages go round its ring and whose last stage K does not fill.
LONG = [(70, 2040, 1600, 32064), (700, 1400, 832, 64064), (760, 2040, 832, 96064), (640, 2400, 832, 64096), (1000, 2040, 832, 128064),
        (1500, 2040, 576, 192064), (1100, 3500, 576, 128128), (1500, 4000, 448, 192128), (1020, 6100, 448, 128192)]
LONG_GATED = [(70, 2040, 1600, 64064), (1000, 2040, 832, 128064), (1500, 2040, 576, 192064), (1100, 3500, 576, 128128), (1500, 4000, 448, 192128)]


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,tile,gated", [(*c, False) for c in LONG] + [(*c, True) for c in LONG_GATED])
def test_sums_are_one_chain_along_k(m, n, k, tile, gated):
    """The bits of the taller tiles' sums (and of the library's, where it does not cut K): which kernel a size goes to does not show
    in a model's logits."""
    from ninfer_amd.kernels import load_ops
    ops = load_ops()
    inner = n // 2 if gated else n
    args = _args(m, inner, k, epilogue=int(gated))
    assert ops.lib.ninfer_gemm_mid_tile(ctypes.byref(args)) == tile and ops.lib.ninfer_gemm_kernel(ctypes.byref(args)) == 4
    g = torch.Generator("cuda").manual_seed(m)
    x, w = (torch.randn(r, k, generator=g, device="cuda").bfloat16() for r in (m, n))
    got, tall, low = (torch.empty(m, inner, device="cuda", dtype=torch.bfloat16) for _ in range(3))
    for out, force in ((got, 0), (low, 2), (tall, 3)):
        with ops.tuned(force_kernel=force, split_min_bytes=1 << 40):
            ops._gemm(x, w, out, m=m, n=inner, k=k, epilogue=int(gated))
    assert torch.equal(got, low) and torch.equal(got, tall)
    if not gated:
        want = x.double() @ w.double().T
        # products exact, k of them added in 32 bits, rounded to bfloat16
        bound = k * 2.0 ** -23 * (x.double().abs() @ w.double().abs().T)
        assert ((got.double() - want).abs() <= bound + 2.0 ** -8 * (want.abs() + bound)).all()
