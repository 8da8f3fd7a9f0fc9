"""What the kernel library decides on the host, without a GPU: which form a step takes and how much scratch
that needs."""
import ctypes

import pytest

BF16 = 1


@pytest.fixture(scope="module")
def lib():
    from ninfer_amd.kernels.build import ensure_built
    lib = ctypes.CDLL(ensure_built())
    lib.ninfer_lightning_chunk_floats.restype = ctypes.c_longlong
    return lib


def test_lightning_scratch_does_not_grow_with_decoding_requests(lib):
    """Single rows beside a portion take no chunk of their own once they are many: the scratch is that
    of the portion's chunks."""
    heads, dim, vdim = 16, 128, 128
    state = heads * dim * vdim
    for singles in (0, 16, 64, 256):
        for rows in (8, 64, 448, 2048):
            floats = lib.ninfer_lightning_chunk_floats(singles + rows, singles + 1, singles, rows, heads, dim, vdim, BF16)
            assert floats in (0, (rows // 64 + 1) * state), (singles, rows)
            assert floats or rows <= 64


def test_lightning_sizes_that_do_not_run_in_chunks(lib):
    floats = lambda dim, vdim, dtype=BF16: lib.ninfer_lightning_chunk_floats(512, 1, 0, 512, 2, dim, vdim, dtype)
    assert floats(128, 128) > 0 and floats(256, 64) > 0
    assert floats(128, 1024) > 0            # (single rows of it are refused, as ever)
    assert floats(257, 16) == -1            # keys too long
    assert floats(256, 256) == -1           # ... and for the walk, with a state too large for single rows
    assert floats(128, 128, 0) == -1        # 32-bit goes token by token


def test_lightning_short_portions(lib):
    """Keys too long for the walk: portions of fewer than 10 rows go token by token. Many short portions of
    shorter ones are walked, without scratch."""
    floats = lambda rows, portions, heads, dim, vdim: lib.ninfer_lightning_chunk_floats(
        rows * portions, portions, 0, rows, heads, dim, vdim, BF16)
    assert floats(8, 1, 4, 256, 64) == -1 and floats(9, 16, 4, 256, 64) == -1
    assert floats(10, 1, 4, 256, 64) > 0
    assert floats(9, 16, 16, 128, 128) == 0
    assert floats(9, 16, 32, 128, 128) > 0


# (an epilogue of 1 is SwiGLU: 2 N rows of weights. 256 CUs, as the library assumes without a GPU)
@pytest.mark.parametrize("m,n,k,gated,beside,rows", [
    (64, 5632, 2048, 1, 0, 64), (640, 5632, 2048, 1, 0, 128), (768, 5632, 2048, 1, 0, 256),
    (1400, 5632, 2048, 1, 0, 128),    # 264 tiles of 256, the last 8 a round of their own, even cut
    (1400, 5632, 2048, 1, 1, 256),    # ... which costs next to nothing beside other products
    (1280, 5632, 2048, 1, 1, 256), (640, 5632, 2048, 1, 1, 128), (2048, 5632, 2048, 1, 1, 256),
    (1531, 12800, 1024, 0, 0, 256), (3000, 6144, 768, 0, 0, 256), (2048, 12800, 512, 0, 0, 256),   # (stores)
    (900, 12800, 512, 0, 0, 128), (1280, 6144, 768, 0, 0, 128), (1280, 8192, 2048, 0, 0, 256)])
def test_height_of_dense_tiles(lib, m, n, k, gated, beside, rows):
    from ninfer_amd.kernels.ops import _GemmArgs
    args = _GemmArgs(M=m, N=n, K=k, lda=k, ldc=n, in_dtype=BF16, out_dtype=BF16 if gated else 0, epilogue=gated,
                     beside=beside)
    assert lib.ninfer_gemm_tile_rows(ctypes.byref(args)) == rows


@pytest.mark.parametrize("m,n,k,gated,kernel", [
    (96, 3072, 768, 1, 4), (64, 4096, 768, 1, 3), (64, 4097, 768, 1, 4), (96, 4096, 1024, 1, 3), (96, 4097, 1024, 1, 4),
    (64, 8192, 768, 0, 3), (128, 4096, 512, 0, 3), (128, 4097, 512, 0, 4)])
def test_which_products_run_in_blocks_of_32_rows(lib, m, n, k, gated, kernel):
    from ninfer_amd.kernels.ops import _GemmArgs
    args = _GemmArgs(A=4096, W=4096, C=4096, M=m, N=n, K=k, lda=k, ldc=n, groups=1, a_div=1, in_dtype=BF16, out_dtype=BF16,
                     epilogue=gated)
    assert lib.ninfer_gemm_kernel(ctypes.byref(args)) == kernel


@pytest.mark.parametrize("rows,n,k,own", [
    (64, 2048, 5632, True), (33, 129, 8192, False), (512, 129, 8192, False), (33, 129, 4096, True), (64, 512, 5632, False),
    (65, 512, 5632, True), (384, 256, 5632, True), (80, 4096, 5632, False), (96, 4096, 5632, True), (112, 3072, 4096, False),
    (80, 3072, 4096, True), (80, 4096, 3584, True), (128, 4096, 4096, True), (160, 1638, 2048, True), (160, 1639, 2048, False),
    (64, 8192, 3072, False), (64, 2048, 2000, False)])
def test_which_plain_products_stay_out_of_the_library(rows, n, k, own):
    from types import SimpleNamespace
    from ninfer_amd.kernels.ops import HipOps
    at = lambda *shape: SimpleNamespace(shape=shape, data_ptr=lambda: 4096)
    assert HipOps._rows_kernel_takes(at(rows, k), at(n, k)) == own


@pytest.mark.parametrize("rows,n,k,cut", [
    (64, 8192, 8192, True), (33, 10240, 3584, True), (32, 10240, 3584, False), (65, 10240, 3584, False), (64, 8192, 3584, False),
    (64, 5120, 5632, True), (64, 4096, 8192, False), (64, 5120, 4864, False), (64, 20480, 3584, True), (64, 20512, 3584, False),
    (64, 16384, 2048, False), (64, 5100, 8192, False), (64, 5120, 5200, False)])
def test_which_products_of_33_to_64_rows_are_cut(rows, n, k, cut):
    import torch
    from types import SimpleNamespace
    from ninfer_amd.kernels.ops import HipOps
    ops = SimpleNamespace(force_generic=False, library_min_rows=32, rows_kernel_max=64, rows_kernel_features=(4096, 32768))
    at = lambda *shape: SimpleNamespace(shape=shape, dtype=torch.bfloat16)
    assert HipOps._rows_cut(ops, at(rows, k), at(rows, n), at(n, k)) == cut
    # (what is asked is what the library keeps from the library)
    assert not cut or not HipOps._use_library(ops, at(rows, k), at(rows, n), at(n, k))


# (experts, chosen, inner, shared inner; rows: does the shared expert start before the routing?)
@pytest.mark.parametrize("sizes,rows,early", [
    ((60, 4, 1408, 5632), 512, True), ((60, 4, 1408, 5632), 600, True), ((60, 4, 1408, 5632), 700, False),
    ((60, 4, 1408, 5632), 1024, False), ((60, 4, 1408, 5632), 2048, False), ((32, 4, 1408, 2816), 1531, True),
    ((32, 4, 1408, 2816), 2048, True), ((16, 2, 704, 1408), 2048, True), ((64, 8, 2560, 20480), 200, True),
    ((64, 8, 2560, 20480), 300, False)])
def test_which_starts_first(sizes, rows, early):
    from types import SimpleNamespace
    from ninfer_amd.kernels.ops import HipOps
    from ninfer_amd.parts.moe import SparseMoE
    experts, top, inner, shared = sizes
    moe = SparseMoE("m.", 2048, experts, top, inner, False, shared_inner=shared)
    assert HipOps.leaves_room(SimpleNamespace(_cus=256), rows, 2 * shared, moe._shared_fills(rows)) == early


# (a short K, where starts and sums outweigh the products, and a model's)
@pytest.mark.parametrize("m,groups,n,k,gated,tile", [
    (128, 32, 512, 384, 0, 412), (264, 32, 768, 256, 0, 412), (2048, 0, 384, 512, 0, 422), (2048, 0, 192, 512, 1, 422),
    (1, 0, 2048, 2048, 0, 811), (173, 0, 2048, 2048, 0, 432), (173, 0, 6144, 2048, 0, 432), (64, 0, 5632, 2048, 1, 822),
    (692, 60, 1408, 2048, 1, 412), (300, 0, 2048, 5632, 0, 432)])
def test_tile_of_32_bit_products(lib, m, groups, n, k, gated, tile):
    from ninfer_amd.kernels.ops import _GemmArgs
    args = _GemmArgs(M=m, N=n, K=k, lda=k, ldc=n, epilogue=gated, groups=groups or 1, offsets=16 if groups else 0)
    assert lib.ninfer_gemm_f32_tile(ctypes.byref(args)) == tile


# (both sides of 40 rows a group and of two tiles of 128 rows a CU; few groups of many features)
@pytest.mark.parametrize("m,groups,n,gated,rows", [
    (60 * 40, 60, 1408, 1, 64), (60 * 41 - 1, 60, 1408, 1, 64), (60 * 41, 60, 1408, 1, 256), (60 * 17, 60, 2048, 0, 64),
    (60 * 137, 60, 1408, 1, 256), (60 * 137, 60, 2048, 0, 256), (16 * 255, 16, 704, 1, 128), (16 * 256, 16, 704, 1, 128),
    (16 * 512, 16, 704, 1, 256), (16 * 512, 16, 1024, 0, 256), (1280, 4, 192, 1, 128), (4 * 256, 4, 2048, 0, 128),
    (4 * 87, 4, 4096, 1, 256), (8 * 87, 8, 2048, 1, 128), (8 * 128, 8, 2048, 1, 256), (8 * 512, 8, 1024, 0, 128),
    (1400, 10, 4096, 1, 256), (8 * 128, 8, 4096, 0, 256), (32 * 512, 32, 256, 1, 256), (64 * 143, 64, 320, 1, 256),
    (40 * 512, 40, 512, 0, 256), (8 * 25, 8, 14336, 1, 256), (16 * 32, 16, 8192, 1, 256), (12 * 25, 12, 2816, 1, 64),
    (17 * 25, 17, 14336, 1, 64)])
def test_height_of_grouped_tiles(lib, m, groups, n, gated, rows):
    from ninfer_amd.kernels.ops import _GemmArgs
    args = _GemmArgs(M=m, N=n, K=1024, lda=1024, ldc=n, in_dtype=BF16, out_dtype=BF16, epilogue=gated, groups=groups,
                     offsets=16)
    assert lib.ninfer_gemm_tile_rows(ctypes.byref(args)) == rows


# (32-bit operands on both sides of 4 GB: an output head, a gated product's weights, a prompt's rows, rows that an
# index gathers)
@pytest.mark.parametrize("m,n,k,gated,indexed", [
    (1, 131056, 8192, 0, 0), (1, 152064, 8192, 0, 0), (200, 152064, 8192, 0, 0), (1, 90000, 8192, 1, 0),
    (150000, 61, 8192, 0, 0), (150000, 1408, 8192, 1, 1)])
def test_large_operands_keep_the_32_bit_kernel(lib, m, n, k, gated, indexed):
    from ninfer_amd.kernels.ops import _GemmArgs
    args = _GemmArgs(A=16, W=16, C=16, M=m, N=n, K=k, lda=k, ldc=n, groups=1, a_div=1, epilogue=gated)
    if indexed:
        args.offsets, args.a_index, args.w_group_stride = 16, 16, 2 * n * k
    assert lib.ninfer_gemm_kernel(ctypes.byref(args)) == 1


@pytest.mark.parametrize("m,n,k,gated,indexed,rows", [
    (40, 262143, 8192, 1, 0, 0), (40, 262200, 8192, 1, 0, 0), (40, 600000, 8192, 0, 0, 0), (600000, 512, 4096, 0, 0, 0),
    (524287, 1408, 4096, 1, 1, 256), (524288, 1408, 4096, 1, 1, 128)])
def test_large_operands_keep_the_many_row_kernel(lib, m, n, k, gated, indexed, rows):
    from ninfer_amd.kernels.ops import _GemmArgs
    args = _GemmArgs(A=16, W=16, C=16, M=m, N=n, K=k, lda=k, ldc=n, groups=1, a_div=1, epilogue=gated, in_dtype=BF16,
                     out_dtype=BF16)
    if indexed:
        args.offsets, args.a_index, args.w_group_stride = 16, 16, 2 * n * k
        assert lib.ninfer_gemm_tile_rows(ctypes.byref(args)) == rows
    assert lib.ninfer_gemm_kernel(ctypes.byref(args)) == 4


def _attention(rows, keys, n_q, n_kv, d, prompt=0, window=0, page=16, **more):
    """The arguments of `rows` single rows (and a prompt's), with the workspace that the single rows ask for."""
    from ninfer_amd.kernels.ops import _AttnArgs
    floats = rows * n_q * (-(-keys // 128)) * (d + 2)
    return _AttnArgs(q=16, kpool=16, vpool=16, out=16, block_table=16, positions=16, row_seq=16, seq_row_start=16, seq_qlen=16,
                     seq_pos0=16, workspace=16, workspace_floats=floats, q_stride=(n_q + 2 * n_kv) * d, bt_stride=999,
                     T=rows + prompt, S=rows + (prompt > 0), Hq=n_q, Hkv=n_kv, D=d, page_size=page, window=window, scale=1.0,
                     dtype=BF16, max_qlen=max(1, prompt), max_kv_len=max(keys, prompt), single_rows=rows, **more)


def _single_rows_plan(lib, a):
    got = [ctypes.c_int() for _ in range(3)]
    assert lib.ninfer_attention_decode_plan(ctypes.byref(a), *map(ctypes.byref, got)) == 0
    return [v.value for v in got]   # kernel (1 scalar, 2 grouped heads, 0 another), keys a chunk, chunks


@pytest.mark.parametrize("more", [{}, {"sink": 1}, {"gate": 16, "gate_stride": 2048}])
@pytest.mark.parametrize("prompt", [2, 1100])
def test_single_rows_beside_a_prompt_run_as_they_would_alone(lib, prompt, more):
    alone = _single_rows_plan(lib, _attention(16, 1500, 16, 4, 128, **more))
    assert alone[0] == 2 and _single_rows_plan(lib, _attention(16, 1500, 16, 4, 128, prompt, **more)) == alone


# (heads of 128 from one and a half blocks a CU on, but not in two uneven chunks nor in a window; heads of 64 from two on
# but for long contexts' smallest)
@pytest.mark.parametrize("rows,keys,n_q,n_kv,d,window,chunk", [
    (16, 1500, 16, 4, 128, 0, 256), (16, 1500, 16, 4, 128, 1500, 256), (16, 1500, 16, 4, 128, 1499, 128),
    (16, 6000, 16, 4, 128, 1024, 512), (16, 6000, 16, 4, 128, 0, 1024), (48, 1200, 16, 4, 128, 0, 512),
    (48, 1535, 16, 4, 128, 0, 512), (48, 1536, 16, 4, 128, 0, 1024), (48, 600, 28, 4, 128, 0, 256),
    (48, 300, 16, 4, 128, 0, 256), (16, 1200, 32, 8, 64, 0, 256), (48, 1200, 12, 4, 64, 0, 512),
    (64, 2600, 16, 4, 128, 1024, 1024), (3, 5000, 64, 8, 64, 0, 256), (3, 5000, 64, 8, 64, 4000, 128), (8, 2999, 32, 4, 64, 0, 128), (8, 3000, 32, 4, 64, 0, 256)])
def test_chunks_of_grouped_heads(lib, rows, keys, n_q, n_kv, d, window, chunk):
    assert _single_rows_plan(lib, _attention(rows, keys, n_q, n_kv, d, window=window)) == [2, chunk, -(-keys // chunk)]


# (prompt rows of one request after single rows of others; requests 0: that many rows of each of several)
@pytest.mark.parametrize("singles,rows,requests,keys,heads,d,vdim,window,taken", [
    (0, 173, 1, 173, 16, 128, 128, 0, 1), (0, 64, 1, 64, 16, 128, 128, 0, 0), (7, 505, 1, 2500, 16, 128, 128, 0, 1),
    (31, 2, 1, 200, 16, 128, 128, 0, 1), (63, 17, 1, 200, 16, 128, 128, 0, 0), (63, 193, 1, 200, 16, 128, 128, 0, 1),
    (63, 192, 1, 200, 16, 128, 128, 0, 0), (0, 2, 16, 66, 16, 128, 128, 0, 1), (0, 2, 16, 66, 32, 100, 100, 0, 0),
    (0, 8, 16, 110, 32, 100, 100, 0, 1), (0, 2, 8, 66, 32, 100, 100, 0, 1), (0, 2, 4, 66, 16, 64, 128, 0, 1),
    (0, 505, 1, 505, 8, 64, 64, 200, 1), (0, 255, 1, 505, 8, 64, 64, 0, 0), (0, 64, 1, 2064, 8, 64, 64, 0, 1),
    (0, 64, 1, 2064, 8, 64, 64, 200, 0), (0, 64, 1, 999, 8, 64, 64, 0, 0), (0, 8, 64, 308, 8, 64, 64, 0, 1),
    (0, 600, 1, 600, 8, 64, 64, 127, 0), (0, 100, 40, 100, 8, 64, 64, 0, 0), (1, 64, 1, 2064, 8, 64, 64, 0, 0),
    (0, 31, 1, 2064, 8, 64, 64, 0, 0), (24, 375, 1, 308, 8, 64, 64, 0, 0), (24, 376, 1, 308, 8, 64, 64, 0, 1), (0, 600, 1, 600, 16, 16, 16, 0, 0)])
def test_which_32_bit_steps_run_eight_rows_to_a_block(lib, singles, rows, requests, keys, heads, d, vdim, window, taken):
    a = _attention(singles, keys, heads, heads, d, window=window, Dv=vdim)
    a.dtype, a.T, a.S, a.max_qlen = 0, singles + rows * requests, singles + requests, rows
    assert lib.ninfer_attention_rows_f32_takes(ctypes.byref(a)) == taken


def test_attention_without_allocation_refuses_sinks_and_gates(lib):
    lib.ninfer_last_error.restype = ctypes.c_char_p
    for more in ({"sink": 1}, {"gate": 16, "gate_stride": 2048}):
        assert lib.ninfer_decode_attention_static(ctypes.byref(_attention(2, 300, 16, 4, 128, **more)), None) != 0
        assert b"sink" in lib.ninfer_last_error()


# (kernel 0: the tiles of heads. Sizes on both sides of the rule's lines, and some far from them)
@pytest.mark.parametrize("rows,keys,n_q,n_kv,d,window,page,kernel", [
    (16, 1500, 16, 4, 128, 0, 16, 2), (128, 64, 64, 8, 128, 0, 16, 0), (128, 1024, 64, 8, 128, 0, 16, 2),
    (64, 2560, 16, 4, 128, 1024, 16, 2), (64, 3584, 16, 4, 128, 1024, 16, 0), (64, 1331, 16, 4, 128, 1024, 16, 0),
    (65, 2560, 16, 4, 128, 1024, 16, 0), (4, 5000, 16, 4, 128, 1024, 16, 2), (128, 512, 16, 4, 128, 256, 16, 2),
    (16, 600, 32, 8, 64, 0, 16, 2), (32, 600, 32, 8, 64, 0, 16, 0), (32, 900, 32, 8, 64, 0, 16, 2), (64, 2600, 32, 8, 64, 0, 16, 2),
    (8, 3072, 32, 8, 64, 1024, 16, 2), (16, 3072, 32, 8, 64, 1024, 16, 0), (16, 600, 32, 8, 64, 256, 16, 2),
    (4, 1000, 32, 8, 64, 0, 4, 0), (64, 600, 8, 8, 64, 0, 16, 1), (128, 600, 8, 8, 64, 0, 16, 0),
    (128, 600, 8, 8, 128, 0, 16, 1), (32, 600, 16, 8, 128, 0, 16, 1), (128, 600, 16, 8, 128, 0, 16, 0),
    (1, 12000, 16, 8, 64, 0, 16, 1), (8, 12000, 16, 8, 64, 0, 16, 0), (32, 2048, 8, 8, 64, 1024, 16, 1),
    (32, 16384, 8, 8, 64, 1024, 16, 0), (4, 1900, 16, 16, 32, 1024, 16, 1), (8, 1900, 16, 16, 32, 1024, 16, 0),
    (8, 4000, 8, 8, 16, 1024, 16, 0), (64, 8192, 8, 8, 16, 4096, 16, 1), (16, 100, 32, 8, 64, 0, 16, 2), (16, 99, 32, 8, 64, 0, 16, 0), (8, 3584, 8, 8, 16, 1024, 16, 1), (4, 4000, 24, 2, 32, 0, 16, 0),
    (4, 4000, 8, 4, 32, 0, 16, 0), (4, 64, 8, 1, 256, 0, 16, 0), (4, 65, 8, 1, 256, 0, 16, 1), (1, 300, 64, 1, 128, 0, 16, 0)])
@pytest.mark.parametrize("more", [{"sink": 1}, {"gate": 16}])
def test_which_rows_with_a_sink_or_a_gate_are_split(lib, rows, keys, n_q, n_kv, d, window, page, kernel, more):
    more = dict(more, gate_stride=n_q * d) if "gate" in more else more
    a = _attention(rows, keys, n_q, n_kv, d, window=window, page=page, **more)
    assert _single_rows_plan(lib, a)[0] == kernel
    plain = _attention(rows, keys, n_q, n_kv, d, window=window, page=page)
    assert _single_rows_plan(lib, plain)[0] != 0   # (plain layers' always are)


# (prompts of their own, portions behind cached keys and decode steps; both heights of blocks measured)
@pytest.mark.parametrize("rank,rd,heads,requests,new,keys,rows", [
    (256, 32, 40, 1, 200, 200, 16), (512, 64, 16, 1, 300, 300, 16), (256, 32, 24, 1, 300, 300, 16),
    (512, 64, 16, 1, 400, 400, 16), (512, 64, 8, 1, 700, 700, 16), (512, 64, 16, 1, 512, 512, 64),
    (512, 64, 24, 1, 400, 400, 64), (256, 32, 40, 1, 300, 300, 64), (512, 64, 16, 1, 2048, 2048, 64),
    (512, 64, 16, 1, 512, 2512, 64), (512, 64, 8, 8, 505, 701, 64), (512, 64, 40, 64, 1, 2500, 64),
    (512, 64, 40, 64, 1, 300, 16), (512, 64, 16, 1, 1, 4000, 16)])
def test_height_of_latent_blocks(lib, rank, rd, heads, requests, new, keys, rows):
    from ninfer_amd.kernels.ops import _LatentArgs
    t = requests if new == 1 else new + requests - 1   # (one portion, the others single rows)
    a = _LatentArgs(pool=16, q_abs=16, out=16, seq_row_start=16, seq_pos0=16, S=requests, T=t, Hq=heads, R=rank, rd=rd,
                    max_kv_len=keys, max_qlen=new, page_size=16, dtype=BF16)
    assert lib.ninfer_latent_attention_block_rows(ctypes.byref(a)) == rows


@pytest.mark.parametrize("rows,keys,heads", [(1, 2600, 40), (40, 2040, 16), (300, 800, 16), (300, 300, 24), (1100, 2100, 16)])
def test_latent_workspace_by_the_sizes_alone(lib, rows, keys, heads):
    """What a step of latent attention asks for does not depend on where its output lies."""
    from ninfer_amd.kernels.ops import _LatentArgs
    lib.ninfer_latent_attention_workspace_floats.restype = ctypes.c_longlong
    plans = set()
    for out in (0, 16, 18):
        a = _LatentArgs(pool=16, q_abs=16, out=out, seq_row_start=16, seq_pos0=16, S=1, T=rows, Hq=heads, R=512, rd=64,
                        max_kv_len=keys, max_qlen=rows, page_size=16, dtype=BF16)
        plans.add((lib.ninfer_latent_attention_workspace_floats(ctypes.byref(a)),
                   lib.ninfer_latent_attention_block_rows(ctypes.byref(a))))
    assert len(plans) == 1


def test_no_block_reads_behind_a_tile_list(lib):
    """The lists hold min(n, n // 16 + experts) and n // 256 + experts tiles of n sorted rows; a launch rounds its
    block rows up and may have more."""
    from ninfer_amd.kernels.ops import _GemmArgs
    for groups in (1, 2, 7, 60, 64, 130):
        for n in list(range(1, 70)) + [100, 255, 256, 257, 1025, 1279, 1280, 4095, 8192]:
            args = _GemmArgs(M=n, N=64, K=64, groups=groups, offsets=16)
            assert lib.ninfer_gemm_last_list_entry(ctypes.byref(args), 0) < min(n, n // 16 + groups), (groups, n)
            assert lib.ninfer_gemm_last_list_entry(ctypes.byref(args), 1) < n // 256 + groups, (groups, n)


def test_a_products_arguments_have_one_size(lib, monkeypatch):
    """The bindings' layout against the library's, compared when the library is loaded."""
    from ninfer_amd.kernels import ops
    assert lib.ninfer_gemm_args_bytes() == ctypes.sizeof(ops._GemmArgs)

    class Longer(ops._GemmArgs):
        _fields_ = [("one_more", ctypes.c_int64)]
    monkeypatch.setattr(ops, "_GemmArgs", Longer)
    with pytest.raises(ops.KernelError, match="lay a product's arguments out differently"):
        ops.HipOps()


# (rows and cached keys, these included, of each portion behind the single rows; does the step form keys and values?)
@pytest.mark.parametrize("heads,rank,rd,vdim,singles,portions,taken", [
    (16, 512, 64, 128, 0, [(2048, 2048)], True), (8, 256, 32, 64, 0, [(2, 2)], True), (16, 512, 64, 128, 0, [(2, 512)], True),
    (16, 512, 64, 128, 0, [(2, 513)], False), (16, 512, 64, 128, 0, [(64, 1024)], True), (16, 512, 64, 128, 0, [(64, 1025)], False),
    (16, 512, 64, 128, 0, [(2048, 16384)], True), (16, 512, 64, 128, 0, [(2048, 16385)], False),
    (16, 512, 64, 128, 0, [(1000, 1000)] + [(2, 502)] * 30, True), (32, 512, 64, 128, 0, [(1000, 1000)] + [(2, 502)] * 30, False),
    (32, 512, 64, 128, 0, [(4, 44)] * 100, False), (32, 512, 64, 128, 0, [(8, 48)] * 60, True), (32, 512, 64, 128, 0, [(2, 32)] * 16, True),
    (16, 512, 64, 128, 1, [(256, 256)], True), (16, 512, 64, 128, 1, [(255, 255)], False), (8, 256, 32, 64, 1, [(511, 511)], False),
    (8, 256, 32, 64, 1, [(512, 512)], True), (16, 512, 64, 128, 32, [(512, 512)], True), (16, 512, 64, 128, 33, [(512, 512)], False),
    (16, 512, 64, 128, 5, [], False), (16, 512, 64, 96, 0, [(64, 64)], False), (16, 512, 32, 128, 0, [(64, 64)], True),
    (16, 512, 0, 128, 0, [(64, 64)], False), (3, 72, 64, 128, 0, [(64, 64)], True), (3, 68, 64, 128, 0, [(64, 64)], False)])
def test_which_prompts_form_keys_and_values_per_head(lib, heads, rank, rd, vdim, singles, portions, taken):
    import torch
    from types import SimpleNamespace
    from ninfer_amd.kernels.ops import HipOps
    rows, keys = sum(r for r, _ in portions), sum(k for _, k in portions)
    ctx = SimpleNamespace(T=singles + rows, S=singles + len(portions), single_rows=singles, portion_keys=keys,
                          act_dtype=torch.bfloat16)
    ops = SimpleNamespace(lib=lib, force_generic=False, conv_pieces_always=False)
    first = lambda **kw: HipOps.latent_heads_rows(SimpleNamespace(**{**vars(ops), **kw}), ctx, heads, 128 - rd, rank, rd, vdim, None)
    assert first() == (singles if taken else ctx.T)
    assert first(force_generic=True) == ctx.T
    assert HipOps.latent_heads_rows(ops, ctx, heads, 128 - rd, rank, rd, vdim, 4096) == ctx.T
    ctx.act_dtype = torch.float32
    assert first() == ctx.T


# (experts, inner, shared inner of width 2,048; bytes a number)
@pytest.mark.parametrize("sizes,size,rows,two", [
    ((60, 1408, 5632), 2, 128, False), ((60, 1408, 5632), 2, 160, True), ((60, 1408, 5632), 4, 16, False), ((60, 1408, 5632), 4, 17, True),
    ((32, 1408, 2816), 2, 384, False), ((32, 1408, 2816), 2, 420, True), ((60, 1408, 5632), 4, 100, True), ((60, 1408, 5632), 4, 101, False), ((32, 1408, 2816), 4, 30, False),
    ((16, 704, 1408), 4, 500, False), ((60, 7040, 28160), 2, 64, False), ((60, 7040, 28160), 2, 65, True)])
def test_which_short_steps_take_two_streams(sizes, size, rows, two):
    import torch
    from types import SimpleNamespace
    from ninfer_amd.kernels.ops import HipOps
    experts, inner, shared = sizes
    weights = 3 * 2048 * (experts * inner + shared) * size
    assert HipOps.pays_beside(SimpleNamespace(), rows, weights, torch.bfloat16 if size == 2 else torch.float32) == two


@pytest.mark.parametrize("min_rows,rows,capturing,two", [(512, 17, False, True), (512, 2048, False, True), (1 << 30, 2048, False, False),
                                                         (1 << 30, 65, False, False), (512, 160, True, False), (1, 1, False, True)])
def test_one_stream_when_it_is_asked_for(monkeypatch, min_rows, rows, capturing, two):
    import torch
    from types import SimpleNamespace
    from ninfer_amd.kernels.ops import HipOps
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
    ops = SimpleNamespace(beside_min_rows=min_rows, pays_beside=lambda *a: True)
    assert HipOps.wants_beside_short(ops, rows, 1 << 40, torch.float32) == two
    ops.pays_beside = lambda *a: False
    assert not HipOps.wants_beside_short(ops, rows, 1 << 40, torch.float32)


# (experts and their inner size, the shared expert's, width 2,048)
@pytest.mark.parametrize("experts,inner,shared,two", [(60, 1408, 5632, True), (16, 7168, 7168, True), (31, 2048, 2048, True),
                                                      (32, 2048, 2048, False), (64, 2048, 2048, False), (128, 1024, 1024, False)])
def test_a_shared_expert_of_little_work_stays_on_the_stream(monkeypatch, experts, inner, shared, two):
    import torch
    from types import SimpleNamespace
    from ninfer_amd.kernels.ops import HipOps
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    ops = SimpleNamespace(beside_min_rows=512, pays_beside=lambda *a: True)
    own = 3 * 2048 * shared * 2
    assert HipOps.wants_beside_short(ops, 128, 3 * 2048 * experts * inner * 2 + own, torch.bfloat16, own) == two


def test_the_bindings_say_how_many_tokens_a_sampled_row_may_keep(lib, monkeypatch):
    from ninfer_amd.kernels.ops import HipOps, KernelError
    assert lib.ninfer_sample_few_tokens() == HipOps.FEW_TOKENS
    monkeypatch.setattr(HipOps, "FEW_TOKENS", 64)
    with pytest.raises(KernelError, match="whole GPU"):
        HipOps()
