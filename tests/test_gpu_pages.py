"""GPU: K/V written into pages by the register-resident quantizers, bit for bit against the oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import flashspec_amd as fa
from flashspec_amd import _lib
from oracle import paged as op
from oracle import quant as oq

from _helpers import assert_quant_equal, from_qt, np_of, randn

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def announce(msg: str) -> None:
    print(f"[case] {msg}", flush=True)


def shifted(x: torch.Tensor) -> torch.Tensor:
    """The same values at an address that is no multiple of 16 bytes."""

    base = torch.empty(x.numel() + 1, dtype=x.dtype, device=DEV)
    base[1:] = x.reshape(-1).to(DEV)
    return base[1:].reshape(x.shape)


# groups of page * D values: 512 multiples (1, 4, 8 chunks), partial chunks (D 80, 96, 112, 24: 2.5,
# 3, 3.5 and under one), 5 and 7 chunks (run as 6 and 8), over 8 chunks and D no multiple of 8
# (element-wise); lengths of one token, whole pages and ragged; 898 pages take two launches
@pytest.mark.parametrize("heads,dim,page,length,dtype", [
    (3, 32, 16, 1, torch.float16),
    (4, 128, 16, 301, torch.float16),
    (2, 256, 16, 32, torch.float32),
    (5, 80, 16, 83, torch.bfloat16),
    (2, 96, 16, 47, torch.float32),
    (2, 112, 16, 65, torch.float16),
    (3, 24, 16, 50, torch.bfloat16),
    (2, 160, 16, 33, torch.float16),
    (2, 224, 16, 40, torch.bfloat16),
    (2, 80, 32, 70, torch.float16),
    (2, 256, 32, 70, torch.float16),
    (2, 36, 16, 35, torch.float16),
    (1, 8, 16, 897 * 16 + 5, torch.float16),
])
def test_prompt_pages_bit_exact(heads, dim, page, length, dtype):
    announce(f"add_request H{heads} D{dim} page{page} L{length} {dtype}")
    pages = -(-length // page)
    alloc = fa.PagedKVAllocator(capacity_blocks=pages + 4, heads=heads, head_dim=dim, block_size=page, device=DEV)
    ora = op.OracleAllocator(pages + 4, heads, dim, page)
    for rid, n in ((0, page), (1, page + 1), (2, 1)):
        k, v = randn((1, heads, n, dim), 10 + rid, dtype), randn((1, heads, n, dim), 20 + rid, dtype)
        alloc.add_request(rid, k.to(DEV), v.to(DEV))
        ora.add_request(rid, np_of(k.float()), np_of(v.float()))
    for a in (alloc, ora):  # the prompt takes the pages in front of request 2 and those behind it
        a.release_request(1)
        a.release_request(0)
    # three rows more than the request keeps
    k, v = randn((1, heads, length + 3, dim), 1, dtype) * 3.0, randn((1, heads, length + 3, dim), 2, dtype)
    alloc.add_request(7, k.to(DEV), v.to(DEV), length=length)
    ora.add_request(7, np_of(k[:, :, :length].float()), np_of(v[:, :, :length].float()))
    torch.cuda.synchronize()
    assert_quant_equal(from_qt(alloc.k_quant), ora.k_quant, "k")
    assert_quant_equal(from_qt(alloc.v_quant), ora.v_quant, "v")


def test_prompt_of_two_dtypes_and_unaligned_sources():
    announce("add_request fp16 K and fp32 V; 2-byte-offset sources")
    heads, dim, page, length = 2, 128, 16, 39
    k, v = randn((1, heads, length, dim), 3), randn((1, heads, length, dim), 4, torch.float32)
    ora = op.OracleAllocator(6, heads, dim, page)
    ora.add_request(0, np_of(k.float()), np_of(v))
    ora.add_request(1, np_of(k.float()), np_of(k.float()))
    alloc = fa.PagedKVAllocator(capacity_blocks=6, heads=heads, head_dim=dim, block_size=page, device=DEV)
    alloc.add_request(0, k.to(DEV), v.to(DEV))
    alloc.add_request(1, shifted(k), shifted(k))
    torch.cuda.synchronize()
    assert_quant_equal(from_qt(alloc.k_quant), ora.k_quant, "k")
    assert_quant_equal(from_qt(alloc.v_quant), ora.v_quant, "v")


@pytest.mark.parametrize("dim,block,seq,dtype", [
    (80, 16, 33, torch.float16),
    (96, 16, 48, torch.bfloat16),
    (24, 8, 21, torch.float32),
    (160, 16, 20, torch.float16),
    (224, 16, 17, torch.float32),
])
def test_partial_chunks_bit_exact(dim, block, seq, dtype):
    """Groups that are no multiple of 512 values, extreme values among them."""

    announce(f"quantize blocks and pages D{dim} block{block} S{seq} {dtype}")
    x = randn((2, 3, seq, dim), dim + seq, dtype) * 2.0
    x[0, 0, 1, 1], x[1, 2, seq - 1, dim - 1] = 60000.0, -60000.0
    x[1] += 100.0  # ranges without zero: a repeated value must not widen them
    ref = oq.quantize_int8_per_block(np_of(x.float()), block)
    got = fa.quantize_int8_per_block(x.to(DEV), block)
    cache = fa.PagedKVCache.from_dense(x.to(DEV), x.to(DEV), block, block_table_pattern="shuffled", layout_seed=1)
    torch.cuda.synchronize()
    assert_quant_equal(from_qt(got), ref, "blocks")
    table = cache.block_table.cpu().numpy()
    for b in range(2):
        for i in range(table.shape[1]):
            assert np.array_equal(np_of(cache.k_quant.values)[table[b, i], :, 0], ref.values[b, :, i])
            assert np.array_equal(np_of(cache.k_quant.scale)[table[b, i]].reshape(-1).view(np.uint32),
                                  ref.scale[b, :, i].reshape(-1).view(np.uint32))


def extreme(dtype: torch.dtype, dim: int) -> torch.Tensor:
    """Blocks of 16 rows with infinities, NaN, both zeros, the type's largest and tiny values."""

    x = randn((10, 1, 16, dim), 5, dtype)
    big = torch.finfo(dtype).max
    x[0, 0, 3, 7] = float("inf")
    x[1, 0, 3, 7] = float("-inf")
    x[2, 0, 3, 7], x[2, 0, 4, 8] = float("inf"), float("-inf")
    x[3, 0, 3, 7] = float("nan")
    x[4] = float("nan")
    x[5, 0, 0, 0], x[5, 0, 1, 0] = big, -big  # a range past fp32 in fp32 and bf16
    x[6] = 0.0
    x[7] = -0.0
    x[8] *= torch.finfo(dtype).tiny
    x[9] = big
    return x


def assert_same_store(a: fa.QuantizedTensor, b: fa.QuantizedTensor, what: str) -> None:
    assert a.block_size == b.block_size and a.original_shape == b.original_shape and a.values.dtype == b.values.dtype
    assert a.values.shape == b.values.shape and a.scale.shape == b.scale.shape, what
    assert torch.equal(a.values.cpu().view(torch.uint8), b.values.cpu().view(torch.uint8)), what
    assert torch.equal(a.scale.cpu().view(torch.int32), b.scale.cpu().view(torch.int32)), what
    assert torch.equal(a.zero_point.cpu(), b.zero_point.cpu()), what


FORMATS = ["affine_block", "fp8_block", "affine_channel", "symmetric_token"]


# chunks of 512 values (block, FP8) or of whole rows (channel, token): 1, 2, 3 (partial), 4, 6, 8 and
# 16 chunks, rows of 1, 2, 4, 8, 10, 12, 16, 28 and 32 lanes, head dims and groups that take the
# element-wise kernel (36, 528; 64-row pages of 256 dims), a last page of one row
@pytest.mark.parametrize("kv_format", FORMATS)
@pytest.mark.parametrize("dim,page,seq,dtype", [
    (8, 16, 17, torch.float16),
    (16, 8, 30, torch.float32),
    (32, 16, 64, torch.bfloat16),
    (64, 16, 49, torch.float16),
    (80, 16, 33, torch.bfloat16),
    (96, 32, 70, torch.float16),
    (128, 16, 301, torch.bfloat16),
    (128, 64, 130, torch.float16),
    (224, 16, 40, torch.float16),
    (256, 16, 48, torch.float32),
    (256, 32, 65, torch.bfloat16),
    (256, 64, 70, torch.float16),
    (36, 16, 35, torch.float16),
    (528, 4, 9, torch.float32),
])
def test_build_matches_the_portable_path_bit_exact(kv_format, dim, page, seq, dtype):
    announce(f"from_dense {kv_format} D{dim} page{page} S{seq} {dtype}")
    k, v = randn((3, 2, seq, dim), 1, dtype) * 2.0, randn((3, 2, seq, dim), 2, dtype) + 3.0
    ref = fa.PagedKVCache.from_dense(k, v, page, block_table_pattern="interleaved", kv_format=kv_format)
    # K aligned, V at an address that takes the element-wise kernel
    got = fa.PagedKVCache.from_dense(k.to(DEV), shifted(v), page, block_table_pattern="interleaved",
                                     kv_format=kv_format)
    both = fa.PagedKVCache.from_dense(k.to(DEV), v.to(DEV), page, block_table_pattern="interleaved",
                                      kv_format=kv_format)
    torch.cuda.synchronize()
    for cache in (got, both):
        assert torch.equal(cache.block_table.cpu(), ref.block_table)
        assert_same_store(cache.k_quant, ref.k_quant, "k")
        assert_same_store(cache.v_quant, ref.v_quant, "v")


@pytest.mark.parametrize("pattern", ["contiguous", "interleaved", "shuffled"])
@pytest.mark.parametrize("batch,seq,dim", [(1, 16, 128), (5, 33, 128), (3, 50, 36)])
def test_build_writes_table_and_lengths(pattern, batch, seq, dim):
    """Both page kernels place the pages, write the table and, without given lengths, the lengths."""

    announce(f"from_dense table and lengths {pattern} B{batch} S{seq} D{dim}")
    k, v = randn((batch, 2, seq, dim), 1), randn((batch, 2, seq, dim), 2, torch.float32)  # two dtypes
    got = fa.PagedKVCache.from_dense(k.to(DEV), v.to(DEV), 16, block_table_pattern=pattern, layout_seed=3)
    given = fa.PagedKVCache.from_dense(k.to(DEV), v.to(DEV), 16, block_table_pattern=pattern, layout_seed=3,
                                       lengths=torch.arange(1, batch + 1, device=DEV))
    torch.cuda.synchronize()
    n = batch * -(-seq // 16)
    if pattern == "shuffled":
        g = torch.Generator(device=DEV)
        g.manual_seed(3)
        want = torch.argsort(torch.randperm(n, generator=g, device=DEV)).cpu().reshape(batch, -1)
    else:
        want = fa.PagedKVCache.from_dense(k, v, 16, block_table_pattern=pattern).block_table
    assert torch.equal(got.block_table.cpu(), want) and torch.equal(given.block_table.cpu(), want)
    assert got.lengths.tolist() == [seq] * batch and given.lengths.tolist() == list(range(1, batch + 1))
    for quant, x in ((got.k_quant, k), (got.v_quant, v)):
        ref = fa.quantize_int8_per_block(x, 16)
        assert torch.equal(quant.values.cpu()[want][:, :, :, 0], ref.values.permute(0, 2, 1, 3, 4))
        assert torch.equal(quant.scale.cpu()[want].reshape(batch, -1, 2), ref.scale[..., 0, 0].permute(0, 2, 1))


@pytest.mark.parametrize("kv_format", FORMATS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim", [80, 128])
def test_extreme_values_match_the_general_path_in_every_format(kv_format, dtype, dim):
    announce(f"extreme values, both page quantizers, {kv_format} {dtype} D{dim}")
    x = extreme(dtype, dim)
    a = fa.PagedKVCache.from_dense(x.to(DEV), x.to(DEV), 16, kv_format=kv_format)
    b = fa.PagedKVCache.from_dense(shifted(x), shifted(x), 16, kv_format=kv_format)
    torch.cuda.synchronize()
    assert_same_store(a.k_quant, b.k_quant, "aligned against unaligned")


@pytest.mark.parametrize("quantize", [fa.quantize_fp8_per_block, fa.quantize_int8_per_channel])
@pytest.mark.parametrize("dim,block,seq,dtype", [(80, 16, 33, torch.float16), (128, 16, 300, torch.bfloat16),
                                                 (256, 32, 40, torch.float32), (64, 8, 21, torch.float16)])
def test_block_formats_match_the_portable_path_bit_exact(quantize, dim, block, seq, dtype):
    announce(f"{quantize.__name__} D{dim} block{block} S{seq} {dtype}")
    x = randn((2, 3, seq, dim), 4, dtype) * 2.0
    got, ref = quantize(x.to(DEV), block), quantize(x, block)
    torch.cuda.synchronize()
    assert_same_store(got, ref, "blocks")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_infinities_nan_and_scratch_ranges_match_the_general_path(dtype):
    """Aligned sources take the register-resident kernel, unaligned ones the element-wise kernel."""

    announce(f"extreme values, both quantizers, {dtype}")
    x = extreme(dtype, 80)
    a, b = fa.quantize_int8_per_block(x.to(DEV), 16), fa.quantize_int8_per_block(shifted(x), 16)
    torch.cuda.synchronize()
    assert torch.equal(a.values, b.values)
    assert torch.equal(a.scale.view(torch.int32), b.scale.view(torch.int32))
    assert torch.equal(a.zero_point, b.zero_point)


# 4 values a lane (D 128, 36, 256, 24) and one (34, 7); pages of one wave, of several (D 256, 64 rows)
# and of a part; whole and cut last pages; more table columns than tokens; -1 entries
@pytest.mark.parametrize("kv_format", FORMATS)
@pytest.mark.parametrize("heads,dim,page,seq,table_dtype", [
    (2, 128, 16, 300, torch.int64),
    (3, 36, 16, 33, torch.int32),
    (2, 256, 64, 130, torch.int64),
    (2, 24, 8, 64, torch.int32),
    (2, 34, 16, 40, torch.int64),
    (1, 7, 4, 10, torch.int64),
])
def test_to_dense_matches_the_portable_path(kv_format, heads, dim, page, seq, table_dtype):
    announce(f"to_dense {kv_format} H{heads} D{dim} page{page} S{seq} {table_dtype}")
    k, v = randn((3, heads, seq, dim), 1) * 2.0, randn((3, heads, seq, dim), 2)
    ref = fa.PagedKVCache.from_dense(k, v, page, block_table_pattern="interleaved", kv_format=kv_format)
    table = ref.block_table.clone()
    table[1, -1] = -1
    table = torch.cat([table, torch.full((3, 1), -1)], dim=1)
    for span in (seq, seq - 3, (table.shape[1] - 1) * page + 1, 10 * table.shape[1] * page):
        want = fa.PagedKVCache(ref.k_quant, ref.v_quant, table, ref.lengths, page, span).to_dense()

        def moved(q):
            return fa.QuantizedTensor(q.values.to(DEV), q.scale.to(DEV), q.zero_point.to(DEV), q.block_size,
                                      q.original_shape)

        got = fa.PagedKVCache(moved(ref.k_quant), moved(ref.v_quant), table.to(DEV, table_dtype),
                              ref.lengths.to(DEV), page, span).to_dense()
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert a.dtype == torch.float32 and a.shape == b.shape
            assert torch.equal(a.cpu().view(torch.int32), b.contiguous().view(torch.int32))


def test_to_dense_of_stores_that_differ_and_of_quant_blocks_in_a_page():
    announce("to_dense: INT8 K with 8-token blocks, FP8 V, page 20 over 16-token blocks")
    x = randn((6, 2, 32, 64), 3)
    table = torch.tensor([[5, 0, 3], [1, 2, 4]])
    k, v = fa.quantize_int8_per_block(x, 8), fa.quantize_fp8_per_block(x, 32)
    y = randn((6, 2, 20, 64), 4)
    short = fa.quantize_int8_per_block(y, 16)  # two blocks of 16 hold a page of 20
    for kq, vq, page in ((k, v, 32), (short, short, 20)):
        want = fa.PagedKVCache(kq, vq, table, torch.tensor([70, 60]), page, 3 * page - 7).to_dense()
        on = [fa.QuantizedTensor(q.values.to(DEV), q.scale.to(DEV), q.zero_point.to(DEV), q.block_size,
                                 q.original_shape) for q in (kq, vq)]
        got = fa.PagedKVCache(on[0], on[1], table.to(DEV), torch.tensor([70, 60], device=DEV), page,
                              3 * page - 7).to_dense()
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a.cpu(), b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim,block,seq", [(128, 16, 301), (34, 8, 21), (3000, 4, 9)])
def test_dequantize_matches_the_portable_path(dtype, dim, block, seq):
    announce(f"dequantize D{dim} block{block} S{seq} {dtype}")
    x = randn((2, 3, seq, dim), 5)
    for quantize in (fa.quantize_int8_per_block, fa.quantize_fp8_per_block):
        q = quantize(x, block)
        on = fa.QuantizedTensor(q.values.to(DEV), q.scale.to(DEV), q.zero_point.to(DEV), block, q.original_shape)
        got, want = fa.dequantize_int8_per_block(on, dtype), fa.dequantize_int8_per_block(q, dtype)
        torch.cuda.synchronize()
        assert torch.equal(got.cpu(), want)


# the C entries that quantize one tensor, which the package itself reaches through fs_build_cache only
@pytest.mark.parametrize("entry,kv_format", [("fs_quantize_pages_i8", "affine_block"),
                                             ("fs_quantize_pages_fp8", "fp8_block"),
                                             ("fs_quantize_pages_i8_channel", "affine_channel")])
@pytest.mark.parametrize("dim", [128, 36])
def test_page_quantizers_of_the_c_interface_match_a_built_cache(entry, kv_format, dim):
    announce(f"{entry} D{dim}")
    x = randn((3, 2, 50, dim), 6, torch.float16).to(DEV)
    cache = fa.PagedKVCache.from_dense(x, x, 16, block_table_pattern="shuffled", layout_seed=5, kv_format=kv_format)
    want = cache.k_quant
    out = [torch.empty_like(t) for t in (want.values, want.scale, want.zero_point)]
    src = torch.empty(12, dtype=torch.int64, device=DEV)
    src[cache.block_table.reshape(-1)] = torch.arange(12, device=DEV)
    _lib.check(getattr(_lib.require(), entry)(x.data_ptr(), _lib.dtype_code(x.dtype), 3, 2, 50, dim, 16, src.data_ptr(), 12,
                                              *(t.data_ptr() for t in out), _lib.stream_ptr(DEV)))
    assert_same_store(fa.QuantizedTensor(*out, want.block_size, want.original_shape), want, entry)


def test_page_update_of_fresh_pages_ignores_what_they_held():
    announce("fs_update_pages_i8 with fresh pages")
    heads, page, dim = 2, 16, 32
    old = fa.quantize_int8_per_block(randn((4, heads, page, dim), 7).to(DEV), page)
    new = randn((1, heads, 3, dim), 8, torch.float16).to(DEV)
    out = [t.clone() for t in (old.values, old.scale, old.zero_point)]
    pages = torch.tensor([3, 1], device=DEV)
    fresh = torch.tensor([1, 0], dtype=torch.uint8, device=DEV)
    rows = torch.full((2, page), -1, dtype=torch.int32)
    rows[0, :2], rows[1, 5] = torch.tensor([0, 1]), 2
    held = fa.dequantize_int8_per_block(old).cpu().reshape(4, heads, page, dim)
    held[3] = 0
    held[3, :, :2], held[1, :, 5] = new[0, :, :2].float().cpu(), new[0, :, 2].float().cpu()
    rows = rows.to(DEV)
    _lib.check(_lib.require().fs_update_pages_i8(
        *(t.data_ptr() for t in out), 4, page, *(t.data_ptr() for t in out), pages.data_ptr(), fresh.data_ptr(), 2,
        rows.data_ptr(), new.data_ptr(), _lib.dtype_code(new.dtype), 3, heads, page, dim, _lib.stream_ptr(DEV)))
    want = fa.quantize_int8_per_block(held, page)
    for name, got, had, w in zip(("values", "scale", "zero"), out, (old.values, old.scale, old.zero_point),
                                 (want.values, want.scale, want.zero_point)):
        assert torch.equal(got[[0, 2]], had[[0, 2]]), name
        assert torch.equal(got[[1, 3]].cpu(), w[[1, 3]]), name


# a launch holds 2^26 - 4 groups of one wave: K's 40 million end inside the first, V's pass into a second
LAUNCH_GROUPS = 4 * (2 ** 24 - 1)


def windows(n: int, *marks: int):
    return [(max(0, m - 40), min(n, m + 40)) for m in (0, *marks, n)]


@pytest.mark.parametrize("kv_format", ["affine_block", "fp8_block"])
def test_more_groups_than_one_launch_holds(kv_format):
    n, dim = 40_000_000, 8
    assert n < LAUNCH_GROUPS < 2 * n
    announce(f"from_dense and to_dense of {n} one-token pages, {kv_format}")
    g = torch.Generator(device=DEV).manual_seed(3)
    k, v = (torch.randn((1, 1, n, dim), generator=g, device=DEV, dtype=torch.float16) for _ in range(2))
    for x in (k, v):
        x[..., 0] = 0  # a group's range holds 0, so that nothing is clipped
    cache = fa.PagedKVCache.from_dense(k, v, 1, kv_format=kv_format)
    dense = cache.to_dense()
    quantize = fa.quantize_int8_per_block if kv_format == "affine_block" else fa.quantize_fp8_per_block
    for name, x, q, d in (("k", k, cache.k_quant, dense[0]), ("v", v, cache.v_quant, dense[1])):
        for a, b in windows(n, LAUNCH_GROUPS % n):
            want = quantize(x[:, :, a:b].cpu(), 1)
            assert torch.equal(q.values[a:b].reshape(-1, dim).cpu().view(torch.uint8),
                               want.values.reshape(-1, dim).view(torch.uint8)), (name, a)
            assert torch.equal(q.scale[a:b].reshape(-1).cpu(), want.scale.reshape(-1)), (name, a)
            assert torch.equal(d[:, :, a:b].cpu(), fa.dequantize_int8_per_block(want)), (name, a)
        # every page of both ranges was written and read: FP8 is off by at most 448 / 16 scales, INT8 by one (half
        # by rounding, half where the rounded zero point clips an end)
        step = q.scale.reshape(1, 1, n, 1) * (32.0 if kv_format == "fp8_block" else 1.01)
        assert bool(((d - x.float()).abs() <= step).all()), name
    ids = torch.arange(n, device=DEV)
    assert torch.equal(cache.block_table.reshape(-1), ids)


def test_block_quantizer_of_more_groups_than_one_launch_holds():
    n, dim = LAUNCH_GROUPS + 5, 8
    announce(f"quantize_int8_per_block of {n} one-token blocks")
    x = torch.randn((n, dim), generator=torch.Generator(device=DEV).manual_seed(4), device=DEV, dtype=torch.float16)
    x[:, 0] = 0  # as above
    q = fa.quantize_int8_per_block(x, 1)
    back = fa.dequantize_int8_per_block(q, dtype=torch.float16)
    for a, b in windows(n, LAUNCH_GROUPS):
        want = fa.quantize_int8_per_block(x[a:b].cpu(), 1)
        assert torch.equal(q.values[a:b].cpu(), want.values) and torch.equal(q.scale[a:b].cpu(), want.scale), a
        assert torch.equal(back[a:b].cpu(), fa.dequantize_int8_per_block(want, dtype=torch.float16)), a
    # one step of the block plus the half-precision rounding of a value under 8 (2^-9 of it at most)
    assert bool(((back - x).abs().float() <= 1.01 * q.scale.reshape(n, 1) + 2.0 ** -8).all())
    announce(f"fs_update_pages_i8 of {n} one-token pages")
    out = [torch.empty_like(t) for t in (q.values, q.scale, q.zero_point)]
    rows = torch.arange(n, dtype=torch.int32, device=DEV)
    _lib.check(_lib.require().fs_update_pages_i8(
        None, None, None, 0, 1, *(t.data_ptr() for t in out), None, None, n, rows.data_ptr(), x.data_ptr(),
        _lib.dtype_code(x.dtype), n, 1, 1, dim, _lib.stream_ptr(DEV)))
    for got, want in zip(out, (q.values, q.scale, q.zero_point)):
        assert torch.equal(got, want)


def test_to_dense_of_more_rows_than_32_bits_count():
    n, pages = 2 ** 30 + 7, 1000  # K and V: 2^31 + 14 rows of one value, each its own wave
    announce(f"to_dense of {n} one-token pages of one value")
    g = torch.Generator(device=DEV).manual_seed(6)
    k, v = (fa.quantize_int8_per_block(torch.randn((pages, 1, 1, 1), generator=g, device=DEV), 1) for _ in range(2))
    table = torch.randint(0, pages, (1, n), generator=g, device=DEV, dtype=torch.int32)
    lengths = torch.tensor([n], device=DEV)
    dense = fa.PagedKVCache(k, v, table, lengths, 1, n).to_dense()
    for q, d in zip((k, v), dense):
        assert d.shape == (1, 1, n, 1)
        page = fa.dequantize_int8_per_block(q).reshape(pages)
        for at in range(0, n, 1 << 27):
            assert torch.equal(d[0, 0, at:at + (1 << 27), 0], page[table[0, at:at + (1 << 27)].long()]), at


def test_token_quantizer_of_more_rows_than_one_launch_holds():
    n, dim = LAUNCH_GROUPS + 5, 4  # a wave per row
    announce(f"quantize_int8_symmetric_per_token of {n} rows")
    x = torch.randn((n, dim), generator=torch.Generator(device=DEV).manual_seed(5), device=DEV, dtype=torch.float16)
    q = fa.quantize_int8_symmetric_per_token(x)
    for a, b in windows(n, LAUNCH_GROUPS):
        want = fa.quantize_int8_symmetric_per_token(x[a:b].cpu())
        assert torch.equal(q.values[a:b].cpu(), want.values) and torch.equal(q.scale[a:b].cpu(), want.scale), a
    back = q.values.reshape(n, dim) * q.scale.reshape(n, 1)
    assert bool(((back - x.float()).abs() <= 0.51 * q.scale.reshape(n, 1)).all())
    assert bool((q.zero_point == 128).all())


def test_prompt_entry_rejects_bad_sizes():
    lib = _lib.require()
    ids = (np.zeros(4, dtype=np.int32)).ctypes.data
    bad = [  # length past the source, page count, head_dim, dtype, null pages
        (1, 1, 1, 8, 9, 2, 64, 16, 1, 1, 1, 1, 1, 1, 4, ids, 1, None),
        (1, 1, 1, 8, 8, 2, 64, 16, 1, 1, 1, 1, 1, 1, 4, ids, 2, None),
        (1, 1, 1, 8, 8, 2, 0, 16, 1, 1, 1, 1, 1, 1, 4, ids, 1, None),
        (1, 1, 9, 8, 8, 2, 64, 16, 1, 1, 1, 1, 1, 1, 4, ids, 1, None),
        (1, 1, 1, 8, 8, 2, 64, 16, 1, 1, 1, 1, 1, 1, 4, None, 1, None),
        (1, 1, 1, 8, 8, 2, 64, 16, 1, 1, 1, 1, 1, 1, 0, ids, 1, None),
    ]
    for args in bad:
        assert lib.fs_write_prompt_i8(*args) == _lib.FS_ERR_INVALID
    past = np.array([4], dtype=np.int32)
    assert lib.fs_write_prompt_i8(1, 1, 1, 8, 8, 2, 64, 16, 1, 1, 1, 1, 1, 1, 4, past.ctypes.data, 1,
                                  None) == _lib.FS_ERR_INVALID
