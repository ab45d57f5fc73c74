"""compress_kv over a cache read in place (compress_retiled_kv) against the
encoder over the padded matrix that the pad_* helpers build: the same streams,
byte for byte, for every layout, ragged token counts, the smallest caches, and
records with more outliers than their slot holds.  Caches that the in-place
path does not take still go through the copy."""
import numpy as np
import pytest

from zs_testutil import kv_bf16, to_torch_bf16

pytestmark = pytest.mark.gpu


def _matrix(za, x, layout, page):
    if layout == "by_kv_head":
        return za.pad_batched_kv_prefix_by_kv_head(x)
    if layout == "paged":
        return za.pad_batched_kv_prefix_paged(x, page)
    return za.pad_batched_kv_prefix(x)


def _same(a, b):
    import torch
    assert (a.rows, a.cols, a.logical_rows, a.logical_cols, a.start_exp, a.num_outliers,
            a.compressed_bytes, a.layout) == (b.rows, b.cols, b.logical_rows, b.logical_cols,
                                              b.start_exp, b.num_outliers, b.compressed_bytes,
                                              b.layout)
    assert torch.equal(a.fixed, b.fixed) and torch.equal(a.exps, b.exps)
    assert torch.equal(a.eoff, b.eoff)


def _compare(x, layout, page=16):
    import zipserv_asplos26_amd as zs
    import zipserv_asplos26_amd.attention as za
    assert za._reads_in_place(x, layout, page)
    m, logical, _ = _matrix(za, x, layout, page)
    _same(za.compress_kv(x, layout, retiled=True, page_block_size=page),
          zs.compress_retiled(m.contiguous(), logical, x.shape[-1], layout=layout))


@pytest.mark.parametrize("layout", ["by_kv_head", "token_major", "dense", "paged"])
@pytest.mark.parametrize("B,T,H,D", [
    (1, 1, 8, 128), (1, 64, 8, 128), (2, 65, 8, 128), (3, 100, 4, 64), (2, 63, 1, 192),
    (1, 1000, 8, 128), (5, 33, 12, 128), (8, 129, 8, 128)])
def test_in_place_bytes(torch_cuda, layout, B, T, H, D):
    x = to_torch_bf16(kv_bf16(np.random.default_rng(T + H), B, T, H, D))
    _compare(x, layout, page=64 if layout == "paged" else 16)


@pytest.mark.parametrize("layout", ["by_kv_head", "token_major"])
def test_in_place_outliers_past_the_slot(torch_cuda, layout):
    # rows of random bits (nearly every element an outlier) among ordinary ones
    rng = np.random.default_rng(5)
    a = kv_bf16(rng, 2, 300, 8, 128)
    a[:, 40:140] = rng.integers(0, 1 << 16, a[:, 40:140].shape, dtype=np.uint16)
    _compare(to_torch_bf16(a), layout)


@pytest.mark.parametrize("layout", ["by_kv_head", "token_major"])
@pytest.mark.parametrize("noise", [False, True])
def test_the_cache_may_change_once_it_is_encoded(torch_cuda, layout, noise):
    # what is written into the cache behind the first phase, by another thread
    # or after the call returned, is not in the stream: also for records with
    # more outliers than an ordinary slot holds (rows of random bits; the band
    # where a sequence ends)
    import zipserv_asplos26_amd as zs
    import zipserv_asplos26_amd.attention as za
    from zipserv_asplos26_amd import codec
    rng = np.random.default_rng(6)
    a = kv_bf16(rng, 2, 301, 8, 128)
    if noise:
        a[:, 40:140] = rng.integers(0, 1 << 16, a[:, 40:140].shape, dtype=np.uint16)
    x = to_torch_bf16(a)
    m, logical, _ = _matrix(za, x, layout, 16)
    want = zs.compress_retiled(m.contiguous(), logical, 128, layout=layout)
    group, _ = za._kv_group(x, layout, 16)
    lid = za.LAYOUT_IDS[layout]
    s = codec._retiled_encode(x, "kv", kv=(lid, *x.shape, group))
    x.copy_(to_torch_bf16(rng.integers(0, 1 << 16, x.shape, dtype=np.uint16)))
    _same(codec._retiled_finish(s, s["meta"].cpu(), logical, 128, layout), want)


@pytest.mark.parametrize("layout", ["by_kv_head", "token_major"])
def test_in_place_bytes_with_ordinary_slots(torch_cuda, layout):
    # zs_compress_retiled_kv_gpu / _kv_exps_gpu, whose second call reads the
    # records past their slots from the cache again
    import zipserv_asplos26_amd as zs
    import zipserv_asplos26_amd.attention as za
    torch, L = torch_cuda, zs.lib()
    rng = np.random.default_rng(7)
    a = kv_bf16(rng, 2, 301, 8, 128)
    a[:, 40:140] = rng.integers(0, 1 << 16, a[:, 40:140].shape, dtype=np.uint16)
    x = to_torch_bf16(a)
    want = za.compress_kv(x, layout, retiled=True)
    shape = (za.LAYOUT_IDS[layout], *x.shape, za._kv_group(x, layout, 16)[0])
    n = want.rows // 16 * (want.cols // 64)
    new = lambda k, dtype: torch.empty(k, dtype=dtype, device="cuda")
    hist, top, work = new(256, torch.int64), new(7, torch.int32), new(
        zs._lib.ZS_RETILED_AUTO_WORK_BYTES, torch.uint8)
    fixed, cnt, eoff = new(n * 1408, torch.uint8), new(n, torch.int32), new(n + 1, torch.int32)
    total, tmp, exps = new(1, torch.int64), new(n * 256, torch.uint8), torch.empty_like(want.exps)
    st = int(torch.cuda.current_stream().cuda_stream)
    ptrs = [t.data_ptr() for t in (hist, top, work, fixed, cnt, eoff, total, tmp)]
    assert L.zs_compress_retiled_kv_gpu(st, x.data_ptr(), *shape, zs._lib.ZS_WINDOW_KV, *ptrs) == 0
    assert int(total) == want.num_outliers
    assert L.zs_compress_retiled_kv_exps_gpu(st, x.data_ptr(), *shape, top.data_ptr(),
                                             eoff.data_ptr(), tmp.data_ptr(), exps.data_ptr()) == 0
    torch.cuda.synchronize()
    for got, ref in ((fixed, want.fixed), (eoff, want.eoff), (exps, want.exps)):
        assert torch.equal(got, ref)


@pytest.mark.parametrize("T", [65, 4097])
def test_in_place_zero_padding_moves_the_window(torch_cuda, T):
    # one or two distinct exponents and much padding: the padding's zeros are
    # part of the histogram that the window is chosen from
    x = torch_cuda.full((2, T, 8, 128), 1.5, dtype=torch_cuda.bfloat16, device="cuda")
    x[:, ::3] = 0.01
    _compare(x, "by_kv_head")


def test_copied_where_it_cannot_be_read_in_place(torch_cuda):
    import zipserv_asplos26_amd as zs
    import zipserv_asplos26_amd.attention as za
    x = to_torch_bf16(kv_bf16(np.random.default_rng(1), 2, 130, 8, 128))
    flat = torch_cuda.empty(x.numel() + 1, dtype=x.dtype, device="cuda")
    flat[1:] = x.view(-1)
    strided = x.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)
    for y in (flat[1:].view(x.shape), strided):
        assert not za._reads_in_place(y, "by_kv_head", 16)
        m, logical, _ = za.pad_batched_kv_prefix_by_kv_head(y)
        _same(za.compress_kv(y, retiled=True), zs.compress_retiled(m, logical, 128))
    narrow = x[..., :80].contiguous()
    assert not za._reads_in_place(narrow, "by_kv_head", 16)
    assert za.compress_kv(narrow, retiled=True).cols == 128
    with pytest.raises(ValueError):
        za.compress_kv(x.float(), retiled=True)
    with pytest.raises(ValueError):
        za.compress_kv(x, "nowhere", retiled=True)
    # pages of 16 tokens of one head: groups of 16 rows, not whole 64-row tiles
    with pytest.raises(ValueError):
        za.compress_kv(x[:1, :16, :1].contiguous(), "paged", retiled=True)
