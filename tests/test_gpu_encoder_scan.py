"""Offsets of the one-pass re-tiled encoder: the exclusive sums of the records'
outlier counts, at the edges of the scan's tiles (1024 records), past the 256
tiles that one step of its sum over earlier tiles takes and past the 4096 that
its one launch takes.  Every bit of the input is random, so nearly all
elements are outliers."""
import pytest

import zipserv_asplos26_amd as zs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K", [(64, 64), (1024, 960), (1024, 1024), (1088, 1024), (4096, 4160),
                                 (16384, 16448), (65536, 65600)])
def test_offsets_are_the_sums_of_the_counts(torch_cuda, M, K):
    torch = torch_cuda
    g = torch.Generator(device="cuda")
    g.manual_seed(M + K)
    x = torch.randint(-2**15, 2**15, (min(M, 4096), K), dtype=torch.int16, device="cuda", generator=g)
    x = x.repeat(M // x.shape[0], 1)
    n = M // 16 * (K // 64)
    st = int(torch.cuda.current_stream().cuda_stream)
    new = lambda shape, dtype: torch.empty(shape, dtype=dtype, device="cuda")
    for rep in range(2):
        hist, top, total = new(256, torch.int64), new(7, torch.int32), new(1, torch.int64)
        counts, eoff = new(n, torch.int32), new(n + 1, torch.int32)
        work = new(zs._lib.ZS_RETILED_AUTO_WORK_BYTES, torch.uint8).fill_(255)
        fixed, tmp = new(n * 1408, torch.uint8), new(n * 256, torch.uint8)
        assert zs.lib().zs_compress_retiled_auto_gpu(
            st, x.data_ptr(), M, K, zs._lib.ZS_WINDOW_KV, hist.data_ptr(), top.data_ptr(),
            work.data_ptr(), fixed.data_ptr(), counts.data_ptr(), eoff.data_ptr(), total.data_ptr(),
            tmp.data_ptr()) == 0
        torch.cuda.synchronize()
        sums = torch.cumsum(counts.to(torch.int64), 0)
        assert int(total) == int(sums[-1])
        assert int(eoff[0]) == 0 and torch.equal(eoff[1:], sums.to(torch.int32))
